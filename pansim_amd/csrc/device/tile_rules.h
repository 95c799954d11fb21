// Tile sizes of the movement and infection launches (host side).
#pragma once
#include <cstdint>

namespace ps {
namespace dev {

constexpr uint32_t MOVE_BLOCK = 256;
// Agents per thread of the movement tile for n agents stepped by one launch.
// Up to 1.5M agents one per lane (move_lane).  Above, the smallest tile whose
// blocks are all resident at once (256 CUs x 5 blocks of 4 waves): a step
// with few movers, bound by one mover's dependent reads, then costs one
// round.  Movement of a weekday, MI355X, by agents per thread 1 / 8 / 16 / 32:
// 100k agents 1.05 / 1.43 / 1.73 / 2.21 ms, 1M 1.79 / 2.10 / 2.35 / 2.90 ms,
// 2M 2.63 / 2.57 / 2.73 / 3.17 ms, 5M 5.45 / 4.50 / 4.14 / 4.58 ms, 10M
// 10.3 / 7.56 / 6.85 / 6.42 ms.  Those are 10-minute steps; with longer ones a
// larger share of the agents moves at each, and the line stands: whole days by
// 1 / 8 / 16, hourly steps 600k agents 0.79 / 0.92 / 1.07 ms, 1M 0.95 / 1.04 /
// 1.15, 2M 1.53 / 1.51 / 1.62; half-hourly 600k 1.06 / 1.31 / 1.50, 1M 1.30 /
// 1.45 / 1.60, 2M 2.02 / 2.03 / 2.15.
constexpr uint32_t MOVE_LANE_MAX = 1500000;
inline uint32_t move_items_for(uint64_t n) {
    const uint64_t resident = 256u * 5u;
    return n <= MOVE_LANE_MAX ? 1u : n <= resident * MOVE_BLOCK * 8u ? 8u : n <= resident * MOVE_BLOCK * 16u ? 16u : 32u;
}

constexpr uint32_t INFECT_BLOCK = 256;
// Agents per thread for n agents stepped by one launch: the fewest that keep
// the launch within one and a half rounds of the resident blocks (256 CUs x 8
// blocks of 4 waves).  Infection of a day, MI355X, by agents per thread
// 1 / 2 / 4 / 8: 100k agents 0.67 / 0.78 / 0.93 / 1.31 ms, 300k 0.74 / 0.76 /
// 0.89 / 1.24 ms, 1M 1.24 / 1.00 / 0.98 / 1.32 ms, 3M 2.82 / 2.13 / 1.74 /
// 1.82 ms, 10M 8.2 / 5.7 / 4.2 / 3.7 ms.  With hazard accumulation at least 4:
// every block clears and flushes its LDS slots (a week of 8 replicas, 2M
// agents: 35.6 ms with 4 agents per thread, 36.4 with 8, 41 with 2).
constexpr uint32_t HAZARD_ITEMS_MIN = 4;
inline uint32_t infect_items_for(uint64_t n, bool hazard) {
    const uint64_t most = 3072u * (uint64_t)INFECT_BLOCK;
    const uint32_t items = n <= most ? 1u : n <= 2u * most ? 2u : n <= 4u * most ? 4u : 8u;
    return hazard && items < HAZARD_ITEMS_MIN ? HAZARD_ITEMS_MIN : items;
}

// Tile sizes of the replica batches' kernels: the autotuner's candidates (and
// what pansim_batch_set_tiles accepts), agents per thread of the movement
// tile (its LDS mover list holds 256 x that many offsets) and of the infection
// tile, and behind them the finer ones.
constexpr uint32_t kMoveCandidates = 3, kInfectCandidates = 2;
constexpr uint32_t kMoveItems[4] = {8, 16, 32, 1};
constexpr uint32_t kInfectItems[4] = {4, 8, 1, 2};
struct BatchTiles {
    int move, infect;  // indices into the lists above
    bool operator==(const BatchTiles& o) const { return move == o.move && infect == o.infect; }
};

// The sizes of a launch for a batch of `agents` agents with candidate c: c
// itself if the caller fixed it.  A pair that the tuner picked (or is timing)
// is cut finer where the batch is too small to fill the chip with its tiles,
// by the rules for one population; with hazard accumulation, which the tuner's
// steps run without, infection takes that rule's size.
inline BatchTiles batch_tiles(uint64_t agents, bool hazard, bool fixed, BatchTiles c) {
    if (fixed) return c;
    if (move_items_for(agents) == 1) c.move = 3;
    const uint32_t fine = infect_items_for(agents, hazard);
    if (hazard) c.infect = 1;
    if (fine < kInfectItems[c.infect]) c.infect = fine == 1 ? 2 : fine == 2 ? 3 : 0;
    return c;
}

// Whether every candidate is cut to one pair, so that there is nothing to tune.
inline bool one_cut(uint64_t agents, bool hazard) {
    return batch_tiles(agents, hazard, false, {0, 0}) ==
           batch_tiles(agents, hazard, false, {(int)kMoveCandidates - 1, (int)kInfectCandidates - 1});
}

}  // namespace dev
}  // namespace ps
