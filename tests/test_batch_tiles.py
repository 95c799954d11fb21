"""The tile sizes of a replica batch's launches (tile_rules.h, compiled here):
a pair fixed by the caller is the pair launched, whatever the size of the batch
and with and without hazard accumulation; a pair that the autotuner picked is
cut finer for a small batch, which is not timed where all are cut to one (CPU
only)."""
import os
import subprocess

import pytest

from pansim_amd import build
from tests.conftest import ROOT

SOURCE = r"""
#include <cstdio>
#include <cstdlib>
#include "tile_rules.h"
using namespace ps::dev;
int main() {
    const uint64_t agents[] = {1, 10000, 786432, 786433, 1500000, 1500001, 1572865, 3145728, 3145729, 10000000};
    for (uint64_t n : agents)
        for (int hazard = 0; hazard < 2; ++hazard)
            for (int fixed = 0; fixed < 2; ++fixed)
                for (int m = 0; m < (int)kMoveCandidates; ++m)
                    for (int i = 0; i < (int)kInfectCandidates; ++i) {
                        const BatchTiles t = batch_tiles(n, hazard, fixed, {m, i});
                        std::printf("%llu %d %d %u %u %u %u %u %u %d\n", (unsigned long long)n, hazard, fixed,
                                    kMoveItems[m], kInfectItems[i], kMoveItems[t.move], kInfectItems[t.infect],
                                    move_items_for(n), infect_items_for(n, hazard), (int)one_cut(n, hazard));
                    }
}
"""


@pytest.fixture(scope="module")
def rows(tmp_path_factory):
    d = tmp_path_factory.mktemp("tiles")
    (d / "t.cpp").write_text(SOURCE)
    subprocess.run([build.CXX, *build.CXXFLAGS, "-I", os.path.join(ROOT, "pansim_amd", "csrc", "device"), "-o", str(d / "t"),
                    str(d / "t.cpp")], check=True)
    out = subprocess.run([str(d / "t")], check=True, capture_output=True, text=True).stdout
    return [tuple(map(int, line.split())) for line in out.splitlines()]


def test_a_fixed_pair_is_launched(rows):
    fixed = [r for r in rows if r[2]]
    assert {(r[3], r[4]) for r in fixed} == {(m, i) for m in (8, 16, 32) for i in (4, 8)}
    for r in fixed:
        assert r[5:7] == r[3:5], r


def test_a_picked_pair_is_cut_by_the_rules(rows):
    for n, hazard, fixed, m, i, move, infect, by_move, by_infect, _ in rows:
        if not fixed:
            assert move == (1 if by_move == 1 else m)
            assert infect == (by_infect if hazard else min(i, by_infect))
            assert not hazard or infect in (4, 8)


def test_one_cut_is_one_pair(rows):
    for n, hazard in {r[:2] for r in rows}:
        picked = [r for r in rows if r[:3] == (n, hazard, 0)]
        assert picked[0][9] == (len({r[5:7] for r in picked}) == 1)
        assert picked[0][9] == (n <= 1_500_000)
