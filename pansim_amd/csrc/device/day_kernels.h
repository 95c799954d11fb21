// Midnight kernels: initial state draws, occupancy rebuild, testing,
// progression, immunity waning, non-COVID hospitalisation, statistics,
// location planning, closure toggles.  Included once, by engine.hip.
#pragma once
#include "step_kernels.h"

namespace ps {
namespace dev {

// ------------------------------------------------------------ common helpers
__device__ __forceinline__ int geometric(double p, Stream& rs) {
    double log1mp = ps_log(1.0 - p);
    const double naf = (1.0 - 2.220446049250313e-16) / 2.0;
    const double thr = 2147483647.0 + naf;
    double cand;
    int guard = 0;
    do {
        cand = floor(ps_log(1.0 - rs.unit()) / log1mp);
    } while (cand >= thr && ++guard < 1000);
    if (cand >= thr) cand = 2147483647.0;
    return (int)(cand + naf);
}

// BasicLengthAbstract::LengthOfState::calculateDays (basicLengthAbstract.cpp:48-53)
__device__ __forceinline__ int calc_days(const Tables& T, uint32_t prog, uint32_t state, uint32_t variant, Stream& rs) {
    size_t k = ((size_t)prog * T.nStates + state) * 7 + variant;
    if (T.lenAvg[k] == -1.0f) return -1;
    double p = T.lenP[k];
    float mx = T.lenMax[k];
    int days = geometric(p, rs);
    int guard = 0;
    while (mx < (float)days && ++guard < 1000) days = geometric(p, rs);
    if (mx < (float)days) days = (int)mx;
    return days;
}

__device__ __forceinline__ float scaling_symptoms(const Agents& A, uint32_t i, uint32_t v, uint32_t s) {
    // scalingSymptoms[v*7 + MAX(6, s)] (agentMeta.cpp:128-129): only slot 6 of
    // each variant is ever written; other slots hold scalingAgeSex
    return s <= 6 ? A.slot6[(size_t)v * A.n + i] : A.scal[i];
}

__device__ __forceinline__ void update_meta(const Agents& A, const Tables& T, uint32_t i, uint8_t st) {
    float sf = T.stSusc[st] ? 1.0f : 0.0f;
    for (uint32_t v = 0; v < T.nVar; ++v) A.susc[(size_t)v * A.suscStride + i] = sf;
}

// ------------------------------------------------------------ init
__global__ void k_init_agents(Agents A, Tables T, uint64_t seed, uint32_t replica, uint32_t qp, uint32_t qlenSteps,
                              uint32_t qlenDays) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= A.n) return;
    uint8_t st = A.rec[i].state;
    A.rec[i].variant = 0;
    update_meta(A, T, i, st);
    for (uint32_t v = 0; v < T.nVar; ++v) A.slot6[(size_t)v * A.n + i] = A.scal[i];
    Stream rs(seed, A.id[i], 0, PH_INIT_DAYS, replica);
    A.days[i] = (int16_t)calc_days(T, A.prog[i], st, 0, rs);
    bool inf = T.stInfected[st] != 0;
    A.infTs[i] = inf ? 0u : NEVER;
    A.infCount[i] = inf ? 1 : 0;
    A.worstState[i] = inf ? (int8_t)st : 0;
    A.worstTs[i] = 0;
    A.worstEndTs[i] = 0;
    A.infLoc[i] = 0;
    A.recTs[i] = NEVER;
    A.rec[i].hospTs = 0;
    A.rec[i].hospUntil = 0;
    A.immTs[i] = 0;
    A.immCount[i] = 0;
    A.statVar[i] = 0;
    A.lastTest[i] = NEVER;
    A.wake[i] = 0;
    uint8_t fl = A.rec[i].flags;  // diagnosed / hcw preset by the host upload
    bool diag = fl & F_DIAGNOSED;
    A.rec[i].diagTs = diag ? 1u : 0u;
    if (diag && qp > 0) {
        A.quarTs[i] = 0;
        A.rec[i].quarUntil = qlenSteps;
        A.daysInQ[i] = qlenDays;
        fl |= F_QUARANTINED;
    } else {
        A.quarTs[i] = 0;
        A.rec[i].quarUntil = 0;
        A.daysInQ[i] = 0;
    }
    fl |= F_STAYED_HOME;
    A.rec[i].flags = fl;
}

// ------------------------------------------------------------ occupancy
__global__ void k_zero_locations(Locs L, uint32_t nVar) {
    uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t l = blockIdx.x * blockDim.x + threadIdx.x; l < L.n; l += stride) {
        L.dyn[l].count = 0u;
        L.dyn[l].sum0 = 0;
        for (uint32_t v = 1; v < nVar; ++v) L.sumX[(size_t)(v - 1) * L.n + l] = 0;
        if ((l & 31u) == 0) L.visited[l >> 5] = 0u;
    }
}

// Runs of equal values among the consecutive lanes of a wave: `head` is set
// on the first lane of each run, the return value is the run's length there.
// Valid lanes form a prefix of the wave.
__device__ __forceinline__ uint32_t lane_run(uint32_t v, bool valid, bool& head) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t prev = __shfl_up(v, 1, 64);
    head = valid && (lane == 0 || prev != v);
    const unsigned long long heads = __ballot(head);
    const uint32_t nValid = (uint32_t)__popcll(__ballot(valid));
    const unsigned long long after = heads & ~((2ull << lane) - 1ull);
    uint32_t next = after ? (uint32_t)(__ffsll((long long)after) - 1) : 64u;
    if (next > nValid) next = nValid;
    return next - lane;
}

__global__ void k_scatter_locations(Agents A, Locs L, Tables T) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool valid = i < A.n;
    const uint32_t loc = valid ? A.location[i] : NOLOC;
    // members of a household are consecutive agents: one occupancy atomic per run
    bool head;
    const uint32_t run = lane_run(loc, valid, head);
    if (!valid) return;
    if (head) atomicAdd(&L.dyn[loc].count, run);
    const AgentRec r = A.rec[i];
    float x = T.stInf[r.state] * T.varMul[r.variant];
    if (x != 0.0f) {
        atomicAdd((unsigned long long*)loc_sum(L, r.variant, loc), (unsigned long long)fixed32(x));
        mark_visited(L, loc);
    }
}

// ------------------------------------------------------------ infectious-list dump
// (BasicInfection::dumpLocationInfectiousList, infectionPolicies.h:262-441)
// The locations of the agents infected since the last collection: flagged
// in a bitmap, and recorded next to each agent.
__global__ void k_dump_mark(Agents A, const uint32_t* agents, const uint32_t* count, uint32_t* locOut, uint32_t* flags) {
    const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= *count) return;
    const uint32_t l = A.location[agents[j]];
    locOut[j] = l;
    atomicOr(&flags[l >> 5], 1u << (l & 31u));
}

// Every agent with non-zero infectiousness at a flagged location.
__global__ void k_dump_infectious(Agents A, Tables T, const uint32_t* flags, uint32_t* outAgent, uint32_t* outLoc,
                                  float* outValue, uint32_t* count) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= A.n) return;
    const uint32_t l = A.location[i];
    if (!((flags[l >> 5] >> (l & 31u)) & 1u)) return;
    const AgentRec r = A.rec[i];
    const float x = T.stInf[r.state] * T.varMul[r.variant];
    if (x == 0.0f) return;
    const uint32_t slot = atomicAdd(count, 1u);
    outAgent[slot] = i;
    outLoc[slot] = l;
    outValue[slot] = x;
}

__global__ void k_count_variants(Agents A, Tables T, unsigned long long* out) {
    __shared__ unsigned int sh[MAXV];
    if (threadIdx.x < MAXV) sh[threadIdx.x] = 0;
    __syncthreads();
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < A.n && T.stInfected[A.rec[i].state]) atomicAdd(&sh[A.rec[i].variant], 1u);
    __syncthreads();
    if (threadIdx.x < T.nVar && sh[threadIdx.x]) atomicAdd(&out[threadIdx.x], (unsigned long long)sh[threadIdx.x]);
}

// ------------------------------------------------------------ testing
struct TestParams {
    uint32_t delay, qlen, usePCR;
    double pRandom, pHome, pWork, pSchool, pHospital, pNursery;
    double pMax;  // at least any agent's probability: all its terms, added in the same order
};

// The testing flags live in a bitmap (1 bit per location, L2 resident): the
// testing pass reads the flags of every agent's home, workplace and school.
__device__ __forceinline__ bool test_flag(const Locs& L, uint32_t l) {
    return ((L.flagBits[l >> 5] >> (l & 31u)) & 1u) != 0u;
}
__device__ __forceinline__ void set_test_flag(const Locs& L, uint32_t l) {
    atomicOr(&L.flagBits[l >> 5], 1u << (l & 31u));
}

__global__ void k_clear_flags(Locs L) {
    uint32_t stride = gridDim.x * blockDim.x;
    const uint32_t words = (L.n + 31u) / 32u;
    for (uint32_t w = blockIdx.x * blockDim.x + threadIdx.x; w < words; w += stride) L.flagBits[w] = 0u;
}

// DetailedTestingOps::flagLocations (testingPolicies.h:59-148) for agent i
__device__ __forceinline__ void flag_agent(const Agents& A, const Locs& L, const Tables& T, uint64_t seed, uint32_t replica,
                                           uint32_t ts, uint32_t dt, const TestParams& p, uint32_t i) {
    const uint32_t day = 24u * 60u / dt;
    if (!(A.rec[i].diagTs > ts - day)) return;
    const pansim_location_types& lt = T.lt;
    const uint32_t ql = p.qlen * 24u * 60u / dt;
    auto ok = [&](uint32_t l) {
        uint32_t q = L.rec[l].quarUntil;
        return q == 0 || (q != 0 && (q - ql >= ts - day || q < ts));
    };
    const CsrReg csr = load_csr(A, i, A.rec[i]);
    uint32_t home = csr.home;
    if (home != NOLOC) set_test_flag(L, home);
    uint32_t work = find_loc(A, L, lt, csr, lt.work, 0, nullptr);
    if (work != NOLOC && ok(work)) set_test_flag(L, work);
    uint32_t school = find_loc(A, L, lt, csr, lt.school, 0, nullptr);
    if (school != NOLOC && ok(school)) {
        set_test_flag(L, school);
        Stream rs(seed, A.id[i], ts, PH_TEST_FLAG, replica);
        uint32_t cls = find_loc(A, L, lt, csr, lt.classroom, 0, &rs);
        if (cls != NOLOC && ok(cls)) set_test_flag(L, cls);
    }
}

// What performTests counts of an agent: 1 tested now, 2 positive now, 4
// positive in the last day.
__device__ __forceinline__ uint32_t test_counts(uint32_t ts, uint32_t day, uint32_t lastTest, uint32_t diagTs) {
    return (lastTest == ts ? 1u : 0u) | (diagTs == ts ? 2u : 0u) | (diagTs < ts && diagTs > ts - day ? 4u : 0u);
}

// Whether the agent may be tested at all: it was not tested lately, is alive
// and not diagnosed, and its draw is below the largest probability there is.
// The test's draw is the first one (unless a classroom is drawn before it), so
// most agents need none of the lookups behind their own probability (a list
// line and three flags per agent).
__device__ __forceinline__ bool may_test(uint64_t seed, uint32_t replica, uint32_t ts, uint32_t dt, const TestParams& p,
                                         const AgentRec& r, uint32_t id, uint32_t lastTest) {
    const uint32_t day = 24u * 60u / dt;
    if (ts > p.delay * day && lastTest != NEVER && lastTest > ts - p.delay * day) return false;
    if ((r.cls & CLS_WB) == 4 || (r.flags & F_DIAGNOSED)) return false;
    if ((r.flags & F_CLASSES) || p.pMax > 1.0) return true;
    Stream rs(seed, id, ts, PH_TESTING, replica);
    return rs.real(1.0) < p.pMax;
}

// DetailedTestingOps::doTesting (testingPolicies.h:157-281) for agent i (record
// r, kept up to date).  Returns test_counts.  The flags of its home, workplace
// and school are read together, so that a thread waits for a few memory round
// trips instead of one per field.
__device__ __forceinline__ uint32_t test_agent(const Agents& A, const Locs& L, const Tables& T, uint64_t seed,
                                               uint32_t replica, uint32_t ts, uint32_t dt, const TestParams& p, uint32_t i,
                                               AgentRec& r, uint32_t id, uint32_t lastTest) {
    const uint32_t day = 24u * 60u / dt;
    const pansim_location_types& lt = T.lt;
    const uint8_t st = r.state;
    if (may_test(seed, replica, ts, dt, p, r, id, lastTest)) {
        Stream rs(seed, id, ts, PH_TESTING, replica);
        const CsrReg csr = load_csr(A, i, r);
        const uint32_t home = csr.home;
        const uint32_t work = find_loc(A, L, lt, csr, lt.work, 0, nullptr);
        const uint32_t school = find_loc(A, L, lt, csr, lt.school, 0, nullptr);
        // flags from the bitmap, the workplace's type from the type bytes
        const bool homeFlag = home != NOLOC && test_flag(L, home);
        const bool workFlag = work != NOLOC && test_flag(L, work);
        const uint32_t workType = work != NOLOC ? (uint32_t)L.type8[work] : (uint32_t)LOC_TYPE_NONE;
        bool schoolFlag = false, classFlag = false;
        if (school != NOLOC) {
            schoolFlag = test_flag(L, school);
            uint32_t cls = find_loc(A, L, lt, csr, lt.classroom, 0, &rs);
            if (cls != NOLOC) classFlag = true;
        }
        double prob = p.pRandom;
        prob += (double)homeFlag * p.pHome;
        prob += (double)workFlag * p.pWork;
        prob += (double)schoolFlag * p.pSchool;
        prob += (double)classFlag * 3.0 * p.pSchool;
        if (work != NOLOC && (workType == lt.doctor || workType == lt.hospital)) prob += p.pHospital;
        if (work != NOLOC && workType == lt.nursery_home) prob += p.pNursery;
        if (r.hospTs <= ts && r.hospUntil > ts) prob += p.pHospital;
        if (prob > 1.0 || rs.real(1.0) < prob) {
            A.lastTest[i] = ts;
            lastTest = ts;
            if (T.stInfected[st]) {
                float pr = p.usePCR ? T.accPCR[st] : T.accAnt[st];
                if ((double)pr > rs.real(1.0)) {
                    A.rec[i].flags = r.flags = (uint8_t)(r.flags | F_DIAGNOSED);
                    A.rec[i].diagTs = r.diagTs = ts;
                }
            } else {
                if (r.quarUntil > ts && (home != NOLOC && L.rec[home].quarUntil < ts)) {
                    if (A.daysInQ[i] > 0) A.daysInQ[i] -= (r.quarUntil - ts) / day;
                    A.rec[i].quarUntil = r.quarUntil = ts;
                }
            }
        }
    }
    return test_counts(ts, day, lastTest, r.diagTs);
}

// ------------------------------------------------------------ progression
// Simulation::updateAgents (simulation.h:425-471), DynamicPPState::update
// (dynamicPPState.cpp:246-303), NextStates::selectNext (multiBadMatrix.cpp:9-31)
// for agent i (record r, kept up to date)
__device__ __forceinline__ void progress_agent(const Agents& A, const Tables& T, uint64_t seed, uint32_t replica, uint32_t ts,
                                               uint32_t dt, uint32_t i, AgentRec& r, uint32_t id, int16_t days) {
    if (days > 0) {
        A.days[i] = (int16_t)(days - 1);
        return;
    }
    if (days != -2 && days != 0) return;
    uint8_t st = r.state;
    uint8_t v = r.variant;
    uint32_t prog = A.prog[i];
    float progS;
    if (st == 7) progS = T.deathScaling[v] / scaling_symptoms(A, i, v, st);
    else progS = T.progScaling[v];
    float scaling = scaling_symptoms(A, i, v, st) * progS;
    Stream rs(seed, id, ts, PH_PROGRESSION, replica);
    if (days == -2) {
        days = (int16_t)calc_days(T, prog, st, v, rs);
        if (v >= 3) {
            double d = days * 0.7;
            days = (int16_t)(d == 0 ? 1.0 : d);
        }
    }
    if (days == 0) {
        uint8_t old = st;
        bool wasInf = T.stInfected[st] != 0;
        // selectNext
        size_t ps_ = (size_t)prog * T.nStates + st;
        uint32_t eb = T.edgeOff[ps_], nb = T.badCount[ps_], ee = T.edgeOff[ps_ + 1];
        uint32_t nNeu = ee - eb - nb;
        float sc = nNeu == 0 ? 1.0f : scaling;
        double random = rs.unit();
        double preSum = 0.0, badSum = 0.0;
        uint32_t next = 0xFFFFFFFFu;
        bool bad = false;
        for (uint32_t j = 0; j < nb; ++j) {
            float term = T.edgeChance[eb + j] * sc;
            preSum += (double)term;
            if (random < preSum) {
                next = T.edgeTo[eb + j];
                bad = true;
                break;
            }
            badSum += (double)T.edgeChance[eb + j];
        }
        if (!bad && nNeu == 0) {  // bad chances summed below the draw
            next = T.edgeTo[eb + nb - 1];
            bad = true;
        }
        if (!bad) {
            double badScaling = 1.0 + ((badSum - preSum) / (1.0 - badSum));
            if (nb == 0) badScaling = 1.0;
            uint32_t idx = 0;
            do {
                preSum += (double)T.edgeChance[eb + nb + idx] * badScaling;
                ++idx;
            } while (preSum < random && idx < nNeu);
            idx--;
            next = T.edgeTo[eb + nb + idx];
        }
        int nd = calc_days(T, prog, next, v, rs);
        st = (uint8_t)next;
        A.rec[i].state = r.state = st;
        A.rec[i].cls = r.cls = T.stCls[st];
        update_meta(A, T, i, st);
        days = (int16_t)nd;
        if (v >= 3 && st < 8) {
            float mul = st < 6 ? 0.7f : 0.5f;
            float d = (float)days * mul;
            days = (int16_t)(d == 0 ? 1.0f : d);
        }
        if (bad) {
            A.worstState[i] = (int8_t)st;
            A.worstTs[i] = ts;
            A.worstEndTs[i] = ts + (uint32_t)((int)days * 60 * 24) / dt;
        } else if (old != st) {
            if (wasInf && !T.stInfected[st]) {
                A.recTs[i] = ts;
                A.rec[i].flags = r.flags = (uint8_t)(r.flags & ~F_DIAGNOSED);
            }
        }
    }
    A.days[i] = days;
}

// ------------------------------------------------------------ immunity
struct ImmParams {
    float eff[5][6][2];  // inf, 2 dose, 3 dose, inf+2, inf+3; rows (comp + 3*different); (waning, level)
    int sim[MAXV];
    float simMul[MAXV];
};

__device__ __forceinline__ float fmin_ref(float a, float b) { return a < b ? a : b; }

// Immunization::update, susceptibility of state-0 agents (immunization.h:547-695):
// agent i, in state 0
__device__ __forceinline__ void immunize_agent(const Agents& A, const Tables& T, uint32_t now, uint32_t dt, const ImmParams& a,
                                               uint32_t i, uint8_t infC, uint8_t immC) {
    // never infected nor immunized: susceptibility 1 for every variant, which
    // it already is when state 0 is a susceptible state (set with that state
    // when the agent was created, and written since only by an infection or
    // by the branches below)
    if (infC == 0 && immC == 0 && T.stSusc[0]) return;
    const uint32_t nVar = T.nVar;
    const uint32_t ts = now == 0 ? 1u : now;
    const uint32_t week = 7u * 24u * 60u / dt;
    float susc[MAXV];
    for (uint32_t v = 0; v < nVar; ++v) susc[v] = 1.0f;
    const uint32_t wImm = (ts - A.immTs[i]) / week;
    const uint32_t wInf = (ts - A.infTs[i]) / week;
    const uint32_t prior = A.statVar[i];
    float scal = A.scal[i];
    auto lin = [&](int e, int row, uint32_t weeks) -> float {
        return -1.0f * a.eff[e][row][0] * (float)weeks + a.eff[e][row][1];
    };
    auto mix = [&](int e, int comp, int similar, uint32_t v, uint32_t weeks) -> float {
        int d = (1 - similar) * 3 + comp, s = similar * 3 + comp;
        return -1.0f * (a.eff[e][d][0] + (a.eff[e][s][0] - a.eff[e][d][0]) * a.simMul[v]) * (float)weeks + a.eff[e][d][1] +
               (a.eff[e][s][1] - a.eff[e][d][1]) * a.simMul[v];
    };
    auto setSlot = [&](uint32_t v, float x) { A.slot6[(size_t)v * A.n + i] = scal * x; };
    if (infC > 0 && (immC == 0 || (immC == 1 && wImm < 4))) {
        for (uint32_t v = 0; v < nVar; ++v) {
            int similar = 0;
            for (uint32_t j = 0; j < nVar; ++j) similar = similar || ((prior & (1u << j)) && a.sim[v] == a.sim[j]);
            int d = (1 - similar) * 3;
            float vsInf = (float)((double)(-1.0f * a.eff[0][d][0] * (float)wInf) +
                                  (((1u << v) & prior) ? 0.95 : (double)a.eff[0][d][1]));
            bool mixIt = similar && !((1u << v) & prior) && a.simMul[v] > 0.0f;
            if (mixIt) vsInf = mix(0, 0, similar, v, wInf);
            susc[v] = 1.0f - vsInf;
            float vsSympt = mixIt ? mix(0, 1, similar, v, wInf) : lin(0, d + 1, wInf);
            float vsHosp = mixIt ? mix(0, 2, similar, v, wInf) : lin(0, d + 2, wInf);
            setSlot(v, fmin_ref(1.0f, (1.0f - vsHosp) / (1.0f - vsSympt)));  // slots 2, 4, 5 share index 6; the last write wins
        }
    } else if (infC == 0 && immC > 0) {
        for (uint32_t v = 0; v < nVar; ++v) {
            int similar = a.sim[v] == 0;
            int d = (1 - similar) * 3;
            if (immC == 1 && wImm == 0) continue;
            if (immC == 1 && wImm < 4) {
                float vsInf = (-1.0f * a.eff[1][d][0] * (float)wImm + a.eff[1][d][1]) / 2.0f;
                susc[v] = 1.0f - vsInf;
                float vsSympt = (-1.0f * a.eff[1][d + 1][0] * (float)wImm + a.eff[1][d + 1][1]) / 2.0f;
                float vsHosp = (-1.0f * a.eff[1][d + 2][0] * (float)wImm + a.eff[1][d + 2][1]) / 2.0f;
                setSlot(v, (1.0f - vsHosp) / (1.0f - vsSympt));
            } else {
                int e = immC == 1 ? 1 : 2;
                bool mixIt = similar && a.simMul[v] > 0.0f;
                float vsInf = mixIt ? mix(e, 0, similar, v, wImm) : lin(e, d + 0, wImm);
                susc[v] = 1.0f - vsInf;
                float vsSympt = mixIt ? mix(e, 1, similar, v, wImm) : lin(e, d + 1, wImm);
                float vsHosp = mixIt ? mix(e, 2, similar, v, wImm) : lin(e, d + 2, wImm);
                setSlot(v, (1.0f - vsHosp) / (1.0f - vsSympt));
            }
        }
    } else if (infC > 0 && immC > 0) {
        uint32_t weeks = wInf < wImm ? wInf : wImm;
        int e = immC == 1 ? 3 : 4;
        for (uint32_t v = 0; v < nVar; ++v) {
            int similar = 0;
            for (uint32_t j = 0; j < nVar; ++j) similar = similar || ((prior & (1u << j)) && a.sim[v] == a.sim[j]);
            int d = (1 - similar) * 3;
            bool mixIt = similar && !((1u << v) & prior) && a.simMul[v] > 0.0f;
            float vsInf = (float)((double)(-1.0f * a.eff[e][d][0] * (float)weeks) +
                                  (((1u << v) & prior) ? 0.95 : (double)a.eff[e][d][1]));
            if (mixIt) vsInf = mix(e, 0, similar, v, weeks);
            susc[v] = 1.0f - vsInf;
            float vsSympt = mixIt ? mix(e, 1, similar, v, weeks) : lin(e, d + 1, weeks);
            float vsHosp = mixIt ? mix(e, 2, similar, v, weeks) : lin(e, d + 2, weeks);
            setSlot(v, fmin_ref(1.0f, (1.0f - vsHosp) / (1.0f - vsSympt)));
        }
    }
    for (uint32_t v = 0; v < nVar; ++v) A.susc[(size_t)v * A.suscStride + i] = fmin_ref(1.0f, susc[v]);
}

// ------------------------------------------------------------ vaccination rollout
// Membership of the ten categories of initCategories (immunization.h:229-339),
// indexed as the reference's pass loop indexes them; location-type ids 2, 3,
// 4, 12, 14 and 22 are literals there.
__device__ __forceinline__ bool in_vacc_category(const Agents& A, const Locs& L, uint32_t i, const AgentRec& r, uint32_t g,
                                                 uint8_t precond) {
    const uint32_t age = r.age;
    auto anyEntry = [&](uint32_t kind) {
        for (uint32_t e = r.csrBegin; e < r.csrBegin + r.csrCount; ++e) {
            const uint32_t t = A.possType[e];
            const LocRec lr = L.rec[A.possLoc[e]];
            bool hit = false;
            if (kind == 0) hit = t == 4 && (lr.type == 12 || lr.type == 14);
            else if (kind == 1) hit = (t == 4 || t == 2) && lr.type == 22;
            else if (kind == 4) hit = t == 4 && lr.essential == 1;
            else hit = t == 4 && lr.type == 3;
            if (hit) return true;
        }
        return false;
    };
    switch (g) {
        case 0: return anyEntry(0);
        case 1: return anyEntry(1);
        case 2: return age >= 60;
        case 3: return precond > 0 && age >= 18 && age < 60;
        case 4: return anyEntry(4);
        case 5: return age > 17 && age < 60;
        case 6: return precond > 0 && age >= 60;
        case 7: return anyEntry(7);
        case 8: return age >= 12 && age < 18;
        case 9: return age >= 5 && age < 12;
    }
    return false;
}

struct VaccCategoryArgs {
    Agents A;
    Locs L;
    uint64_t seed;
    uint32_t replica;
    uint32_t nPasses;
    uint8_t passes[10];   // group indices in visiting order
    uint8_t round[10];    // round of each group (its immunizationOrder value)
    float level[10];      // willingness of each group
};

// initCategories: an agent is decided by the first visited group it belongs
// to, with one draw.
__global__ void k_vacc_categories(VaccCategoryArgs a) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.A.n) return;
    const AgentRec r = a.A.rec[i];
    const uint8_t pre = a.A.precond[i];
    uint8_t round = 0;
    for (uint32_t p = 0; p < a.nPasses; ++p) {
        const uint32_t g = a.passes[p];
        if (!in_vacc_category(a.A, a.L, i, r, g, pre)) continue;
        Stream rs(a.seed, a.A.id[i], 0, PH_IMM_CATEGORY, a.replica);
        round = rs.unit() < (double)a.level[g] ? a.round[g] : (uint8_t)255;
        break;
    }
    a.A.immRound[i] = round;
}

__device__ __forceinline__ int age_group_of(uint32_t age) { return age < 90 ? (int)(age / 10) : (age < 200 ? 9 : -1); }

// ages per 10-year group (initAgeGroups, immunization.h:421-479)
__global__ void k_age_groups(Agents A, unsigned long long* out) {
    __shared__ unsigned int sh[10];
    if (threadIdx.x < 10) sh[threadIdx.x] = 0;
    __syncthreads();
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < A.n; i += gridDim.x * blockDim.x) {
        int g = age_group_of(A.rec[i].age);
        if (g >= 0) atomicAdd(&sh[g], 1u);
    }
    __syncthreads();
    if (threadIdx.x < 10 && sh[threadIdx.x]) atomicAdd(&out[threadIdx.x], (unsigned long long)sh[threadIdx.x]);
}

struct VaccDayArgs {
    Agents A;
    Tables T;
    uint64_t seed;
    uint32_t replica;
    uint32_t ts;     // timestamp, 1 at timestamp 0 (immunization.h:485)
    uint32_t tsKey;  // timestamp of the draws
    uint32_t spd;    // steps per day
    uint32_t round;  // booster round / category round
    uint32_t draw;   // draw index of this pass
    uint32_t anyRound;
    float prob[10];
};

// booster eligibility (immunization.h:707-717)
__device__ __forceinline__ bool booster_eligible(const VaccDayArgs& a, uint32_t i, const AgentRec& r) {
    const uint32_t it = a.A.immTs[i];
    return it > 0 && a.A.immCount[i] >= 1 && (a.ts - it) / a.spd > 4u * 30u && a.T.stWB[r.state] == 0 &&
           (a.ts >= a.spd * 3u * 30u && r.diagTs < a.ts - a.spd * 4u * 30u);
}

// first-dose eligibility (immunization.h:849-854)
__device__ __forceinline__ bool vacc_eligible(const VaccDayArgs& a, uint32_t i, const AgentRec& r) {
    return a.A.immCount[i] == 0 && a.T.stWB[r.state] == 0 &&
           ((a.ts < a.spd * 3u * 30u && r.diagTs == 0) || (a.ts >= a.spd * 3u * 30u && r.diagTs < a.ts - a.spd * 3u * 30u));
}

__global__ void k_booster_count(VaccDayArgs a, unsigned long long* out) {
    __shared__ unsigned int sh[10];
    if (threadIdx.x < 10) sh[threadIdx.x] = 0;
    __syncthreads();
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < a.A.n; i += gridDim.x * blockDim.x) {
        const AgentRec r = a.A.rec[i];
        int g = age_group_of(r.age);
        if (g >= 0 && booster_eligible(a, i, r)) atomicAdd(&sh[g], 1u);
    }
    __syncthreads();
    if (threadIdx.x < 10 && sh[threadIdx.x]) atomicAdd(&out[threadIdx.x], (unsigned long long)sh[threadIdx.x]);
}

// the age groups are disjoint, so one pass applies all ten in the
// reference's group-by-group order
__global__ void k_booster_apply(VaccDayArgs a) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.A.n) return;
    const AgentRec r = a.A.rec[i];
    int g = age_group_of(r.age);
    if (g < 0 || !booster_eligible(a, i, r)) return;
    const float prob = a.prob[g];
    Stream rs(a.seed, a.A.id[i], a.tsKey, PH_VACCINATION, a.replica);
    rs.draw = a.draw;
    if (prob == 1.0f || rs.unit() < (double)prob) {
        a.A.immTs[i] = a.ts;
        a.A.immCount[i] = (uint8_t)(a.A.immCount[i] + 1);
    }
}

// per-thread counts, one LDS atomic per thread and one global atomic per block
__device__ __forceinline__ void block_count_add(unsigned int mine, unsigned long long* out) {
    __shared__ unsigned int sh;
    if (threadIdx.x == 0) sh = 0;
    __syncthreads();
    if (mine) atomicAdd(&sh, mine);
    __syncthreads();
    if (threadIdx.x == 0 && sh) atomicAdd(out, (unsigned long long)sh);
}

__global__ void k_vacc_count(VaccDayArgs a, unsigned long long* out) {
    unsigned int mine = 0;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < a.A.n; i += gridDim.x * blockDim.x) {
        const AgentRec r = a.A.rec[i];
        mine += ((a.A.immRound[i] == a.round || a.anyRound) && vacc_eligible(a, i, r)) ? 1u : 0u;
    }
    block_count_add(mine, out);
}

__global__ void k_vacc_apply(VaccDayArgs a) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.A.n) return;
    if (a.A.immRound[i] != a.round) return;
    const AgentRec r = a.A.rec[i];
    if (!vacc_eligible(a, i, r)) return;
    Stream rs(a.seed, a.A.id[i], a.tsKey, PH_VACCINATION, a.replica);
    rs.draw = a.draw;
    if (a.prob[0] == 1.0f || rs.unit() < (double)a.prob[0]) {
        a.A.immTs[i] = a.ts;
        a.A.immCount[i] = 1;
    }
}

__global__ void k_count_immunized(Agents A, uint32_t ts, unsigned long long* out) {
    unsigned int mine = 0;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < A.n; i += gridDim.x * blockDim.x)
        mine += A.immTs[i] == ts ? 1u : 0u;
    block_count_add(mine, out);
}

// ------------------------------------------------------------ non-COVID hospitalisation
__constant__ double c_randomHospProbs[84] = {
    0.00017785,  0.000118567, 0.000614453, 0.003174864, 0.001016573, 0.0011019,   0.000926381, 9.52062E-05,
    6.34708E-05, 0.000328928, 0.000986754, 0.00044981,  0.000623826, 0.000855563, 0.006333678, 0.004222452,
    0.008444904, 0.030227275, 0.036202732, 0.03924143,  0.032990764, 0.003390532, 0.002260355, 0.00452071,
    0.009394699, 0.016018856, 0.022216016, 0.030468759, 0.000364207, 0.000242805, 0.001240249, 0.006390329,
    0.002081773, 0.002256508, 0.001897075, 9.97603E-05, 6.65068E-05, 0.000335,    0.000999373, 0.000471326,
    0.000653666, 0.000896488, 0.002751133, 0.001834089, 0.003668178, 0.013129695, 0.015725228, 0.017045135,
    0.014330059, 0.001472731, 0.000981821, 0.001963642, 0.004080736, 0.006958043, 0.009649877, 0.013234587,
    0.00036181,  0.000241207, 0.001237053, 0.006378891, 0.002068074, 0.002241659, 0.001884591, 9.84773E-05,
    6.56515E-05, 0.000333289, 0.000995818, 0.000465264, 0.000645259, 0.000884959, 0.012211473, 0.008140982,
    0.016281963, 0.058278861, 0.069799674, 0.075658351, 0.063606928, 0.006537022, 0.004358015, 0.008716029,
    0.018113189, 0.030884712, 0.042832973, 0.058744446};

constexpr double MAX_HOSP_PROB = 0.08;  // above every entry

// The day's factor of the admission probabilities (simulation.h:206-422).
__device__ __forceinline__ double other_factor(uint32_t ts, uint32_t dt, float probabilityMul) {
    const int multDay[4] = {99, 99 + 365, 99 + 2 * 365, 99 + 3 * 365};
    const double mult[4] = {0.82, 0.67, 0.9, 0.9};
    int day = (int)(ts / (24u * 60u / dt));
    int d = 0;
    while (d < 3 && day > multDay[d]) d++;
    return probabilityMul > 0.0f ? (double)probabilityMul : mult[d];
}

// Whether anything may happen to the agent: a stay of its ends now, or its
// admission draw (the second; the first is unused) is below any probability
// of the table, so that most agents need no table entry.
__device__ __forceinline__ bool may_other(uint64_t seed, uint32_t replica, uint32_t ts, double factor, const AgentRec& r,
                                          uint32_t id) {
    const uint8_t w = r.cls & CLS_WB;
    if (w == 4) return false;
    if (ts > 0 && r.hospUntil == ts) return true;
    if (w == 3 || ts < r.hospUntil) return false;
    Stream rs(seed, id, ts, PH_OTHER_DISEASE, replica);
    rs.skip();
    return rs.real(1.0) < MAX_HOSP_PROB * factor;
}

// Simulation::otherDisease per-agent part (simulation.h:206-422)
// for agent i (record r, kept up to date)
__device__ __forceinline__ void other_agent(const Agents& A, const Tables& T, uint64_t seed, uint32_t replica, uint32_t ts,
                                            uint32_t dt, double factor, uint32_t i, AgentRec& r, uint32_t id) {
    if (!may_other(seed, replica, ts, factor, r, id)) return;
    const uint8_t w = r.cls & CLS_WB;
    Stream rs(seed, id, ts, PH_OTHER_DISEASE, replica);
    uint8_t age = r.age;
    uint32_t ag = age < 5 ? 0 : age < 15 ? 1 : age < 30 ? 2 : age < 60 ? 3 : age < 70 ? 4 : age < 80 ? 5 : 6;
    uint32_t notSex = A.sex[i] ? 0u : 1u;
    uint8_t pc = A.precond[i];
    uint32_t type = pc == 2 ? 1 : (pc == 4 ? 2 : 0);
    if (ts > 0 && r.hospUntil == ts) {
        if (rs.real(1.0) < c_randomHospProbs[type * 4 * 7 + 2 * 7 + notSex * 7 + ag]) {
            // die(false) (dynamicPPState.cpp:313-325)
            uint8_t dead = (uint8_t)T.nonCOVIDDead;
            A.rec[i].state = r.state = dead;
            A.rec[i].cls = r.cls = T.stCls[dead];
            A.days[i] = -1;
            update_meta(A, T, i, dead);
            A.worstState[i] = (int8_t)dead;
            A.worstTs[i] = ts;
            return;
        }
    }
    if (w == 3 || ts < r.hospUntil) return;
    rs.skip();  // sudden death: disabled in the reference, its draw still made (and unused)
    double probability = c_randomHospProbs[type * 4 * 7 + notSex * 7 + ag] * factor;
    if (rs.real(1.0) < probability) {
        const double avgLengths[3] = {5.55, 2.78, 5.24};
        unsigned avg = (unsigned)avgLengths[type];
        double p = 1.0 / (double)avg;
        unsigned length = (unsigned)geometric(p, rs);
        if (length == 0) length = 1;
        A.rec[i].hospTs = r.hospTs = ts;
        A.rec[i].hospUntil = r.hospUntil = ts + length * 24u * 60u / dt;
    }
}

__global__ void k_count_covid_hospital(Agents A, Locs L, Tables T, uint32_t ts, uint32_t dueWith,
                                       unsigned long long* out) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    bool c = false;
    if (i < A.n) {
        uint8_t st = A.rec[i].state;
        if (dueWith == 0) c = st >= 6 && st <= 8;
        else
            c = T.stInfected[st] && L.rec[A.location[i]].type == T.lt.hospital &&
                !(T.stWB[st] < 3 && ts > 0 && A.rec[i].hospUntil == ts);
    }
    unsigned long long m = __ballot(c);
    if ((threadIdx.x & 63u) == 0 && m) atomicAdd(out, (unsigned long long)__popcll(m));
}

// ------------------------------------------------------------ statistics
enum StatSlot {
    S_HOSP = 0, S_STAYED, S_Q, S_QT, S_NQ, S_ALLINF, S_NI, S_INF, S_REINF, S_BSTR, S_HCI, S_HCE, S_INFH, S_VNI,
    S_VARINF = 14,            // + v
    S_INFV = S_VARINF + MAXV, // + v
    S_IMM = S_INFV + MAXV,    // + v (2^-24 fixed point)
    S_STATE = S_IMM + MAXV,   // + state
    S_COUNT = S_STATE + 128,
    // after the statistics: performTests' three counts, agents immunized today
    S_TESTS = S_COUNT, S_IMMUNIZED = S_TESTS + 3, DAY_COUNTERS
};
constexpr uint32_t DAY_COPIES = 16;  // of the day pass's counters at most, summed by the host

// ------------------------------------------------------------ the day's agent passes
// Testing, progression, immunity, the other disease and the statistics touch
// only the agent's own fields (and location flags that none of them writes),
// so one pass over the agents makes whichever of them are asked for
// (`stages`), in the reference's order for each agent, reading its record
// once.  A midnight of 10M agents took 574 us in five passes, and takes 352; of
// 600k with hourly steps 152 and 78.
enum DayStage : uint32_t {
    DAY_TEST = 1, DAY_PROGRESS = 2, DAY_IMMUNITY = 4, DAY_OTHER = 8, DAY_STATS = 16, DAY_IMMUNIZED = 32
};
struct DayArgs {
    Agents A;
    Locs L;
    Tables T;
    uint64_t seed;
    uint32_t replica, ts, dt, stages;
    TestParams test;
    ImmParams imm;
    float probabilityMul;
    unsigned long long* counters;  // [copies][DAY_COUNTERS]
    uint32_t copies;               // at most DAY_COPIES
};

// The flag word of one agent: bit k set counts it in counter dayFlagSlot(k).
// 0-6 infected with variant v, 7-13 ever infected by variant v, then:
enum DayFlag : uint32_t {
    DF_HOSP = 14, DF_STAYED, DF_Q, DF_QT, DF_NQ, DF_ALLINF, DF_NI, DF_INF, DF_HCI, DF_HCE, DF_INFH, DF_VNI, DF_TEST0,
    DF_IMMUNIZED = DF_TEST0 + 3, DAY_FLAGS
};
static_assert(DAY_FLAGS <= 32, "one word");
__device__ __forceinline__ uint32_t day_flag_slot(uint32_t k) {
    constexpr uint8_t slot[DAY_FLAGS] = {S_VARINF, S_VARINF + 1, S_VARINF + 2, S_VARINF + 3, S_VARINF + 4, S_VARINF + 5, S_VARINF + 6,
                                         S_INFV, S_INFV + 1, S_INFV + 2, S_INFV + 3, S_INFV + 4, S_INFV + 5, S_INFV + 6,
                                         S_HOSP, S_STAYED, S_Q, S_QT, S_NQ, S_ALLINF, S_NI, S_INF, S_HCI, S_HCE, S_INFH, S_VNI,
                                         S_TESTS, S_TESTS + 1, S_TESTS + 2, S_IMMUNIZED};
    return slot[k];
}

// One agent's stages in order, then its flag word.
struct DaySums {
    uint32_t reinf = 0, bstr = 0;
    unsigned long long imm[MAXV] = {0};
};
struct DayLoads {
    AgentRec r;
    uint32_t id, lastTest;
    int16_t days;
    uint8_t ic, mc;
};
__device__ __forceinline__ uint32_t day_flags(const Agents& A, const Locs& L, const Tables& T, uint32_t ts, uint32_t day,
                                              uint32_t i, const AgentRec& r, uint8_t ic, uint8_t mc, DaySums& sums) {
    uint32_t f = 0;
    const uint8_t w = r.cls & CLS_WB;
    const bool inf = (r.cls & CLS_INFECTED) != 0;
    bool isQ = false, newInf = false;
    if (r.quarUntil > ts) isQ = A.quarTs[i] <= ts;
    if (ic != 0) {  // infected once or more: only then an infection time and variants
        const uint32_t it = A.infTs[i];
        newInf = it > ts - day && it <= ts;
        f |= ((uint32_t)A.statVar[i] & 0x7Fu) << 7 | 1u << DF_INF;
        sums.reinf += ic - 1u;
    }
    if (inf) {
        f |= 1u << r.variant | 1u << DF_ALLINF | (isQ ? 1u << DF_QT : 1u << DF_NQ);
        if (L.type8[A.location[i]] == T.lt.hospital) f |= 1u << DF_INFH;
    }
    f |= w != 4 && w != 3 && ts < r.hospUntil ? 1u << DF_HOSP : 0u;
    f |= r.flags & F_STAYED_HOME ? 1u << DF_STAYED : 0u;
    f |= isQ ? 1u << DF_Q : 0u;
    f |= newInf ? 1u << DF_NI : 0u;
    if (r.flags & F_HCW) f |= (inf || (r.flags & F_QUARANTINED) ? 1u << DF_HCI : 0u) | (newInf ? 1u << DF_HCE : 0u);
    if (mc != 0) {
        f |= ic == 0 ? 1u << DF_VNI : 0u;
        sums.bstr += mc - 1u;
    }
    return f;
}

// The 256-agent chunks blk, blk + nBlk, ... of one population, at most
// DAY_MOST of them, in groups of DAY_GROUP.  On most days nothing happens to
// most agents (no test, no transition, full susceptibility, no admission):
// the first pass over a group streams the agents, decides that from one round
// of loads and two draws, counts them, and appends the others to an LDS list;
// the second runs all stages for the listed ones, 64 at a time, instead of
// having every wave wait for the dependent reads of one lane after another.
// Each agent's yes/no counts are one flag word, and a lane adds words in
// bit-sliced counters (plane j holds bit j of all 32 counts: a few logic
// operations per agent for all of them); the sums go through LDS to one of
// a.copies copies of the counters, because many blocks that end together would
// queue at one copy's words.  STAGES: the stages, if the compiler is to know
// them, else 0 (a.stages).
constexpr uint32_t DAY_PLANES = 7, DAY_MOST = ((1u << DAY_PLANES) - 1u) / 2u, DAY_GROUP = 8;
template <uint32_t STAGES>
__device__ __forceinline__ void day_pass(const Agents& A, const Locs& L, const Tables& T, const DayArgs& a, uint32_t blk,
                                         uint32_t nBlk) {
    __shared__ unsigned long long sh[DAY_COUNTERS];
    __shared__ uint16_t list[256 * DAY_GROUP];  // (chunk of the group << 8) | agent of the chunk
    __shared__ uint32_t nList;
    for (uint32_t k = threadIdx.x; k < DAY_COUNTERS; k += blockDim.x) sh[k] = 0;
    if (threadIdx.x == 0) nList = 0;
    __syncthreads();
    const uint32_t stages = STAGES ? STAGES : a.stages, ts = a.ts, dt = a.dt;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t day = 24u * 60u / dt;
    const uint32_t nVar = T.nVar, n = A.n;
    const double factor = other_factor(ts, dt, a.probabilityMul);
    const bool full0 = T.stSusc[0] != 0;  // state 0 is susceptible: 1 for whoever was never infected nor immunized
    const unsigned long long below = (1ull << lane) - 1ull;
    uint32_t plane[DAY_PLANES] = {0};
    DaySums sums;
    auto add_flags = [&](uint32_t f) {
#pragma unroll
        for (uint32_t j = 0; j < DAY_PLANES; ++j) {
            const uint32_t carry = plane[j] & f;
            plane[j] ^= f;
            f = carry;
        }
    };
    // state histogram: one LDS atomic per distinct state of the wave
    auto add_states = [&](bool valid, uint32_t st) {
        unsigned long long todo = __ballot(valid);
        while (todo) {
            const uint32_t first = (uint32_t)(__ffsll((long long)todo) - 1);
            const uint32_t s0 = (uint32_t)__builtin_amdgcn_readlane((int)st, (int)first);
            const unsigned long long m = __ballot(valid && st == s0);
            if (lane == first) atomicAdd(&sh[S_STATE + s0], (unsigned long long)__popcll(m));
            todo &= ~m;
        }
    };
    auto load = [&](uint32_t i) {
        DayLoads d{};
        d.r = A.rec[i];
        d.id = A.id[i];
        if (stages & DAY_TEST) d.lastTest = A.lastTest[i];
        if (stages & DAY_PROGRESS) d.days = A.days[i];
        if (stages & (DAY_IMMUNITY | DAY_STATS)) {
            d.ic = A.infCount[i];
            d.mc = A.immCount[i];
        }
        return d;
    };
    for (uint32_t group = blk; group * 256u < n; group += DAY_GROUP * nBlk) {
        uint32_t state0 = 0;  // of the wave
        for (uint32_t c = 0; c < DAY_GROUP; ++c) {
            const uint32_t i = (group + c * nBlk) * 256u + threadIdx.x;
            if (i - threadIdx.x >= n) break;
            const bool valid = i < n;
            bool rare = false, light = false;
            uint32_t f = 0;
            if (valid) {
                const DayLoads d = load(i);
                rare = (d.days == 0 || d.days == -2) && (stages & DAY_PROGRESS);
                if (stages & DAY_TEST) rare = rare || may_test(a.seed, a.replica, ts, dt, a.test, d.r, d.id, d.lastTest);
                if (stages & (DAY_IMMUNITY | DAY_STATS))
                    rare = rare || d.ic != 0 || d.mc != 0 || d.r.state != 0 || !full0 || (d.r.cls & CLS_INFECTED);
                if (stages & DAY_OTHER) rare = rare || may_other(a.seed, a.replica, ts, factor, d.r, d.id);
                if (stages & DAY_IMMUNIZED) rare = rare || A.immTs[i] == (ts == 0 ? 1u : ts);
                light = !rare;
                if (light) {
                    if (stages & DAY_TEST) f = test_counts(ts, day, d.lastTest, d.r.diagTs) << DF_TEST0;
                    if ((stages & DAY_PROGRESS) && d.days > 0) A.days[i] = (int16_t)(d.days - 1);
                    if (stages & DAY_STATS) f |= day_flags(A, L, T, ts, day, i, d.r, 0, 0, sums);
                }
            }
            if (stages & DAY_STATS) state0 += (uint32_t)__popcll(__ballot(light));  // in state 0
            add_flags(f);
            const unsigned long long m = __ballot(rare);
            if (m != 0ull) {
                uint32_t pos = 0;
                if (lane == 0) pos = atomicAdd(&nList, (uint32_t)__popcll(m));
                pos = (uint32_t)__builtin_amdgcn_readfirstlane((int)pos) + (uint32_t)__popcll(m & below);
                if (rare) list[pos] = (uint16_t)((c << 8) | threadIdx.x);
            }
        }
        if (lane == 0 && state0) atomicAdd(&sh[S_STATE], (unsigned long long)state0);
        __syncthreads();
        const uint32_t cnt = nList;
        for (uint32_t j0 = 0; j0 < cnt; j0 += 256u) {
            const uint32_t j = j0 + threadIdx.x;
            const bool valid = j < cnt;
            uint32_t st = 0, f = 0;
            if (valid) {
                const uint32_t e = list[j];
                const uint32_t i = (group + (e >> 8) * nBlk) * 256u + (e & 0xFFu);
                DayLoads d = load(i);
                AgentRec& r = d.r;
                if (stages & DAY_TEST)
                    f = test_agent(A, L, T, a.seed, a.replica, ts, dt, a.test, i, r, d.id, d.lastTest) << DF_TEST0;
                if (stages & DAY_PROGRESS) progress_agent(A, T, a.seed, a.replica, ts, dt, i, r, d.id, d.days);
                if ((stages & DAY_IMMUNITY) && r.state == 0) immunize_agent(A, T, ts, dt, a.imm, i, d.ic, d.mc);
                if (stages & DAY_OTHER) other_agent(A, T, a.seed, a.replica, ts, dt, factor, i, r, d.id);
                if (stages & DAY_IMMUNIZED) f |= A.immTs[i] == (ts == 0 ? 1u : ts) ? 1u << DF_IMMUNIZED : 0u;
                st = r.state;
                if (stages & DAY_STATS) {
                    f |= day_flags(A, L, T, ts, day, i, r, d.ic, d.mc, sums);
#pragma unroll
                    for (uint32_t v = 0; v < (uint32_t)MAXV; ++v) {
                        if (v >= nVar) break;
                        const float s = A.susc[(size_t)v * A.suscStride + i];
                        sums.imm[v] += (unsigned long long)(long long)((double)(1.0f - s) * 16777216.0);
                    }
                }
            }
            if (stages & DAY_STATS) add_states(valid, st);
            add_flags(f);
        }
        __syncthreads();
        if (threadIdx.x == 0) nList = 0;
        __syncthreads();
    }
    // the wave's counts
    uint32_t any = 0;
#pragma unroll
    for (uint32_t j = 0; j < DAY_PLANES; ++j) any |= plane[j];
#pragma unroll
    for (uint32_t k = 0; k < DAY_FLAGS; ++k) {
        if (__ballot((any >> k) & 1u) == 0ull) continue;
        uint32_t c = 0;
#pragma unroll
        for (uint32_t j = 0; j < DAY_PLANES; ++j) c += (uint32_t)__popcll(__ballot((plane[j] >> k) & 1u)) << j;
        if (lane == 0) atomicAdd(&sh[day_flag_slot(k)], (unsigned long long)c);
    }
    if (sums.reinf) atomicAdd(&sh[S_REINF], (unsigned long long)sums.reinf);
    if (sums.bstr) atomicAdd(&sh[S_BSTR], (unsigned long long)sums.bstr);
#pragma unroll
    for (uint32_t v = 0; v < (uint32_t)MAXV; ++v) {
        unsigned long long x = sums.imm[v];
        if (__ballot(x != 0ull) == 0ull) continue;
        for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
        if (lane == 0) atomicAdd(&sh[S_IMM + v], x);
    }
    __syncthreads();
    unsigned long long* out = a.counters + (size_t)(blk % a.copies) * DAY_COUNTERS;
    for (uint32_t k = threadIdx.x; k < DAY_COUNTERS; k += blockDim.x)
        if (sh[k]) atomicAdd(&out[k], sh[k]);
}

// amdgpu_waves_per_eu(8): bound by the latency of the listed agents' dependent
// reads, the pass gains more from resident waves than it loses to spilled
// registers (10M agents 421 us at the compiler's 4 waves per SIMD, 352 at 8).
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8))) k_day(DayArgs a) { day_pass<0>(a.A, a.L, a.T, a, blockIdx.x, gridDim.x); }

// A stage asked for by itself (a host loop that calls the routines one by one)
// carries nothing of the others: the statistics as a pass whose stages the
// compiler knows, the others one agent per thread, without lists or bit-sliced
// counters.  Per call, MI355X, as k_day / this: 16k agents testing 41 / 28 us,
// progression 23 / 16, immunity 26 / 19, other disease 22 / 14, statistics
// 39 / 26; 1M 67 / 44, 38 / 21, 47 / 28, 43 / 21, 60 / 42; 10M 241 / 220,
// 58 / 40, 166 / 106, 152 / 90, 165 / 117.
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8))) k_day_stats(DayArgs a) {
    day_pass<DAY_STATS>(a.A, a.L, a.T, a, blockIdx.x, gridDim.x);
}

template <uint32_t STAGE>
__global__ void __launch_bounds__(256) k_stage(DayArgs a) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    const Agents& A = a.A;
    const bool valid = i < A.n;
    if constexpr (STAGE == DAY_PROGRESS) {
        if (!valid) return;
        const int16_t days = A.days[i];
        if (days > 0) A.days[i] = (int16_t)(days - 1);
        if (days != -2 && days != 0) return;
        AgentRec r = A.rec[i];
        progress_agent(A, a.T, a.seed, a.replica, a.ts, a.dt, i, r, A.id[i], days);
    }
    if constexpr (STAGE == DAY_IMMUNITY)
        if (valid && A.rec[i].state == 0) immunize_agent(A, a.T, a.ts, a.dt, a.imm, i, A.infCount[i], A.immCount[i]);
    if constexpr (STAGE == DAY_OTHER)
        if (valid) {
            AgentRec r = A.rec[i];
            other_agent(A, a.T, a.seed, a.replica, a.ts, a.dt, other_factor(a.ts, a.dt, a.probabilityMul), i, r, A.id[i]);
        }
    if constexpr (STAGE == DAY_TEST) {
        __shared__ uint32_t sh[3];
        if (threadIdx.x < 3) sh[threadIdx.x] = 0;
        __syncthreads();
        uint32_t f = 0;
        if (valid) {
            AgentRec r = A.rec[i];
            f = test_agent(A, a.L, a.T, a.seed, a.replica, a.ts, a.dt, a.test, i, r, A.id[i], A.lastTest[i]);
        }
#pragma unroll
        for (uint32_t k = 0; k < 3; ++k) {
            const unsigned long long b = __ballot((f >> k) & 1u);
            if (b != 0ull && (threadIdx.x & 63u) == 0u) atomicAdd(&sh[k], (uint32_t)__popcll(b));
        }
        __syncthreads();
        if (threadIdx.x < 3 && sh[threadIdx.x]) atomicAdd(&a.counters[S_TESTS + threadIdx.x], (unsigned long long)sh[threadIdx.x]);
    }
}

// performTests' first pass: the locations of the agents diagnosed in the last
// day are flagged for day_pass's testing.
__global__ void k_flag_locations(DayArgs a) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < a.A.n) flag_agent(a.A, a.L, a.T, a.seed, a.replica, a.ts, a.dt, a.test, i);
}

// ------------------------------------------------------------ planning
struct PlanArgs {
    Agents A;
    Locs L;
    Tables T;
    uint64_t seed;
    uint32_t replica, ts, dt, curfewEnd, schoolAge;
    uint32_t policy;                // quarantine policy
    const uint32_t* adults;         // the agents aged 27-64
    uint32_t nAdults;
};

// checkSchoolQuarantine (movementPolicies.h:1285-1310), one thread per school
__device__ __forceinline__ void plan_school(const PlanArgs& a, uint32_t s) {
    if (s >= a.L.nSchools) return;
    LocRec* q = a.L.rec;
    uint32_t school = a.L.schools[s];
    if (q[school].quarUntil > a.ts) return;
    uint32_t counter = 0, mx = 0;
    for (uint32_t c = a.L.classOff[s]; c < a.L.classOff[s + 1]; ++c) {
        uint32_t cu = q[a.L.classrooms[c]].quarUntil;
        if (cu > a.ts) {
            counter++;
            mx = mx > cu ? mx : cu;
        }
    }
    if (counter > 1) {
        q[school].quarUntil = mx;
        mark_special(a.L, school);
        for (uint32_t c = a.L.classOff[s]; c < a.L.classOff[s + 1]; ++c) {
            q[a.L.classrooms[c]].quarUntil = mx;
            mark_special(a.L, a.L.classrooms[c]);
        }
    }
}

// Per-agent part of planLocations in one pass: the resets of
// movementPolicies.h:1446-1451 (stepsUntilMove := curfewEnd, stayedHome,
// noWorkAgent) and, with quarantinePolicy > 2, checkSchoolWorkQuarantine
// (movementPolicies.h:1188-1240).
__device__ __forceinline__ void plan_agent(const PlanArgs& a, uint32_t i) {
    const Agents& A = a.A;
    if (i >= A.n) return;
    const bool schoolwork = a.policy > 2;
    A.wake[i] = a.curfewEnd < 1440u / a.dt ? (uint16_t)a.curfewEnd : WAKE_NONE;
    const AgentRec r = A.rec[i];
    uint8_t fl = (uint8_t)((r.flags | F_STAYED_HOME) & ~F_NO_WORK);
    if (schoolwork && !(fl & F_QUARANTINED) && !(r.diagTs > 0 && !a.T.stInfected[r.state])) {
        const pansim_location_types& lt = a.T.lt;
        Stream rs(a.seed, a.A.id[i], a.ts, PH_PLAN_SCHOOLWORK, a.replica);
        const CsrReg csr = load_csr(A, i, r);
        // the planning lookup (home, school, classroom first-match): a
        // workplace is drawn when the agent has several, in this order
        uint32_t wl = find_loc(A, a.L, lt, csr, lt.work, 0, &rs, true);
        uint32_t sl = find_loc(A, a.L, lt, csr, lt.school, 0, nullptr, true);
        uint32_t cl = find_loc(A, a.L, lt, csr, lt.classroom, 0, nullptr, true);
        // the three quarantine times loaded together, then the first that
        // applies; a location whose special bit is clear was last quarantined
        // until at most the first step of the day that ends now (every
        // quarantine write since, tonight's school quarantines included, sets
        // the bit), so its record is not read
        const LocRec* q = a.L.rec;
        const uint32_t qs = sl != NOLOC && loc_special(a.L, sl) ? q[sl].quarUntil : 0u;
        const uint32_t qc = cl != NOLOC && loc_special(a.L, cl) ? q[cl].quarUntil : 0u;
        const uint32_t qw = wl != NOLOC && loc_special(a.L, wl) ? q[wl].quarUntil : 0u;
        uint32_t until = 0;
        if (qs > a.ts) until = qs;
        else if (qc > a.ts) until = qc;
        else if (qw > a.ts) until = qw;
        if (until > 0) {
            fl |= F_QUARANTINED;
            A.quarTs[i] = a.ts;
            A.rec[i].quarUntil = until;
            A.daysInQ[i] += (until - a.ts) / (24u * 60u / a.dt);
        }
    }
    if (fl != r.flags) A.rec[i].flags = fl;
}

// Per-location part: noWork reset (movementPolicies.h:1449) and, with
// quarantinePolicy > 2, the quarantine -> closedUntil conversion
// (movementPolicies.h:1544-1557).
// Also recomputes the special-location bits for the day (loc_special), clears
// the testing flags, and clears the infectiousness sums with the visited bits:
// no agent changes location between the day's last movement step and the
// planning, so the occupancy counts stand, and plan_sums_underage refills the
// sums (which the midnight passes change through state and variant) from the
// infectious agents alone.  64 consecutive lanes cover 64 consecutive
// locations (l0 = the first lane's) and write their bitmap words from a ballot.
__device__ __forceinline__ void plan_loc(const PlanArgs& a, uint32_t l) {
    const pansim_location_types& lt = a.T.lt;
    const uint32_t dayStart = a.ts - a.ts % (1440u / a.dt);
    const bool valid = l < a.L.n;
    bool sp = false;
    if (valid) {
        LocRec* lr = &a.L.rec[l];
        const LocRec r = *lr;
        uint32_t q = r.quarUntil, closed = r.closedUntil;
        if (a.policy > 2 && q > a.ts) {
            if (r.type == lt.school || r.type == lt.classroom) {
                closed = q;
                q = 0;
            } else if (r.type == lt.work) {
                q = 0;
            }
        }
        if (r.noWork != 0u) lr->noWork = 0u;
        if (q != r.quarUntil) lr->quarUntil = q;
        if (closed != r.closedUntil) lr->closedUntil = closed;
        sp = q > dayStart || closed > dayStart || r.open == 0;
        a.L.dyn[l].sum0 = 0;
        for (uint32_t v = 1; v < a.T.nVar; ++v) a.L.sumX[(size_t)(v - 1) * a.L.n + l] = 0;
    }
    const unsigned long long bits = __ballot(sp);
    if (valid && (l & 31u) == 0u) {
        a.L.special[l >> 5] = (uint32_t)((l & 32u) ? bits >> 32 : bits);
        a.L.noWorkBits[l >> 5] = 0u;  // with noWork above
        a.L.flagBits[l >> 5] = 0u;
        a.L.visited[l >> 5] = 0u;
    }
}

constexpr uint32_t NOWORK_FLAGGED = 0xFFFFFFFFu;

// The sums of agent i's location, and checkUnderageAtHome
// (movementPolicies.h:1056-1094) for an agent aged 14 or less
__device__ __forceinline__ void plan_sums_underage(const PlanArgs& a, uint32_t i) {
    const Agents& A = a.A;
    if (i >= A.n) return;
    const AgentRec r = A.rec[i];
    if (r.cls & CLS_INFECTIOUS) {
        const float x = a.T.stInf[r.state] * a.T.varMul[r.variant];
        if (x != 0.0f) {
            const uint32_t loc = A.location[i];
            atomicAdd((unsigned long long*)loc_sum(a.L, r.variant, loc), (unsigned long long)fixed32(x));
            mark_visited(a.L, loc);
        }
    }
    if (r.age > 14) return;
    const pansim_location_types& lt = a.T.lt;
    bool flag = false;
    if (r.flags & F_QUARANTINED) flag = true;
    else {
        const CsrReg csr = load_csr(A, i, r);
        uint32_t sl = find_loc(A, a.L, lt, csr, lt.school, 0, nullptr, true);
        uint32_t cl = find_loc(A, a.L, lt, csr, lt.classroom, 0, nullptr, true);
        bool tooOld = r.age >= a.schoolAge;
        // (a location that is not special is open and not closed today)
        auto shut = [&](uint32_t l) {
            return l != NOLOC && loc_special(a.L, l) && (a.L.rec[l].open == 0 || a.L.rec[l].closedUntil > a.ts);
        };
        flag = tooOld || shut(sl) || shut(cl);
    }
    if (flag) {
        uint32_t h = r.home;
        if (h != NOLOC) {
            a.L.rec[h].noWork = NOWORK_FLAGGED;
            atomicOr(&a.L.noWorkBits[h >> 5], 1u << (h & 31u));
        }
    }
}

// A home flagged by tonight's planning (an L2-resident bitmap read before the
// home's location record)
__device__ __forceinline__ bool nowork_flagged(const Locs& L, uint32_t h) {
    return h != NOLOC && ((L.noWorkBits[h >> 5] >> (h & 31u)) & 1u) != 0u;
}

// setNoWorkToday (movementPolicies.h:1137-1158): the lowest eligible agent of
// a flagged home claims it (claim pass, then resolve pass), over the list of
// the agents aged 27-64 (`adults`, n entries)
__device__ __forceinline__ void plan_nowork_claim(const PlanArgs& a, uint32_t j) {
    const Agents& A = a.A;
    if (j >= a.nAdults) return;
    const uint32_t i = a.adults[j];
    uint32_t h = A.rec[i].home;
    // 0 = not flagged, NOWORK_FLAGGED = flagged, else (claiming agent's
    // input index + 1)
    if (nowork_flagged(a.L, h)) atomicMin(&a.L.rec[h].noWork, A.id[i] + 1u);
}

__device__ __forceinline__ void plan_nowork_resolve(const PlanArgs& a, uint32_t j) {
    const Agents& A = a.A;
    if (j >= a.nAdults) return;
    const uint32_t i = a.adults[j];
    uint32_t h = A.rec[i].home;
    if (nowork_flagged(a.L, h) && a.L.rec[h].noWork == A.id[i] + 1u) A.rec[i].flags = (uint8_t)(A.rec[i].flags | F_NO_WORK);
}

// The planning's passes, in order; each runs over one kind of unit.
enum PlanPass { PLAN_SCHOOL, PLAN_AGENT, PLAN_LOC, PLAN_SUMS_UNDERAGE, PLAN_CLAIM, PLAN_RESOLVE };
template <PlanPass P>
__device__ __forceinline__ void plan_unit(const PlanArgs& a, uint32_t u) {
    if constexpr (P == PLAN_SCHOOL) plan_school(a, u);
    if constexpr (P == PLAN_AGENT) plan_agent(a, u);
    if constexpr (P == PLAN_LOC) plan_loc(a, u);
    if constexpr (P == PLAN_SUMS_UNDERAGE) plan_sums_underage(a, u);
    if constexpr (P == PLAN_CLAIM) plan_nowork_claim(a, u);
    if constexpr (P == PLAN_RESOLVE) plan_nowork_resolve(a, u);
}
template <PlanPass P>
__global__ void __launch_bounds__(256) k_plan(PlanArgs a) {
    plan_unit<P>(a, blockIdx.x * 256u + threadIdx.x);
}

// The same passes for every replica of a batch by one launch each: block b
// works on replica rep[b], its (b - first[rep[b]])-th block.  A replica whose
// midnight is made on its own (stages 0, null counters) is skipped.
struct BlockTable {
    const uint32_t* rep;    // [blocks]
    const uint32_t* first;  // [replicas + 1]
};
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8))) k_day_batch(const DayArgs* args, BlockTable t) {
    const uint32_t r = t.rep[blockIdx.x];
    const DayArgs& a = args[r];
    if (a.stages == 0u) return;
    Agents A = a.A;
    Locs L = a.L;
    Tables T = a.T;
    globalize(A), globalize(L), globalize(T);
    day_pass<0>(A, L, T, a, blockIdx.x - t.first[r], t.first[r + 1] - t.first[r]);
}
__global__ void __launch_bounds__(256) k_flag_batch(const DayArgs* args, BlockTable t) {
    const uint32_t r = t.rep[blockIdx.x];
    const DayArgs& a = args[r];
    const uint32_t i = (blockIdx.x - t.first[r]) * 256u + threadIdx.x;
    Agents A = a.A;
    Locs L = a.L;
    Tables T = a.T;
    globalize(A), globalize(L), globalize(T);
    if ((a.stages & DAY_TEST) && i < A.n) flag_agent(A, L, T, a.seed, a.replica, a.ts, a.dt, a.test, i);
}
template <PlanPass P>
__global__ void __launch_bounds__(256) k_plan_batch(const PlanArgs* args, BlockTable t) {
    const uint32_t r = t.rep[blockIdx.x];
    PlanArgs a = args[r];
    globalize(a.A), globalize(a.L), globalize(a.T);
    gptr(a.adults);
    if (P == PLAN_SCHOOL && a.policy <= 3) return;
    plan_unit<P>(a, (blockIdx.x - t.first[r]) * 256u + threadIdx.x);
}

// ------------------------------------------------------------ closures
struct TypeList {
    uint32_t t[16];
};
__global__ void k_set_open(Locs L, TypeList types, uint32_t n, uint8_t open) {
    uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t l = blockIdx.x * blockDim.x + threadIdx.x; l < L.n; l += stride) {
        if (L.rec[l].essential == 1) continue;
        for (uint32_t k = 0; k < n; ++k)
            if (L.rec[l].type == types.t[k]) {
                L.rec[l].open = open;
                if (!open) mark_special(L, l);
            }
    }
}

__global__ void k_scale_inf(Locs L, uint32_t homeType, double factor, uint32_t divide, const float* typeMul) {
    uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t l = blockIdx.x * blockDim.x + threadIdx.x; l < L.n; l += stride) {
        const uint32_t t = L.rec[l].type;
        if (t == homeType) continue;
        const float v = divide ? (float)((double)L.infRaw[l] / factor) : (float)((double)L.infRaw[l] * factor);
        L.infRaw[l] = v;
        L.dyn[l].inf = v * typeMul[t];
    }
}

// The infection factor of every location after a change of the type
// multipliers.
__global__ void k_loc_infm(Locs L, const float* typeMul) {
    uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t l = blockIdx.x * blockDim.x + threadIdx.x; l < L.n; l += stride)
        L.dyn[l].inf = L.infRaw[l] * typeMul[L.rec[l].type];
}

// ExposeToMutation (closurePolicies.h:356-390)
__global__ void k_expose_mutation(Agents A, Tables T, uint64_t seed, uint32_t replica, uint32_t ts, uint32_t v,
                                  double fraction) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= A.n) return;
    float s = A.susc[(size_t)v * A.suscStride + i];
    if (!(s > 0.0f)) return;
    Stream rs(seed, A.id[i], ts, PH_MUTATION, replica);
    if (rs.unit() < fraction * (double)s) {
        uint8_t fi = (uint8_t)T.firstInfected;
        A.rec[i].state = fi;
        A.rec[i].cls = T.stCls[fi];
        A.rec[i].variant = (uint8_t)v;
        A.days[i] = -2;
        update_meta(A, T, i, fi);
        A.infTs[i] = ts;
        A.infLoc[i] = A.location[i];
        A.infCount[i] = (uint8_t)(A.infCount[i] + 1);
        A.worstState[i] = (int8_t)fi;
        A.worstTs[i] = ts;
        A.statVar[i] = (uint8_t)(A.statVar[i] | (1u << v));
    }
}

// ------------------------------------------------------------ hazard gradient
// The sums over the copies, in one order.
__global__ void __launch_bounds__(256) k_hazard_sum(const double* copies, double* out) {
    const uint32_t j = blockIdx.x * 256u + threadIdx.x;
    if (j >= HAZARD_SLOTS) return;
    double s = 0.0;
    for (uint32_t c = 0; c < HAZARD_COPIES; ++c) s += copies[(size_t)c * HAZARD_SLOTS + j];
    out[j] = s;
}

// ------------------------------------------------------------ field downloads
// One member of an array of records (or an array: pitch = width) as 32-bit
// values in input order, where `id` maps stored to input index (null: as
// stored).  A record is read for one of its members, so this is bound by the
// record's bytes; the host then receives 4 B per value, contiguous, instead of
// whole records that it takes apart and scatters (a snapshot of 400k agents,
// 11 fields and the sums: 8.6 ms that way).
enum FieldKind : uint32_t { FIELD_U8, FIELD_I8, FIELD_U16, FIELD_I16, FIELD_U32, FIELD_BIT, FIELD_WAKE };
struct FieldArgs {
    const uint8_t* base;
    uint32_t pitch, offset, kind;
    uint32_t param;  // FIELD_BIT: the bit; FIELD_WAKE: the day's first step minus the timestamp
    const uint32_t* id;
    uint32_t n;
    uint32_t* out;
};
__global__ void __launch_bounds__(256) k_field(FieldArgs a) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= a.n) return;
    const uint8_t* p = a.base + (size_t)i * a.pitch + a.offset;
    uint32_t v = 0;
    switch (a.kind) {
    case FIELD_U8: v = *p; break;
    case FIELD_I8: v = (uint32_t)(int32_t)(int8_t)*p; break;
    case FIELD_U16: v = *(const uint16_t*)p; break;
    case FIELD_I16: v = (uint32_t)(int32_t)*(const int16_t*)p; break;
    case FIELD_U32: v = *(const uint32_t*)p; break;
    case FIELD_BIT: v = (*p & a.param) ? 1u : 0u; break;
    default: {
        const uint16_t w = *(const uint16_t*)p;
        v = w == WAKE_NONE ? NEVER : a.param + w;
    }
    }
    a.out[a.id ? a.id[i] : i] = v;
}

// The variant-0 sums, contiguous.
__global__ void __launch_bounds__(256) k_sums0(const LocDyn* dyn, uint32_t n, long long* out) {
    const uint32_t l = blockIdx.x * 256u + threadIdx.x;
    if (l < n) out[l] = dyn[l].sum0;
}

// ------------------------------------------------------------ test helpers
__global__ void k_expf(const float* in, float* out, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = ps_expf(in[i]);
}
__global__ void k_log(const double* in, double* out, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = ps_log(in[i]);
}
__global__ void k_philox(const uint32_t* ctr, uint32_t k0, uint32_t k1, uint32_t* out, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    u32x4 c;
    for (int j = 0; j < 4; ++j) c.v[j] = ctr[4 * i + j];
    u32x4 r = philox4x32_10(c, k0, k1);
    for (int j = 0; j < 4; ++j) out[4 * i + j] = r.v[j];
}

}  // namespace dev
}  // namespace ps
