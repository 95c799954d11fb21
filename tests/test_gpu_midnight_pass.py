"""The midnight's one pass over the agents (pansim_midnight_day) against the
routines called one by one (pansim_testing_day, pansim_progression_day,
pansim_immunization_day, pansim_other_disease_day, pansim_stats_day): the same
fields, counts and statistics, at sizes around a wave, a block, a group of
blocks and past the lines of its launch, with probabilities that test nobody,
a few and everybody (the fast reject off, in use and never taken).  Every
compared value is whole."""
import ctypes

import numpy as np
import pytest

import pansim_amd

pytestmark = pytest.mark.gpu

u32, f32, f64, i32 = ctypes.c_uint32, ctypes.c_float, ctypes.c_double, ctypes.c_int32


class Midnight(ctypes.Structure):
    _fields_ = [("timestamp", u32), ("time_step", u32), ("testing", u32), ("progression", u32), ("immunization", u32),
                ("other_disease", u32), ("statistics", u32), ("test_probs", f64 * 6), ("testing_delay", u32),
                ("quarantine_length", u32), ("use_pcr", u32), ("protection", f32 * 60), ("similarity", i32 * 7),
                ("similar_multiplier", f32 * 7), ("probability_mul", f32), ("count_immunized", u32), ("tests", u32 * 3),
                ("immunized", u32), ("stats_len", u32), ("stats", u32 * 256)]


PROBS = {"none": (0.0,) * 6, "default": (0.00005, 0.01, 0.0005, 0.0005, 0.005, 0.05), "all": (1.0, 1.0, 0.2, 0.2, 0.005, 0.05),
         "negative": (0.3, -0.2, 0.1, 0.1, 0.0, 0.0)}
PROTECTION = [0.85, 0.5, 0.77, 0.4, 0.85, 0.63, 0.9, 0.65, 0.92, 0.7, 0.003, 0.006, 0.01, 0.02, 0.005, 0.02, 0.002, 0.004,
              0.002, 0.004] * 3
FIELDS = [f for f in pansim_amd.AGENT_FIELDS if f != "stepsUntilMove"]


@pytest.mark.parametrize("n,probs", [(1, "default"), (63, "all"), (257, "negative"), (2049, "default"), (70_001, "none"),
                                     (70_001, "all"), (540_001, "default")])
def test_pass_equals_the_separate_routines(n, probs):
    args = pansim_amd.synthetic_args(n, 1, 3, 5, extra=["-k", "0.05", "--synthInfected", "0.05", "--immunizationStart", "2",
                                                        "--immunizationsPerWeek", str(max(7, n // 3))])
    one, apart = pansim_amd.Simulation(args), pansim_amd.Simulation(args)
    L = pansim_amd.lib()
    L.pansim_midnight_day.argtypes = [ctypes.c_void_p, ctypes.POINTER(Midnight)]
    try:
        for s in (one, apart):
            s.steps(6 * 144 + 70)
        ts, dt = 7 * 144, 10
        m = Midnight(timestamp=ts, time_step=dt, testing=1, progression=1, immunization=1, other_disease=1, statistics=1,
                     testing_delay=5, quarantine_length=10, use_pcr=1, count_immunized=0, immunized=17)
        m.test_probs[:] = PROBS[probs]
        m.protection[:] = PROTECTION
        m.similarity[:] = (0, 0, 0, 1, 1, 1, 1)
        assert L.pansim_midnight_day(one.ctx, ctypes.byref(m)) == 0

        c = ctypes.c_void_p(apart.ctx)
        tests, out, ln = (u32 * 3)(), (u32 * 256)(), ctypes.c_size_t()
        assert L.pansim_testing_day(c, u32(ts), u32(dt), m.test_probs, u32(5), u32(10), u32(1), tests) == 0
        assert L.pansim_progression_day(c, u32(ts), u32(dt)) == 0
        assert L.pansim_immunization_day(c, u32(ts), u32(dt), m.protection, m.similarity, m.similar_multiplier) == 0
        assert L.pansim_other_disease_day(c, u32(ts), u32(dt), f32(0.0)) == 0
        assert L.pansim_stats_day(c, u32(ts), u32(dt), tests, u32(17), out, ctypes.c_size_t(256), ctypes.byref(ln)) == 0
        assert list(m.tests) == list(tests)
        assert m.stats_len == ln.value and list(m.stats)[:ln.value] == list(out)[:ln.value]
        for f in FIELDS:
            assert np.array_equal(one.field(f), apart.field(f)), f
    finally:
        one.close()
        apart.close()
