"""The midnight routines called one by one run kernels of their own: the same
fields, counts and statistics as the one pass at the sizes where their launches
change (a block and its neighbours, the last size whose pass shares one copy of
the counters and the first with several), and one stage of the one-pass call
alone is the routine itself.  Every compared value is whole."""
import ctypes

import numpy as np
import pytest

import pansim_amd
from tests import test_gpu_midnight_pass as one_pass

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [255, 256, 257, 131_072, 131_073])
@pytest.mark.parametrize("probs", ["default", "all"])
def test_routines_equal_the_pass_where_launches_change(n, probs):
    one_pass.test_pass_equals_the_separate_routines(n, probs)


def test_one_stage_of_the_pass_is_the_routine():
    args = pansim_amd.synthetic_args(3001, 1, 3, 5, extra=["-k", "0.05", "--synthInfected", "0.05", "--immunizationStart", "2",
                                                           "--immunizationsPerWeek", "1000"])
    one, apart = pansim_amd.Simulation(args), pansim_amd.Simulation(args)
    L = pansim_amd.lib()
    L.pansim_midnight_day.argtypes = [ctypes.c_void_p, ctypes.POINTER(one_pass.Midnight)]
    u32, f32 = ctypes.c_uint32, ctypes.c_float
    try:
        for s in (one, apart):
            s.steps(6 * 144 + 70)
        ts, dt, c = 7 * 144, 10, ctypes.c_void_p(apart.ctx)
        m = one_pass.Midnight(timestamp=ts, time_step=dt, testing_delay=5, quarantine_length=10, use_pcr=1, immunized=17)
        m.test_probs[:] = one_pass.PROBS["all"]
        m.protection[:] = one_pass.PROTECTION
        m.similarity[:] = (0, 0, 0, 1, 1, 1, 1)
        tests, out, ln = (u32 * 3)(), (u32 * 256)(), ctypes.c_size_t()
        stages = ("testing", "progression", "immunization", "other_disease", "statistics")
        for stage in stages:
            for s in stages:
                setattr(m, s, 1 if s == stage else 0)
            assert L.pansim_midnight_day(one.ctx, ctypes.byref(m)) == 0
            if stage == "testing":
                assert L.pansim_testing_day(c, u32(ts), u32(dt), m.test_probs, u32(5), u32(10), u32(1), tests) == 0
                assert list(m.tests) == list(tests) and tests[0] > 0
            elif stage == "progression":
                assert L.pansim_progression_day(c, u32(ts), u32(dt)) == 0
            elif stage == "immunization":
                assert L.pansim_immunization_day(c, u32(ts), u32(dt), m.protection, m.similarity, m.similar_multiplier) == 0
            elif stage == "other_disease":
                assert L.pansim_other_disease_day(c, u32(ts), u32(dt), f32(0.0)) == 0
            else:
                assert L.pansim_stats_day(c, u32(ts), u32(dt), tests, u32(17), out, ctypes.c_size_t(256), ctypes.byref(ln)) == 0
                assert m.stats_len == ln.value and list(m.stats)[:ln.value] == list(out)[:ln.value]
            for f in one_pass.FIELDS:
                assert np.array_equal(one.field(f), apart.field(f)), (stage, f)
    finally:
        one.close()
        apart.close()
