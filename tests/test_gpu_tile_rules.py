"""The tile sizes chosen by the number of agents (one agent per lane, tiles of
8, 16 or 32 agents per thread in movement; 1, 2, 4 or 8 in infection): the
first size past each line of the rules against the oracle, and batches large
enough for every batch tile against the same populations run alone (small
batches are cut into the finest tiles).  Every compared value is whole."""
import numpy as np
import pytest

import pansim_amd
from tests.parity_util import run_parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [786_433, 1_572_865, 2_621_441, 3_145_729])
def test_parity_past_each_line(n):
    # movement / infection agents per thread: 1 / 2, 8 / 4, 16 / 4, 16 / 8
    run_parity(pansim_amd.synthetic_args(n, 1, 3, 5, extra=["-k", "0.02", "--synthInfected", "0.01"]), [50])


FIELDS = ["state", "location", "infectedTimestamp", "infectedLocation", "diagnosed", "quarantined", "locCount"]


@pytest.mark.parametrize("tiles", [(8, 4), (16, 8), (32, 8)])
def test_large_batches_match_each_replica_alone(tiles):
    args = [pansim_amd.synthetic_args(n, 1, j, j + 3, extra=["-k", "0.01", "--synthInfected", "0.01"])
            for j, n in enumerate((2_000_003, 1_300_001))]
    ens = pansim_amd.Ensemble(args)
    try:
        ens.set_tiles(*tiles)
        ens.steps(144)
        ens.days(1)
        for r, a in enumerate(args):
            solo = pansim_amd.Simulation(a)
            solo.steps(2 * 144)
            for f in FIELDS:
                assert np.array_equal(ens.replica(r).field(f), solo.field(f)), (r, f)
            assert np.array_equal(ens.replica(r).location_sums(0), solo.location_sums(0))
            assert [ens.replica(r).day_stats(d) for d in range(2)] == [solo.day_stats(d) for d in range(2)]
            solo.close()
    finally:
        ens.close()
