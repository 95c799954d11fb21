"""Runs of steps whose launches read their arguments from device memory (eight
steps or more of a small population) equal the same steps asked for one by one,
field by field, for every quarantine policy, one and several variants, runs
shorter and longer than that line, and populations of less than a wave, of a
block and a lane, and of several blocks."""
import json

import numpy as np
import pytest

import pansim_amd

pytestmark = pytest.mark.gpu

FIELDS = ["state", "variant", "location", "infectedTimestamp", "infectedLocation", "infectedCount", "statsVariant",
          "worstStateTimestamp", "susceptible0", "diagnosed", "quarantined", "quarantinedUntilTimestamp", "daysInQuarantine",
          "locCount", "locQuarantineUntil"]


@pytest.mark.parametrize("agents", [50, 257, 6001])
@pytest.mark.parametrize("policy", [0, 1, 2, 3])
@pytest.mark.parametrize("variants", [False, True])
def test_runs_equal_single_steps(tmp_path, agents, policy, variants):
    rules = [{"name": "Curfew", "conditionType": "afterDays", "threshold": 0, "threshold2": 0, "parameter": "2000-0500",
              "openAfter": 2, "closeAfter": -1, "locationTypesToClose": []}]
    if variants:
        rules += [{"name": "ExposeToMutation", "conditionType": "afterDays", "threshold": 0, "threshold2": v,
                   "parameter": "0.1", "openAfter": 1, "closeAfter": -1, "locationTypesToClose": []} for v in (1, 2)]
    p = tmp_path / "rules.json"
    p.write_text(json.dumps({"rules": rules}))
    args = pansim_amd.synthetic_args(agents, 1, 4, 9, extra=["-k", "0.003", "--synthInfected", "0.2", "--quarantinePolicy",
                                                             str(policy), "--testingProbabilities",
                                                             "0.05,0.05,0.05,0.05,0.05,0.05", "--closures", str(p)])
    one, many = pansim_amd.Simulation(args), pansim_amd.Simulation(args)
    try:
        # whole days, then runs that end anywhere in the waking hours
        for n in (5 * 144, 50, 4, 5, 6, 7, 8, 9, 3, 10, 11, 31, 144):
            for _ in range(n):
                one.steps(1)
            many.steps(n)
            for f in FIELDS:
                assert np.array_equal(one.field(f), many.field(f)), (n, f)
            for v in range(one.n_variants):
                assert np.array_equal(one.location_sums(v), many.location_sums(v))
        assert one.movement_counters() == many.movement_counters()
        assert [one.day_stats(d) for d in range(one.num_days)] == [many.day_stats(d) for d in range(many.num_days)]
        if policy > 1 and agents > 1000:
            assert np.any(one.field("locQuarantineUntil") > 0)
    finally:
        one.close()
        many.close()


@pytest.mark.parametrize("agents", [63, 256, 3001, 131072, 131073])
def test_direct_infection_equals_general(agents):
    """The infection pass of small populations (up to 131072 agents it reads
    the locations' records outright) infects whom the general pass does, which
    the hazard instance runs."""
    args = pansim_amd.synthetic_args(agents, 1, 4, 9, extra=["-k", "0.003", "--synthInfected", "0.1"])
    plain, general = pansim_amd.Simulation(args), pansim_amd.Simulation(args)
    try:
        general.hazard_enable(True)
        plain.steps(2 * 144 + 60)
        general.steps(2 * 144 + 60)
        for f in FIELDS:
            assert np.array_equal(plain.field(f), general.field(f)), f
    finally:
        plain.close()
        general.close()
