"""Quiet ranges: a run of steps given to one call (steps at which nobody moves
share one infection launch) equals the same steps asked for one by one, field
by field, with one and several active variants, with and without a curfew,
with few exposed agents (draws spread over a wave) and many (draws in a row),
and with hazard accumulation."""
import json

import numpy as np
import pytest

import pansim_amd

pytestmark = pytest.mark.gpu

FIELDS = ["state", "variant", "location", "infectedTimestamp", "infectedLocation", "infectedCount", "statsVariant",
          "worstStateTimestamp", "susceptible0", "diagnosed", "quarantined", "locCount"]


def _args(tmp_path, infected, variants, curfew):
    rules = []
    if variants:
        rules += [{"name": "ExposeToMutation", "conditionType": "afterDays", "threshold": 0, "threshold2": v,
                   "parameter": "0.05", "openAfter": 3, "closeAfter": -1, "locationTypesToClose": []} for v in (1, 2)]
    if curfew:
        rules.append({"name": "Curfew", "conditionType": "afterDays", "threshold": 0, "threshold2": 0,
                      "parameter": "2000-0500", "openAfter": 3, "closeAfter": -1, "locationTypesToClose": []})
    p = tmp_path / "rules.json"
    p.write_text(json.dumps({"rules": rules}))
    return pansim_amd.synthetic_args(5003, 1, 4, 9, extra=["-k", "0.002", "--synthInfected", str(infected),
                                                           "--closures", str(p)])


@pytest.mark.parametrize("infected", [0.005, 0.4])
@pytest.mark.parametrize("variants", [False, True])
@pytest.mark.parametrize("curfew", [False, True])
@pytest.mark.parametrize("hazard", [False, True])
def test_ranges_equal_single_steps(tmp_path, infected, variants, curfew, hazard):
    args = _args(tmp_path, infected, variants, curfew)
    one, many = pansim_amd.Simulation(args), pansim_amd.Simulation(args)
    try:
        if hazard:
            for s in (one, many):
                s.hazard_enable(True)
                s.hazard_set_probe(1e-3, 4)
        # whole days, then a range that starts and ends inside a night
        for n in (3 * 144, 7, 11, 126, 150):
            for _ in range(n):
                one.steps(1)
            many.steps(n)
            for f in FIELDS:
                assert np.array_equal(one.field(f), many.field(f)), (n, f)
            for v in range(one.n_variants):
                assert np.array_equal(one.location_sums(v), many.location_sums(v))
        assert [one.day_stats(d) for d in range(one.num_days)] == [many.day_stats(d) for d in range(many.num_days)]
        if hazard:
            # the same non-negative (J, gradient) or same-signed (probe) FP32
            # terms in another order: at most 5003 agents x 726 steps x 3
            # variants of them, each sum within that many roundings of 2^-53
            a, b = one.hazard_with_probes(), many.hazard_with_probes()
            assert a[0] > 0
            assert np.all(np.abs(a - b) <= 5003 * 726 * 3 * 2.0 ** -53 * np.maximum(np.abs(a), np.abs(b)))
    finally:
        one.close()
        many.close()
