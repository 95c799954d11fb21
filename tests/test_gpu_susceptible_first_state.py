"""A progression whose first infected state is susceptible: an agent infected
at one step of a night may be infected again at the next, so a run of steps
given to one call, a whole day of a batch and the oracle agree with the steps
asked for one by one.  Every compared value is whole."""
import json
import os
import shutil

import numpy as np
import pytest

import pansim_amd
from oracle.oracle import OracleSim

pytestmark = pytest.mark.gpu

FIELDS = ["state", "variant", "location", "infectedTimestamp", "infectedLocation", "infectedCount", "statsVariant", "locCount"]


def _args(tmp_path, variants):
    d = tmp_path / "progressions"
    shutil.copytree(os.path.join(pansim_amd.DATA_DIR, "inputConfigFiles", "progressions"), d)
    path = d / "transition_config.json"
    cfg = json.load(open(path))
    info = cfg["stateInformation"]
    info["susceptibleStates"].append(info["firstInfectedState"])
    path.write_text(json.dumps(cfg))
    rules = [{"name": "ExposeToMutation", "conditionType": "afterDays", "threshold": 0, "threshold2": v, "parameter": "0.05",
              "openAfter": 3, "closeAfter": -1, "locationTypesToClose": []} for v in ((1, 2) if variants else ())]
    rpath = tmp_path / "rules.json"
    rpath.write_text(json.dumps({"rules": rules}))
    return pansim_amd.synthetic_args(3001, 1, 4, 9, extra=["-k", "0.01", "--synthInfected", "0.2", "-P", str(path),
                                                           "--closures", str(rpath)])


@pytest.mark.parametrize("variants", [False, True])
def test_runs_days_and_single_steps_agree(tmp_path, variants):
    args = _args(tmp_path, variants)
    one, many, ens, ora = pansim_amd.Simulation(args), pansim_amd.Simulation(args), pansim_amd.Ensemble([args]), OracleSim(args)
    try:
        for _ in range(2 * 144):
            one.steps(1)
        many.steps(2 * 144)
        ens.days(2)
        ora.steps(2 * 144)
        # (several infections within a day: the case is met)
        assert one.field("infectedCount").max() > 1
        for f in FIELDS:
            assert np.array_equal(ora.field(f), one.field(f)), ("single steps", f)
            assert np.array_equal(ora.field(f), many.field(f)), ("run of steps", f)
            assert np.array_equal(ora.field(f), ens.replica(0).field(f)), ("batch day", f)
        for v in range(one.n_variants):
            assert np.array_equal(one.location_sums(v), many.location_sums(v))
    finally:
        for s in (one, many, ens, ora):
            s.close()
