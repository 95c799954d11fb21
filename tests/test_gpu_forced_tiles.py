"""Every movement and infection tile with every policy.  Populations of these
sizes would be cut into the finest tiles, so the larger ones are forced on a
batch of them: curfew, several variants, closure rules, every quarantine
policy, long location lists, other time steps, tiny populations, quiet ranges
and hazard accumulation, each replica against its own oracle run.  Larger
populations alone, with the tiles of their size, equal a batch of another tile.
Every compared value but the hazard sums is whole."""
import json

import numpy as np
import pytest

import pansim_amd
from oracle.oracle import OracleSim
from tests.parity_util import compare_days, compare_state
from tests.test_gpu_parity import _long_list_world

pytestmark = pytest.mark.gpu

TILES = [(8, 4), (16, 8), (32, 8)]


def _rules(path):
    rules = [{"name": "ExposeToMutation", "conditionType": "afterDays", "threshold": 0, "threshold2": v, "parameter": "0.05",
              "openAfter": 2, "closeAfter": -1, "locationTypesToClose": []} for v in (1, 2)]
    rules.append({"name": "Curfew", "conditionType": "afterDays", "threshold": 1, "threshold2": 0, "parameter": "2000-0500",
                  "openAfter": 2, "closeAfter": -1, "locationTypesToClose": []})
    path.write_text(json.dumps({"rules": rules}))
    return ["--closures", str(path)]


def _replicas(tmp_path, dt):
    rules = _rules(tmp_path / "rules.json")
    tests = ["--testingProbabilities", "0.05,0.05,0.05,0.05,0.05,0.05"]
    step = ["-t", str(dt)]
    args = [
        pansim_amd.synthetic_args(9001, 1, 3, 5, extra=["-k", "0.005", "--synthInfected", "0.05", "--quarantinePolicy", "3",
                                                        *tests, *rules, *step]),
        pansim_amd.synthetic_args(63, 1, 4, 6, extra=["-k", "0.05", "--synthInfected", "0.3", *rules, *step]),
        pansim_amd.config1_args(2500, 500, 1, 9, extra=["-k", "0.03", "--quarantinePolicy", "4", *tests, *step]),
        pansim_amd.config1_args(2049, 400, 1, 8, extra=["-k", "0.03", "--quarantinePolicy", "1", *tests, *rules, *step]),
    ]
    if dt == 10:
        args.append(_long_list_world(tmp_path))
    return args


@pytest.mark.parametrize("tiles", TILES)
@pytest.mark.parametrize("dt,hazard", [(10, False), (10, True), (5, False), (60, False)])
def test_small_populations_on_every_tile(tmp_path, tiles, dt, hazard):
    args = _replicas(tmp_path, dt)
    spd = 1440 // dt
    ens = pansim_amd.Ensemble(args)
    oracles = [OracleSim(a) for a in args]
    solos = [pansim_amd.Simulation(a) for a in args] if hazard else []
    try:
        ens.set_tiles(*tiles)
        assert ens.tiles() == tiles
        for s in [ens.replica(r) for r in range(len(args))] + solos if hazard else []:
            s.hazard_enable(True)
        # a day step by step, two whole days, then into a day with a curfew
        for what, n in ((ens.steps, spd), (ens.days, 2), (ens.steps, spd // 2)):
            what(n)
            ens.sync()
            for o in oracles:
                o.steps(n * spd if what == ens.days else n)
            for r, o in enumerate(oracles):
                compare_state(ens.replica(r), o, f"replica {r}, tiles {tiles}")
        for r, o in enumerate(oracles):
            compare_days(ens.replica(r), o)
        for r, s in enumerate(solos):
            s.steps(3 * spd + spd // 2)
            a, b = ens.replica(r).hazard_with_probes(), s.hazard_with_probes()
            assert b[0] > 0
            # the same non-negative terms in another order: at most one per
            # agent, step and variant, each sum within that many roundings
            assert np.all(np.abs(a - b) <= s.n_agents * s.timestamp * s.n_variants * 2.0 ** -53 * np.abs(b))
    finally:
        ens.close()
        for o in oracles + solos:
            o.close()


FIELDS = ["state", "variant", "location", "infectedTimestamp", "infectedLocation", "infectedCount", "diagnosed", "quarantined",
          "daysInQuarantine", "locCount", "locQuarantineUntil"]


@pytest.mark.parametrize("n,tiles", [(800_003, (16, 4)), (1_600_001, (32, 8)), (3_200_003, (8, 4))])
def test_large_populations_alone_equal_other_tiles(tmp_path, n, tiles):
    """Alone (movement / infection agents per thread 1 / 2, 8 / 4, 16 / 8) with
    a curfew and several variants, quiet ranges included."""
    args = pansim_amd.synthetic_args(n, 1, 3, 5, extra=["-k", "0.005", "--synthInfected", "0.02", *_rules(tmp_path / "r.json")])
    solo, ens = pansim_amd.Simulation(args), pansim_amd.Ensemble([args])
    try:
        ens.set_tiles(*tiles)
        ens.days(2)
        ens.steps(40)
        solo.steps(2 * 144)
        solo.steps(40)
        for f in FIELDS:
            assert np.array_equal(ens.replica(0).field(f), solo.field(f)), f
        for v in range(solo.n_variants):
            assert np.array_equal(ens.replica(0).location_sums(v), solo.location_sums(v))
        assert [ens.replica(0).day_stats(d) for d in range(3)] == [solo.day_stats(d) for d in range(3)]
        assert len(np.unique(solo.field("variant"))) > 1
    finally:
        solo.close()
        ens.close()
