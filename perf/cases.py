"""The work that a user of pansim_amd has it do, as cases that can be timed.

A simulation is built from command-line flags (the reference's), advanced in
days or weeks, and read through its per-day statistics; a calibration script
drives it day by day through runForDay; an ensemble advances many uneven
populations in lockstep; a gradient evaluation accumulates the expected
infections and their derivatives; a monitoring program reads whole fields.
Every case is one of these calls on a population that has been running for a
while (`spin` days), so that the epidemic is under way, people are diagnosed,
quarantined and in hospital, and every midnight routine has work.

Populations: "dummy" is the reference's -n / -N generator (uniform random
locations, config1_args); "synth" the household population of
synthetic_args (schools, classrooms, workplaces, shifted schedules).
"""
import math

import numpy as np

import pansim_amd

# the shipped closure rules, the shipped two-year scenario (variants exposed
# at given days, school age limits, curfew, masks), and no rules at all
RULES = {
    "default": "inputConfigFiles/closureRules.json",
    "scenario": "inputConfigFiles/closureJun6_real_later3_delta_omicronBA2_earlier8.json",
    "none": "inputConfigFiles/noRules.json",
}
# the scenario exposes six variants to the original one's population
SCENARIO_VARIANTS = [
    "--infectiousnessMultiplier", "1.03,1.79,2.45,2.7,3.6,3.6,3.6",
    "--diseaseProgressionScaling", "0.9,1.05,0.9,0.8,0.8,0.8,0.8",
    "--diseaseProgressionDeathScaling", "1.0,1.03,1.3,0.6,0.6,0.6,0.6",
]

# the calibration script's daily flags: everything open, and the strictest set
FLAGS_OPEN = "TPdef PLNONE CFNONE SONONE QU3 MA1.0"
FLAGS_STRICT = "TP035 PL0 CF2000-0500 SO12 QU2 MA0.8"


def _case(name, **kw):
    c = {
        "name": name, "kind": "run", "pop": "synth", "agents": 100_000, "replicas": 1, "dt": 10, "days": 7,
        "spin": 14, "quarantine": 3, "rules": "default", "flags": "", "infected": 0.001,
    }
    c.update(kw)
    return c


def listed():
    return [
        # one calibration day of a village: the smallest call, where only
        # launches and dependent reads cost anything
        _case("village_2k_interface_day", kind="interface", pop="dummy", agents=2_000, days=1, spin=7, flags=FLAGS_OPEN),
        # a small town of the size of the reference's example population
        _case("town_16k_week", agents=16_365, quarantine=2),
        # the CPU-runnable workload: -n 100000 -N 20000, closures off
        _case("dummy_100k_week", pop="dummy", agents=100_000, rules="none"),
        # one calibration day of the reference's city under the strictest flags
        # (curfew, closed sites, school age limit, masks)
        _case("city_180k_strict_day", kind="interface", agents=179_500, days=1, spin=7, flags=FLAGS_STRICT),
        # a week of the shipped two-year scenario while two variants circulate,
        # vaccination runs and the curfew holds
        _case("city_300k_two_variants_week", agents=300_001, rules="scenario", spin=140),
        # five-minute steps: twice the steps per day, few movers in each
        _case("city_250k_5min_week", agents=250_007, dt=5, quarantine=1),
        # hourly steps with no quarantine and no rules: few steps, each with a
        # large share of the population moving
        _case("region_600k_hourly_4weeks", agents=600_011, dt=60, days=28, quarantine=0, rules="none"),
        # one member of a calibration ensemble at the common size
        _case("region_1M_week", agents=1_000_000),
        # the headline population: 10M agents, 4.6M locations, all policies on
        _case("country_10M_week", agents=10_000_000),
        # an ensemble of sixteen uneven cities, in lockstep
        _case("ensemble_16_week", kind="ensemble", agents=2_000_000, replicas=16),
        # one week of a gradient evaluation over eight replicas
        _case("gradient_8_week", kind="gradient", agents=2_000_000, replicas=8),
        # a day's run followed by a read of the agents' and locations' state
        _case("snapshot_400k_day", kind="snapshot", agents=400_003, days=1),
    ]


def draw(rng):
    kind = rng.choice(["run", "run", "run", "run", "interface", "snapshot", "ensemble", "gradient"])
    batch = kind in ("ensemble", "gradient")
    # 1,500 to 1,500,000 agents, uniform in the logarithm
    agents = int(math.exp(rng.uniform(math.log(1_500), math.log(1_500_000))))
    c = _case("", kind=kind, agents=agents)
    del c["name"]
    if batch:
        c["agents"] = max(agents, 4_000)
        c["replicas"] = rng.randint(2, 12)
    elif kind != "snapshot" and rng.random() < 0.3:
        c["pop"] = "dummy"
        c["agents"] = min(agents, 200_000)
    c["dt"] = rng.choice([10, 10, 10, 10, 5, 15, 20, 30, 60])
    c["days"] = rng.choice([1, 2, 7]) if c["dt"] >= 10 or not batch else rng.choice([1, 2])
    c["spin"] = rng.randint(2, 20)
    c["quarantine"] = rng.randint(0, 4)
    c["rules"] = rng.choice(["default", "default", "none", "scenario"])
    if c["rules"] == "scenario" and c["replicas"] == 1:
        c["spin"] = rng.randint(30, 200)  # curfew and school limits from day 49, vaccination from 96, a variant from 125
    c["infected"] = round(math.exp(rng.uniform(math.log(0.0005), math.log(0.02))), 6)
    if kind == "interface":
        c["days"] = 1
        c["flags"] = rng.choice([FLAGS_OPEN, FLAGS_STRICT, "TP015 CF2000-0500 SONONE QU3", "TPdef PL0 SO3 QU1 MA0.8"])
    return c


def _args(case, seed, agents, member=0):
    """The command line of one population; every random choice comes from the
    seed (and the ensemble member)."""
    s = int(seed) * 64 + member
    rules = RULES[case["rules"]]
    extra = ["-t", str(case["dt"]), "--quarantinePolicy", str((case["quarantine"] + member) % 5)]
    if case["rules"] == "none" or (case["replicas"] > 1 and member % 2):
        extra += ["--enableClosures", "0"]
        rules = RULES["none"]
    extra += ["--closures", rules]
    if case["rules"] == "scenario":
        extra += SCENARIO_VARIANTS
    if case["pop"] == "dummy":
        return pansim_amd.config1_args(agents, max(1, agents // 5), 4, s, extra=extra)
    # replicas differ in their infection coefficient, as in a calibration
    extra += ["--synthInfected", str(case["infected"]), "-k",
              "%.6g" % (3.74e-4 * (0.7 + 0.6 * (member % 8) / 7.0)) if case["replicas"] > 1 else "0.000374"]
    # a snapshot's population is one that a program knows: its draws differ,
    # its number of locations does not
    return pansim_amd.synthetic_args(agents, 4, s, 1 if case["kind"] == "snapshot" else s + 1, extra=extra)


def _sizes(case):
    """Uneven replica sizes, a factor of 16 between the smallest and the
    largest, adding up to about case["agents"]."""
    n = case["replicas"]
    w = [16.0 ** (j / max(1, n - 1)) for j in range(n)]
    return [max(257, int(case["agents"] * x / sum(w)) | 1) for x in w]


def prepare(case, seed):
    kind, spin = case["kind"], case["spin"]
    if kind == "interface":
        si = pansim_amd.SimulatorInterface()
        si.initSimulation(["panSim"] + _args(case, seed, case["agents"]))
        for _ in range(spin):
            si.runForDay(FLAGS_OPEN.split())
        return {"kind": kind, "si": si, "flags": case["flags"].split()}
    if kind in ("ensemble", "gradient"):
        ens = pansim_amd.Ensemble([_args(case, seed, n, j) for j, n in enumerate(_sizes(case))])
        ens.steps(1440 // case["dt"])  # the first day step by step
        ens.days(max(1, spin - 1))
        views = [ens.replica(r) for r in range(case["replicas"])]
        if kind == "gradient":
            for v in views:
                v.set_location_type_multipliers(np.ones(256, dtype=np.float32))
                v.hazard_enable(True)
        ens.sync()
        return {"kind": kind, "ens": ens, "views": views, "days": case["days"]}
    sim = pansim_amd.Simulation(_args(case, seed, case["agents"]))
    sim.steps(spin * sim.steps_per_day)
    sim.sync()
    return {"kind": kind, "sim": sim, "days": case["days"]}


def _stats(view, first):
    return np.array([view.day_stats(d) for d in range(first, view.num_days)], dtype=np.int64)


def run(state):
    kind = state["kind"]
    if kind == "interface":
        return np.array(state["si"].runForDay(state["flags"]), dtype=np.int64)
    if kind in ("ensemble", "gradient"):
        views = state["views"]
        first = views[0].num_days
        state["ens"].days(state["days"])
        out = {"stats": np.stack([_stats(v, first) for v in views])}
        if kind == "gradient":
            # per replica: expected infections, d/dk, d/dm of every location type
            g = [v.hazard(reset=True) for v in views]
            out["J"] = np.array([x[0] for x in g])
            out["dk"] = np.array([x[1] for x in g])
            out["dm"] = np.stack([x[2] for x in g])
        return out
    sim = state["sim"]
    first = sim.num_days
    sim.steps(state["days"] * sim.steps_per_day)
    out = {"stats": _stats(sim, first)}
    if kind == "snapshot":
        for f in ("state", "variant", "location", "diagnosed", "quarantined", "infectedTimestamp", "infectedLocation",
                  "daysInQuarantine", "worstState", "susceptible0", "locCount", "locQuarantineUntil"):
            out[f] = sim.field(f)
        out["sums"] = sim.location_sums(0)
    return out


# Per agent and simulated day, counted on the synthetic population (the dummy
# population's figures are within 3 %): 7.7 movement evaluations and 3.4
# relocations, nearly independent of the population's size.
EVALUATIONS, RELOCATIONS = 7.7, 3.4
# susceptible agents met at a location with infectious visitors, per agent and
# step: about 1.5 % on average over a day of the third week
EXPOSURES = 0.015


def work(case):
    """Bytes of one pass that no implementation of the pipeline can do
    without: each movement evaluation reads the agent's 32-byte record, its
    location and the chosen entry of its list and writes its next evaluation
    time (42 B); each relocation writes the location and updates the occupancy
    of two places (20 B); each exposure reads location, sum, occupancy,
    infectiousness and susceptibility (24 B); each midnight reads and writes
    the agent's state once (64 B); a snapshot writes its fields.  The path has
    no contraction: its arithmetic is counted as the 10-round counter-based
    draws (about 60 operations each), one per evaluation and exposure."""
    spd = 1440 / case["dt"]
    n = case["agents"]
    exposures = EXPOSURES * spd
    day = EVALUATIONS * 42 + RELOCATIONS * 20 + exposures * 24 + 64
    b = n * day * case["days"]
    if case["kind"] == "snapshot":
        b += n * 4 * 10 + (n // 2) * 16
    return {"bytes": b, "flops": n * case["days"] * (EVALUATIONS + exposures) * 60.0}


def exact(case, seed):
    """Every output but the gradient's is a whole number.  The expected
    infections and their derivatives are sums over a simulated trajectory that
    only the engine's own random streams define, so plain 64-bit arithmetic
    has no value for them."""
    return None
