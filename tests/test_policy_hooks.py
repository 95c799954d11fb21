"""The hooks of the policy template Simulation<...>: a policy that replaces a
hook has it called at every step or midnight, in the reference's order
(simulation.h:899-926), and the shipped policies reach the engine by its calls
for runs of steps and whole midnights.  A C++ program over an engine of stubs, compiled here (CPU only)."""
import os
import subprocess

import pytest

import pansim_amd
from pansim_amd import build
from tests.conftest import ROOT


@pytest.fixture(scope="module")
def order(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("hooks") / "policy_hooks")
    host = os.path.join(ROOT, "pansim_amd", "csrc", "host")
    sources = [os.path.join(host, s) for s in ("json.cpp", "scenario.cpp", "synthpop.cpp", "model.cpp")]
    r = subprocess.run([build.CXX, *build.CXXFLAGS, "-O0", "-o", exe, os.path.join(ROOT, "tests", "policy_hooks.cpp"), *sources],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    # hourly steps: 24 per day
    args = pansim_amd.with_data_dir(pansim_amd.config1_args(200, 50, 1, 0, extra=["-t", "60"]))
    r = subprocess.run([exe, *args], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    out = dict(line.split(": ", 1) for line in r.stdout.splitlines())
    assert not [k for k, v in out.items() if v == "wrong time"]
    return {k: v.split() for k, v in out.items()}


def _steps(log):
    """What follows the first day's planning."""
    return log[log.index("plan") + 1:]


def test_shipped_policies_give_runs_of_steps(order):
    for name in ("shipped", "selectable"):
        assert order[name] == ["midnight(ios)", "plan", "run24", "midnight(tpios)", "plan", "run2"], name
    # a derived policy may say that it changes no hook
    assert _steps(order["named"]) == ["run2"]


def test_derived_movement_policy_is_called_every_step(order):
    assert _steps(order["movement"]) == ["hook:movement", "move", "infect"] * 2


def test_derived_infection_policy_is_called_every_step(order):
    assert _steps(order["infection"]) == ["move", "hook:infection", "infect"] * 2


def test_infection_policy_needs_only_the_hooks(order):
    assert _steps(order["minimal"]) == ["move", "hook:infection"] * 2


def test_closure_policy_acts_between_movement_and_infection(order):
    assert _steps(order["closure"]) == ["move", "hook:closure", "infect"] * 2


def test_derived_testing_policy_is_called_every_midnight(order):
    routines = ["immunization", "other", "statistics", "plan"]
    assert order["testing"] == [*routines, "run24", "hook:testing", "testing", "progression", *routines, "run1"]
