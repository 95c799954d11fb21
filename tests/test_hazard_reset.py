"""Clearing the hazard sums is ordered with the launches around it.

The engine works on a stream of its own that the null stream is not ordered
against, so memory that its launches write is cleared on that stream.  CPU: no
clearing call of the engine leaves the stream out.  GPU: the sums read with a
reset after every few steps add up to the sums of an undisturbed run."""
import os
import re

import numpy as np
import pytest

import pansim_amd
from tests.conftest import ROOT


def test_every_clearing_is_on_a_stream():
    text = open(os.path.join(ROOT, "pansim_amd", "csrc", "device", "engine.hip")).read()
    assert not re.findall(r"\bhipMemset(?:D8|D16|D32)?\s*\(", text)


@pytest.mark.gpu
def test_read_with_reset_after_every_few_steps_adds_up():
    agents, steps = 6001, 300
    args = pansim_amd.synthetic_args(agents, 1, 4, 9, extra=["-k", "0.002", "--synthInfected", "0.05"])
    whole, parts = pansim_amd.Simulation(args), pansim_amd.Simulation(args)
    try:
        for s in (whole, parts):
            s.steps(40)
            s.hazard_enable(True)
        total, done, n = np.zeros(262), 0, 1
        while done < steps:
            n = min(n, steps - done)
            parts.steps(n)
            total += parts.hazard_with_probes(reset=True)
            done += n
            n = n % 7 + 1
        whole.steps(steps)
        ref = whole.hazard_with_probes()
        assert ref[0] > 0
        # the same non-negative terms in another order: at most one per agent
        # and step, each sum within that many roundings of 2^-53
        assert np.all(np.abs(total - ref) <= agents * steps * 2.0 ** -53 * np.abs(ref))
        # enabling starts from zero again
        whole.hazard_enable(True)
        assert not np.any(whole.hazard_with_probes())
    finally:
        whole.close()
        parts.close()
