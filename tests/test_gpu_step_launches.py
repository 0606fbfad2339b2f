"""Captured periods whose steps share launches (no synaptic input) against the same steps called one by one."""
from __future__ import annotations

import numpy as np
import pytest

from relearn_amd import RL_PREC_FP64, BarnesHutHIP, StepParams

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("steps,h", [(1, 10), (2, 10), (3, 7), (256, 10), (257, 10), (300, 1)])
@pytest.mark.parametrize("networks", [1, 5])
def test_captured_steps_match_single_steps(steps, h, networks):
    n = 333 * networks
    print("[gpu-case] captured steps,", steps, "steps,", h, "substeps,", networks, "networks", flush=True)
    rng = np.random.default_rng(steps + networks)
    xyz = rng.random((n, 3)) * 500.0
    signal = (rng.random(n) < 0.2).astype(np.uint8)
    enabled = (rng.random(n) < 0.9).astype(np.uint8)
    x, u, ca, target = rng.uniform(-70, -45, n), rng.uniform(-15, -10, n), rng.uniform(0, 0.3, n), rng.uniform(0.05, 0.3, n)
    p = StepParams.izhikevich(input_mode=1)
    p.h = h
    p.input_stddev = 4.0
    out = []
    for captured in (False, True):
        g = BarnesHutHIP((0, 0, 0), (500, 500, 500), seed=9, precision=RL_PREC_FP64)
        if networks > 1:
            g.init_networks(np.arange(networks + 1) * 333, np.tile([0.0, 0, 0, 500, 500, 500], (networks, 1)), xyz, signal)
        else:
            g.init(xyz, signal)
        g.set_enabled(enabled)
        zero = np.zeros(n, np.uint32)
        g.prepare_update_connectivity(zero, zero, zero)
        g.neurons_init(p, target, x=x, u=u, ca=ca, grown=np.zeros(3 * n))
        g.neurons_step(1000)   # a status that the disabled neurons carry
        states = []
        if captured:
            g.graph_create(steps, 4 * n)
        for k in range(2):
            if captured:
                g.graph_launch(k * steps, k)
            else:
                for s in range(steps):
                    g.neurons_step(k * steps + s)
                g.neurons_commit_elements(k)
            states.append({key: np.array(v) for key, v in g.neurons_get().items() if key in ("x", "u", "ca", "fired", "grown")})
        out.append(states)
        g.close()
    for a, b in zip(*out):
        for key in ("x", "u", "ca", "fired"):
            assert np.array_equal(a[key], b[key]), key
    # the periods' grown elements (no vacant element bound: the first update has nothing to connect)
    assert np.array_equal(out[0][0]["grown"], out[1][0]["grown"])
