"""The neuron step kernel's instances and edges against the CPU oracle: the unrolled 10 substeps and other
numbers, launches that end inside a wave or a block, calcium values that are infinite, NaN or far
outside the growth curve, targets equal to the minimum calcium; and waves that hold many networks."""
from __future__ import annotations

import numpy as np
import pytest

from relearn_amd import BarnesHutHIP, StepParams
from relearn_amd._lib import network_seed
from tests.test_gpu_parity import _izh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("h", [1, 7, 10])
@pytest.mark.parametrize("n", [1, 63, 257, 1000])
def test_step_sizes_and_substeps(oracle, n, h):
    print("[gpu-case] step,", n, "neurons,", h, "substeps", flush=True)
    rng = np.random.default_rng(n + h)
    po, pg = _izh(oracle), StepParams()
    po.h = h
    for f in ("a", "b", "c", "d", "v_spike", "k1", "k2", "k3", "h", "tau_ca", "beta_ca"):
        setattr(pg, f, getattr(po, f))
    for k in range(3):
        pg.eta[k], pg.nu[k] = po.eta[k], po.nu[k]
    pg.input_mode = 0
    x, u, ca = rng.uniform(-70, 20, n), rng.uniform(-15, 5, n), rng.uniform(0, 1, n)
    special = np.array([np.nan, np.inf, -np.inf, 1e200, -1e200, 0.4, 0.1, 0.0, -0.0, 1e-310])
    ca[:min(n, len(special))] = special[:n]
    tca = rng.uniform(0.05, 0.9, n)
    tca[::5] = 0.4   # the axons' minimum calcium: the curve's degenerate case
    g = BarnesHutHIP((0, 0, 0), (1, 1, 1))
    g.init(rng.random((n, 3)), np.zeros(n, np.uint8))
    g.neurons_init(pg, tca, x=x, u=u, ca=ca)
    fo, do = np.zeros(n, np.uint8), np.zeros(3 * n)
    for s in range(4):
        inp = rng.normal(5.0, 2.0, n)
        oracle.neuron_step(po, x, u, ca, inp, fo, tca, do)
        g.neurons_step(s, inp)
    st = g.neurons_get()
    g.close()
    for k, o in (("x", x), ("u", u), ("ca", ca)):
        assert np.array_equal(st[k], o, equal_nan=True), k
    assert np.array_equal(st["fired"], fo)
    # four deltas of nu * (2 exp - 1), each exp within 1 unit in the last place: 4 * 1e-4 * 2 * 2^-52
    assert np.allclose(st["delta"].ravel(), do, rtol=1e-9, atol=2e-19, equal_nan=True)


def test_step_many_networks_in_a_wave():
    sizes = [1 + (7 * k) % 5 for k in range(60)]
    off = np.concatenate([[0], np.cumsum(sizes)])
    n = int(off[-1])
    print("[gpu-case] step,", len(sizes), "networks of 1 to 5 neurons", flush=True)
    rng = np.random.default_rng(3)
    xyz, sig = rng.random((n, 3)), np.zeros(n, np.uint8)
    boxes = np.tile(np.array([0.0, 0, 0, 1, 1, 1]), (len(sizes), 1))
    p = StepParams.izhikevich(input_mode=1)
    big = BarnesHutHIP((0, 0, 0), (1, 1, 1), seed=5)
    big.init_networks(off, boxes, xyz, sig)
    big.neurons_init(p, np.full(n, 0.7))
    for s in range(6):
        big.neurons_step(s)
    e = big.neurons_get()
    big.close()
    for k in (0, 1, 13, 37, 59):
        a, b = int(off[k]), int(off[k + 1])
        one = BarnesHutHIP((0, 0, 0), (1, 1, 1), seed=network_seed(5, k))
        one.init(xyz[a:b], sig[a:b])
        one.neurons_init(p, np.full(b - a, 0.7))
        for s in range(6):
            one.neurons_step(s)
        o = one.neurons_get()
        one.close()
        for f in ("x", "u", "ca", "fired"):
            assert np.array_equal(e[f][a:b], o[f]), (k, f)
        assert np.array_equal(e["delta"][:, a:b], o["delta"]), k
