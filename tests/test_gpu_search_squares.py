"""The search's decisions on squared distances, at the places where they hand over to the reference's own
comparison: neurons on an exact grid (sides and distances are small integers, so theta * distance
equals the side in many tests), boxes so small that squared distances underflow, and Gaussian sums
close to the smallest FP64 numbers.  FP64 picks against the CPU oracle; draws within 1e-12 of a boundary
are exempt, as in the other parity tests."""
from __future__ import annotations

import numpy as np
import pytest

from relearn_amd import RL_PREC_FP64, BarnesHutHIP
from relearn_amd.workloads import Network
from tests.test_gpu_parity import _check_search

pytestmark = pytest.mark.gpu


def _grid(per_side, spacing, seed):
    rng = np.random.default_rng(seed)
    g = np.stack(np.meshgrid(*[np.arange(per_side)] * 3, indexing="ij"), axis=-1).reshape(-1, 3).astype(np.float64)
    n = len(g)
    side = per_side * spacing
    return Network((g + 0.5) * spacing, (rng.random(n) < 0.2).astype(np.uint8), rng.poisson(1.0, n).astype(np.uint32),
                   np.ones(n, np.uint32), np.ones(n, np.uint32), (0.0, 0.0, 0.0), (side, side, side))


@pytest.mark.parametrize("mu", [0.0, 2.5])
@pytest.mark.parametrize("spacing,sigma", [(1.0, 6.0),          # exact ties between theta * distance and side
                                           (2.0 ** -466, 6.0 * 2.0 ** -466),   # squares below 1e-250
                                           (2.0 ** 400, 6.0 * 2.0 ** 400),
                                           (1.0, 0.0445),       # sums from 1e-219 down past 1e-250 to 0
                                           (1.0, 0.0417)])      # nearest neighbour: exp(-575) = 1e-250
def test_search_parity_on_squares(oracle, spacing, sigma, mu):
    print("[gpu-case] squares, spacing", spacing, "sigma", sigma, "mu", mu, flush=True)
    net = _grid(16, spacing, 5)
    m = mu * spacing
    t = oracle.Tree(net.xyz, net.box_min, net.box_max)
    t.update(net.vac_exc, net.vac_inh, None)
    # theta 0.25: side 1, 2, 4 against distances 4, 8, 16
    ref = t.find_targets(net.signal, net.vac_axon, None, theta=0.25, sigma=sigma, mu=m, seed=3, step=1, threads=0)
    t.close()
    g = BarnesHutHIP(net.box_min, net.box_max, theta=0.25, sigma=sigma, mu=m, seed=3, precision=RL_PREC_FP64)
    g.init(net.xyz, net.signal)
    g.prepare_update_connectivity(net.vac_axon, net.vac_exc, net.vac_inh)
    nreq = g.find_target_neurons(1)
    tgt, tests, cnt = g.get_search_slots(int(net.vac_axon.sum()))
    g.close()
    bad, near = _check_search(ref, tgt, tests, cnt, net)
    print("[gpu-case]   near-boundary", near, "mismatches", len(bad), bad[:5], flush=True)
    assert not bad
    assert nreq == int(cnt.sum())
