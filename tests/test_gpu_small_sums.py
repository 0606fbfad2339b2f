"""FP64 searches whose probabilities sum to nearly nothing: only lists whose sum is 0 go to the per-lane search,
and all pick as the oracle does."""
from __future__ import annotations

import numpy as np
import pytest

from relearn_amd import RL_PREC_FP64
from relearn_amd.workloads import uniform_cube
from tests.test_gpu_parity import _check_search, _search_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sigma", [3.0, 4.0])
def test_search_parity_with_small_sums(oracle, sigma):
    print("[gpu-case] small sums, 4,000 neurons, sigma", sigma, flush=True)
    net = uniform_cube(4000, 1000.0 * 4.0 ** (1 / 3), 3)
    t = oracle.Tree(net.xyz, net.box_min, net.box_max)
    t.update(net.vac_exc, net.vac_inh)
    sums = []
    for s in np.flatnonzero(net.vac_axon):
        nodes, _, total, fallback, _ = t.candidate_list(0, net.xyz[s], int(s), int(net.signal[s]), 0.3, sigma, cap=8192)
        assert len(nodes) > 0
        sums.append(0.0 if fallback else total)
    t.close()
    sums = np.array(sums)
    assert (sums == 0.0).sum() > 20 and ((sums > 0.0) & (sums < 1e-306)).sum() > 20   # FP64 loses bits below 2e-308
    assert ((sums > 1e-306) & (sums < 1e-250)).sum() > 100
    ref, g, nreq, tgt, tests, cnt = _search_pair(oracle, net, seed=2, step=1, sigma=sigma, precision=RL_PREC_FP64)
    lane_sources = g.last_search_stats()["lane_sources"]
    g.close()
    bad, near = _check_search(ref, tgt, tests, cnt, net)
    print("[gpu-case]   near-boundary", near, "mismatches", len(bad), bad[:5], flush=True)
    assert not bad
    assert lane_sources == (sums == 0.0).sum()
