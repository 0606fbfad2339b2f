"""Work distribution of the persistent search waves: every active source is searched exactly once,
whatever the number of sources per segment (none, fewer than one per XCD, one grab, several grabs)
and the grab size.  Picks and test counts against the CPU oracle; the flat kernel (sigma = 10^12 um)
makes the FP32-mixed picks the oracle's."""
from __future__ import annotations

import numpy as np
import pytest

from relearn_amd import RL_FLAG_WALK_ALWAYS, RL_FLAG_WAVE_PER_SOURCE, RL_PREC_FP32_MIXED, RL_PREC_FP64, BarnesHutHIP
from relearn_amd.workloads import uniform_cube
from tests.test_gpu_parity import _check_search

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,flags", [(RL_PREC_FP64, 0), (RL_PREC_FP32_MIXED, RL_FLAG_WAVE_PER_SOURCE),
                                             (RL_PREC_FP32_MIXED, RL_FLAG_WALK_ALWAYS)])
@pytest.mark.parametrize("active", [0, 1, 7, 8, 9, 513, 4097])
def test_every_source_searched_once(oracle, active, precision, flags):
    print("[gpu-case] queue,", active, "sources, precision", precision, "flags", flags, flush=True)
    net = uniform_cube(6000, 1817.0, 21)
    rng = np.random.default_rng(active)
    va = np.zeros(net.n, np.uint32)
    va[rng.choice(net.n, active, replace=False)] = 1 + rng.poisson(1.0, active).astype(np.uint32)
    net.vac_axon = va
    t = oracle.Tree(net.xyz, net.box_min, net.box_max)
    t.update(net.vac_exc, net.vac_inh, None)
    ref = t.find_targets(net.signal, va, None, sigma=1.0e12, seed=11, step=2, threads=0)
    t.close()
    g = BarnesHutHIP(net.box_min, net.box_max, sigma=1.0e12, seed=11, precision=precision, flags=flags)
    g.init(net.xyz, net.signal)
    for chunk in (1, 8):
        g.set_tuning(16, chunk)
        g.prepare_update_connectivity(va, net.vac_exc, net.vac_inh)
        nreq = g.find_target_neurons(2)
        tgt, tests, cnt = g.get_search_slots(int(va.sum()))
        bad, _ = _check_search(ref, tgt, tests, cnt, net)
        assert not bad
        assert nreq == int(cnt.sum())
    g.close()
