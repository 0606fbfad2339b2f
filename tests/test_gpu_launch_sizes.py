"""Sizes at which the update's launches change: prefix sums by one block or by tiles (counts of 32,768
and around), and tree levels taken together by one block or launched one by one (levels of 1,024 nodes
and around, forests with many roots).  Trees, searches and commits against the CPU oracle."""
from __future__ import annotations

import numpy as np
import pytest

from relearn_amd import RL_PREC_FP64, BarnesHutHIP
from relearn_amd.workloads import uniform_cube
from tests.test_gpu_ensemble import _ensemble
from tests.test_gpu_parity import _check_search, _compare_trees, _tree_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [16384, 16385, 32768, 32769])
def test_update_at_scan_sizes(oracle, n):
    print("[gpu-case] update,", n, "neurons", flush=True)
    net = uniform_cube(n, 1000.0 * (n / 1000.0) ** (1 / 3), n % 11)
    net.vac_axon[:] = 0
    net.vac_axon[::17] = 3   # few searches for the oracle, targets still collide
    net.vac_axon[-1] = 2
    t, g = _tree_pair(oracle, net.xyz, net.signal, net.box_min, net.box_max, net.vac_exc, net.vac_inh)
    _compare_trees(t.export(), g.export_tree())
    ref = t.find_targets(net.signal, net.vac_axon, None, seed=0, step=6, threads=0)
    for rep in range(2):   # the second update reuses every buffer
        g.prepare_update_connectivity(net.vac_axon, net.vac_exc, net.vac_inh)
        m = g.find_target_neurons(6)
        tgt, tests, cnt = g.get_search_slots(int(net.vac_axon.sum()))
        bad, _ = _check_search(ref, tgt, tests, cnt, net)
        assert not bad
        rt, rs, rg, rj = g.get_requests(m)
        created = g.commit(6)
        ok = g.get_commit_result(m)
        va, ve, vi = g.get_vacancies()
        e, i, a = net.vac_exc.copy(), net.vac_inh.copy(), net.vac_axon.copy()
        ok_ref, created_ref = oracle.commit(rt, rs, rg, rj, e, i, a, seed=0, step=6)
        assert created == created_ref and np.array_equal(ok, ok_ref)
        assert np.array_equal(ve, e) and np.array_equal(vi, i) and np.array_equal(va, a)
    g.close()


@pytest.mark.parametrize("n", [700, 1500, 3000])
def test_tree_at_level_sizes(oracle, n):
    print("[gpu-case] tree,", n, "neurons", flush=True)
    net = uniform_cube(n, 1500.0, n)
    t, g = _tree_pair(oracle, net.xyz, net.signal, net.box_min, net.box_max, net.vac_exc, net.vac_inh)
    _compare_trees(t.export(), g.export_tree())
    g.close()


@pytest.mark.parametrize("networks", [1023, 1025])
def test_forest_with_many_roots(networks):
    print("[gpu-case] forest,", networks, "networks", flush=True)
    off, boxes, xyz, sig, va, ve, vi = _ensemble([2 + k % 3 for k in range(networks)], 13)
    g = BarnesHutHIP(boxes[:, :3].min(0), boxes[:, 3:].max(0), precision=RL_PREC_FP64)
    g.init_networks(off, boxes, xyz, sig)
    g.prepare_update_connectivity(va, ve, vi)
    e = g.export_tree()
    g.close()
    # roots are nodes 0 .. networks - 1 and count their network's vacant dendrites
    first = off[:-1].astype(np.int64)
    assert np.array_equal(e["cnt_exc"][:networks], np.add.reduceat(ve, first))
    assert np.array_equal(e["cnt_inh"][:networks], np.add.reduceat(vi, first))
