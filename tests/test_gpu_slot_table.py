"""The wave-per-source search at the end of its slot table: a wave holds 2,047 expanded nodes of a source, and a
source with more goes to the per-lane search.  The expanded nodes are counted on the oracle's tree."""
from __future__ import annotations

import numpy as np
import pytest

from relearn_amd import RL_PREC_FP32_MIXED, RL_PREC_FP64
from relearn_amd.workloads import Network, uniform_cube
from tests.test_gpu_parity import _check_search, _search_pair

pytestmark = pytest.mark.gpu
MOST = 2047


def _expanded(export, xyz, signal, source, theta):
    """Nodes that the source expands in its list from the root, the root among them, and the most of one level."""
    cnt = export["cnt_inh" if signal[source] else "cnt_exc"]
    pos = export["pos_inh" if signal[source] else "pos_exc"]
    level, total, widest = np.array([0]), 1, 1
    while len(level):
        nc = export["nchild"][level].astype(np.int64)
        kids = np.repeat(export["link"][level] - (np.cumsum(nc) - nc), nc) + np.arange(nc.sum())
        kids = kids[(cnt[kids] != 0) & (export["nchild"][kids] != 0)]
        d = np.sqrt(((pos[kids] - xyz[source]) ** 2).sum(axis=1))
        level = kids[(d != 0) & ~(export["side"][kids] < theta * d)]
        total += len(level)
        widest = max(widest, len(level))
    return total, widest


def _concentric(n, seed):
    """Neurons at log-uniform distances from one point: a source expands many nodes, few of them of one level."""
    rng = np.random.default_rng(seed)
    d = rng.normal(size=(n, 3))
    d *= (360.0 * 10.0 ** (-4.0 * rng.random(n)) / np.linalg.norm(d, axis=1))[:, None]
    vac_axon = np.zeros(n, np.uint32)
    vac_axon[::5] = 1 + rng.poisson(1.0, n // 5)
    return Network(np.array([437.1, 611.3, 389.7]) + d, (rng.random(n) < 0.2).astype(np.uint8), vac_axon,
                   rng.poisson(1.5, n).astype(np.uint32), rng.poisson(1.5, n).astype(np.uint32), (0.0, 0.0, 0.0),
                   (1000.0, 1000.0, 1000.0))


def _run(oracle, net, theta, precision):
    t = oracle.Tree(net.xyz, net.box_min, net.box_max)
    t.update(net.vac_exc, net.vac_inh)
    export = t.export()
    t.close()
    counts = np.array([_expanded(export, net.xyz, net.signal, s, theta) for s in np.flatnonzero(net.vac_axon)])
    ref, g, nreq, tgt, tests, cnt = _search_pair(oracle, net, seed=3, step=1, theta=theta, precision=precision)
    stats = g.last_search_stats()
    g.close()
    if precision == RL_PREC_FP64:
        bad, near = _check_search(ref, tgt, tests, cnt, net)
        print("[gpu-case]   near-boundary", near, "mismatches", len(bad), bad[:5], flush=True)
        assert not bad
    else:   # picks may differ by FP32 probabilities; the decisions, and so the tests, are the FP64 ones
        target = np.asarray(ref["target"])
        both = (target != 0xFFFFFFFF) & (tgt != 0xFFFFFFFF)
        same = both & (target == tgt)
        assert np.mean(target[both] != tgt[both]) <= 1e-3
        assert np.array_equal(np.asarray(ref["node_tests"])[same], tests[same])
    assert nreq == int(cnt.sum())
    return counts, stats["lane_sources"]


@pytest.mark.parametrize("precision", [RL_PREC_FP64, RL_PREC_FP32_MIXED])
def test_search_parity_at_the_tables_end(oracle, precision):
    print("[gpu-case] slot table, concentric 20,000, theta 0.3, precision", precision, flush=True)
    counts, lane_sources = _run(oracle, _concentric(20_000, 6), 0.3, precision)
    slots, widest = counts[:, 0], counts[:, 1]
    assert widest.max() < 256   # the ring holds every level
    assert ((slots >= 1900) & (slots <= MOST)).sum() > 100 and (slots > MOST).sum() > 100
    for k in (MOST - 1, MOST, MOST + 1, MOST + 2):
        assert (slots == k).any()
    assert lane_sources == (slots > MOST).sum()


@pytest.mark.parametrize("theta", [0.2, 0.15])
@pytest.mark.parametrize("precision", [RL_PREC_FP64, RL_PREC_FP32_MIXED])
def test_search_parity_with_levels_wider_than_the_ring(oracle, precision, theta):
    print("[gpu-case] slot table, uniform 52,000, theta", theta, "precision", precision, flush=True)
    net = uniform_cube(52_000, 10_000.0 * (0.052 ** (1 / 3)), 4)
    net.vac_axon[np.arange(net.n) % 32 != 0] = 0
    counts, lane_sources = _run(oracle, net, theta, precision)
    slots, widest = counts[:, 0], counts[:, 1]
    assert (widest[slots <= MOST] > 520).sum() > 50   # more than the ring's 512 slots wait at once
    assert (slots > MOST).any() == (theta == 0.15)
    assert lane_sources == (slots > MOST).sum()
