"""The pairs grouped by source: what fired sources push and what axons are deleted among, at the sizes
where the grouping changes (one block, bins of 256 to 1,024 sources), with uneven lists and pairs whose weight is 0;
and the append to lists that are empty, long or hold pairs whose weight is 0."""
from __future__ import annotations

import numpy as np
import pytest

from relearn_amd import BarnesHutHIP, StepParams

pytestmark = pytest.mark.gpu


def _graph(n, rng):
    """In-edges without repeated pairs: targets without and with hundreds of sources, a source of half of the targets."""
    degree = rng.integers(0, 12, n)
    degree[rng.integers(0, n, 3)] = min(n // 2, 700)
    degree[rng.random(n) < 0.2] = 0
    tgt = np.repeat(np.arange(n), degree)
    src = rng.integers(0, n, len(tgt))
    tgt, src = np.concatenate([tgt, np.arange(0, n, 2)]), np.concatenate([src, np.full((n + 1) // 2, n - 1)])
    key = np.unique(tgt.astype(np.int64) * n + src)
    tgt, src = key // n, key % n
    w = np.where(src % 5 == 0, -1, 1) * rng.integers(1, 4, len(src))
    off = np.concatenate([[0], np.cumsum(np.bincount(tgt, minlength=n))]).astype(np.uint64)
    return off, src.astype(np.uint32), w.astype(np.int32)


@pytest.mark.parametrize("n,room", [(1, 0), (65, 10), (2048, 0), (2048, 100000), (2049, 0), (131072, 5), (300001, 0)])
def test_pushes_and_axon_deletion(oracle, n, room):
    print("[gpu-case] pairs by source,", n, "neurons, room", room, flush=True)
    rng = np.random.default_rng(n + room)
    off, src, w = _graph(n, rng)
    tgt = np.repeat(np.arange(n), np.diff(off.astype(np.int64)))
    p = StepParams.izhikevich(input_mode=0)
    p.synaptic_input, p.synapse_conductance = 1, 0.5
    po = oracle.StepParams()
    for f in ("a", "b", "c", "d", "v_spike", "k1", "k2", "k3", "h", "tau_ca", "beta_ca"):
        setattr(po, f, getattr(p, f))
    for k in range(3):
        # axons shrink by about three elements, dendrites stay
        p.eta[k], p.nu[k] = 0.0, (3.0 if k == 0 else 0.0)
        po.eta[k], po.nu[k] = p.eta[k], p.nu[k]
    conn = np.zeros((3, n), np.uint32)
    np.add.at(conn[0], src, np.abs(w).astype(np.uint32))
    np.add.at(conn[1], tgt[w > 0], w[w > 0].astype(np.uint32))
    np.add.at(conn[2], tgt[w < 0], np.abs(w[w < 0]).astype(np.uint32))
    x, u, ca = rng.uniform(-70, -50, n), rng.uniform(-15, -10, n), np.full(n, 0.9)
    tca = np.full(n, 0.1)
    g = BarnesHutHIP((0, 0, 0), (1, 1, 1))
    g.init(rng.random((n, 3)), (np.arange(n) % 5 == 0).astype(np.uint8))
    g.net_init(len(src) + room, off, src, w)
    g.neurons_init(p, tca, x=x, u=u, ca=ca, grown=conn.astype(np.float64).ravel(), connected=conn.ravel())
    fired, delta = np.zeros(n, np.uint8), np.zeros(3 * n)

    def step(k):
        # a third of the neurons fires; integer sums are exact in FP64
        syn = np.bincount(tgt, weights=w * fired[src], minlength=n)
        bg = np.where(rng.random(n) < 0.3, 400.0, 5.0)
        g.neurons_step(k, bg)
        oracle.neuron_step(po, x, u, ca, bg + syn * 0.5, fired, tca, delta)
        st = g.neurons_get()
        assert np.array_equal(st["fired"], fired) and np.array_equal(st["x"], x) and np.array_equal(st["u"], u)

    step(0)
    step(1)
    deleted = np.asarray(g.neurons_commit_elements(3)).reshape(3, n)
    off2, src2, w2 = g.net_get_edges()
    assert np.array_equal(off2, off) and np.array_equal(src2, src)
    gone = np.abs(w) - np.abs(w2)
    assert (gone >= 0).all() and (w2 * w >= 0).all()
    lost = np.zeros(n, np.uint32)
    np.add.at(lost, src, gone.astype(np.uint32))
    assert np.array_equal(lost, deleted[0]) and not deleted[1:].any()
    assert n < 64 or ((w2 == 0).any() and (gone > 0).any())
    after = np.zeros((2, n), np.uint32)
    np.add.at(after[0], tgt[w > 0], np.abs(w2[w > 0]).astype(np.uint32))
    np.add.at(after[1], tgt[w < 0], np.abs(w2[w < 0]).astype(np.uint32))
    assert np.array_equal(np.asarray(g.neurons_get()["connected"]).reshape(3, n)[1:], after)
    w = w2
    step(2)   # the lists hold the pairs that are left
    step(3)
    g.close()


@pytest.mark.parametrize("n,room", [(2, 40), (63, 400), (64, 400), (65, 0), (3001, 0), (3001, 20000)])
def test_append_to_uneven_lists(n, room):
    print("[gpu-case] append to uneven lists,", n, "neurons, room", room, flush=True)
    rng = np.random.default_rng(n + room)
    off, src, w = _graph(n, rng)
    tgt = np.repeat(np.arange(n), np.diff(off.astype(np.int64)))
    signal = (np.arange(n) % 5 == 0).astype(np.uint8)
    conn = np.zeros((3, n), np.uint32)
    np.add.at(conn[0], src, np.abs(w).astype(np.uint32))
    np.add.at(conn[1], tgt[w > 0], w[w > 0].astype(np.uint32))
    np.add.at(conn[2], tgt[w < 0], np.abs(w[w < 0]).astype(np.uint32))
    p = StepParams.izhikevich(input_mode=0)
    for k in range(3):
        p.eta[k], p.nu[k] = 0.0, (3.0 if k == 0 else 0.0)   # axons shrink by about three elements
    g = BarnesHutHIP((0, 0, 0), (1000, 1000, 1000), seed=4)
    g.init(rng.random((n, 3)) * 1000.0, signal)
    g.net_init(len(src) + room, off, src, w)
    g.neurons_init(p, np.full(n, 0.1), ca=np.full(n, 0.9), grown=conn.astype(np.float64).ravel(), connected=conn.ravel())
    gaps = 0
    for update in range(3):
        if update == 1:
            g.neurons_step(0, np.full(n, 5.0))
            g.neurons_commit_elements(update)
        off, src, w = g.net_get_edges()
        tgt = np.repeat(np.arange(n), np.diff(off.astype(np.int64)))
        gaps += int((w == 0).sum())
        expect = {k: v for k, v in zip(zip(tgt.tolist(), src.tolist()), w.tolist()) if v != 0}
        g.prepare_update_connectivity(*[rng.poisson(m, n).astype(np.uint32) for m in (2.0, 1.5, 1.5)])
        m = g.find_target_neurons(update)
        g.commit(update)
        req, ok = g.get_requests(m), np.asarray(g.get_commit_result(m))
        new_tgt, new_src = np.asarray(req[0])[ok != 0], np.asarray(req[1])[ok != 0]
        for t, s in zip(new_tgt.tolist(), new_src.tolist()):
            expect[(t, s)] = expect.get((t, s), 0) + (-1 if signal[s] else 1)
        off, src, w = g.net_get_edges()
        tgt = np.repeat(np.arange(n), np.diff(off.astype(np.int64)))
        assert len(src) == len(expect)
        assert dict(zip(zip(tgt.tolist(), src.tolist()), w.tolist())) == expect
    assert n < 65 or gaps > 0
    g.close()
