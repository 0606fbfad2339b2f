"""The pairs grouped by source in networks of over a million neurons, whose bins hold 256 to 8,192 sources (with
more than 4,096 sources, or more than 8,192 pairs, they are sorted without a staging area): a few thousand
connected neurons among them behave as the same neurons alone, and sources lose the synapses they delete."""
from __future__ import annotations

import numpy as np
import pytest

from relearn_amd import BarnesHutHIP, StepParams

pytestmark = pytest.mark.gpu
CONNECTED = 4000


def _graph(rng):
    """In-edges of the connected neurons without repeated pairs; the first 32 sources reach a fifth of them each."""
    src = np.concatenate([rng.integers(0, CONNECTED, 30_000), np.repeat(np.arange(32), CONNECTED // 5)])
    key = np.unique(rng.integers(0, CONNECTED, len(src)) * CONNECTED + src)
    tgt, src = key // CONNECTED, key % CONNECTED
    return tgt, src, np.where(src % 5 == 0, -1, 1) * rng.integers(1, 4, len(src))


def _run(n, ids, tgt, src, w, rng_seed):
    """Two steps and an element commit, whose deletions are checked; the connected neurons' states."""
    p = StepParams.izhikevich(input_mode=0)
    p.synaptic_input, p.synapse_conductance = 1, 0.5
    for k in range(3):
        p.eta[k], p.nu[k] = 0.0, (3.0 if k == 0 else 0.0)   # axons shrink by about three elements
    conn = np.zeros((3, n), np.uint32)
    np.add.at(conn[0], ids[src], np.abs(w).astype(np.uint32))
    np.add.at(conn[1], ids[tgt[w > 0]], w[w > 0].astype(np.uint32))
    np.add.at(conn[2], ids[tgt[w < 0]], np.abs(w[w < 0]).astype(np.uint32))
    off = np.zeros(n + 1, np.uint64)
    off[ids + 1] = np.bincount(tgt, minlength=CONNECTED)
    off = np.cumsum(off).astype(np.uint64)
    rng = np.random.default_rng(rng_seed)
    signal = np.zeros(n, np.uint8)
    signal[ids] = np.arange(CONNECTED) % 5 == 0
    g = BarnesHutHIP((0, 0, 0), (1, 1, 1))
    g.init(np.random.default_rng(n).random((n, 3)), signal)
    g.net_init(len(src), off, ids[src], w)
    state = [np.full(n, v) for v in (-65.0, -13.0, 0.9)]
    state[0][ids] = rng.uniform(-70, -50, CONNECTED)
    g.neurons_init(p, np.full(n, 0.1), x=state[0], u=state[1], ca=state[2], grown=conn.astype(np.float64).ravel(),
                   connected=conn.ravel())
    given, states = np.full(n, 5.0), []
    for k in range(2):
        given[ids] = np.where(rng.random(CONNECTED) < 0.3, 400.0, 5.0)
        g.neurons_step(k, given)
        s = g.neurons_get()
        states.append([s[f][ids] for f in ("x", "u", "ca", "fired")])
    assert 0 < states[0][3].sum() < CONNECTED   # what these fired reaches the others in the second step
    deleted = np.asarray(g.neurons_commit_elements(3)).reshape(3, n)
    left = g.net_get_edges()[2]
    connected = np.asarray(g.neurons_get()["connected"])
    g.close()
    lost = np.zeros(CONNECTED, np.int64)
    np.add.at(lost, src, np.abs(w) - np.abs(left))
    assert (left * w >= 0).all() and (lost > 0).any()
    assert np.array_equal(lost, deleted[0, ids]) and deleted.sum() == lost.sum()
    after = np.zeros((2, CONNECTED), np.uint32)
    np.add.at(after[0], tgt[w > 0], np.abs(left[w > 0]).astype(np.uint32))
    np.add.at(after[1], tgt[w < 0], np.abs(left[w < 0]).astype(np.uint32))
    assert np.array_equal(connected[1:, ids], after) and connected[1:].sum() == after.sum()
    return states


@pytest.mark.parametrize("n", [2 ** 20 - 1, 2 ** 20, 2 ** 21 + 1, 2 ** 23 + 5, 2 ** 24 + 3])
def test_connected_neurons_among_many(n):
    print("[gpu-case] pairs by source in large bins,", n, "neurons", flush=True)
    rng = np.random.default_rng(n)
    tgt, src, w = _graph(rng)
    edges = np.concatenate([256 * rng.integers(1, n // 256, 1500), [1, n - 1]])   # on both sides of bins' ends
    ids = np.unique(np.concatenate([np.arange(40), edges, edges - 1, rng.integers(0, n, 2 * CONNECTED)]))
    ids = np.sort(np.concatenate([ids[:40], rng.permutation(ids[40:])[:CONNECTED - 40]]))
    large, alone = _run(n, ids, tgt, src, w, 1), _run(CONNECTED, np.arange(CONNECTED), tgt, src, w, 1)
    for a, b in zip(large, alone):
        for x, y in zip(a, b):
            assert np.array_equal(x, y)
