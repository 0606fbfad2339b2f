"""The allocation-free commit on requests in source order and shuffled, at counts around a wave and a block: the
vacancies and connected counts follow from the accept flags, and the flags do not depend on the order."""
import numpy as np
import pytest

from relearn_amd._lib import commit_requests_noalloc
from tests.test_zz_no_alloc import _Hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1, 63, 64, 65, 1023, 1025, 5000])
@pytest.mark.parametrize("connected", [True, False])
def test_axons_of_runs_of_requests(m, connected):
    print("[gpu-case] no-alloc commit,", m, "requests, connected counts", connected, flush=True)
    rng = np.random.default_rng(m)
    n = max(2, m // 3)
    axons = np.bincount(rng.integers(0, n, m), minlength=n).astype(np.uint32)
    axons[n // 2] += 130   # runs longer than a wave
    source = np.repeat(np.arange(n), axons)[:m].astype(np.uint32)
    m = len(source)
    ordinal = (np.arange(m) - (np.cumsum(axons) - axons)[source]).astype(np.uint32)
    target = rng.integers(0, n, m).astype(np.uint32)
    signal = (source % 5 == 0).astype(np.uint8)
    vacant = [axons] + [rng.poisson(1.5, n).astype(np.uint32) for _ in range(2)]
    flags = []
    for order in (np.arange(m), rng.permutation(m)):
        hip = _Hip()
        d_req = [hip.dev(a[order]) for a in (target, source, signal, ordinal)]
        d_vac = [hip.dev(v) for v in vacant]
        d_conn = [hip.dev(np.zeros(n, np.uint32)) for _ in range(3)] if connected else [0, 0, 0]
        d_ok = hip.dev(np.full(m, 7, np.uint8))
        hip.sync()
        created = commit_requests_noalloc(n, m, *d_req, 11, 3, d_vac, d_conn, d_ok, wait=True)
        hip.sync()
        ok = np.empty(m, np.uint8)
        ok[order] = hip.host(d_ok)
        left = [hip.host(p) for p in d_vac]
        taken = [hip.host(p) for p in d_conn] if connected else None
        hip.free()
        yes = ok == 1
        assert np.array_equal(ok, yes.astype(np.uint8)) and created == yes.sum()
        count = [np.bincount(source[yes], minlength=n),
                 np.bincount(target[yes & (signal == 0)], minlength=n), np.bincount(target[yes & (signal != 0)], minlength=n)]
        for k in range(3):
            assert np.array_equal(left[k], vacant[k] - count[k])
            assert taken is None or np.array_equal(taken[k], count[k])
        flags.append(ok)
    assert np.array_equal(flags[0], flags[1])
