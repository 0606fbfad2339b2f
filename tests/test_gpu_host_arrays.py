"""Caller arrays in page-locked and in pageable host memory, whole and from odd addresses: the same results."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from relearn_amd import BarnesHutHIP, StepParams

pytestmark = pytest.mark.gpu


class _Arrays:
    """Numpy arrays in memory from hipHostMalloc, or pageable; given back on exit."""

    def __init__(self, locked):
        self.hip, self.locked, self.held = C.CDLL("libamdhip64.so.7"), locked, []

    def __enter__(self):
        return self

    def __exit__(self, *a):
        for p in self.held:
            assert self.hip.hipHostFree(p) == 0

    def new(self, n, dtype, shift=0):
        """n zeros that start `shift` elements into their allocation."""
        size = (n + shift + 8) * np.dtype(dtype).itemsize
        if not self.locked:
            return np.zeros(n + shift + 8, dtype)[shift:shift + n]
        p = C.c_void_p()
        assert self.hip.hipHostMalloc(C.byref(p), C.c_size_t(size), 0) == 0
        self.held.append(p)
        whole = np.frombuffer((C.c_char * size).from_address(p.value), dtype)
        whole[:] = 0
        return whole[shift:shift + n]


@pytest.mark.parametrize("n", [1, 65, 1000, 100003])
@pytest.mark.parametrize("shift", [0, 1])
def test_step_input_memory(n, shift):
    print("[gpu-case] step input in page-locked memory,", n, "neurons, shift", shift, flush=True)
    rng = np.random.default_rng(n)
    given = rng.normal(5.0, 3.0, (3, n))
    xyz, ca = rng.random((n, 3)), rng.uniform(0, 0.3, n)
    out = []
    for locked in (False, True):
        g = BarnesHutHIP((0, 0, 0), (1, 1, 1))
        g.init(xyz, np.zeros(n, np.uint8))
        g.neurons_init(StepParams.izhikevich(input_mode=0), np.full(n, 0.2), ca=ca)
        with _Arrays(locked) as memory:
            for k, v in enumerate(given):
                a = memory.new(n, np.float64, shift)
                a[:] = v
                assert g.L.rl_neurons_step(g.h, k, a.ctypes.data_as(C.POINTER(C.c_double))) == 0
            out.append(g.neurons_get())
        g.close()
    for k in out[0]:
        assert np.array_equal(out[0][k], out[1][k]), k


def _pointer(a, kind):
    return a.ctypes.data_as(C.POINTER(kind))


@pytest.mark.parametrize("n", [2, 65, 3001, 70001])
@pytest.mark.parametrize("shift", [0, 1])
def test_update_arrays_memory(n, shift):
    print("[gpu-case] update through page-locked arrays,", n, "neurons, shift", shift, flush=True)
    rng = np.random.default_rng(n)
    xyz = rng.random((n, 3)) * 3000.0
    signal = (rng.random(n) < 0.2).astype(np.uint8)
    vacant = [rng.poisson(m, n).astype(np.uint32) for m in (2.0, 1.5, 1.5)]
    grown = rng.random(3 * n)
    out = []
    for locked in (False, True):
        g = BarnesHutHIP((0, 0, 0), (3000, 3000, 3000), seed=3)
        g.init(xyz, signal)
        g.neurons_init(StepParams.izhikevich(input_mode=1), np.full(n, 0.2), grown=grown)
        g.neurons_step(0)
        with _Arrays(locked) as memory:
            u32 = lambda k: memory.new(k, np.uint32, shift)  # noqa: E731
            u8 = lambda k: memory.new(k, np.uint8, shift)  # noqa: E731
            f64 = lambda k: memory.new(k, np.float64, shift)  # noqa: E731
            given = [u32(n) for _ in vacant]
            for a, v in zip(given, vacant):
                a[:] = v
            P32, P8, P64 = C.c_uint32, C.c_uint8, C.c_double
            assert g.L.rl_bh_prepare_update_connectivity(g.h, *[_pointer(a, P32) for a in given]) == 0
            m = g.find_target_neurons(2)
            created = g.commit(2)
            target, source, ordinal, sig, ok = u32(m), u32(m), u32(m), u8(m), u8(m)
            assert g.L.rl_bh_get_requests(g.h, m, _pointer(target, P32), _pointer(source, P32), _pointer(sig, P8),
                                          _pointer(ordinal, P32)) == 0
            assert g.L.rl_bh_get_commit_result(g.h, m, _pointer(ok, P8)) == 0
            left = [u32(n) for _ in vacant]
            assert g.L.rl_bh_get_vacancies(g.h, *[_pointer(a, P32) for a in left]) == 0
            x, u, ca, fired = f64(n), f64(n), f64(n), u8(n)
            delta, grown_now, connected = f64(3 * n), f64(3 * n), u32(3 * n)
            assert g.L.rl_neurons_get(g.h, _pointer(x, P64), _pointer(u, P64), _pointer(ca, P64), _pointer(fired, P8),
                                      _pointer(delta, P64), _pointer(grown_now, P64), _pointer(connected, P32)) == 0
            out.append([np.array(a) for a in (m, created, target, source, ordinal, sig, ok, *left, x, u, ca, fired, delta,
                                              grown_now, connected)])
        g.close()
    assert n < 65 or (out[0][0] > 0 and out[0][6].any() and not np.array_equal(out[0][7], vacant[0]))
    for a, b in zip(*out):
        assert np.array_equal(a, b)
