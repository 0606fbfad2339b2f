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
