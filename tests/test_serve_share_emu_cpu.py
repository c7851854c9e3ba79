"""A request's share of a step's tables: the shares of the requests of a step add
up to at least the bytes that the step takes from the arena."""
import ctypes

import numpy as np
import pytest

from test_emu_cpu import emu  # noqa: F401


@pytest.mark.parametrize("K", [8, 24, 32])
@pytest.mark.parametrize("sizes", [[1], [50_000], [1 << 22], [1 << 27], [3, 70_000, 1 << 20, 0, 5_000_000],
                                   [6144] * 40])
@pytest.mark.parametrize("log_b", [1, 6, 8])
@pytest.mark.parametrize("wide", [0, 1, 2])
def test_shares_cover_the_step(emu, K, sizes, log_b, wide):  # noqa: F811
    n = np.array(sizes, np.uint32)
    lb = np.full(n.size, log_b, np.uint32)
    w = np.array([i % 2 if wide == 2 else wide for i in range(n.size)], np.uint32)
    shares, step = ctypes.c_size_t(), ctypes.c_size_t()
    f = emu.gms_emu_step_bytes
    f.argtypes = [ctypes.c_void_p] * 3 + [ctypes.c_uint32] * 2 + [ctypes.POINTER(ctypes.c_size_t)] * 2
    assert f(n.ctypes.data, lb.ctypes.data, w.ctypes.data, n.size, K, ctypes.byref(shares),
             ctypes.byref(step)) == 0
    assert shares.value >= step.value > 0
