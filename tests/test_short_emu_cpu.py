"""The short-input kernels on the CPU emulation, at the edges of their tiles,
against the oracle: one-workgroup and two-launch forms, one to three ranking
passes, grouped count tiles, and 64-bit elements (packed ranking)."""
import ctypes

import numpy as np
import pytest

import gpumultisplit_amd as gms
import oracle
from gpumultisplit_amd import workloads as W
from test_emu_cpu import emu, emu_multisplit, p  # noqa: F401


@pytest.mark.parametrize("B,n", [(2, 1025), (6, 12_289), (33, 8193), (256, 24_577), (1000, 4097),
                                 (1000, 21_505)])
@pytest.mark.parametrize("kv", [False, True])
def test_emulated_short_multisplit(emu, B, n, kv):  # noqa: F811
    keys = W.uniform_keys(n, seed=B + n)
    keys[n // 2:n // 2 + 700] = 0xFFFFFFFF
    got = emu_multisplit(emu, keys, B, gms.range_bucket(B), kv)
    wk, wv, wo = oracle.multisplit(keys, B, oracle.RANGE, 0,
                                   np.arange(n, dtype=np.uint32) if kv else None)
    np.testing.assert_array_equal(got[0], wk)
    np.testing.assert_array_equal(got[2], wo)
    if kv:
        np.testing.assert_array_equal(got[1], wv)


@pytest.mark.parametrize("kind,param,width", [(0, 0, 0), (1, (1 << 57) + 3, 0), (2, 33, 6)])
@pytest.mark.parametrize("n", [1500, 9001])
def test_emulated_short_multisplit_64bit(emu, kind, param, width, n):  # noqa: F811
    B = 100
    keys = W.rng(n).integers(0, 1 << 64, size=n, dtype=np.uint64, endpoint=False)
    vals = np.arange(n, dtype=np.uint64)
    if kind == 0:
        ids = np.array([(int(k) * B) >> 64 for k in keys])
    elif kind == 1:
        ids = np.array([min(int(k) // param, B - 1) for k in keys])
    else:
        ids = ((keys >> np.uint64(param)) & np.uint64((1 << width) - 1)).astype(np.int64)
    order = np.argsort(ids, kind="stable")
    kout, vout, offs = np.zeros_like(keys), np.zeros_like(vals), np.zeros(B, np.uint32)
    h = ctypes.c_void_p()
    assert emu.gms_multisplit_create(B, ctypes.byref(h)) == 0
    assert emu.gms_multisplit_allocate(h, n, 1) == 0
    d = gms.gms_bucket_desc64(kind, width, param)
    assert emu.gms_multisplit_wide(h, p(keys), p(vals), p(kout), p(vout), n, 8, 8, d, None, p(offs),
                                   None) == 0
    emu.gms_multisplit_destroy(h)
    np.testing.assert_array_equal(kout, keys[order])
    np.testing.assert_array_equal(vout, order)
    np.testing.assert_array_equal(offs, np.searchsorted(ids[order], np.arange(B)))
