"""Bucket starts written over an input or an output of the same call.

The call reads its inputs before any start is handed out, so a program may let
the starts overwrite the key or value input (which it needs no more), and the
starts win where they overlap an output.  On the emulation, workgroups run one
after another: a kernel that writes the starts while later workgroups still
read the input gives other results than the oracle."""
import ctypes

import numpy as np
import pytest

import gpumultisplit_amd as gms
import oracle
from gpumultisplit_amd import workloads as W
from test_emu_cpu import emu, p  # noqa: F401


def _place(where, kin, vin, kout, vout, B):
    """The words of the starts: the last B of an input, read by the call's last
    tile, or the first B of an output, written by its first one."""
    a = {"keys": kin, "values": vin, "kout": kout, "vout": vout}[where].view(np.uint32)
    return a[a.size - B:] if where in ("keys", "values") else a[:B]


def _check(kout, vout, offs, where, B, want):
    wk, wv, wo = want
    np.testing.assert_array_equal(offs, wo)
    np.testing.assert_array_equal(kout[B if where == "kout" else 0:], wk[B if where == "kout" else 0:])
    np.testing.assert_array_equal(vout[B if where == "vout" else 0:], wv[B if where == "vout" else 0:])


@pytest.mark.parametrize("entry", ["context", "noalloc"])
@pytest.mark.parametrize("where", ["keys", "values", "kout", "vout"])
@pytest.mark.parametrize("B,n", [(3, 900), (64, 30_001), (256, 30_001), (1000, 20_001)])
def test_starts_over_a_buffer(emu, B, n, where, entry):  # noqa: F811
    keys = W.uniform_keys(n, seed=B + n)
    want = oracle.multisplit(keys, B, oracle.RANGE, 0, np.arange(n, dtype=np.uint32))
    kin, vin = keys.copy(), np.arange(n, dtype=np.uint32)
    kout, vout = np.zeros(max(n, B), np.uint32), np.zeros(max(n, B), np.uint32)
    offs = _place(where, kin, vin, kout, vout, B)
    d = gms.range_bucket(B).desc()
    if entry == "noalloc":
        assert emu.gms_multisplit_noalloc(p(kin), p(vin), p(kout), p(vout), n, B, d, p(offs), None) == 0
    else:
        h = ctypes.c_void_p()
        assert emu.gms_multisplit_create(B, ctypes.byref(h)) == 0
        assert emu.gms_multisplit_allocate(h, n, 1) == 0
        assert emu.gms_multisplit(h, p(kin), p(vin), p(kout), p(vout), n, d, p(offs), None) == 0
        emu.gms_multisplit_destroy(h)
    _check(kout[:n], vout[:n], offs, where, B, want)


@pytest.mark.parametrize("where", ["keys", "values"])
def test_starts_over_an_input_many_buckets(emu, where):  # noqa: F811
    for B, n in ((3000, 4000), (3000, 20_001)):
        keys = W.uniform_keys(n, seed=B + n)
        want = oracle.multisplit(keys, B, oracle.RANGE, 0, np.arange(n, dtype=np.uint32))
        kin, vin = keys.copy(), np.arange(n, dtype=np.uint32)
        kout, vout = np.zeros(n, np.uint32), np.zeros(n, np.uint32)
        offs = _place(where, kin, vin, kout, vout, B)
        h = ctypes.c_void_p()
        assert emu.gms_multisplit_create(B, ctypes.byref(h)) == 0
        assert emu.gms_multisplit_allocate(h, n, 1) == 0
        assert emu.gms_multisplit(h, p(kin), p(vin), p(kout), p(vout), n, gms.range_bucket(B).desc(),
                                  p(offs), None) == 0
        emu.gms_multisplit_destroy(h)
        _check(kout, vout, offs, where, B, want)


@pytest.mark.parametrize("where", ["keys", "values", "kout", "vout"])
@pytest.mark.parametrize("B,n", [(3, 900), (64, 20_001), (256, 20_001)])
def test_starts_over_a_64bit_buffer(emu, B, n, where):  # noqa: F811
    keys = W.rng(n).integers(0, 1 << 64, size=n, dtype=np.uint64, endpoint=False)
    ids = np.array([(int(k) * B) >> 64 for k in keys])
    order = np.argsort(ids, kind="stable")
    starts = np.searchsorted(ids[order], np.arange(B))
    kin, vin = keys.copy(), np.arange(n, dtype=np.uint64)
    kout, vout = np.zeros(n, np.uint64), np.zeros(n, np.uint64)
    offs = _place(where, kin, vin, kout, vout, B)
    h = ctypes.c_void_p()
    assert emu.gms_multisplit_create(B, ctypes.byref(h)) == 0
    assert emu.gms_multisplit_allocate(h, n, 1) == 0
    assert emu.gms_multisplit_wide(h, p(kin), p(vin), p(kout), p(vout), n, 8, 8,
                                   gms.gms_bucket_desc64(0, 0, 0), p(offs), None, None) == 0
    emu.gms_multisplit_destroy(h)
    np.testing.assert_array_equal(offs, starts)
    k0, v0 = (B + 1) // 2 if where == "kout" else 0, (B + 1) // 2 if where == "vout" else 0
    np.testing.assert_array_equal(kout[k0:], keys[order][k0:])
    np.testing.assert_array_equal(vout[v0:], order[v0:])
