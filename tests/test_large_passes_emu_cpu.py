"""Widths of the digit passes of multisplits into more than 1024 buckets."""
import ctypes

import numpy as np
import pytest

import gpumultisplit_amd as gms
import oracle
from gpumultisplit_amd import workloads as W
from test_emu_cpu import emu, p  # noqa: F401

SIZES = [1, 5000, 1 << 20, (1 << 20) + 1, 3 << 19, (3 << 19) + 1, 1 << 21, (1 << 21) + 1, 1 << 25,
         (1 << 26) - 1, 1 << 26, 1 << 27]


def _passes(emu, bits, kv, n, wide=0):  # noqa: F811
    w = np.zeros(3, np.uint32)
    k = emu.gms_emu_large_passes(bits, kv, wide, ctypes.c_uint32(n), w.ctypes.data_as(ctypes.c_void_p))
    return [int(x) for x in w[:k]]


def test_widths_cover_the_id(emu):  # noqa: F811
    for wide in (0, 1):
        for bits in range(9 if wide else 11, 21):
            for kv in (0, 1):
                for n in SIZES:
                    w = _passes(emu, bits, kv, n, wide)
                    assert sum(w) == bits and min(w) >= 1
                    assert max(w) <= (9 if bits in (17, 18) and not wide else 8)


def test_no_width_that_measured_slower(emu):  # noqa: F811
    assert _passes(emu, 18, 0, 1 << 27) == [6, 6, 6]       # 9 + 9: sorted keys a third slower
    assert _passes(emu, 17, 0, 1 << 26) == [6, 6, 5]
    assert _passes(emu, 18, 1, 1 << 27) == [9, 9] and _passes(emu, 18, 0, 1 << 25) == [9, 9]
    assert _passes(emu, 18, 1, 1_300_000) == [8, 8, 2] and _passes(emu, 18, 1, 1 << 20) == [9, 9]
    for kv in (0, 1):
        for n in (1, 1 << 21, 1 << 26, 1 << 27):
            assert _passes(emu, 14, kv, n) == [8, 6]
        assert _passes(emu, 14, kv, 3_000_000) == [7, 7]
    assert _passes(emu, 12, 0, 9_000_000) == [8, 4] == _passes(emu, 12, 1, 2_600_000)
    assert _passes(emu, 12, 1, 3_000_000) == [6, 6] == _passes(emu, 12, 0, 1 << 21)
    assert _passes(emu, 19, 1, 3_000_000) == [8, 8, 3] and _passes(emu, 20, 1, 1_900_000) == [8, 8, 4]


@pytest.mark.parametrize("cap", [5000, 1 << 20, 1_300_000])
@pytest.mark.parametrize("B", [1 << 12, 1 << 14, 1 << 17, 1 << 18, 1 << 20])
def test_calls_below_the_capacity(emu, B, cap):  # noqa: F811
    """A context's matrix holds the passes of every shorter call, also where those
    are wider than the ones of a call at the capacity."""
    h = ctypes.c_void_p()
    assert emu.gms_multisplit_create(B, ctypes.byref(h)) == 0
    assert emu.gms_multisplit_allocate(h, cap, 1) == 0
    for n in (4500, 9000):
        if n > cap:
            continue
        keys = W.uniform_keys(n, seed=B + n)
        vals = np.arange(n, dtype=np.uint32)
        kout, vout, offs = np.zeros_like(keys), np.zeros_like(vals), np.zeros(B, np.uint32)
        assert emu.gms_multisplit_key_value(h, p(keys), p(vals), p(kout), p(vout), n,
                                            gms.range_bucket(B).desc(), p(offs), None) == 0
        wk, wv, wo = oracle.multisplit(keys, B, oracle.RANGE, 0, vals)
        np.testing.assert_array_equal(kout, wk)
        np.testing.assert_array_equal(vout, wv)
        np.testing.assert_array_equal(offs, wo)
    emu.gms_multisplit_destroy(h)
