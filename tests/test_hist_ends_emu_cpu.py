"""Ragged ends of the histograms on the CPU emulation, against the oracle."""
import numpy as np
import pytest

import gpumultisplit_amd as gms
import oracle
from gpumultisplit_amd import workloads as W
from hist_ends import sizes
from test_emu_cpu import emu, p  # noqa: F401


def _at(x, off):
    """The address of a copy of x that starts `off` words behind a 16-byte boundary."""
    x = x.view(np.uint32)
    big = np.zeros(x.size + 8, np.uint32)
    a = (-big.ctypes.data // 4) % 4 + off
    big[a:a + x.size] = x
    return big, big.ctypes.data + 4 * a


@pytest.mark.parametrize("tiles", [0, 2])
def test_ragged_ends(emu, tiles):  # noqa: F811
    lv = np.sort(W.uniform_keys(65, seed=8))
    for n, off in sizes(tiles):
        keys = W.uniform_keys(n, seed=n)
        keep, at = _at(keys, off)
        h = np.zeros(100, np.uint32)
        assert emu.gms_histogram_u32(at, n, p(h), 100, gms.range_bucket(100).desc(), None) == 0
        np.testing.assert_array_equal(h, oracle.histogram(keys, 100), err_msg=f"bins {n} {off}")
        h = np.zeros(64, np.int32)
        assert emu.gms_histogram_range_u32(at, n, p(h), 65, p(lv), None) == 0
        np.testing.assert_array_equal(h, oracle.histogram_range(keys, lv), err_msg=f"range {n} {off}")
        x = (keys.astype(np.float64) / 2.0 ** 32 * 80.0 - 8.0).astype(np.float32)
        keep, at = _at(x, off)
        h = np.zeros(32, np.int32)
        assert emu.gms_histogram_even_f32(at, n, p(h), 32, 0.0, 64.0, 0.5, None) == 0
        np.testing.assert_array_equal(h, oracle.histogram_even_f32(x, 32, 0.0, 0.5), err_msg=f"even {n} {off}")


@pytest.mark.parametrize("tiles", [0, 1])
def test_ragged_ends_64bit(emu, tiles):  # noqa: F811
    for words, off in sizes(tiles):
        if words % 2 or off % 2:
            continue
        n = words // 2
        keys = W.rng(n).integers(0, 1 << 64, size=n, dtype=np.uint64, endpoint=False)
        keep, at = _at(keys, off)
        h = np.zeros(64, np.uint32)
        assert emu.gms_histogram_wide(at, n, 8, p(h), 64, gms.gms_bucket_desc64(0, 0, 0), None) == 0
        np.testing.assert_array_equal(h, np.bincount((keys >> np.uint64(58)).astype(np.int64), minlength=64))
