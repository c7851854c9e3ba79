"""Histograms on the GPU: ragged ends, and the streamed cell-table form of large
inputs, with inputs that start off a 16-byte boundary."""
import numpy as np
import pytest

import gpumultisplit_amd as gms
import oracle
from gpumultisplit_amd import workloads as W
from gpu_util import banner, from_dev, to_dev
from hist_ends import sizes

pytestmark = pytest.mark.gpu


def _off(a, dev, off):
    """The array, `off` words into a device allocation."""
    import torch
    big = torch.zeros(a.size + off, dtype=torch.float32 if a.dtype == np.float32 else torch.int32,
                      device=dev)
    big[off:] = torch.from_numpy(a if a.dtype == np.float32 else a.view(np.int32)).to(dev)
    return big[off:]


def _levels(n, seed):
    lv = np.sort(W.rng(seed).random(n, dtype=np.float32) * np.float32(1024))
    lv[0], lv[-1] = np.float32(0), np.float32(1024)
    return lv


# 0 and 3 whole tiles, and one more than the resident grids of 512 and 768
@pytest.mark.parametrize("tiles", [0, 3, 513, 769])
def test_ragged_ends(dev, tiles):
    import torch
    lv = _levels(257, tiles)
    d_lv = torch.from_numpy(lv).to(dev)
    todo = sizes(tiles)
    for n, off in todo if tiles < 100 else todo[::5]:
        banner(f"histogram ends n={n} off={off}")
        keys = W.uniform_keys(n, seed=n)
        h = torch.zeros(100, dtype=torch.int32, device=dev)
        gms.histogram(_off(keys, dev, off), n, h, 100, gms.range_bucket(100))
        np.testing.assert_array_equal(from_dev(h), oracle.histogram(keys, 100))
        x = (W.rng(n).random(n, dtype=np.float32) * np.float32(1100) - np.float32(30)).astype(np.float32)
        d_x = _off(x, dev, off)
        h = torch.zeros(256, dtype=torch.int32, device=dev)
        gms.multisplit2_histogram_range(d_x, n, h, d_lv, 257)
        np.testing.assert_array_equal(from_dev(h).view(np.int32), oracle.histogram_range(x, lv))
        h = torch.zeros(64, dtype=torch.int32, device=dev)
        gms.multisplit2_histogram_even(d_x, n, h, 0.0, 1024.0, 0.0625, 64)
        np.testing.assert_array_equal(from_dev(h).view(np.int32),
                                      oracle.histogram_even_f32(x, 64, 0.0, 0.0625))


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("kind", ["float", "uint"])
def test_streamed_range_table(dev, kind, off):
    import torch
    n = (1 << 26) + 1
    banner(f"streamed range histogram {kind} off={off}")
    if kind == "float":
        x, lv = W.rng(off).random(n, dtype=np.float32) * np.float32(1100), _levels(257, 3)
        d_lv = torch.from_numpy(lv).to(dev)
    else:
        x, lv = W.uniform_keys(n, seed=off), np.sort(W.uniform_keys(200, seed=4))
        d_lv = to_dev(lv, dev)
    h = torch.zeros(lv.size - 1, dtype=torch.int32, device=dev)
    gms.multisplit2_histogram_range(_off(x, dev, off), n, h, d_lv, lv.size)
    np.testing.assert_array_equal(from_dev(h).view(np.int32), oracle.histogram_range(x, lv))
