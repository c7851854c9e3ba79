"""GPU parity of the LDS-loaded postscan (few buckets, large inputs) with the
oracle: around the size it is taken from, with whole and ragged last tiles,
aligned and unaligned inputs, in the streamed form, and the bucket starts that
the postscans write."""
import numpy as np
import pytest

import gpumultisplit_amd as gms
import oracle
from gpumultisplit_amd import workloads as W
from gpu_util import banner, filled_u32, from_dev, to_dev

pytestmark = pytest.mark.gpu

FROM = 9 << 20


@pytest.mark.parametrize("kv", [False, True])
@pytest.mark.parametrize("B,n,shift", [(2, FROM - 1, 0), (2, FROM, 0), (3, FROM + 1, 1),
                                       (8, 1537 * 6144, 0), (8, 1537 * 6144 + 1, 0),
                                       (16, 12_345_677, 0), (16, 12_345_677, 3),
                                       (10, (1 << 26) + 5, 0), (32, (1 << 26) + 6143, 0),
                                       (256, 3_000_001, 0), (1000, 3_000_001, 1)])
def test_postscan_reg(dev, B, n, shift, kv):
    import torch
    banner(f"postscan B={B} n={n} shift={shift} kv={kv}")
    keys = W.uniform_keys(n + shift, seed=n)
    keys[1000:9000] = 0xFFFFFFFF
    kin = to_dev(keys, dev)[shift:]
    vin = torch.arange(n + shift, dtype=torch.int32, device=dev)[shift:] if kv else None
    kout, vout = filled_u32(n, dev), filled_u32(n, dev) if kv else None
    offs = filled_u32(B, dev, 0xFFFFFFFF)
    ctx = gms.multisplit_context(B)
    gms.multisplit_allocate_key_value(n, ctx)
    gms.multisplit(kin, kout, n, ctx, gms.range_bucket(B), d_value_in=vin, d_value_out=vout,
                   d_offsets=offs)
    torch.cuda.synchronize()
    vals = np.arange(shift, n + shift, dtype=np.uint32) if kv else None
    wk, wv, wo = oracle.multisplit(keys[shift:], B, oracle.RANGE, 0, vals)
    np.testing.assert_array_equal(from_dev(kout)[:n], wk)
    np.testing.assert_array_equal(from_dev(offs), wo)
    if kv:
        np.testing.assert_array_equal(from_dev(vout)[:n], wv)


@pytest.mark.parametrize("kv", [False, True])
@pytest.mark.parametrize("starts", [False, True])
@pytest.mark.parametrize("B,n,shift", [
    (2, 2_300_001, 0), (8, (1 << 22) + 1, 1), (16, 2_100_001, 0), (32, (3 << 20) - 1, 0),
    (64, 3 << 20, 0), (64, (7 << 20) - 1, 1), (33, 7 << 20, 0), (128, 1_600_001, 3),
    (256, 6144 * 300, 0), (256, 6144 * 300 + 1, 2), (200, (7 << 20) - 1, 0), (256, 7 << 20, 0),
    (256, (9 << 20) - 1, 0), (64, 9 << 20, 0), (31, (1 << 26) + 7167, 0),
    (129, (7 << 20) + 1, 1)])
def test_postscan_forms(dev, B, n, shift, starts, kv):
    """Both forms on both sides of every size where the choice between them
    changes, with and without the bucket starts, against the oracle."""
    import torch
    banner(f"postscan forms B={B} n={n} shift={shift} starts={starts} kv={kv}")
    keys = W.uniform_keys(n + shift, seed=n)
    keys[1000:9000] = 0xFFFFFFFF
    keys[n // 2:n // 2 + 20000] = 0
    kin = to_dev(keys, dev)[shift:]
    vin = torch.arange(n + shift, dtype=torch.int32, device=dev)[shift:] if kv else None
    kout, vout = filled_u32(n, dev), filled_u32(n, dev) if kv else None
    offs = filled_u32(B, dev, 0xFFFFFFFF) if starts else None
    ctx = gms.multisplit_context(B)
    gms.multisplit_allocate_key_value(n, ctx)
    gms.multisplit(kin, kout, n, ctx, gms.range_bucket(B), d_value_in=vin, d_value_out=vout,
                   d_offsets=offs)
    torch.cuda.synchronize()
    vals = np.arange(shift, n + shift, dtype=np.uint32) if kv else None
    wk, wv, wo = oracle.multisplit(keys[shift:], B, oracle.RANGE, 0, vals)
    np.testing.assert_array_equal(from_dev(kout)[:n], wk)
    if starts:
        np.testing.assert_array_equal(from_dev(offs), wo)
    if kv:
        np.testing.assert_array_equal(from_dev(vout)[:n], wv)
