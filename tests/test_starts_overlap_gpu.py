"""Bucket starts over the key or value input of the same call, on the GPU: one
workgroup, two launches, and both forms of the three stages, 32- and 64-bit."""
import numpy as np
import pytest

import gpumultisplit_amd as gms
import oracle
from gpumultisplit_amd import workloads as W
from gpu_util import banner, filled_u32, from_dev, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("where", ["keys", "values"])
@pytest.mark.parametrize("B,n", [(8, 900), (256, 30_001), (1000, 300_007), (256, 3_000_001),
                                 (2, (9 << 20) + 5), (4096, 5000)])
def test_starts_over_an_input(dev, B, n, where):
    import torch
    banner(f"starts over {where} B={B} n={n}")
    keys = W.uniform_keys(n, seed=B + n)
    vals = np.arange(n, dtype=np.uint32)
    kin, vin = to_dev(keys, dev), to_dev(vals, dev)
    kout, vout = filled_u32(n, dev), filled_u32(n, dev)
    offs = (kin if where == "keys" else vin)[n - B:n]
    ctx = gms.multisplit_context(B)
    gms.multisplit_allocate_key_value(n, ctx)
    gms.multisplit(kin, kout, n, ctx, gms.range_bucket(B), d_value_in=vin, d_value_out=vout,
                   d_offsets=offs)
    torch.cuda.synchronize()
    wk, wv, wo = oracle.multisplit(keys, B, oracle.RANGE, 0, vals)
    np.testing.assert_array_equal(from_dev(kout)[:n], wk)
    np.testing.assert_array_equal(from_dev(vout)[:n], wv)
    np.testing.assert_array_equal(from_dev(offs), wo)


@pytest.mark.parametrize("n", [5000, 300_007, 2_000_003])
def test_starts_over_a_64bit_input(dev, n):
    import torch
    banner(f"starts over 64-bit values n={n}")
    B = 100
    g = torch.Generator(device=dev)
    g.manual_seed(n)
    kin = torch.randint(-(1 << 63), (1 << 63) - 1, (n,), dtype=torch.int64, device=dev, generator=g)
    vin = torch.arange(n, dtype=torch.int64, device=dev)
    kout, vout = torch.zeros_like(kin), torch.zeros_like(vin)
    ids = (kin >> 57) & 63
    want = torch.sort(ids, stable=True)
    offs = vin.view(torch.int32)[2 * n - B:]
    ctx = gms.multisplit_context(B)
    gms.multisplit_allocate_key_value(n, ctx)
    gms.multisplit(kin, kout, n, ctx, gms.digit_bucket(57, 6), d_value_in=vin, d_value_out=vout,
                   d_offsets=offs)
    torch.cuda.synchronize()
    assert torch.equal(vout, want.indices)
    assert torch.equal(kout, kin[want.indices])
    np.testing.assert_array_equal(offs.cpu().numpy(),
                                  np.searchsorted(want.values.cpu().numpy(), np.arange(B)))
