"""GPU parity of the digit passes above 1024 buckets on both sides of the sizes
where their widths change, against a stable sort of the ids."""
import pytest

import gpumultisplit_amd as gms
from gpu_util import banner

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits,n", [(12, 1 << 21), (12, (1 << 21) + 1), (12, 1 << 25), (14, 1_900_001),
                                    (17, 1_300_001), (18, 1 << 20), (18, (1 << 20) + 1), (18, 3 << 19),
                                    (18, (3 << 19) + 1), (17, (1 << 26) + 3), (18, 1 << 26),
                                    (19, (1 << 21) + 1), (20, 3 << 19), (20, (3 << 19) + 1)])
@pytest.mark.parametrize("kv", [False, True])
def test_pass_widths(dev, bits, n, kv):
    import torch
    banner(f"pass widths bits={bits} n={n} kv={kv}")
    g = torch.Generator(device=dev)
    g.manual_seed(n + bits)
    kin = torch.randint(-(1 << 31), 1 << 31, (n,), dtype=torch.int32, device=dev, generator=g)
    kin[n // 3:n // 3 + 5000] = -1
    B = 1 << bits
    ids = (kin.to(torch.int64) & 0xFFFFFFFF) >> (32 - bits)
    want = torch.sort(ids, stable=True)
    vin = torch.arange(n, dtype=torch.int32, device=dev) if kv else None
    kout = torch.zeros_like(kin)
    vout = torch.zeros_like(vin) if kv else None
    offs = torch.zeros(B, dtype=torch.int32, device=dev)
    ctx = gms.multisplit_context(B)
    gms.multisplit_allocate_key_value(n, ctx)
    gms.multisplit(kin, kout, n, ctx, gms.range_bucket(B), d_value_in=vin, d_value_out=vout,
                   d_offsets=offs)
    torch.cuda.synchronize()
    assert torch.equal(kout, kin[want.indices])
    if kv:
        assert torch.equal(vout.to(torch.int64), want.indices)
    starts = torch.searchsorted(want.values, torch.arange(B, dtype=torch.int64, device=dev))
    assert torch.equal(offs.to(torch.int64), starts)
