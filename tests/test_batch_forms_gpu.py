"""Batched steps on both sides of the sizes where a tile's ranking changes between
register and LDS counters, under every shape, against a stable sort of the ids."""
import pytest

import gpumultisplit_amd as gms
from gpu_util import banner

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,persistent", [(0, 0), (8, 0), (16, 0), (24, 0), (24, 1), (8, 1)])
@pytest.mark.parametrize("kv,total", [(False, (1 << 26) - 1), (False, (1 << 26) + 1),
                                      (True, (3 << 23) - 1), (True, (3 << 23) + 1)])
def test_large_steps(dev, K, persistent, kv, total):
    import torch
    banner(f"batch forms K={K} persistent={persistent} kv={kv} total={total}")
    g = torch.Generator(device=dev)
    g.manual_seed(total)
    buckets = (2, 8, 32, 64, 100, 256)
    big = total // 6
    sizes = [big] * 5 + [total - 5 * big]
    starts = [sum(s + 3 & ~3 for s in sizes[:i]) + (1 if i == 3 else 0) for i in range(6)]  # one unaligned
    span = starts[-1] + sizes[-1] + 8
    kin = torch.randint(-(1 << 31), 1 << 31, (span,), dtype=torch.int32, device=dev, generator=g)
    kin[starts[5] + 1000:starts[5] + 50000] = 7
    vin = torch.arange(span, dtype=torch.int32, device=dev) if kv else None
    # instance 3 starts a word late: its span is one word shorter
    sizes[3] -= 1
    sizes[5] += 1
    kout = torch.zeros_like(kin)
    vout = torch.zeros_like(vin) if kv else None
    offs = [torch.zeros(B, dtype=torch.int32, device=dev) for B in buckets]
    items = []
    for a, n, B, o in zip(starts, sizes, buckets, offs):
        v = dict(d_value_in=vin[a:a + n], d_value_out=vout[a:a + n]) if kv else {}
        items.append(gms.BatchItem(kin[a:a + n], kout[a:a + n], n, B, gms.range_bucket(B), d_offsets=o,
                                   **v))
    assert sum(sizes) == total
    b = gms.Batch(items)
    if K:
        b.tuning = {"items_per_thread": K, "persistent": persistent}
    b.run()
    torch.cuda.synchronize()
    for a, n, B, o in zip(starts, sizes, buckets, offs):
        ids = ((kin[a:a + n].to(torch.int64) & 0xFFFFFFFF) * B) >> 32
        want = torch.sort(ids, stable=True)
        assert torch.equal(kout[a:a + n], kin[a:a + n][want.indices]), B
        if kv:
            assert torch.equal(vout[a:a + n], vin[a:a + n][want.indices]), B
        assert torch.equal(o.to(torch.int64),
                           torch.searchsorted(want.values, torch.arange(B, device=dev))), B
