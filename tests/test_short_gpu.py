"""GPU parity of the short-input forms (one workgroup, or a count and a scatter
launch) with the oracle, at the sizes where their dispatch and tiles change:
the last size of the one-workgroup form, of every tile length and of the form
itself, and one element to either side; keys that all share a bucket, and
inputs that start off a 16-byte boundary.
"""
import numpy as np
import pytest

import gpumultisplit_amd as gms
import oracle
from gpumultisplit_amd import workloads as W
from gpu_util import banner, filled_u32, from_dev, to_dev

pytestmark = pytest.mark.gpu

EDGES = (1, 1023, 1024, 1025, 2048, 2049, 4095, 4096, 4097, 6144, 6145, 8192, 8193)


def _around(*sizes):
    return [s + d for s in sizes for d in (-1, 0, 1)]


def _sizes(B):
    top = (1 << 21) if B <= 64 else (3 << 19) if B <= 256 else (1 << 20)
    return list(EDGES) + [60_013] + _around(1 << 18, 1 << 20, top)


def _off(a, dev, shift):
    """The array, `shift` elements into a device allocation."""
    import torch
    t = to_dev(a, dev)
    big = torch.empty(t.numel() + shift, dtype=t.dtype, device=dev)
    big[shift:] = t
    return big[shift:]


@pytest.mark.parametrize("kv", [False, True])
@pytest.mark.parametrize("B,dist", [(2, "uniform"), (7, "onehot"), (16, "uniform"), (33, "uniform"),
                                    (64, "onehot"), (100, "uniform"), (256, "uniform"),
                                    (256, "onehot"), (400, "uniform"), (1000, "uniform")])
def test_short_multisplit(dev, B, dist, kv):
    import torch
    ctx = gms.multisplit_context(B)
    gms.multisplit_allocate_key_value((1 << 22) + 1, ctx)
    offs = filled_u32(B, dev, 0xFFFFFFFF)
    for i, n in enumerate(_sizes(B)):
        shift = (0, 1, 0, 3)[i % 4]
        banner(f"short B={B} {dist} kv={kv} n={n} shift={shift}")
        keys = W.uniform_keys(n, seed=B + n)
        if dist == "onehot":
            keys[np.arange(n) % 11 != 0] = np.uint32(0xFFFFFFFF)
        vals = W.uniform_keys(n, seed=B + n + 1)
        kin, vin = _off(keys, dev, shift), _off(vals, dev, shift) if kv else None
        kout, vout = filled_u32(n, dev), filled_u32(n, dev) if kv else None
        gms.multisplit(kin, kout, n, ctx, gms.range_bucket(B), d_value_in=vin, d_value_out=vout,
                       d_offsets=offs)
        torch.cuda.synchronize()
        wk, wv, wo = oracle.multisplit(keys, B, oracle.RANGE, 0, vals if kv else None)
        np.testing.assert_array_equal(from_dev(kout)[:n], wk)
        np.testing.assert_array_equal(from_dev(offs), wo)
        if kv:
            np.testing.assert_array_equal(from_dev(vout)[:n], wv)


@pytest.mark.parametrize("kb,vb", [(8, 0), (8, 4), (8, 8), (4, 8)])
@pytest.mark.parametrize("B,ident", [(5, "range"), (64, "digit"), (200, "delta"), (256, "identity"),
                                     (5000, "range")])
def test_short_multisplit_64bit(dev, kb, vb, B, ident):
    import torch
    ctx = gms.multisplit_context(B)
    gms.multisplit_allocate_key_value(1 << 19, ctx)
    offs = filled_u32(B, dev, 0xFFFFFFFF)
    f = {"range": gms.range_bucket(B), "digit": gms.digit_bucket(7, 6),
         "delta": gms.delta_func(-(-(1 << (8 * kb)) // B)), "identity": gms.identity_bucket()}[ident]
    for n in (1, 1025, 4096, 4097, 8192, 8193, 30_001, (1 << 18) + 1):
        banner(f"short 64-bit {kb}/{vb} B={B} {ident} n={n}")
        g = W.rng(n + B)
        hi = 400 if ident == "identity" else 1 << (8 * kb)
        keys = g.integers(0, hi, size=n, dtype=np.uint64, endpoint=False)
        ids = np.array([min(int(f(int(k))) if ident != "range" else (int(k) * B) >> (8 * kb), B - 1)
                        for k in keys])
        order = np.argsort(ids, kind="stable")
        kdt = torch.int64 if kb == 8 else torch.int32
        kin = to_dev(keys.view(np.int64) if kb == 8 else keys.astype(np.uint32), dev)
        vin = torch.arange(n, dtype=torch.int64 if vb == 8 else torch.int32, device=dev) if vb else None
        kout = torch.zeros(n, dtype=kdt, device=dev)
        vout = torch.zeros_like(vin) if vb else None
        gms.multisplit(kin, kout, n, ctx, f, d_value_in=vin, d_value_out=vout, d_offsets=offs)
        torch.cuda.synchronize()
        assert torch.equal(kout, kin[torch.from_numpy(order).to(dev)])
        if vb:
            np.testing.assert_array_equal(vout.cpu().numpy(), order)
        np.testing.assert_array_equal(from_dev(offs), np.searchsorted(ids[order], np.arange(B)))


@pytest.mark.parametrize("kb,vb", [(4, 0), (4, 4), (4, 8), (8, 0), (8, 4), (8, 8)])
@pytest.mark.parametrize("bits", [8, 5])
def test_short_sort(dev, kb, vb, bits):
    import torch
    ctx = gms.ms_sort_context()
    alloc = getattr(gms, f"multisplit_sort_{bits}bit_allocate" + ("_pairs" if vb else ""))
    sort = getattr(gms, f"multisplit_sort_{bits}bit" + ("_pairs" if vb else ""))
    alloc(1 << 19, ctx, **(dict(key_bytes=kb, value_bytes=vb) if vb else dict(key_bytes=kb)))
    for n in EDGES + (20_001, 1 << 18, (1 << 18) + 1):
        banner(f"short sort {kb}/{vb} bits={bits} n={n}")
        keys = W.rng(n).integers(0, 1 << (8 * kb), size=n, dtype=np.uint64, endpoint=False)
        keys[::3] = keys[0]  # ties: stability shows in the values
        if n > 2:
            keys[1], keys[2] = 0, (1 << (8 * kb)) - 1
        order = np.argsort(keys, kind="stable")
        kin = to_dev(keys.view(np.int64) if kb == 8 else keys.astype(np.uint32), dev)
        kout = torch.zeros_like(kin)
        if vb:
            vin = torch.arange(n, dtype=torch.int64 if vb == 8 else torch.int32, device=dev)
            vout = torch.zeros_like(vin)
            sort(kin, kout, vin, vout, n, ctx)
        else:
            sort(kin, kout, n, ctx)
        torch.cuda.synchronize()
        assert torch.equal(kout, kin[torch.from_numpy(order).to(dev)])
        if vb:
            np.testing.assert_array_equal(vout.cpu().numpy(), order)


@pytest.mark.parametrize("B", [2, 1024])
def test_host_results_of_many_contexts(dev, B):
    """More contexts alive than pinned result slots: the calls beyond them take
    the copy, and slots given back are taken again."""
    n = 5000
    keys = W.uniform_keys(n, seed=B)
    wk, _, wo = oracle.multisplit(keys, B, oracle.RANGE, 0, None)
    kin, kout = to_dev(keys, dev), filled_u32(n, dev)
    for _ in range(2):
        ctxs = [gms.multisplit_context(B) for _ in range(67)]
        for c in ctxs:
            gms.multisplit_allocate_key_only(n, c)
            offs = np.full(B, 0xFFFFFFFF, dtype=np.uint32)
            gms.multisplit_key_only(kin, kout, n, c, gms.range_bucket(B), offs)
            np.testing.assert_array_equal(offs, wo)
        np.testing.assert_array_equal(from_dev(kout)[:n], wk)
        for c in ctxs:
            gms.multisplit_release_memory(c)


@pytest.mark.parametrize("kv", [False, True])
@pytest.mark.parametrize("B", [2048, 4096, 5000, 100_000, 200_000, 500_000, 1 << 20])
def test_many_buckets_pass_widths(dev, B, kv):
    """Bucket counts of 11, 12, 13, 17, 18, 19 and 20 bits, whose LSD passes have
    different widths, below and above the two-launch sizes, with the starts of
    both search kernels."""
    ctx = gms.multisplit_context(B)
    gms.multisplit_allocate_key_value(2_200_001, ctx)
    for n in (8193, 300_007, 2_200_001):
        banner(f"many buckets B={B} kv={kv} n={n}")
        keys = W.uniform_keys(n, seed=B + n)
        keys[:n // 7] = keys[0]
        vals = np.arange(n, dtype=np.uint32)
        kout, vout = filled_u32(n, dev), filled_u32(n, dev) if kv else None
        offs = filled_u32(B, dev, 0xFFFFFFFF)
        gms.multisplit(to_dev(keys, dev), kout, n, ctx, gms.range_bucket(B),
                       d_value_in=to_dev(vals, dev) if kv else None, d_value_out=vout,
                       d_offsets=offs)
        wk, wv, wo = oracle.multisplit(keys, B, oracle.RANGE, 0, vals if kv else None)
        np.testing.assert_array_equal(from_dev(kout)[:n], wk)
        np.testing.assert_array_equal(from_dev(offs), wo)
        if kv:
            np.testing.assert_array_equal(from_dev(vout)[:n], wv)


@pytest.mark.gpu
def test_stream_and_pointer_of_tensors(dev):
    """The stream a call goes to is the current one of the tensor's device, for
    plain tensors and subclasses alike; what was refused stays refused."""
    import torch
    t = torch.zeros(8, dtype=torch.int32, device=dev)
    sub = torch.nn.Parameter(t, requires_grad=False)
    side = torch.cuda.Stream()
    for _ in range(2):
        for stream in (torch.cuda.default_stream(), side):
            with torch.cuda.stream(stream):
                assert gms._stream(None, t) == stream.cuda_stream
                assert gms._stream(sub) == stream.cuda_stream
    assert gms._ptr(t) == gms._ptr(sub) == t.data_ptr()
    for bad in (t[::2], t.cpu(), t.to(torch.int64), t.to(torch.int16)):
        with pytest.raises(ValueError):
            gms._ptr(bad)
