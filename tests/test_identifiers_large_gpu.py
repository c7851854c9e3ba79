"""Every identifier through the three stages, at sizes above those of the short
forms and on both sides of the limits of the postscan's forms, against a stable
sort of the ids."""
import pytest

import gpumultisplit_amd as gms
from gpu_util import banner

pytestmark = pytest.mark.gpu

KINDS = {
    "delta": (lambda B: gms.delta_func(-(-(1 << 32) // B) + 12345),
              lambda k, B: (k // (-(-(1 << 32) // B) + 12345)).clamp(max=B - 1)),
    "delta_small": (lambda B: gms.delta_func(3), lambda k, B: (k // 3).clamp(max=B - 1)),
    "digit": (lambda B: gms.digit_bucket(9, (B - 1).bit_length()),
              lambda k, B: (k >> 9) & ((1 << (B - 1).bit_length()) - 1)),
    "identity": (lambda B: gms.identity_bucket(), lambda k, B: k.clamp(max=B - 1)),
    "lowbits": (lambda B: gms.test_bucket((B - 1).bit_length()),
                lambda k, B: k & ((1 << (B - 1).bit_length()) - 1)),
}


@pytest.mark.parametrize("kv", [False, True])
@pytest.mark.parametrize("kind", list(KINDS))
@pytest.mark.parametrize("B,n,shift", [(2, 2_300_001, 0), (8, (1 << 24) + 5, 0), (16, (1 << 25) + 6143, 0),
                                       (16, 1 << 25, 1), (8, (1 << 26) + 1, 0), (64, 6_300_000, 0),
                                       (256, 2_300_001, 3), (256, (9 << 20) + 7, 0), (1024, 3_000_001, 0)])
def test_identifiers(dev, kind, B, n, shift, kv):
    import torch
    f, ids_of = KINDS[kind]
    g = torch.Generator(device=dev)
    g.manual_seed(n + B)
    top = (B + B // 4) if kind == "identity" else 4 * B if kind == "delta_small" else 1 << 32
    k64 = torch.randint(0, top, (n + shift,), device=dev, generator=g)
    kin = k64.to(torch.int32)[shift:] if top < 1 << 31 else (k64 - ((k64 >> 31) << 32)).to(torch.int32)[shift:]
    want = torch.sort(ids_of(k64[shift:], B), stable=True)
    del k64
    vin = torch.arange(n + shift, dtype=torch.int32, device=dev)[shift:] if kv else None
    for starts in (True, False):
        banner(f"{kind} B={B} n={n} shift={shift} kv={kv} starts={starts}")
        kout = torch.zeros(n, dtype=torch.int32, device=dev)
        vout = torch.zeros_like(kout) if kv else None
        offs = torch.zeros(B, dtype=torch.int32, device=dev) if starts else None
        ctx = gms.multisplit_context(B)
        gms.multisplit_allocate_key_value(n, ctx)
        gms.multisplit(kin, kout, n, ctx, f(B), d_value_in=vin, d_value_out=vout, d_offsets=offs)
        torch.cuda.synchronize()
        assert torch.equal(kout, kin[want.indices])
        if kv:
            assert torch.equal(vout.to(torch.int64), want.indices + shift)
        if starts:
            edges = torch.arange(B, dtype=want.values.dtype, device=dev)
            assert torch.equal(offs.to(torch.int64), torch.searchsorted(want.values, edges))
        gms.multisplit_release_memory(ctx)


@pytest.mark.parametrize("kb,vb", [(8, 0), (8, 4), (8, 8), (4, 8)])
@pytest.mark.parametrize("ident", ["range", "delta", "digit"])
@pytest.mark.parametrize("B,n", [(8, 1_300_001), (100, (1 << 20) + 1), (256, 5_000_003)])
def test_identifiers_64bit(dev, kb, vb, ident, B, n):
    import torch
    banner(f"64-bit {kb}/{vb} {ident} B={B} n={n}")
    g = torch.Generator(device=dev)
    g.manual_seed(n + B)
    bits = (B - 1).bit_length() if B & (B - 1) == 0 else (B - 1).bit_length() - 1
    if kb == 8:  # the upper word decides the range and the quotient by a multiple of 2^32
        kin = torch.randint(-(1 << 63), (1 << 63) - 1, (n,), dtype=torch.int64, device=dev, generator=g)
        hi = (kin >> 32) & 0xFFFFFFFF
    else:
        hi = torch.randint(0, 1 << 32, (n,), device=dev, generator=g)
        kin = (hi - ((hi >> 31) << 32)).to(torch.int32)
    delta = -(-(1 << 32) // B) + 77
    if ident == "range":  # floor(k * B / 2^64) needs the lower word only where hi * B's fraction is near 1
        ids = (hi * B) >> 32
        if kb == 8:
            lo = kin & 0xFFFFFFFF
            ids = (hi * B + ((lo * B) >> 32)) >> 32
        f = gms.range_bucket(B)
    elif ident == "delta":
        ids = (hi // delta).clamp(max=B - 1)
        f = gms.delta_func(delta << 32 if kb == 8 else delta)
    else:
        ids = (hi >> 5) & ((1 << bits) - 1)
        f = gms.digit_bucket(37 if kb == 8 else 5, bits)
    want = torch.sort(ids, stable=True)
    vin = torch.arange(n, dtype=torch.int64 if vb == 8 else torch.int32, device=dev) if vb else None
    for starts in (True, False):
        kout = torch.zeros_like(kin)
        vout = torch.zeros_like(vin) if vb else None
        offs = torch.zeros(B, dtype=torch.int32, device=dev) if starts else None
        ctx = gms.multisplit_context(B)
        gms.multisplit_allocate_key_value(n, ctx)
        gms.multisplit(kin, kout, n, ctx, f, d_value_in=vin, d_value_out=vout, d_offsets=offs)
        torch.cuda.synchronize()
        assert torch.equal(kout, kin[want.indices])
        if vb:
            assert torch.equal(vout.to(torch.int64), want.indices)
        if starts:
            edges = torch.arange(B, dtype=want.values.dtype, device=dev)
            assert torch.equal(offs.to(torch.int64), torch.searchsorted(want.values, edges))
