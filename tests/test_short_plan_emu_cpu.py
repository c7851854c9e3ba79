"""The rule of the two-launch form: its shapes by size, and matrices that hold
every shorter call of a context."""
import ctypes

import pytest

from test_emu_cpu import emu  # noqa: F401


def _plan(emu, n, B, kw=1, vw=1):  # noqa: F811
    f = emu.gms_emu_short_plan
    f.argtypes = [ctypes.c_uint32] * 4 + [ctypes.c_void_p] * 3
    items, group, words = ctypes.c_uint32(), ctypes.c_uint32(), ctypes.c_uint64()
    f(n, B, kw, vw, ctypes.byref(items), ctypes.byref(group), ctypes.byref(words))
    return items.value, group.value, words.value


def test_shapes(emu):  # noqa: F811
    # 16 elements per thread are slower than 8 and than the three stages above 2^20
    for B in (2, 8, 16, 64, 256):
        for n in ((1 << 18) + 1, 1 << 20, (1 << 20) + 1, 1_100_000, 1_530_000):
            assert _plan(emu, n, B)[0] == 8, (B, n)
        assert _plan(emu, 1 << 18, B)[0] == 4
    assert _plan(emu, 1 << 21, 64)[:2] == (8, 4)
    assert _plan(emu, 1_530_000, 256)[:2] == (8, 4)
    assert _plan(emu, 1 << 21, 8)[:2] == (8, 1)
    # whole tiles of the three stages: those
    for B in (2, 8, 128, 256):
        assert _plan(emu, 3 << 19, B)[0] == 0
        assert _plan(emu, (3 << 19) - 1, B)[0] == 8
    assert _plan(emu, 3 << 19, 64)[0] == 8
    assert _plan(emu, 3 << 18, 1000)[0] == 0 and _plan(emu, 3 << 18, 256)[0] == 8
    # above: the three stages
    for B, top in ((64, 1 << 21), (256, 3 << 19), (1024, 1 << 20)):
        assert _plan(emu, top + 1, B)[0] == 0


@pytest.mark.parametrize("B", [2, 8, 16, 64, 128, 256, 1000, 4096, 1 << 17, 1 << 20])
def test_matrix_holds_every_shorter_call(emu, B):  # noqa: F811
    emu.gms_emu_matrix_words.restype = ctypes.c_uint64
    sizes = sorted({1, 8193, 3 << 18, 3 << 19, (1 << 21) + 1, 5_000_000} |
                   {s + d for s in (1 << 18, 1 << 20, 3 << 19, 1 << 21) for d in (-1, 0)} |
                   {100_000 * i for i in range(1, 22)})
    pass_buckets = [B] if B <= 1024 else [1 << w for w in range(2, 10)]
    for i, cap in enumerate(sizes):
        have = emu.gms_emu_matrix_words(cap, B)
        for n in sizes[:i + 1]:
            for b in pass_buckets:
                assert _plan(emu, n, b)[2] <= have, (cap, n, b)
