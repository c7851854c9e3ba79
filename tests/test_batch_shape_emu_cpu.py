"""The tile shape of a batch's step that was not tuned, by the keys of the step
and the classes that hold most of them.  Planning touches no buffer."""
import ctypes

import pytest

import gpumultisplit_amd as gms
from test_emu_cpu import emu  # noqa: F401


def _shape(emu, parts):  # noqa: F811
    """items_per_thread of the first step of a batch of (n, buckets, kv) instances."""
    items, at = [], 1 << 40
    for n, B, kv in parts:
        a = [at + i * (1 << 32) for i in range(4)]
        at += 4 << 32
        items.append(gms.gms_batch_item(a[0], a[1] if kv else None, a[2], a[3] if kv else None, n, B,
                                        gms.range_bucket(B).desc(), None))
    h = ctypes.c_void_p()
    assert emu.gms_batch_create(ctypes.byref(h)) == 0
    try:
        arr = (gms.gms_batch_item * len(items))(*items)
        assert emu.gms_batch_plan(h, arr, len(items), None) == 0
        t = gms.gms_batch_tuning()
        assert emu.gms_batch_get_tuning(h, ctypes.byref(t)) == 0
        return t.items_per_thread
    finally:
        emu.gms_batch_destroy(h)


@pytest.mark.parametrize("parts,items", [
    ([(1_000_000, 64, 1)] * 11, 8), ([(1_000_000, 256, 0)] * 16, 8),
    ([(1_000_000, 64, 1)] * 42, 16), ([(1_000_000, 128, 0)] * 42, 16),
    ([(1_000_000, 256, 0)] * 42, 24),   # 16: 151 us against 143, and 141 before shapes by size
    ([(1_000_000, 256, 1)] * 21, 24),
    ([(1_000_000, 256, 1)] * 20 + [(1_000_000, 64, 1)] * 22, 16),
    ([(1_000_000, 256, 1)] * 22 + [(1_000_000, 64, 1)] * 20, 24),
    ([(1_000_000, 64, 1)] * 72, 24), ([(1_000_000, 64, 0)] * 72, 24),
    ([(1_000_000, 32, 0)] * 72, 16),    # 24: 199 us against 187
    ([(1_000_000, 32, 1)] * 72, 24),
    ([(1_000_000, 32, 0)] * 35 + [(1_000_000, 64, 0)] * 37, 24)])
def test_default_shape(emu, parts, items):  # noqa: F811
    assert _shape(emu, parts) == items


def test_by_size_can_be_restored(emu):  # noqa: F811
    """Reading the tuning and writing it back fixes the first step's shape for every
    step; 0 returns to shapes by size."""
    items = [gms.gms_batch_item((1 << 40) + (i << 34), None, (2 << 40) + (i << 34), None, 1_000_000, 64,
                                gms.range_bucket(64).desc(), None) for i in range(42)]
    arr = (gms.gms_batch_item * len(items))(*items)
    sort = gms.gms_batch_sort_item(3 << 40, None, 4 << 40, None, 5000, 8)
    h, t = ctypes.c_void_p(), gms.gms_batch_tuning()
    work = ctypes.c_uint32()

    def tiles():
        assert emu.gms_batch_stats(h, None, ctypes.byref(work), None, None) == 0
        return work.value

    assert emu.gms_batch_create(ctypes.byref(h)) == 0
    try:
        assert emu.gms_batch_plan_mixed(h, arr, len(items), ctypes.byref(sort), 1, None) == 0
        assert emu.gms_batch_get_tuning(h, ctypes.byref(t)) == 0
        assert t.items_per_thread == 16
        # step 0: the multisplits and the first digit, 16 keys per thread; three more digits, 8
        first = 42 * -(-1_000_000 // 4096) + 2
        assert tiles() == first + 3 * 3
        assert emu.gms_batch_set_tuning(h, t) == 0
        assert tiles() == first + 3 * 2
        assert emu.gms_batch_set_tuning(h, gms.gms_batch_tuning(0, 0)) == 0
        assert tiles() == first + 3 * 3
        assert emu.gms_batch_set_tuning(h, gms.gms_batch_tuning(12, 0)) == 1
    finally:
        emu.gms_batch_destroy(h)
