"""Every form of the kernels at emulated sizes, which the rules leave to one of
them: the three stages (which short calls skip) with both postscans, the
range histogram's cell table, and LDS counters in batched tiles.  The cases of
the other emulation tests run again with the form forced."""
import ctypes

import numpy as np
import pytest

import gpumultisplit_amd as gms
import oracle
import test_emu_cpu as E
from gpumultisplit_amd import workloads as W
from hist_cases import range_level_sets, range_samples
from test_emu_cpu import emu, p  # noqa: F401

SHORT, REG, TABLE, BATCH_LDS = range(4)


@pytest.fixture
def force(emu):  # noqa: F811
    emu.gms_emu_force.argtypes = [ctypes.c_int, ctypes.c_int]
    yield emu.gms_emu_force
    for i in range(4):
        emu.gms_emu_force(i, -1)


@pytest.fixture(params=["lds", "registers"])
def stages(force, request):
    force(SHORT, 0)
    force(REG, int(request.param == "registers"))
    return request.param


def _call(emu, keys, B, desc, kind, param, kv, starts, shift):  # noqa: F811
    """One device call; `shift`: the inputs start this many words into their arrays."""
    n = keys.size
    kin, vin = np.empty(n + 8, np.uint32), np.empty(n + 8, np.uint32)
    a = (-kin.ctypes.data // 4) % 4 + shift  # `shift` words behind a 16-byte boundary
    b = (-vin.ctypes.data // 4) % 4 + shift
    k, v = kin[a:a + n], vin[b:b + n]
    k[:], v[:] = keys, np.arange(n, dtype=np.uint32)
    kout, vout = np.full(n, 0x5A5A5A5A, np.uint32), np.full(n, 0x5A5A5A5A, np.uint32)
    offs = np.full(B, 77, np.uint32)
    h = ctypes.c_void_p()
    assert emu.gms_multisplit_create(B, ctypes.byref(h)) == 0
    assert emu.gms_multisplit_allocate(h, n, 1) == 0
    assert emu.gms_multisplit(h, p(k), p(v) if kv else None, p(kout), p(vout) if kv else None, n, desc,
                              p(offs) if starts else None, None) == 0
    emu.gms_multisplit_destroy(h)
    wk, wv, wo = oracle.multisplit(keys, B, kind, param, np.arange(n, dtype=np.uint32))
    np.testing.assert_array_equal(kout, wk)
    if kv:
        np.testing.assert_array_equal(vout, wv)
    if starts:
        np.testing.assert_array_equal(offs, wo)


@pytest.mark.parametrize("B", [2, 3, 8, 17, 64, 100, 256, 1000])
@pytest.mark.parametrize("kv", [False, True])
def test_three_stages(emu, stages, B, kv):  # noqa: F811
    tile = gms.tile_keys(B, kv, 0)
    for i, n in enumerate((1, 65, tile - 1, tile, tile + 1, 3 * tile + 17)):
        keys = W.uniform_keys(n, seed=B + n)
        keys[n // 2:n // 2 + 500] = 0xFFFFFFFF
        for starts, shift in ((i % 2 == 0, 0), (i % 2 == 1, 1 + i % 3)):
            _call(emu, keys, B, gms.range_bucket(B).desc(), oracle.RANGE, 0, kv, starts, shift)


@pytest.mark.parametrize("f,B,kind,param", [
    (gms.delta_func(1 << 26), 64, oracle.DELTA, 1 << 26), (gms.delta_func(3), 7, oracle.DELTA, 3),
    (gms.digit_bucket(24, 8), 256, oracle.DIGIT, 24), (gms.identity_bucket(), 16, oracle.IDENTITY, 0),
    (gms.test_bucket(3), 8, oracle.LOWBITS, 3)])
@pytest.mark.parametrize("kv", [False, True])
def test_three_stages_identifiers(emu, stages, f, B, kind, param, kv):  # noqa: F811
    n = 2 * 6144 + 777
    keys = W.uniform_keys(n, seed=B)
    if kind == oracle.IDENTITY:
        keys = keys % np.uint32(B + 5)  # some ids past B - 1: clamped
    if kind == oracle.DELTA and param == 3:
        keys = keys % np.uint32(30)
    _call(emu, keys, B, f.desc(), kind, param, kv, True, 0)


def test_three_stages_many_tiles(emu, stages):  # noqa: F811
    for B, kv, extra in ((2, True, 0), (8, False, 5), (256, True, 6143)):
        E.test_emulated_many_tiles_ragged_last(emu, B, kv, extra)
    E.test_emulated_skewed_and_delta(emu)


@pytest.mark.parametrize("bits", [4, 5, 7, 8])
def test_three_stages_sort(emu, stages, bits):  # noqa: F811
    E.test_emulated_sort(emu, bits)


@pytest.mark.parametrize("B,kind,param,width", [(257, oracle.RANGE, 0, 0), (4096, oracle.DIGIT, 7, 12),
                                                (70000, oracle.IDENTITY, 0, 0), (1 << 18, oracle.RANGE, 0, 0),
                                                (1 << 20, oracle.RANGE, 0, 0)])
def test_three_stages_more_than_256_buckets(emu, stages, B, kind, param, width):  # noqa: F811
    E.test_emulated_more_than_256_buckets(emu, B, kind, param, width)


@pytest.mark.parametrize("kb,vb", [(8, 0), (8, 4), (8, 8), (4, 8)])
@pytest.mark.parametrize("B", [2, 100, 256])
def test_three_stages_64bit(emu, force, kb, vb, B):  # noqa: F811
    """Whole, ragged and single tiles, with the starts on the device and none."""
    force(SHORT, 0)
    for n in (1, 1024, 4096, 9000):
        g = W.rng(n + B)
        keys = g.integers(0, 1 << (8 * kb), size=n, dtype=np.uint64, endpoint=False)
        ids = np.array([(int(k) * B) >> (8 * kb) for k in keys])
        order = np.argsort(ids, kind="stable")
        kin = keys if kb == 8 else keys.astype(np.uint32)
        vin = np.arange(n, dtype=np.uint64 if vb == 8 else np.uint32) if vb else None
        for starts in (True, False):
            kout = np.zeros_like(kin)
            vout = np.zeros_like(vin) if vb else None
            offs = np.zeros(B, np.uint32)
            h = ctypes.c_void_p()
            assert emu.gms_multisplit_create(B, ctypes.byref(h)) == 0
            assert emu.gms_multisplit_allocate(h, n, 1) == 0
            assert emu.gms_multisplit_wide(h, p(kin), p(vin), p(kout), p(vout), n, kb, vb,
                                           gms.gms_bucket_desc64(0, 0, 0), p(offs) if starts else None,
                                           None, None) == 0
            emu.gms_multisplit_destroy(h)
            np.testing.assert_array_equal(kout, kin[order])
            if vb:
                np.testing.assert_array_equal(vout, order)
            if starts:
                np.testing.assert_array_equal(offs, np.searchsorted(ids[order], np.arange(B)))


def test_compaction(emu, stages):  # noqa: F811
    n = 3 * 6144 + 100
    keys = W.uniform_keys(n, seed=9)
    for kv in (False, True):
        vals = np.arange(n, dtype=np.uint32)
        kout, vout, count = np.zeros_like(keys), np.zeros_like(vals), ctypes.c_uint32()
        h = ctypes.c_void_p()
        assert emu.gms_compaction_create(ctypes.byref(h)) == 0
        assert emu.gms_compaction_allocate(h, n, int(kv)) == 0
        assert emu.gms_compaction(h, p(keys), p(vals) if kv else None, p(kout), p(vout) if kv else None, n,
                                  gms.delta_func(1 << 30).desc(), ctypes.addressof(count), None, None) == 0
        emu.gms_compaction_destroy(h)
        kept = np.flatnonzero(keys < np.uint32(1 << 30))
        assert count.value == kept.size
        np.testing.assert_array_equal(kout[:kept.size], keys[kept])
        if kv:
            np.testing.assert_array_equal(vout[:kept.size], kept)


@pytest.mark.parametrize("where", ["keys", "values", "kout", "vout"])
@pytest.mark.parametrize("B", [3, 256])
def test_starts_over_a_buffer(emu, stages, B, where):  # noqa: F811
    import test_starts_overlap_emu_cpu as S
    S.test_starts_over_a_buffer(emu, B, 30_001, where, "context")
    if stages == "lds":
        S.test_starts_over_a_64bit_buffer(emu, B, 20_001, where)


@pytest.mark.parametrize("table", [0, 1])
def test_range_histogram_edge_sets(emu, force, table):  # noqa: F811
    """The cell table, and the search without it, on the edge sets that stress
    the table; inputs that start off a 16-byte boundary."""
    force(TABLE, table)
    E.test_emulated_histogram_range_edge_sets(emu)
    sets, isets = range_level_sets()
    for lv, fn in ((sets[1], emu.gms_histogram_range_f32), (isets[2], emu.gms_histogram_range_u32)):
        x = range_samples(lv, 2 * 4096 + 55, seed=11)
        for off in (1, 2, 3):
            big = np.zeros(x.size + 8, x.dtype)
            a = (-big.ctypes.data // 4) % 4 + off
            big[a:a + x.size] = x
            h = np.zeros(lv.size - 1, np.int32)
            assert fn(big.ctypes.data + 4 * a, x.size, p(h), lv.size, p(lv), None) == 0
            np.testing.assert_array_equal(h, oracle.histogram_range(x, lv))


@pytest.mark.parametrize("tuning", [(8, 0), (8, 1), (16, 0), (16, 1), (24, 0), (24, 1)])
def test_batch_lds_counters(emu, force, tuning):  # noqa: F811
    force(BATCH_LDS, 1)
    E._emu_batch(emu, E.BATCH_CASES, tuning, seed=5 + sum(tuning))
    E._emu_batch(emu, [(n, B, f, kind, param, not kv) for n, B, f, kind, param, kv in E.BATCH_CASES],
                 tuning, seed=6 + sum(tuning))
