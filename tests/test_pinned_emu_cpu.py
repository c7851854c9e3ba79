"""Host results through pinned memory, on the emulated runtime: calls must give
the same results where no pinned memory can be had."""
import ctypes

import numpy as np
import pytest

import gpumultisplit_amd as gms
import oracle
from gpumultisplit_amd import workloads as W
from test_emu_cpu import emu, p  # noqa: F401


def _multisplit_ctx(emu, B, n):  # noqa: F811
    h = ctypes.c_void_p()
    assert emu.gms_multisplit_create(B, ctypes.byref(h)) == 0
    assert emu.gms_multisplit_allocate(h, n, 0) == 0
    return h


def _host_starts(emu, h, keys, B):  # noqa: F811
    kout, offs = np.zeros_like(keys), np.full(B, 77, np.uint32)
    assert emu.gms_multisplit_key_only(h, p(keys), p(kout), keys.size, gms.range_bucket(B).desc(),
                                       p(offs), None) == 0
    wk, _, wo = oracle.multisplit(keys, B, oracle.RANGE, 0, None)
    np.testing.assert_array_equal(kout, wk)
    np.testing.assert_array_equal(offs, wo)


@pytest.fixture
def refuse(emu):  # noqa: F811
    emu.gms_emu_refuse_pinned.argtypes = [ctypes.c_uint32]
    yield emu.gms_emu_refuse_pinned
    emu.gms_emu_refuse_pinned(0)


def test_refused_pinned_memory_falls_back_to_the_copy(emu, refuse):  # noqa: F811
    refuse(1000)
    for B in (2, 64, 1024):
        keys = W.uniform_keys(3000, seed=B)
        h = _multisplit_ctx(emu, B, keys.size)
        for _ in range(2):
            _host_starts(emu, h, keys, B)
        emu.gms_multisplit_destroy(h)
    keys = W.uniform_keys(3000, seed=3)
    kout, count = np.zeros_like(keys), ctypes.c_uint32(7)
    h = ctypes.c_void_p()
    assert emu.gms_compaction_create(ctypes.byref(h)) == 0
    assert emu.gms_compaction_allocate(h, keys.size, 0) == 0
    d = gms.delta_func(1 << 31).desc()
    assert emu.gms_compaction(h, p(keys), None, p(kout), None, keys.size, d,
                              ctypes.addressof(count), None, None) == 0
    emu.gms_compaction_destroy(h)
    kept = keys[keys < np.uint32(1 << 31)]
    assert count.value == kept.size
    np.testing.assert_array_equal(kout[:kept.size], kept)


def test_calls_with_host_results_allocate_nothing(emu):  # noqa: F811
    """Allocations belong to *_allocate: another thread may be capturing a graph
    while a call runs."""
    emu.gms_emu_alloc_calls.restype = ctypes.c_uint64
    keys = W.uniform_keys(3000, seed=1)
    for _ in range(2):
        h = _multisplit_ctx(emu, 64, keys.size)
        before = emu.gms_emu_alloc_calls()
        for _ in range(2):
            _host_starts(emu, h, keys, 64)
        assert emu.gms_emu_alloc_calls() == before
        emu.gms_multisplit_destroy(h)
    kout, count = np.zeros_like(keys), ctypes.c_uint32(7)
    h = ctypes.c_void_p()
    assert emu.gms_compaction_create(ctypes.byref(h)) == 0
    assert emu.gms_compaction_allocate(h, keys.size, 0) == 0
    before = emu.gms_emu_alloc_calls()
    assert emu.gms_compaction(h, p(keys), None, p(kout), None, keys.size, gms.delta_func(1 << 31).desc(),
                              ctypes.addressof(count), None, None) == 0
    assert emu.gms_emu_alloc_calls() == before
    emu.gms_compaction_destroy(h)
    assert count.value == np.count_nonzero(keys < np.uint32(1 << 31))


def test_refused_pinned_memory_is_asked_for_once(emu, refuse):  # noqa: F811
    """Calls do not ask again; a context allocated after the last one of the
    device was released does, and contexts that outlive others keep their
    results."""
    emu.gms_emu_alloc_calls.restype = ctypes.c_uint64
    keys = W.uniform_keys(3000, seed=5)
    refuse(1)
    h = _multisplit_ctx(emu, 64, keys.size)
    before = emu.gms_emu_alloc_calls()
    for _ in range(3):
        _host_starts(emu, h, keys, 64)
    assert emu.gms_emu_alloc_calls() == before
    emu.gms_multisplit_destroy(h)
    a, b = _multisplit_ctx(emu, 64, keys.size), _multisplit_ctx(emu, 8, keys.size)
    _host_starts(emu, a, keys, 64)
    _host_starts(emu, b, keys, 8)
    assert emu.gms_multisplit_allocate(a, 2 * keys.size, 0) == 0  # anew: its slot goes back
    _host_starts(emu, a, keys, 64)
    emu.gms_multisplit_destroy(a)
    _host_starts(emu, b, keys, 8)
    emu.gms_multisplit_release(b)
    emu.gms_multisplit_release(b)  # twice is harmless
    emu.gms_multisplit_destroy(b)
