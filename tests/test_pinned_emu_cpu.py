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
