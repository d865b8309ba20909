"""A table that was created with an allocator takes all memory that it keeps from it."""
import ctypes as C

import numpy as np
import pytest
import torch

import workloads as w
from gpu_util import dev, hip
from hierarchicalkv_amd import HashTable, default_options
from hierarchicalkv_amd import table as table_module
from hierarchicalkv_amd._capi import lib

pytestmark = pytest.mark.gpu
ALLOC = C.CFUNCTYPE(C.c_int, C.c_void_p, C.c_int, C.POINTER(C.c_void_p), C.c_size_t)
FREE = C.CFUNCTYPE(C.c_int, C.c_void_p, C.c_int, C.c_void_p)


class Allocator(C.Structure):
    _fields_ = [("ctx", C.c_void_p), ("alloc", ALLOC), ("free", FREE)]


class Counting:
    """hipMalloc and hipHostMalloc with a count of what is out; blocks of `refuse_from` bytes and more are refused."""

    def __init__(self):
        self.out, self.refuse_from = {}, None
        self.struct = Allocator(None, ALLOC(self._alloc), FREE(self._free))

    def _alloc(self, _ctx, kind, where, size):
        if self.refuse_from is not None and size >= self.refuse_from:
            return 1
        p = C.c_void_p()
        h = hip()
        rc = (h.hipMalloc(C.byref(p), C.c_size_t(size)) if kind == 0 else
              h.hipHostMalloc(C.byref(p), C.c_size_t(size), 3))  # portable, mapped
        if rc == 0:
            where[0] = p.value
            self.out[p.value] = (kind, size)
        return rc

    def _free(self, _ctx, kind, p):
        assert self.out.pop(p)[0] == kind
        return hip().hipFree(C.c_void_p(p)) if kind == 0 else hip().hipHostFree(C.c_void_p(p))

    def device_bytes(self):
        return sum(size for kind, size in self.out.values() if kind == 0)

    def table(self, **kw):
        t = HashTable()
        h = C.c_void_p()
        table_module._check(lib.hkv_table_create_with_allocator(C.byref(default_options(**kw)), C.byref(self.struct),
                                                                C.byref(h)))
        t._h = h
        return t


def pool_bytes():
    """What is in use of the device's stream-ordered pool."""
    torch.cuda.synchronize()
    pool, used = C.c_void_p(), C.c_uint64()
    assert hip().hipDeviceGetDefaultMemPool(C.byref(pool), 0) == 0
    assert hip().hipMemPoolGetAttribute(pool, 7, C.byref(used)) == 0  # hipMemPoolAttrUsedMemCurrent
    return used.value


def repeated_calls(t, sizes, ids=1000):
    universe = w.unique_keys(71, 0, ids)
    rng = np.random.default_rng(5)
    for n in sizes:
        keys = universe[rng.integers(0, len(universe), n)]
        rows = dev(w.values_from_keys(keys, 4))
        t.insert_or_assign(n, dev(keys), rows, unique_key=False)
        torch.cuda.synchronize()
        rows.zero_()
        torch.cuda.synchronize()
        t.find_or_insert(n, dev(keys), rows, unique_key=False)
        torch.cuda.synchronize()
        assert np.array_equal(rows.cpu().numpy(), w.values_from_keys(keys, 4))


def test_index_of_repeated_keys_comes_from_the_allocator():
    cap = 1 << 18
    c = Counting()
    t = c.table(init_capacity=cap, max_capacity=cap, max_hbm_for_vectors=1 << 30, dim=4)
    table_bytes, blocks, before = c.device_bytes(), len(c.out), pool_bytes()
    for n in (5000, 3000, 70000, 100000):  # grows twice
        repeated_calls(t, (n, n))
        assert pool_bytes() == before
        assert c.device_bytes() >= table_bytes + 4 * 8 * n
        assert len(c.out) == blocks + 1
    t.close()
    assert not c.out


def test_calls_go_on_where_the_allocator_has_no_room_for_the_index():
    cap = 1 << 18
    c = Counting()
    t = c.table(init_capacity=cap, max_capacity=cap, max_hbm_for_vectors=1 << 30, dim=4)
    blocks = len(c.out)
    repeated_calls(t, (3000,))
    assert len(c.out) == blocks + 1
    c.refuse_from = 4 * 8 * 50000
    repeated_calls(t, (50000, 50000))
    assert len(c.out) == blocks
    repeated_calls(t, (3000,))
    assert len(c.out) == blocks + 1
    c.refuse_from = None
    repeated_calls(t, (50000, 3000))
    assert len(c.out) == blocks + 1
    t.close()
    assert not c.out


def test_a_small_table_keeps_a_small_index():
    for slots in (1 << 10, 3 << 9):
        c = Counting()
        t = c.table(init_capacity=slots, max_capacity=slots, max_hbm_for_vectors=1 << 30, dim=4)
        slots, table_bytes, before = t.capacity(), c.device_bytes(), pool_bytes()
        for n in (60000, 30, slots, 500, slots + 1):
            repeated_calls(t, (n,), ids=200)  # (far from filling a bucket)
            assert c.device_bytes() <= table_bytes + 68 * slots and pool_bytes() == before
        assert c.device_bytes() > table_bytes
        t.close()
        assert not c.out
