"""The upserts at the batch sizes where their kernels change: the keys of a tile and of a wavefront,
and the sizes up to which a tile takes one or two keys.  Half of a batch is new and half was
written recently, so nothing depends on the order within the batch; the oracle has every answer."""
import numpy as np
import pytest
import torch

import workloads as w
from gpu_util import DEV, assert_same_table, dev, host_bytes, host_u64
from hierarchicalkv_amd import HashTable, default_options

pytestmark = pytest.mark.gpu


def bytes_of(a):
    return np.ascontiguousarray(a).view(np.uint8).reshape(len(a), -1)


# full tables (victims through the score bounds; one key per tile up to 2^15 keys, two up to 2^18) and
# tables with free slots (2^14, 2^17); rows of 36 and 40 bytes: accum_or_assign adds them in units of 4 and 8
@pytest.mark.parametrize("full,cap_bits,dim,sizes", [
    (True, 14, 9, (1, 9, 65, 1000)),
    (True, 14, 10, (1, 9, 65, 1000)),
    (True, 18, 8, (1, 7, 8, 9, 16, 17, 65, 1 << 15, (1 << 15) + 1)),
    (True, 21, 8, (1 << 18, (1 << 18) + 1)),
    # up to 2^16 keys two per tile are at most four wavefronts per SIMD, above that more; rows of 12 and 256 bytes, and longer ones
    (True, 19, 3, (1 << 16, (1 << 16) + 1)),
    (True, 19, 64, (1 << 16, (1 << 16) + 1)),
    (True, 19, 65, (1 << 16, (1 << 16) + 1)),
    (False, 18, 8, (1, 8, 9, 17, 1 << 14, (1 << 14) + 1)),
    (False, 21, 8, (1 << 17, (1 << 17) + 1)),
])
def test_every_upsert_at_the_edges(oracle, full, cap_bits, dim, sizes):
    cap = 1 << cap_bits
    o = default_options(init_capacity=cap, max_capacity=cap, max_hbm_for_vectors=1 << 30, dim=dim)
    t = HashTable()
    t.init(o)
    ot = oracle.OracleTable(o)
    t.set_clock(1, 1 << 44)
    ot.set_clock(1, 1 << 44)
    at = 0

    def new_keys(n):
        nonlocal at
        at += n
        return w.unique_keys(90, at - n, n)

    rng = np.random.default_rng(cap_bits)
    fill = cap + cap // 4 if full else cap // 4
    while at < fill:
        keys = new_keys(cap // 8)
        rows = rng.random((len(keys), dim), dtype=np.float32)
        t.insert_or_assign(len(keys), dev(keys), dev(rows))
        ot.insert_or_assign_mt(keys, bytes_of(rows), None)
    assert_same_table(t, ot, dim * 4)
    recent = keys
    for n in sizes:
        for op in ("insert_or_assign", "find_or_insert", "accum_or_assign", "insert_and_evict"):
            hits = rng.choice(recent, n // 2, replace=False)
            keys = np.concatenate([hits, new_keys(n - n // 2)])
            is_hit = np.arange(n) < n // 2
            order = rng.permutation(n)
            keys, is_hit = keys[order], is_hit[order]
            rows = rng.random((n, dim), dtype=np.float32)
            dk, dv = dev(keys), dev(rows)
            if op == "insert_or_assign":
                t.insert_or_assign(n, dk, dv)
                ot.insert_or_assign(keys, bytes_of(rows), None)
            elif op == "find_or_insert":
                t.find_or_insert(n, dk, dv)
                want = bytes_of(rows).copy()
                ot.find_or_insert(keys, want, None)
                assert (host_bytes(dv, n, dim * 4) == want).all(), (n, op)
            elif op == "accum_or_assign":
                t.accum_or_assign(n, dk, dv, dev(is_hit))
                ot.accum_or_assign(keys, bytes_of(rows), is_hit.astype(np.uint8), None)
            else:
                ek = torch.zeros(n, dtype=torch.int64, device=DEV)
                ev = torch.zeros(n, dim, dtype=torch.float32, device=DEV)
                es = torch.zeros(n, dtype=torch.int64, device=DEV)
                gone = t.insert_and_evict(n, dk, dv, None, ek, ev, es)
                wk, wv, ws = ot.insert_and_evict(keys, bytes_of(rows), None)[:3]
                assert gone == len(wk), (n, op)
                a, b = np.argsort(host_u64(ek)[:gone]), np.argsort(wk)
                assert (host_u64(ek)[:gone][a] == wk[b]).all(), (n, op)
                assert (host_bytes(ev, n, dim * 4)[:gone][a] == wv[b]).all(), (n, op)
                assert (host_u64(es)[:gone][a] == ws[b]).all(), (n, op)
            assert t.size() == ot.size(), (n, op)
        assert_same_table(t, ot, dim * 4)
    t.close()
