"""The upserts over row sizes and caller addresses, on a table with free slots and on a full one: every
row of the table is the oracle's byte for byte, and nothing is written beside a caller's rows."""
import numpy as np
import pytest
import torch

import workloads as w
from gpu_util import DEV, assert_same_table, dev, host_u64
from hierarchicalkv_amd import HashTable, default_options

pytestmark = pytest.mark.gpu
PAD = 64


def placed(rows, shift):
    """the rows in device memory, `shift` bytes off a 64-byte boundary, between guard bytes"""
    buf = torch.full((PAD + shift + rows.size + PAD,), 0xA5, dtype=torch.uint8, device=DEV)
    buf[PAD + shift:PAD + shift + rows.size] = dev(rows.reshape(-1))
    return buf, buf[PAD + shift:]


def body(buf, shift, n, vb):
    got = buf.cpu().numpy()
    assert (got[:PAD + shift] == 0xA5).all() and (got[PAD + shift + n * vb:] == 0xA5).all()
    return got[PAD + shift:PAD + shift + n * vb].reshape(n, vb)


# units of 1, 2, 4 and 8 bytes; 16 and around it; last units that overlap; the edges of one, two, four
# and eight units per lane (128, 256, 512, 1024 bytes); addresses off by nothing, by 4, by 1
@pytest.mark.parametrize("row_bytes,shift", [
    (1, 0), (2, 1), (3, 0), (4, 0), (6, 1), (8, 4), (12, 0), (15, 1), (16, 0), (16, 1), (17, 0), (40, 0), (66, 1), (128, 4),
    (132, 0), (200, 0), (256, 0), (260, 4), (512, 1), (516, 0), (1024, 0), (1030, 0), (2100, 1)])
def test_rows_of_every_size(oracle, row_bytes, shift):
    check(oracle, row_bytes, shift, 1 << 30)


# no row in HBM and half of them: unaligned units to and from host memory, slots held to the end of the launch
@pytest.mark.parametrize("hbm_share", [0, 0.5])
@pytest.mark.parametrize("row_bytes,shift", [
    (1, 0), (2, 1), (3, 0), (6, 1), (12, 0), (15, 1), (16, 0), (17, 4), (40, 0), (66, 1), (200, 0), (260, 4), (516, 1), (1030, 0)])
def test_rows_in_host_memory(oracle, row_bytes, shift, hbm_share):
    check(oracle, row_bytes, shift, int((1 << 13) * row_bytes * hbm_share))


def check(oracle, row_bytes, shift, hbm):
    cap = 1 << 13
    hybrid = hbm < cap * row_bytes
    o = default_options(init_capacity=cap, max_capacity=cap, max_hbm_for_vectors=hbm, dim=row_bytes,
                        value_kind=0, value_size=1)
    t = HashTable()
    t.init(o)
    assert t.is_pure_hbm() != hybrid
    ot = oracle.OracleTable(o, hybrid)
    t.set_clock(1, 1 << 44)
    ot.set_clock(1, 1 << 44)
    rng = np.random.default_rng(row_bytes * 8 + shift)
    at, n = 0, 1003
    recent = np.zeros(0, np.uint64)
    # new keys come in over free slots first and evict later on; hits are keys of the last batch
    for step in range(18):
        n_hit = n // 2 if len(recent) else 0
        fresh = w.unique_keys(95, at, n - n_hit)
        at += n - n_hit
        keys = rng.permutation(np.concatenate([rng.choice(recent, n_hit, replace=False) if n_hit else recent, fresh]))
        rows = rng.integers(0, 256, (n, row_bytes), dtype=np.uint8)
        buf, dv = placed(rows, shift)
        op = ("insert_or_assign", "find_or_insert", "insert_and_evict")[step % 3]
        if hybrid and op == "insert_and_evict":  # (pure HBM only)
            op = "insert_or_assign"
        if op == "insert_or_assign":
            t.insert_or_assign(n, dev(keys), dv)
            ot.insert_or_assign(keys, rows, None)
        elif op == "find_or_insert":
            t.find_or_insert(n, dev(keys), dv)
            ot.find_or_insert(keys, rows, None)
        else:
            ek = torch.zeros(n, dtype=torch.int64, device=DEV)
            ebuf, ev = placed(np.full((n, row_bytes), 0xA5, np.uint8), shift)
            gone = t.insert_and_evict(n, dev(keys), dv, None, ek, ev, None)
            wk, wv, _ = ot.insert_and_evict(keys, rows, None)
            assert gone == len(wk)
            a, b = np.argsort(host_u64(ek)[:gone]), np.argsort(wk)
            assert (host_u64(ek)[:gone][a] == wk[b]).all()
            assert (body(ebuf, shift, gone, row_bytes)[a] == wv[b]).all()
        assert (body(buf, shift, n, row_bytes) == rows).all()  # find_or_insert: with the table's rows
        recent = fresh
    assert ot.size() > cap * 9 // 10
    assert_same_table(t, ot, row_bytes)
    t.close()
