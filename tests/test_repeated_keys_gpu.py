"""Batches that repeat keys (unique_key=False): every occurrence gets what the first one gets, the
table holds each key once.  Expected values are worked out here with numpy."""
import numpy as np
import pytest
import torch

import workloads as w
from gpu_util import DEV, dev, export_table, sort_by_key
from hierarchicalkv_amd import HashTable, default_options

pytestmark = pytest.mark.gpu
RESERVED = np.uint64(0xFFFFFFFFFFFFFFFF)


# batch sizes at the edges of a workgroup's 1024 keys and of the 64 keys of a wavefront; distinct
# keys from one (all repetitions of one word) to about all; rows of 256 and 16 bytes (copies in
# units of 16 bytes), of 40 (units of 4), of 10 and 3 (single bytes)
@pytest.mark.parametrize("n,distinct,value_size,dim", [
    (2, 1, 4, 64), (63, 7, 2, 5), (64, 64, 4, 64), (1023, 1, 1, 3), (1024, 300, 4, 64), (1025, 1024, 2, 5),
    (4097, 2, 4, 10), (50001, 20000, 4, 64), (262144, 1000, 4, 4),
])
def test_first_occurrence_stands_for_the_key(n, distinct, value_size, dim):
    cap = 1 << 18
    t = HashTable()
    t.init(default_options(init_capacity=cap, max_capacity=cap, max_hbm_for_vectors=1 << 32, dim=dim,
                           value_kind=0, value_size=value_size))
    vb = dim * value_size
    rng = np.random.Generator(np.random.PCG64(n + distinct))
    universe = w.unique_keys(41, n, distinct)
    known = universe[:distinct // 3]
    rows0 = rng.integers(0, 256, (len(known), vb), dtype=np.uint8)
    if len(known):
        t.insert_or_assign(len(known), dev(known), dev(rows0))
    keys = universe[rng.integers(0, distinct, n)]
    keys[n // 2] = RESERVED
    rows = rng.integers(0, 256, (n, vb), dtype=np.uint8)

    want, first, table = rows.copy(), {}, {int(k): r for k, r in zip(known, rows0)}
    for i, k in enumerate(keys):
        if k == RESERVED:
            continue
        i0 = first.setdefault(int(k), i)
        want[i] = table.setdefault(int(k), rows[i0])

    d_keys, d_rows = dev(keys), dev(rows)
    t.find_or_insert(n, d_keys, d_rows, unique_key=False)
    torch.cuda.synchronize()
    assert (d_rows.cpu().numpy() == want).all()
    gk, gv, _ = sort_by_key(*export_table(t, vb, chunk=cap))
    assert gk.tolist() == sorted(table)
    assert (gv == np.stack([table[int(k)] for k in gk])).all()

    # insert_or_assign leaves the first occurrence's row
    rows2 = rng.integers(0, 256, (n, vb), dtype=np.uint8)
    t.insert_or_assign(n, d_keys, dev(rows2), unique_key=False)
    for k, i0 in first.items():
        table[k] = rows2[i0]
    gk, gv, _ = sort_by_key(*export_table(t, vb, chunk=cap))
    assert gk.tolist() == sorted(table)
    assert (gv == np.stack([table[int(k)] for k in gk])).all()

    ptrs = torch.zeros(n, dtype=torch.int64, device=DEV)
    founds = torch.zeros(n, dtype=torch.bool, device=DEV)
    t.find_or_insert_ptr(n, d_keys, ptrs, founds, unique_key=False)
    torch.cuda.synchronize()
    p, f = ptrs.cpu().numpy(), founds.cpu().numpy()
    live = keys != RESERVED
    assert f[live].all()
    at = {}
    for k, q in zip(keys[live], p[live]):
        assert at.setdefault(int(k), q) == q
    assert len(set(at.values())) == len(first)
    t.close()


# rows of 4 GiB in units of one byte and of 16 GiB in units of four: as many units as a launch may not have threads
@pytest.mark.parametrize("n,value_size,dim", [(1 << 22, 1, 1026), (1 << 24, 4, 257)])
def test_rows_of_many_gigabytes(n, value_size, dim):
    cap, distinct, vb = 1 << 13, 3001, dim * value_size
    assert n * vb // (4 if vb % 4 == 0 else 1) >= 1 << 32
    t = HashTable()
    t.init(default_options(init_capacity=cap, max_capacity=cap, max_hbm_for_vectors=1 << 32, dim=dim,
                           value_kind=0, value_size=value_size))
    rng = np.random.default_rng(dim)
    universe = w.unique_keys(43, 0, distinct)
    pick = rng.integers(0, distinct, n)
    seen, at = np.unique(pick, return_index=True)
    first = np.zeros(distinct, np.int64)
    first[seen] = at
    given = torch.empty(n, vb // 2, dtype=torch.int16, device=DEV).random_()
    rows = given.clone()
    keys, source = dev(universe[pick]), dev(first[pick])
    t.find_or_insert(n, keys, rows, unique_key=False)
    assert t.size() == len(seen)
    for lo in range(0, n, 1 << 20):
        assert torch.equal(rows[lo:lo + (1 << 20)], given[source[lo:lo + (1 << 20)]]), lo
    t.close()
