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
# keys from one (all repetitions of one word) to about all; rows of 256, 10 and 3 bytes (16-byte,
# 2-byte and single-byte copies)
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
