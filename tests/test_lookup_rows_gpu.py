"""find over row sizes, output addresses and batch sizes: the rows of keys that are present come back
byte for byte, everything else in the output buffer stays as it was."""
import numpy as np
import pytest
import torch

import workloads as w
from gpu_util import DEV, dev
from hierarchicalkv_amd import HashTable, default_options

pytestmark = pytest.mark.gpu
PAD = 64


# rows below 16 bytes (units of 1, 2, 4, 8), at and around 16, with a last unit that overlaps, of 512
# bytes and more (one key per tile); addresses off by nothing, by 4, by 1; batches at the edges of a
# tile's and a wavefront's keys and where the keys per tile change (2^14)
@pytest.mark.parametrize("row_bytes,shift", [
    (1, 0), (2, 0), (3, 1), (5, 0), (7, 1), (8, 0), (12, 4), (15, 0), (16, 0), (16, 4), (17, 0), (31, 1), (32, 1), (66, 0),
    (200, 4), (256, 0), (512, 0), (516, 0), (1028, 1), (4100, 0)])
def test_rows_of_every_size(row_bytes, shift):
    check(row_bytes, shift, 1 << 34, (1, 2, 7, 8, 9, 15, 16, 17, 63, 65, 1000, 16384, 16385, 16400))


# the other form of the row copy: no row in HBM (where a miss must not reach over the host link), and half of them;
# 2^14 and 2^14 + 1 keys are one and two per tile
@pytest.mark.parametrize("hbm_share", [0, 0.5])
@pytest.mark.parametrize("row_bytes,shift", [
    (1, 0), (2, 1), (3, 0), (6, 0), (12, 1), (15, 0), (16, 0), (17, 4), (40, 0), (66, 1), (256, 4), (516, 0), (1030, 1)])
def test_rows_in_host_memory(row_bytes, shift, hbm_share):
    check(row_bytes, shift, int((1 << 15) * row_bytes * hbm_share), (1, 9, 65, 1000, 16384, 16385))


# no key found, few, half of them, nearly all and all: the copy's list of found keys at its edges, for rows of less
# than a unit's 16 bytes, of a part of a wavefront's step of 1024 bytes, of one step and of more; the missed-keys
# form too.  A quarter missed: wavefronts on both sides of the line where misses are listed as well; rows of 383 and 384
# bytes: two keys and one per tile
@pytest.mark.parametrize("missed_form", [False, True])
@pytest.mark.parametrize("row_bytes", [4, 12, 16, 40, 64, 256, 383, 384, 512, 1024, 1040, 4096])
def test_any_share_of_hits(row_bytes, missed_form):
    for miss_share in (1.0, 0.97, 0.5, 0.25, 0.03, 0.0):
        check(row_bytes, 0, 1 << 34, (1, 8, 17, 65, 1000, 16385), miss_share, missed_form)


def check(row_bytes, shift, hbm, sizes, miss_share=0.2, missed_form=False):
    cap, resident = 1 << 15, 20000
    t = HashTable()
    t.init(default_options(init_capacity=cap, max_capacity=cap, max_hbm_for_vectors=hbm, dim=row_bytes,
                           value_kind=0, value_size=1))
    assert t.is_pure_hbm() == (hbm >= cap * row_bytes)
    keys = w.unique_keys(61, 0, resident)
    rng = np.random.Generator(np.random.PCG64(row_bytes))
    rows = rng.integers(0, 256, (resident, row_bytes), dtype=np.uint8)
    t.insert_or_assign(resident, dev(keys), dev(rows))
    assert t.size() == resident
    absent = w.unique_keys(62, 0, 3000)
    for n in sizes:
        if n > 1000 and row_bytes > 2000:
            continue
        pick = rng.integers(0, resident, n)
        miss = rng.random(n) < miss_share
        q = np.where(miss, absent[np.arange(n) % len(absent)], keys[pick])
        buf = torch.full((PAD + shift + n * row_bytes + PAD,), 0xA5, dtype=torch.uint8, device=DEV)
        founds = torch.zeros(n, dtype=torch.bool, device=DEV)
        d_q = dev(q)
        if missed_form:
            mk, mi = torch.zeros(n, dtype=torch.int64, device=DEV), torch.zeros(n, dtype=torch.int32, device=DEV)
            ms = torch.zeros(1, dtype=torch.int32, device=DEV)
            t.find_missed(n, d_q, buf[PAD + shift:], mk, mi, ms)
            count = int(ms.item())
            where = np.sort(mi[:count].cpu().numpy())
            assert (where == np.flatnonzero(miss)).all()
            assert (mk[:count] == d_q[mi[:count].long()]).all()
        else:
            t.find(n, d_q, buf[PAD + shift:], founds)
            torch.cuda.synchronize()
            assert (founds.cpu().numpy() == ~miss).all()
        got = buf.cpu().numpy()
        body = got[PAD + shift:PAD + shift + n * row_bytes].reshape(n, row_bytes)
        assert (body[~miss] == rows[pick[~miss]]).all()
        assert (body[miss] == 0xA5).all()
        assert (got[:PAD + shift] == 0xA5).all() and (got[PAD + shift + n * row_bytes:] == 0xA5).all()
    t.close()


# more keys than one launch takes at two keys per tile (2^29); at 2^30 a single one would have 2^32 threads
@pytest.mark.parametrize("call", ["contains", "find_ptr", "find"])
def test_more_than_2_30_keys(call):
    part, n = 1 << 20, (1 << 30) + 4097
    t = HashTable()
    t.init(default_options(init_capacity=1 << 20, max_capacity=1 << 20, max_hbm_for_vectors=1 << 30, dim=1))
    universe = dev(w.unique_keys(63, 0, part))
    rows = torch.arange(part, dtype=torch.float32, device=DEV)
    t.insert_or_assign(part // 4, universe, rows)
    there = torch.arange(part, device=DEV) < part // 4
    keys = universe.repeat(n // part + 1)[:n]
    founds = torch.zeros(n, dtype=torch.bool, device=DEV)
    out = torch.full((n,), -1, dtype=torch.int64 if call == "find_ptr" else torch.int32, device=DEV)
    if call == "contains":
        t.contains(n, keys, founds)
        want = out[:part]
    elif call == "find":
        t.find(n, keys, out, founds)
        want = torch.where(there, rows.view(torch.int32), -1)
    else:
        t.find_ptr(n, keys, out, founds)
        want = torch.zeros(part, dtype=torch.int64, device=DEV)
        t.find_ptr(part, universe, want, torch.zeros(part, dtype=torch.bool, device=DEV))
        assert torch.equal(want != 0, there)
    for lo in range(0, n, part):
        m = min(part, n - lo)
        if not (torch.equal(founds[lo:lo + m], there[:m]) and torch.equal(out[lo:lo + m], want[:m])):
            raise AssertionError(f"keys {lo} to {lo + m}")
    t.close()
