"""Many keys of one call in every bucket, as in test_contention_gpu.py, at the sizes where the upserts take two
and eight keys per tile, and where a call brings so many keys per bucket that the victims are searched by
the scan again.  The outcome depends on the order in which the keys get their turn; what must hold in any
order is checked on the device after every call (see check())."""
import os

import pytest
import torch

import workloads_device as wd
from gpu_util import DEV
from hierarchicalkv_amd import EvictStrategy, HashTable, Predicate, default_options
from test_score_bounds_gpu import bounds_hold

pytestmark = pytest.mark.gpu
LRU, LFU, ELRU, ELFU, CUSTOM = (EvictStrategy.kLru, EvictStrategy.kLfu, EvictStrategy.kEpochLru,
                                EvictStrategy.kEpochLfu, EvictStrategy.kCustomized)


class Model:
    """The keys a table may hold and what is known of each: whether it is in, and which write its row is from."""

    def __init__(self, seed, cap, dim):
        self.cap, self.dim = cap, dim
        self.keys = torch.sort(wd.dev_keys(seed, 0, 2 * cap)).values
        self.resident = torch.zeros(2 * cap, dtype=torch.bool, device=DEV)
        self.write = torch.full((2 * cap,), -1, dtype=torch.int64, device=DEV)  # -1: not known
        self.out = [torch.zeros(cap, dtype=torch.int64, device=DEV), torch.zeros(cap, dim, device=DEV),
                    torch.zeros(cap, dtype=torch.int64, device=DEV), torch.zeros(1, dtype=torch.int64, device=DEV)]

    def rows(self, which, write):
        return ((which * 31 + write * 7919)[:, None] + torch.arange(self.dim, device=DEV)).bitwise_and(0xFFFFF).float()

    def index(self, keys):
        i = torch.searchsorted(self.keys, keys).clamp(max=len(self.keys) - 1)
        assert bool((self.keys[i] == keys).all())
        return i

    def check(self, t, batch, upsert, all_in, erased=None, evicted=None):
        """No key is in the table twice; the table holds nothing but keys it held before and keys of the call;
        under LRU (`all_in`) every key of the call; erase removes exactly its keys; insert_and_evict hands back
        every key that left, once, and every key of the call that did not get in; a key whose last write is
        known carries that row."""
        k, v, s, c = self.out
        t.export_batch_if(Predicate.kAlways, 0, 0, self.cap, 0, c, k, v, s)
        m = int(c.item())
        at = self.index(k[:m])
        now = torch.zeros_like(self.resident)
        now[at] = True
        assert int(now.sum()) == m == t.size() <= self.cap
        mine = torch.zeros_like(now)
        mine[batch] = True
        if erased is not None:
            assert torch.equal(now, self.resident & ~mine)
        elif not upsert:
            assert torch.equal(now, self.resident)
        else:
            assert not bool((now & ~self.resident & ~mine).any())
            if all_in:
                assert bool(now[batch].all())
        if evicted is not None:
            gone = self.index(evicted)
            left = gone[~mine[gone]]
            out = torch.zeros_like(now)
            out[left] = True
            assert int(out.sum()) == len(left) and bool(self.resident[left].all())
            assert torch.equal(now & ~mine, self.resident & ~mine & ~out)
            out[gone] = True
            assert bool(out[mine & ~now].all())
        self.resident = now
        known = self.write[at] >= 0
        assert torch.equal(v[:m][known], self.rows(at[known], self.write[at[known]]))


def run(strategy, cap, n, dim, hybrid=False, steps=7):
    buckets = cap // 128
    t = HashTable()
    t.init(default_options(init_capacity=cap, max_capacity=cap, dim=dim, evict_strategy=strategy,
                           max_hbm_for_vectors=cap * dim if hybrid else 1 << 34))
    assert t.is_pure_hbm() != hybrid
    if strategy in (ELRU, ELFU):
        t.set_global_epoch(5)
    from_clock = strategy in (LRU, ELRU)
    gen = torch.Generator(device=DEV)
    gen.manual_seed(cap + n + int(strategy))
    m = Model(500 + int(strategy), cap, dim)
    at, write = 0, 0
    order = torch.randperm(2 * cap, device=DEV, generator=gen)
    while at < cap * 5 // 4:  # past load factor 1.0
        batch = order[at:at + min(n, cap // 8)]
        sc = None if from_clock else torch.randint(1, 1 << 20, (len(batch),), device=DEV, generator=gen)
        t.insert_or_assign(len(batch), m.keys[batch], m.rows(batch, torch.zeros_like(batch)), sc)
        m.write[batch] = 0
        at += len(batch)
    t.contains(len(m.keys), m.keys, m.resident)
    ops = ["insert_or_assign", "find_or_insert", "accum_or_assign"] + ([] if hybrid else ["insert_and_evict"])
    crowded = n > (32 if strategy == LRU else 48) * buckets
    for step in range(steps):
        op = ops[step % len(ops)] if step != 4 else "erase"
        size = n // 8 if op == "erase" else n
        batch = torch.randperm(2 * cap, device=DEV, generator=gen)[:size]
        keys = m.keys[batch]
        sc = None if from_clock else torch.randint(1, 1 << (4, 20, 40)[step % 3], (size,), device=DEV, generator=gen)
        write += 1
        rows = m.rows(batch, torch.full_like(batch, write))
        gone = None
        if op == "insert_or_assign":
            t.insert_or_assign(size, keys, rows, sc)
            m.write[batch] = write
        elif op == "insert_and_evict":
            ek, ev, es = torch.zeros_like(keys), torch.zeros_like(rows), torch.zeros_like(keys)
            gone = ek[:t.insert_and_evict(size, keys, rows, sc, ek, ev, es)]
            m.write[batch] = write
        elif op == "find_or_insert":
            t.find_or_insert(size, keys, rows, sc)
            m.write[batch] = -1
        elif op == "accum_or_assign":
            t.accum_or_assign(size, keys, rows, torch.rand(size, device=DEV, generator=gen) < 0.5, sc)
            m.write[batch] = -1
        else:
            t.erase(size, keys)
            m.write[batch] = -1
        m.check(t, batch, op != "erase", strategy == LRU and op != "accum_or_assign", op == "erase" or None, gone)
        bounded = os.environ.get("HKV_SCORE_BOUNDS") != "0" and op != "erase" and (strategy == LRU or not crowded)
        if bounded and (strategy != CUSTOM or dim % 4 == 0):
            ok, bad, _ = bounds_hold(t)
            assert ok, (step, op, bad)
    t.close()


# some nine keys of a call per bucket: the searches through the bounds, with two tries in a trip where tiles have
# two keys and with one where they have eight, which make two with five keys per bucket; rows of 16 bytes and of 36
# (whose units overlap)
@pytest.mark.parametrize("strategy,dim", [(LRU, 4), (LRU, 9), (ELRU, 9), (CUSTOM, 4), (CUSTOM, 9), (LFU, 4), (ELFU, 9)])
@pytest.mark.parametrize("cap,n", [(1 << 19, 40000), (1 << 22, (1 << 18) + 33000), (1 << 23, (1 << 18) + 33000)],
                         ids=["two-per-tile", "eight-per-tile", "eight-per-tile-two-tries"])
def test_bounded_searches(cap, n, strategy, dim):
    run(strategy, cap, n, dim)


# 37 to 62 keys of a call per bucket: LRU takes the scan, the others one try per trip
@pytest.mark.parametrize("strategy,dim", [(LRU, 4), (LRU, 9), (ELRU, 4), (CUSTOM, 4), (LFU, 9)])
@pytest.mark.parametrize("cap,n", [(1 << 13, 4000), (1 << 17, 40000), (1 << 20, 300000)],
                         ids=["one-per-tile", "two-per-tile", "eight-per-tile"])
def test_crowded_buckets(cap, n, strategy, dim):
    run(strategy, cap, n, dim)


# a quarter of the rows in HBM: insert_or_assign and find_or_insert hold their slots to the end of the launch
@pytest.mark.parametrize("strategy,dim", [(LRU, 4), (CUSTOM, 4), (LFU, 9)])
@pytest.mark.parametrize("cap,n", [(1 << 19, 40000), (1 << 22, (1 << 18) + 33000)], ids=["two-per-tile", "eight-per-tile"])
def test_held_slots(cap, n, strategy, dim):
    run(strategy, cap, n, dim, hybrid=True)
