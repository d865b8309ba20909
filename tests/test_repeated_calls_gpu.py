"""Batches that repeat keys, call after call on one table: the index of the batch's keys is the
table's and is not cleared between calls.  Expected values are worked out here with numpy."""
import threading

import numpy as np
import pytest
import torch

import workloads as w
from gpu_util import DEV, dev, export_table, sort_by_key
from hierarchicalkv_amd import HashTable, default_options

pytestmark = pytest.mark.gpu
VB = 16


def make(cap, **kw):
    t = HashTable()
    t.init(default_options(init_capacity=cap, max_capacity=cap, max_hbm_for_vectors=kw.pop("hbm", 1 << 32), dim=4, **kw))
    return t


def check_call(t, model, universe, n, rng, stream=None):
    """One find_or_insert and one insert_or_assign of n keys drawn with repetitions; every occurrence reads
    what the first one reads or brings, and the first one's row stays."""
    pick = rng.integers(0, len(universe), n)
    seen, first = np.unique(pick, return_index=True)
    keys, rows = universe[pick], rng.integers(0, 256, (n, VB), dtype=np.uint8)
    stand = np.empty(len(universe), np.int64)
    stand[seen] = first
    present, stored = model
    want = np.where(present[pick][:, None], stored[pick], rows[stand[pick]])
    d_keys, d_rows = dev(keys), dev(rows)
    torch.cuda.synchronize()
    t.find_or_insert(n, d_keys, d_rows, unique_key=False, stream=stream)
    torch.cuda.synchronize()
    assert (d_rows.cpu().numpy() == want).all(), n
    present[seen] = True
    rows2 = rng.integers(0, 256, (n, VB), dtype=np.uint8)
    d_rows2 = dev(rows2)
    torch.cuda.synchronize()
    t.insert_or_assign(n, d_keys, d_rows2, unique_key=False, stream=stream)
    stored[seen] = rows2[first]
    torch.cuda.synchronize()


def check_table(t, model, universe, cap):
    present, stored = model
    gk, gv, _ = sort_by_key(*export_table(t, VB, chunk=cap))
    o = np.argsort(universe[present])
    assert (gk == universe[present][o]).all() and (gv == stored[present][o]).all()


# sizes that make the index grow, that use a part of it, and that are too long for it to be kept (above 2^21); at 2^15
# the workgroups of the pass change; on two streams the index goes from one to the other
@pytest.mark.parametrize("streams", [1, 2])
def test_index_is_used_again(streams):
    cap = 1 << 18
    t = make(cap)
    rng = np.random.default_rng(streams)
    universe = w.unique_keys(51, 0, 60000)
    model = np.zeros(len(universe), bool), np.zeros((len(universe), VB), np.uint8)
    s = [torch.cuda.Stream() for _ in range(streams)]
    for k, n in enumerate((3, 1 << 12, (1 << 12) + 1, 40, 1 << 15, (1 << 15) - 1, 70000, 5, (1 << 21) + 3, 1 << 15, 300000, 64)):
        check_call(t, model, universe, n, rng, s[k % streams])
    check_table(t, model, universe, cap)
    t.close()


def test_more_calls_than_the_index_can_count():
    cap = 1 << 10
    t = make(cap)
    universe = w.unique_keys(52, 0, 7)
    model = np.zeros(len(universe), bool), np.zeros((len(universe), VB), np.uint8)
    rng = np.random.default_rng(3)
    check_call(t, model, universe, 30, rng)
    keys = dev(universe[[0, 1, 0, 2, 1, 6]])
    rows = dev(np.arange(6 * VB, dtype=np.uint8).reshape(6, VB))
    for _ in range((1 << 16) - 4):  # 65 535 numbers; the next calls see the last of them and the first again
        t.insert_or_assign(6, keys, rows, unique_key=False)
    h = rows.cpu().numpy()
    for k, at in ((0, 0), (1, 1), (2, 3), (6, 5)):
        model[0][k], model[1][k] = True, h[at]
    for n in (30, 6, 64, 1, 2, 17):
        check_call(t, model, universe, n, rng)
    check_table(t, model, universe, cap)
    t.close()


@pytest.mark.parametrize("kw", [{"api_lock": 0}, {"hbm": 0, "io_by_cpu": 1}], ids=["no_group_lock", "io_by_cpu"])
def test_index_that_goes_with_the_call(kw):
    cap = 1 << 14
    t = make(cap, **kw)
    rng = np.random.default_rng(9)
    universe = w.unique_keys(53, 0, 3000)
    model = np.zeros(len(universe), bool), np.zeros((len(universe), VB), np.uint8)
    for n in (2, 5000, 33, 9000):
        check_call(t, model, universe, n, rng)
    check_table(t, model, universe, cap)
    t.close()


def test_recorded_calls_beside_eager_ones():
    """A recorded call runs again with the number it was recorded with, on an index of its own."""
    cap, n = 1 << 14, 5000
    t = make(cap)
    rng = np.random.default_rng(4)
    universe = w.unique_keys(54, 0, 2000)
    model = np.zeros(len(universe), bool), np.zeros((len(universe), VB), np.uint8)
    s = torch.cuda.Stream()
    keys = torch.zeros(n, dtype=torch.int64, device=DEV)
    rows = torch.zeros(n, VB, dtype=torch.uint8, device=DEV)

    def load():
        pick = rng.integers(0, len(universe), n)
        given = rng.integers(0, 256, (n, VB), dtype=np.uint8)
        keys.copy_(dev(universe[pick]))
        rows.copy_(dev(given))
        seen, first = np.unique(pick, return_index=True)
        model[0][seen], model[1][seen] = True, given[first]
        torch.cuda.synchronize()

    with torch.cuda.stream(s):
        check_call(t, model, universe, n, rng)
        load()
        t.insert_or_assign(n, keys, rows, unique_key=False)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            t.insert_or_assign(n, keys, rows, unique_key=False)
        for _ in range(4):
            load()
            g.replay()
            torch.cuda.synchronize()
            check_table(t, model, universe, cap)
            check_call(t, model, universe, 4000, rng)
        check_table(t, model, universe, cap)
    torch.cuda.synchronize()
    t.close()


def check_evict(t, model, universe, n, rng):
    """insert_and_evict where nothing has to leave: the first occurrence's row stays."""
    pick = rng.integers(0, len(universe), n)
    seen, first = np.unique(pick, return_index=True)
    rows = rng.integers(0, 256, (n, VB), dtype=np.uint8)
    ek = torch.full((n,), -1, dtype=torch.int64, device=DEV)
    ev = torch.full((n, VB), 0xA5, dtype=torch.uint8, device=DEV)
    es = torch.full((n,), -1, dtype=torch.int64, device=DEV)
    assert t.insert_and_evict(n, dev(universe[pick]), dev(rows), None, ek, ev, es, unique_key=False) == 0
    assert bool((ek == -1).all()) and bool((ev == 0xA5).all()) and bool((es == -1).all())
    model[0][seen], model[1][seen] = True, rows[first]


def check_ptr(t, model, universe, n, rng):
    """find_or_insert by pointer: every occurrence gets the slot's row address, and whether the key was there before."""
    pick = rng.integers(0, len(universe), n)
    keys = dev(universe[pick])
    ptrs, want = (torch.zeros(n, dtype=torch.int64, device=DEV) for _ in range(2))
    founds, found_now = (torch.zeros(n, dtype=torch.bool, device=DEV) for _ in range(2))
    t.find_or_insert_ptr(n, keys, ptrs, founds, unique_key=False)
    t.find_ptr(n, keys, want, found_now)
    torch.cuda.synchronize()
    assert bool(found_now.all()) and torch.equal(ptrs, want)
    assert (founds.cpu().numpy() == model[0][pick]).all()
    model[0][pick] = True
    # the rows of keys that came in this way are the caller's to write
    rows = rng.integers(0, 256, (len(universe), VB), dtype=np.uint8)
    t.assign(n, keys, dev(rows[pick]), unique_key=False)
    model[1][pick] = rows[pick]
    torch.cuda.synchronize()


# sizes on both sides of those where the keys per tile and the workgroups change (2^15, 2^16, 2^17, 2^18)
@pytest.mark.parametrize("cap", [1 << 17, 1 << 20])
def test_every_call_that_takes_repeated_keys(cap):
    t = make(cap)
    rng = np.random.default_rng(cap)
    universe = w.unique_keys(55, 0, 40000)
    model = np.zeros(len(universe), bool), np.zeros((len(universe), VB), np.uint8)
    for n in (2, 300, (1 << 15) - 1, (1 << 15) + 1, (1 << 16) + 1, (1 << 17) - 1, (1 << 17) + 1, 1 << 18, (1 << 18) + 1, 77):
        check_ptr(t, model, universe, n, rng)
        check_evict(t, model, universe, n, rng)
        check_call(t, model, universe, n, rng)
        check_table(t, model, universe, cap)
    t.close()


def planned_calls(universe, model, sizes, rng):
    """Alternating find_or_insert and insert_or_assign with repeated keys: per call the keys, the rows and what has to be in the
    rows afterwards, on the device and on the host."""
    present, stored = model
    plan = []
    for k, n in enumerate(sizes):
        pick = rng.integers(0, len(universe), n)
        seen, first = np.unique(pick, return_index=True)
        rows = rng.integers(0, 256, (n, VB), dtype=np.uint8)
        stand = np.empty(len(universe), np.int64)
        stand[seen] = first
        want = rows
        if k % 2 == 0:
            want = np.where(present[pick][:, None], stored[pick], rows[stand[pick]])
            new = ~present[seen]
            stored[seen[new]] = rows[first[new]]
        else:
            stored[seen] = rows[first]
        present[seen] = True
        plan.append((n, dev(universe[pick]), dev(rows), want))
    return plan


def issue(t, k, call, stream):
    n, keys, rows, _ = call
    (t.find_or_insert if k % 2 == 0 else t.insert_or_assign)(n, keys, rows, unique_key=False, stream=stream)


def check_plan(plan):
    for k, (n, _, rows, want) in enumerate(plan):
        assert (rows.cpu().numpy() == want).all(), (k, n)


# the index grows, and is used by the next stream, while the calls of the one before are under way
def test_streams_share_the_index_without_waiting():
    cap = 1 << 19
    t = make(cap)
    rng = np.random.default_rng(12)
    universe = w.unique_keys(56, 0, 50000)
    model = np.zeros(len(universe), bool), np.zeros((len(universe), VB), np.uint8)
    streams = [torch.cuda.Stream() for _ in range(3)]
    sizes = [5000, 300, 70000, 4000, 150000, 2, 1 << 15, 300000, 300, 200000, 90000, 1000, 300000, 65, 40000, 250000] * 2
    plan = planned_calls(universe, model, sizes, rng)
    torch.cuda.synchronize()
    for k, call in enumerate(plan):  # one after the other on the host, so the group lock orders them in this order
        issue(t, k, call, streams[k % 3])
    torch.cuda.synchronize()
    check_plan(plan)
    check_table(t, model, universe, cap)
    t.close()


def test_host_threads_share_the_index():
    cap, threads = 1 << 19, 4
    t = make(cap)
    errors, work = [], []
    for tid in range(threads):
        universe = w.unique_keys(57 + tid, 0, 15000)
        model = np.zeros(len(universe), bool), np.zeros((len(universe), VB), np.uint8)
        sizes = [(1 << (6 + (3 * k + tid) % 13)) + k for k in range(40)]
        work.append((universe, model, planned_calls(universe, model, sizes, np.random.default_rng(tid))))
    torch.cuda.synchronize()

    def worker(tid):
        try:
            torch.cuda.set_device(0)
            s = torch.cuda.Stream()
            for k, call in enumerate(work[tid][2]):
                issue(t, k, call, s)
            s.synchronize()
        except BaseException as e:  # noqa: BLE001 - reported by the main thread
            errors.append((tid, repr(e)))

    running = [threading.Thread(target=worker, args=(i,)) for i in range(threads)]
    for th in running:
        th.start()
    for th in running:
        th.join()
    assert not errors, errors
    torch.cuda.synchronize()
    for _, _, plan in work:
        check_plan(plan)
    universe = np.concatenate([u for u, _, _ in work])
    check_table(t, (np.concatenate([m[0] for _, m, _ in work]), np.concatenate([m[1] for _, m, _ in work])), universe, cap)
    t.close()
