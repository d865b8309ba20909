"""When a table grows.  An inserting call takes a sample of the load unless the last one, with all keys that have come
since, rules growth out; a table without the group lock takes one at every call.  Both must have the
same capacity after every call."""
import threading

import numpy as np
import pytest
import torch

import workloads as w
from gpu_util import DEV, dev
from hierarchicalkv_amd import HashTable, default_options

pytestmark = pytest.mark.gpu
DIM = 4


def make(init, most, load, api_lock):
    t = HashTable()
    t.init(default_options(init_capacity=init, max_capacity=most, max_hbm_for_vectors=1 << 30, dim=DIM,
                           max_load_factor=load, api_lock=api_lock))
    return t


# tables of less and of more buckets than the sample has (1024); small calls, calls as large as the room that is left
@pytest.mark.parametrize("init,most,load,sizes", [
    (1 << 10, 1 << 16, 0.5, (1, 7, 64, 300)),
    (1 << 12, 1 << 18, 0.75, (3, 500, 2000, 4096)),
    (1 << 17, 1 << 19, 0.75, (1000, 16000, 33000)),
    (1 << 18, 1 << 20, 0.5, (5000, 20000, 70001)),
])
def test_grows_with_the_call_that_has_to(init, most, load, sizes):
    kept, always = make(init, most, load, 1), make(init, most, load, 0)
    rng = np.random.default_rng(init)
    universe = w.unique_keys(61, 0, most)
    rows = torch.zeros(max(sizes), DIM, dtype=torch.float32, device=DEV)
    ptrs = torch.zeros(max(sizes), dtype=torch.int64, device=DEV)
    founds = torch.zeros(max(sizes), dtype=torch.bool, device=DEV)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    at, capacities = 0, []
    torch.cuda.synchronize()
    for step in range(150):
        n = int(rng.choice(sizes))
        lo = at if rng.random() < 0.7 else int(rng.integers(0, max(1, at - n)))  # new keys, or some that came before
        op = rng.choice(["insert_or_assign", "find_or_insert", "find_or_insert_ptr", "erase", "clear", "reserve"],
                        p=[0.4, 0.2, 0.1, 0.28, 0.01, 0.01])
        if op != "erase" and lo + n > most:
            break
        keys = dev(universe[lo:lo + n])
        n = min(n, len(keys))
        torch.cuda.synchronize()
        s = streams[step // 20 % 2]
        wanted = kept.capacity() + 1
        for t in (kept, always):
            if op == "insert_or_assign":
                t.insert_or_assign(n, keys, rows, stream=s)
            elif op == "find_or_insert":
                t.find_or_insert(n, keys, rows, stream=s)
            elif op == "find_or_insert_ptr":
                t.find_or_insert_ptr(n, keys, ptrs, founds, stream=s)
            elif op == "erase":
                t.erase(n, keys, stream=s)
            elif op == "clear":
                t.clear(stream=s)
            else:
                t.reserve(wanted, stream=s)
            torch.cuda.synchronize()
        if op.startswith(("insert", "find")):
            at = max(at, lo + n)
        capacities.append(kept.capacity())
        assert kept.capacity() == always.capacity(), (step, op, n)
    assert len(set(capacities)) > 1  # it did grow
    kept.close()
    always.close()


def test_replays_of_a_recorded_call_are_not_counted():
    """A call that was recorded while the table could not grow brings keys with every replay; once the table may
    grow, every call looks at the load."""
    cap, n = 1 << 12, 512
    t = make(cap, cap, 0.75, 1)
    s = torch.cuda.Stream()
    keys = torch.zeros(n, dtype=torch.int64, device=DEV)
    rows = torch.zeros(n, DIM, dtype=torch.float32, device=DEV)
    with torch.cuda.stream(s):
        keys.copy_(dev(w.unique_keys(62, 0, n)))
        t.insert_or_assign(n, keys, rows)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            t.insert_or_assign(n, keys, rows)
        t.set_max_capacity(2 * cap)
        t.insert_or_assign(8, dev(w.unique_keys(63, 0, 8)), rows)
        assert t.capacity() == cap
        for k in range(1, 7):  # 3592 keys of 4096
            keys.copy_(dev(w.unique_keys(62, k * n, n)))
            g.replay()
        torch.cuda.synchronize()
        assert t.size() > 0.75 * cap
        t.insert_or_assign(8, dev(w.unique_keys(63, 8, 8)), rows)
        assert t.capacity() == 2 * cap
    torch.cuda.synchronize()
    t.close()


def test_host_threads_insert_into_one_table_that_grows():
    """Eight threads, each on a stream and with keys of its own: whatever sample a call goes by, the table has grown
    whenever it had to, so that no bucket ever was full and every key is there with its row."""
    threads, rounds, n, dim = 8, 80, 50, 4
    t = HashTable()
    t.init(default_options(init_capacity=1 << 13, max_capacity=1 << 18, max_hbm_for_vectors=1 << 30, dim=dim,
                           max_load_factor=0.5))
    errors = []

    def worker(tid):
        try:
            torch.cuda.set_device(0)
            s = torch.cuda.Stream()
            for r in range(rounds):
                keys = w.unique_keys(6400 + tid, r * n, n)
                dk, dv = dev(keys), dev(w.values_from_keys(keys, dim))
                torch.cuda.current_stream().synchronize()
                if r % 3 == 2:
                    t.find_or_insert(n, dk, dv, stream=s)
                else:
                    t.insert_or_assign(n, dk, dv, stream=s, unique_key=r % 3 == 0)
                s.synchronize()  # the buffers go away
        except BaseException as e:  # noqa: BLE001 - reported by the main thread
            errors.append((tid, repr(e)))

    running = [threading.Thread(target=worker, args=(i,)) for i in range(threads)]
    for th in running:
        th.start()
    for th in running:
        th.join()
    assert not errors, errors[:3]
    torch.cuda.synchronize()
    assert t.size() == threads * rounds * n and t.capacity() >= 2 * (threads * rounds - threads) * n
    for tid in range(threads):
        keys = w.unique_keys(6400 + tid, 0, rounds * n)
        out = torch.zeros(rounds * n, dim, dtype=torch.float32, device=DEV)
        founds = torch.zeros(rounds * n, dtype=torch.bool, device=DEV)
        t.find(rounds * n, dev(keys), out, founds)
        torch.cuda.synchronize()
        assert bool(founds.all()) and np.array_equal(out.cpu().numpy(), w.values_from_keys(keys, dim))
    t.close()
