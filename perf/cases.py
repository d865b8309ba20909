"""The work that programs on top of this table do, as cases that can be timed and compared.

A case is one step of such a program, on the table and with the batches that it keeps:

  lookup    an inference server reads the rows of a request (find); most keys are in the table
  refresh   a server that is kept up to date: a batch of new and changed rows comes in
            (insert_or_assign) and requests are answered from the table (find).  The table is full,
            so every new key evicts the one that was not used for the longest time.  With
            hbm_share < 1 the other rows are in host memory
  train     one step of embedding training: rows are fetched, and made for keys seen for the first
            time (find_or_insert), the gradients are added (accum_or_assign), the updated rows are
            read (find)
  raw_ids   the same for ids as they come from the features, repeated within the batch
            (find_or_insert and insert_or_assign with unique_key=False)
  evict     the table as a cache in front of a larger store: what a batch pushes out is written
            back (insert_and_evict, scores from the caller)
  publish   rows changed since a given step leave the trained table (export_batch_if) and enter a
            serving table (insert_or_assign), which answers requests (find)
  window    the keys of a sliding time window: the oldest batch leaves (erase), a new one comes in
            (insert_or_assign), requests are answered (find).  The table may still grow, and has
            room: the state of most tables between their creation and their largest size

Keys are 64-bit mixes of a counter, so they fall into buckets at random.  Batches come from a ring
that a case walks along, one row a pass: a key of a row is new again when the ring comes back to
it, because as many keys as the table holds nearly twice have been inserted in between, and a key
that a row expects in the table was used so recently that it cannot have been evicted.  What a pass
returns therefore does not depend on the order in which the keys of a batch are handled.

Rows are float32 or, as bytes to the table, float16; every call moves rows without arithmetic except
accum_or_assign, which adds one float32 to another once: outputs are exact.
"""
import math

import torch

from hierarchicalkv_amd import EvictStrategy, HashTable, Predicate, default_options

DEV = "cuda:0"
_M63 = (1 << 63) - 1
_CHUNK = 1 << 20  # keys per call while a table is being filled
_MOST_BYTES = 1.1e9  # of a drawn case: work() of the largest listed one


def listed():
    return [
        # one key of one user, the smallest call there is: latency only
        {"name": "find-1", "kind": "lookup", "n": 1, "dim": 64, "half": False, "capacity": 1 << 20, "load": 1.0},
        # the features of one scored request, in half precision
        {"name": "find-request", "kind": "lookup", "n": 3001, "dim": 32, "half": True, "capacity": 1 << 22, "load": 1.0},
        # a large inference batch on a large table: the shape the framework is benchmarked on
        {"name": "find-bulk", "kind": "lookup", "n": 1 << 20, "dim": 64, "half": False, "capacity": 1 << 26, "load": 1.0},
        # a ragged batch of rows of 200 bytes, which are not a multiple of 16, in a table with free slots
        {"name": "find-ragged", "kind": "lookup", "n": 200003, "dim": 50, "half": False, "capacity": 1 << 24, "load": 0.75},
        # the benchmark's step: insert_or_assign with half of the keys new, and find, in a full table
        {"name": "refresh-bulk", "kind": "refresh", "n": 1 << 20, "dim": 64, "half": False, "capacity": 1 << 26, "hbm_share": 1.0},
        # an ordinary update of a table of short rows (40 bytes)
        {"name": "refresh-short-rows", "kind": "refresh", "n": 60000, "dim": 10, "half": False, "capacity": 1 << 22, "hbm_share": 1.0},
        # half of the rows do not fit into device memory
        {"name": "refresh-host-rows", "kind": "refresh", "n": 32768, "dim": 64, "half": False, "capacity": 1 << 21, "hbm_share": 0.5},
        # a training step on wide rows
        {"name": "train", "kind": "train", "n": 131072, "dim": 128, "half": False, "capacity": 1 << 23},
        # a training step on ids as they come, Zipf-distributed
        {"name": "train-raw-ids", "kind": "raw_ids", "n": 262144, "dim": 32, "half": False, "capacity": 1 << 22},
        # a cache that writes back what it evicts
        {"name": "cache-evict", "kind": "evict", "n": 131072, "dim": 32, "half": False, "capacity": 1 << 22},
        # changed rows go from the trained table to the serving table
        {"name": "publish", "kind": "publish", "n": 65536, "dim": 16, "half": False, "capacity": 1 << 22},
        # a sliding window of keys in a table that can still grow
        {"name": "window", "kind": "window", "n": 30000, "dim": 16, "half": False, "capacity": 1 << 21},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["lookup", "lookup", "lookup", "refresh", "refresh", "train", "raw_ids", "evict", "publish", "window"])
    dim = rng.choice([4, 8, 10, 16, 18, 32, 33, 50, 64, 100, 128, 200])
    half = kind != "train" and rng.random() < 0.3
    most_rows = (1 << 28) // _row_bytes({"dim": dim, "half": half})  # 256 MB of rows at the most
    if kind == "lookup":
        n = _log_uniform(rng, 1, min(1 << 20, most_rows))
        capacity = 1 << rng.randint(max(18, n.bit_length() + 2), 26 if dim * (2 if half else 4) <= 256 else 24)
        return {"kind": kind, "n": n, "dim": dim, "half": half, "capacity": capacity, "load": rng.choice([0.5, 0.75, 1.0, 1.0])}
    n = _log_uniform(rng, 2000, min(1 << 19, most_rows))
    capacity = 1 << min(25, rng.randint(n.bit_length() + 4, n.bit_length() + 6))
    case = {"kind": kind, "n": n, "dim": dim, "half": half, "capacity": capacity}
    if kind == "refresh":
        case["hbm_share"] = 1.0
        if rng.random() < 0.2:
            n = min(n, 40000)
            case.update(n=n, capacity=1 << (n.bit_length() + 4), hbm_share=0.5)
    while work(case)["bytes"] > _MOST_BYTES:
        case.update(n=case["n"] // 2, capacity=case["capacity"] // 2)
    return case


def _row_bytes(case):
    return case["dim"] * (2 if case["half"] else 4)


# -- keys, rows, tables ------------------------------------------------------------------------

def _lsr(x, k):
    return (x >> k) & ((1 << (64 - k)) - 1)


def _mix64(x):
    """splitmix64 finaliser on int64 tensors: a bijection of 64-bit words."""
    z = x - 0x61C8864680B583EB
    z = (z ^ _lsr(z, 30)) * -0x40A7B892E31B1A47
    z = (z ^ _lsr(z, 27)) * -0x6B2FB644ECCEEE15
    return z ^ _lsr(z, 31)


def _keys(seed, counters):
    """The keys of counters below 2^40; the four reserved words are folded away."""
    k = _mix64(counters + ((seed & 0x7FFFF) << 40))
    return torch.where((k | 3) == -1, k & _M63, k)


def _counters(lo, hi):
    return torch.arange(lo, hi, dtype=torch.int64, device=DEV)


def _generator(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _rows(case, n, gen):
    return torch.randn(n, case["dim"], device=DEV, generator=gen, dtype=torch.float16 if case["half"] else torch.float32)


def _zeros(case, n):
    return torch.zeros(n, case["dim"], device=DEV, dtype=torch.float16 if case["half"] else torch.float32)


def _table(case, strategy=EvictStrategy.kLru, hbm_share=1.0, grows=False):
    rows = case["capacity"] * _row_bytes(case)
    half = {"value_kind": 0, "value_size": 2} if case["half"] else {}  # float16 rows are bytes to the table
    t = HashTable()
    t.init(default_options(init_capacity=case["capacity"], max_capacity=case["capacity"] * (4 if grows else 1),
                           max_hbm_for_vectors=4 * rows if hbm_share == 1.0 else int(rows * hbm_share),
                           max_load_factor=0.75 if grows else 0.5, dim=case["dim"], evict_strategy=strategy, **half))
    return t


def _fill(case, table, keys, gen, scores=None):
    chunk = min(_CHUNK, max(1024, case["capacity"] // 16))
    rows = _rows(case, min(chunk, keys.numel()), gen)
    for at in range(0, keys.numel(), chunk):
        part = keys[at:at + chunk]
        table.insert_or_assign(part.numel(), part, rows, None if scores is None else scores[at:at + chunk])


class _State:
    """What the program holds between its calls."""

    def __init__(self, case):
        self.kind = case["kind"]
        self.n = case["n"]
        self.pos = 0

    def turn(self, ring):
        return ring[self.pos % len(ring)]


def _ring(case, new_share, seed, gen):
    """Counters of the batches of a full table, one row per batch, in random order within a row:
    `w` new keys, and keys of the rows `d` to `d + r - 1` before it.  Returns the rows, w and d."""
    n, capacity = case["n"], case["capacity"]
    w = max(1, round(n * new_share))
    r = -(-(n - w) // w)  # rows that the other keys come from
    d = max(1, min(64, int(0.2 * capacity / w)))
    m = -(-int(1.9 * capacity) // w) + d + r
    col = torch.randperm(n, device=DEV, generator=gen)
    age = torch.where(col < w, 0, d + (col - w) // w)  # rows ago, of each column
    at = torch.where(col < w, col, (col - w) % w)
    row = torch.arange(m, dtype=torch.int64, device=DEV)[:, None]
    return (row - age[None, :]) % m * w + at[None, :], w, d


def _prepare_lookup(case, s, seed, gen):
    n, capacity = case["n"], case["capacity"]
    s.table = _table(case)
    offered = int(capacity * (1.5 if case["load"] == 1.0 else case["load"]))
    _fill(case, s.table, _keys(seed, _counters(0, offered)), gen)
    recent = min(capacity, offered) // 2  # keys that are certainly still there
    batches = max(4, min(64, (1 << 22) // n))
    c = torch.randint(offered - recent, offered, (batches, n), device=DEV, generator=gen)
    absent = torch.rand(batches, n, device=DEV, generator=gen) < 0.125
    s.batches = list(_keys(seed, torch.where(absent, c + offered, c)).unbind(0))
    s.out = _zeros(case, n)
    s.found = torch.zeros(n, dtype=torch.bool, device=DEV)


def _run_lookup(s):
    s.table.find(s.n, s.turn(s.batches), s.out, s.found)
    return s.out, s.found


def _prepare_refresh(case, s, seed, gen):
    n = case["n"]
    c, w, d = _ring(case, 0.5, seed, gen)
    s.table = _table(case, hbm_share=case["hbm_share"])
    _fill(case, s.table, _keys(seed, _counters(0, c.shape[0] * w)), gen)
    # requests: keys that came in with the batch, and keys of an earlier one
    q = torch.roll(c, d // 2 + 1, 0)
    q[:, :n // 4] = c[:, :n // 4]
    s.batches = list(_keys(seed, c).unbind(0))
    s.requests = list(_keys(seed, q).unbind(0))
    s.rows = [_rows(case, n, gen) for _ in range(2)]
    s.out = _zeros(case, n)
    s.found = torch.zeros(n, dtype=torch.bool, device=DEV)


def _run_refresh(s):
    s.table.insert_or_assign(s.n, s.turn(s.batches), s.turn(s.rows))
    s.table.find(s.n, s.turn(s.requests), s.out, s.found)
    return s.out, s.found


def _prepare_train(case, s, seed, gen):
    n = case["n"]
    c, w, _ = _ring(case, 0.125, seed, gen)
    s.table = _table(case)
    _fill(case, s.table, _keys(seed, _counters(0, c.shape[0] * w)), gen)
    s.batches = list(_keys(seed, c).unbind(0))
    s.emb = _zeros(case, n)
    s.grads = _rows(case, n, gen) * -0.01
    s.present = torch.ones(n, dtype=torch.bool, device=DEV)
    s.out = _zeros(case, n)
    s.found = torch.zeros(n, dtype=torch.bool, device=DEV)


def _run_train(s):
    keys = s.turn(s.batches)
    s.emb.zero_()  # where a key's row starts
    s.table.find_or_insert(s.n, keys, s.emb)
    s.table.accum_or_assign(s.n, keys, s.grads, s.present)
    s.table.find(s.n, keys, s.out, s.found)
    return s.emb, s.out, s.found


def _prepare_raw_ids(case, s, seed, gen):
    n, universe = case["n"], case["capacity"] // 2
    s.table = _table(case)
    _fill(case, s.table, _keys(seed, _counters(0, universe * 3 // 4)), gen)
    batches = max(4, min(64, (1 << 22) // n))
    a = 1.0 - 1.05  # Zipf(1.05) over the universe, by inversion of the continuous law
    u = torch.rand(batches, n, dtype=torch.float64, device=DEV, generator=gen)
    rank = torch.floor((1.0 + u * (float(universe) ** a - 1.0)) ** (1.0 / a)).to(torch.int64).clamp_(1, universe) - 1
    s.batches = list(_keys(seed, rank).unbind(0))
    s.emb = _zeros(case, n)


def _run_raw_ids(s):
    ids = s.turn(s.batches)
    s.emb.zero_()
    s.table.find_or_insert(s.n, ids, s.emb, unique_key=False)
    s.emb.mul_(0.98)  # the optimizer's part: the same for every occurrence of an id
    s.table.insert_or_assign(s.n, ids, s.emb, unique_key=False)
    return s.emb


def _prepare_evict(case, s, seed, gen):
    n = case["n"]
    c, w, _ = _ring(case, 0.5, seed, gen)
    ids = c.shape[0] * w
    # here keys are the row numbers of the store, in random order
    order = torch.randperm(ids, device=DEV, generator=gen)
    s.table = _table(case, strategy=EvictStrategy.kCustomized)
    _fill(case, s.table, order, gen, _counters(0, ids))
    s.store = _zeros(case, ids)
    s.batches = list(order[c].unbind(0))
    s.rows = [_rows(case, n, gen) for _ in range(2)]
    s.score_in_batch = torch.randperm(n, device=DEV, generator=gen)
    s.scores = torch.zeros(n, dtype=torch.int64, device=DEV)
    s.out_keys = torch.zeros(n, dtype=torch.int64, device=DEV)
    s.out_rows = _zeros(case, n)
    s.out_scores = torch.zeros(n, dtype=torch.int64, device=DEV)


def _run_evict(s):
    torch.add(s.score_in_batch, (s.pos + 1) << 32, out=s.scores)  # later steps score higher
    gone = s.table.insert_and_evict(s.n, s.turn(s.batches), s.turn(s.rows), s.scores,
                                    s.out_keys, s.out_rows, s.out_scores)
    s.store.index_copy_(0, s.out_keys[:gone], s.out_rows[:gone])
    return s.store, gone


def _prepare_publish(case, s, seed, gen):
    n, capacity = case["n"], case["capacity"]
    offered = int(capacity * 0.75)
    keys = _keys(seed, _counters(0, offered))
    s.table = _table(case, strategy=EvictStrategy.kCustomized)
    # the step a row was last changed at: evenly spread over 2^32
    _fill(case, s.table, keys, gen, _lsr(_mix64(keys ^ 0x5555), 32))
    s.replica = _table(case)
    s.thresholds = [int((1.0 - share) * 2 ** 32) for share in (0.125, 0.1875, 0.25, 0.15625)]
    s.count = torch.zeros(1, dtype=torch.int64, device=DEV)
    s.out_keys = torch.zeros(capacity, dtype=torch.int64, device=DEV)
    s.out_rows = _zeros(case, capacity)
    c = torch.randint(0, offered, (8, n), device=DEV, generator=gen)
    s.requests = list(_keys(seed, c).unbind(0))
    s.out = _zeros(case, n)
    s.found = torch.zeros(n, dtype=torch.bool, device=DEV)
    s.capacity = capacity


def _run_publish(s):
    s.table.export_batch_if(Predicate.kScoreGe, 0, s.turn(s.thresholds), s.capacity, 0, s.count, s.out_keys, s.out_rows)
    changed = int(s.count.item())
    s.replica.insert_or_assign(changed, s.out_keys, s.out_rows)
    s.replica.find(s.n, s.turn(s.requests), s.out, s.found)
    return s.out, s.found, changed


def _prepare_window(case, s, seed, gen):
    n, capacity = case["n"], case["capacity"]
    live = max(2, capacity // 2 // n)  # batches in the window: half of the slots are in use
    s.table = _table(case, grows=True)
    _fill(case, s.table, _keys(seed, _counters(0, live * n)), gen)
    s.batches = list(_keys(seed, _counters(0, 2 * live * n)).view(2 * live, n).unbind(0))
    s.live = live
    s.pos = live
    s.rows = [_rows(case, n, gen) for _ in range(2)]
    s.out = _zeros(case, n)
    s.found = torch.zeros(n, dtype=torch.bool, device=DEV)


def _run_window(s):
    ring = s.batches
    s.table.erase(s.n, ring[(s.pos - s.live) % len(ring)])
    s.table.insert_or_assign(s.n, ring[s.pos % len(ring)], s.turn(s.rows))
    asked = s.pos if s.pos % 2 == 0 else s.pos - s.live // 2  # the newest batch, one from the middle of the window
    s.table.find(s.n, ring[asked % len(ring)], s.out, s.found)
    return s.out, s.found


_PREPARE = {"lookup": _prepare_lookup, "refresh": _prepare_refresh, "train": _prepare_train, "raw_ids": _prepare_raw_ids,
            "evict": _prepare_evict, "publish": _prepare_publish, "window": _prepare_window}
_RUN = {"lookup": _run_lookup, "refresh": _run_refresh, "train": _run_train, "raw_ids": _run_raw_ids,
        "evict": _run_evict, "publish": _run_publish, "window": _run_window}


def prepare(case, seed):
    s = _State(case)
    _PREPARE[case["kind"]](case, s, seed, _generator(seed))
    torch.cuda.synchronize()
    return s


def run(state):
    out = _RUN[state.kind](state)
    state.pos += 1
    return out


def work(case):
    """Bytes of a step: every key, row, flag and score of the batch that goes in or out, and every
    stored key, row and score of the table that is read or written, once; no digests, no search."""
    n, row = case["n"], _row_bytes(case)
    find = n * (8 + 8 + 1 + 2 * row)        # key, stored key, flag, row
    assign = n * (8 + 8 + 8 + 2 * row)      # key, stored key, score, row
    kind = case["kind"]
    if kind == "lookup":
        b = find - n // 8 * 2 * row
    elif kind == "refresh":
        b = assign + n // 2 * (8 + 1) + find  # a new key also changes the stored key and its digest
    elif kind == "train":
        b = n * row + assign + n * (8 + 8 + 8 + 1 + 3 * row) + find
    elif kind == "raw_ids":
        b = n * row + 2 * assign + 2 * n * row
    elif kind == "evict":
        b = 3 * 8 * n + assign + n * 8 + n // 2 * (16 + 8 + 2 * row) + n // 2 * (8 + 2 * row)
    elif kind == "publish":
        slots, changed = case["capacity"], int(0.75 * case["capacity"] * 0.18)
        b = slots * 16 + changed * (8 + 2 * row) + changed * (24 + 2 * row) + find
    else:
        b = n * (8 + 8 + 8 + 1) + assign + find
    return {"bytes": b, "flops": n * case["dim"] if kind == "train" else 0}


def tolerance(case):
    return "exact"
