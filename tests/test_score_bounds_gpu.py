"""The score bounds of a table (hkv_table_view::bounds): for every line of 16 slots a value that
is not above any score in the line, which the upserts use to find a bucket's lowest score from
one or two of its eight score lines.  LRU and EpochLRU scores only grow, so their bounds stay right
by themselves; under Customized, LFU and EpochLFU a key that writes a score below its line's bound
lowers the bound itself.  Checked here:
  * the invariant itself, read back from device memory after mixed call sequences, on the
    deterministic and on the hardware clock (a bound above a score would send an eviction to the
    wrong slot sooner or later);
  * that erase and the calls which may lower scores (upserts with ignore_evict_strategy,
    set_clock) leave the bounds right;
  * parity with the oracle through all of this (deterministic clock), which is the parity of the
    bounded search with the full scan: the oracle scans all 128 scores."""
import numpy as np
import pytest
import torch

import workloads as w
from gpu_util import DEV, assert_same_table, dev, read_device
from hierarchicalkv_amd import EvictStrategy, HashTable, default_options

import os

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(os.environ.get("HKV_SCORE_BOUNDS") == "0", reason="score bounds switched off")]


def bytes_of(a):
    return np.ascontiguousarray(a).view(np.uint8).reshape(len(a), -1)


def bounds_hold(t):
    """bound[line] <= the score of every key (or tombstone) of the line, for all lines of the table.
    A free slot does not count: it gets a score of the time when it is taken."""
    torch.cuda.synchronize()
    v = t.view()
    cap = v.capacity
    scores = read_device(v.scores, cap * 8).view(np.uint64).reshape(cap // 16, 16).copy()
    keys = read_device(v.keys, cap * 8).view(np.uint64).reshape(cap // 16, 16)
    bounds = read_device(v.bounds, cap // 16 * 8).view(np.uint64)
    scores[keys == np.uint64(v.empty_key)] = np.uint64((1 << 64) - 1)
    bad = np.flatnonzero(bounds > scores.min(axis=1))
    return len(bad) == 0, bad[:5], int((bounds > 0).sum())


def make(cap, dim, strategy=EvictStrategy.kLru, **kw):
    o = default_options(init_capacity=cap, max_capacity=cap, max_hbm_for_vectors=1 << 30, dim=dim,
                        evict_strategy=strategy, **kw)
    t = HashTable()
    t.init(o)
    return t, o


@pytest.mark.parametrize("clock", ["deterministic", "hardware"])
def test_bounds_stay_below_the_scores(oracle, clock):
    cap, dim = 1 << 13, 8
    t, o = make(cap, dim)
    ot = oracle.OracleTable(o)
    det = clock == "deterministic"
    if det:
        t.set_clock(1, 1 << 44)
        ot.set_clock(1, 1 << 44)
    rng = np.random.default_rng(77)
    universe = w.unique_keys(610, 0, 4 * cap)
    tight = 0
    for step in range(60):
        n = int(rng.choice([64, 700, 3000]))
        keys = rng.choice(universe, size=n, replace=False)
        vals = rng.random((n, dim), dtype=np.float32)
        op = rng.choice(["insert_or_assign", "find_or_insert", "insert_and_evict", "assign", "erase"],
                        p=[0.4, 0.15, 0.2, 0.1, 0.15])
        if op == "find_or_insert":  # all resident or all new: see test_random_ops_gpu.py
            present = ot.contains(keys) if det else np.ones(n, bool)
            keep = present if present.sum() else ~present
            keys, vals = keys[keep], vals[keep]
            n = len(keys)
        dk, dv = dev(keys), dev(vals)
        if op == "insert_or_assign":
            t.insert_or_assign(n, dk, dv)
            ot.insert_or_assign(keys, bytes_of(vals), None)
        elif op == "find_or_insert":
            t.find_or_insert(n, dk, dv.clone())
            ot.find_or_insert(keys, bytes_of(vals).copy(), None)
        elif op == "insert_and_evict":
            ek = torch.zeros(n, dtype=torch.int64, device=DEV)
            ev = torch.zeros(n, dim, dtype=torch.float32, device=DEV)
            t.insert_and_evict(n, dk, dv, None, ek, ev, None)
            ot.insert_and_evict(keys, bytes_of(vals), None)
        elif op == "assign":
            t.assign(n, dk, dv)
            ot.assign(keys, bytes_of(vals), None)
        else:
            t.erase(n, dk)
            ot.erase(keys)
        ok, bad, n_tight = bounds_hold(t)
        assert ok, (step, op, bad)
        tight = max(tight, n_tight)
        if det:
            assert t.size() == ot.size(), (step, op)
            if step % 10 == 9:
                assert_same_table(t, ot, dim * 4)
    assert tight > cap // 16 // 4  # the bounds are in use, not all zero
    if det:
        assert_same_table(t, ot, dim * 4)
    t.close()


def test_scores_from_outside_the_clock(oracle):
    """An upsert with ignore_evict_strategy (what load() uses) writes the caller's scores into an
    LRU table, lower than what is there; the clock can be set back.  Evictions afterwards must
    still take the lowest score of the bucket."""
    cap, dim = 1 << 12, 4
    t, o = make(cap, dim)
    ot = oracle.OracleTable(o)
    t.set_clock(1, 1 << 44)
    ot.set_clock(1, 1 << 44)
    keys = w.unique_keys(620, 0, 8 * cap)
    for b in range(6):  # fill and evict: the bounds tighten
        k = keys[b * 2000:(b + 1) * 2000]
        v = w.values_from_keys(k, dim)
        t.insert_or_assign(len(k), dev(k), dev(v))
        ot.insert_or_assign(k, bytes_of(v), None)
    assert bounds_hold(t)[0]
    # caller's scores, far below the clock's
    k = keys[500:2500]
    v = w.uniform_values(621, 0, len(k), dim)
    sc = np.arange(1, len(k) + 1, dtype=np.uint64)
    t.insert_or_assign(len(k), dev(k), dev(v), dev(sc), ignore_evict_strategy=True)
    ot.insert_or_assign(k, bytes_of(v), sc, ignore=True)
    assert_same_table(t, ot, dim * 4)
    # the next clocked upserts evict those low scores first
    for b in range(6, 9):
        k = keys[b * 2000:(b + 1) * 2000]
        v = w.values_from_keys(k, dim)
        t.insert_or_assign(len(k), dev(k), dev(v))
        ot.insert_or_assign(k, bytes_of(v), None)
        assert bounds_hold(t)[0]
        assert_same_table(t, ot, dim * 4)
    # the clock goes back: new scores below the old ones
    t.set_clock(1, 1 << 30)
    ot.set_clock(1, 1 << 30)
    for b in range(9, 12):
        k = keys[18000 + (b - 9) * 1000:18000 + (b - 8) * 1000]
        v = w.values_from_keys(k, dim)
        t.insert_or_assign(len(k), dev(k), dev(v))
        ot.insert_or_assign(k, bytes_of(v), None)
        assert bounds_hold(t)[0]
        assert_same_table(t, ot, dim * 4)
    t.close()


@pytest.mark.parametrize("dim", [64, 128])
def test_bounded_kernels_with_wide_rows(oracle, dim):
    """The bounded search in the instantiations that move rows of 256 and 512 bytes (two and four
    16-byte units per lane, which is what a table of dim 64 / 128 runs): insert_or_assign,
    find_or_insert, insert_and_evict (two wavefronts per workgroup) and accum_or_assign on a table
    filled past load factor 1.0, LRU on the deterministic clock, every call against the oracle."""
    from gpu_util import canonical_evicted, export_table, host_bytes, host_u64, sort_by_key
    cap, bs = 1 << 14, 3000
    t, o = make(cap, dim)
    ot = oracle.OracleTable(o)
    t.set_clock(1, 1 << 44)
    ot.set_clock(1, 1 << 44)
    seed, pos = 630 + dim, 0
    vb = dim * 4
    while pos < cap + 4 * bs:  # past load factor 1.0: the last batches evict
        k = w.unique_keys(seed, pos, bs)
        v = w.uniform_values(seed, pos, bs, dim)
        t.insert_or_assign(bs, dev(k), dev(v))
        ot.insert_or_assign(k, bytes_of(v), None)
        pos += bs
    assert t.size() == ot.size()
    assert_same_table(t, ot, vb)
    ok, _, n_tight = bounds_hold(t)
    assert ok and n_tight > 0  # the bounded kernel has been at work
    for rep in range(3):
        # insert_or_assign: half from the latest batch (highest scores: no key of this batch can
        # evict one of them before its turn), half new
        k = np.concatenate([w.unique_keys(seed, pos - bs // 2, bs // 2), w.unique_keys(seed, pos, bs // 2)])
        pos += bs // 2
        v = w.uniform_values(seed + 1, pos, len(k), dim)
        t.insert_or_assign(len(k), dev(k), dev(v))
        ot.insert_or_assign(k, bytes_of(v), None)
        assert_same_table(t, ot, vb)
        # find_or_insert: the same mix; hits hand their rows back, misses insert
        k = np.concatenate([w.unique_keys(seed, pos - bs // 2, bs // 2), w.unique_keys(seed, pos, bs // 2)])
        pos += bs // 2
        v = w.uniform_values(seed + 2, pos, len(k), dim)
        dv = dev(v)
        t.find_or_insert(len(k), dev(k), dv)
        ov = bytes_of(v).copy()
        ot.find_or_insert(k, ov, None)
        torch.cuda.synchronize()
        assert (host_bytes(dv, len(k), vb) == ov).all()
        assert_same_table(t, ot, vb)
        # insert_and_evict: evicted keys, rows and scores
        k = np.concatenate([w.unique_keys(seed, pos - bs // 2, bs // 2), w.unique_keys(seed, pos, bs // 2 + 37)])
        pos += bs // 2 + 37
        n = len(k)
        v = w.uniform_values(seed + 3, pos, n, dim)
        ek = torch.zeros(n, dtype=torch.int64, device=DEV)
        ev = torch.zeros(n, dim, dtype=torch.float32, device=DEV)
        es = torch.zeros(n, dtype=torch.int64, device=DEV)
        cnt = t.insert_and_evict(n, dev(k), dev(v), None, ek, ev, es)
        oek, oev, oes = ot.insert_and_evict(k, bytes_of(v), None)
        assert cnt == len(oek) and cnt > 0
        gk, _, _ = sort_by_key(*export_table(t, vb))
        a = canonical_evicted(host_u64(ek[:cnt]), host_bytes(ev[:cnt], cnt, vb), host_u64(es[:cnt]), gk)
        b = canonical_evicted(oek, oev, oes, gk)
        assert (a[0] == b[0]).all() and (a[1] == b[1]).all() and (a[2] == b[2]).all()
        assert_same_table(t, ot, vb)
        # accum_or_assign: recent keys accumulate, new keys are assigned, flags from contains
        k = np.concatenate([w.unique_keys(seed, pos - bs // 2, bs // 2), w.unique_keys(seed, pos, bs // 2)])
        pos += bs // 2
        d = (w.uniform_values(seed + 4, pos, len(k), dim) * np.float32(0.01)).astype(np.float32)
        founds = torch.zeros(len(k), dtype=torch.bool, device=DEV)
        t.contains(len(k), dev(k), founds)
        torch.cuda.synchronize()
        flags = founds.cpu().numpy()
        assert (flags == ot.contains(k)).all() and flags.any() and not flags.all()
        t.accum_or_assign(len(k), dev(k), dev(d), founds)
        ot.accum_or_assign(k, bytes_of(d), flags.astype(np.uint8))
        assert_same_table(t, ot, vb)
        ok, bad, _ = bounds_hold(t)
        assert ok, (rep, bad)
    t.close()


# ---- strategies whose scores come from the caller, and EpochLRU ---------------------------------

def upsert(t, ot, k, v, sc):
    t.insert_or_assign(len(k), dev(k), dev(v), dev(sc))
    ot.insert_or_assign(k, bytes_of(v), sc)


def one_per_bucket(oracle, keys, buckets):
    """The first key of `keys` for every bucket that any of them falls into."""
    seen, keep = set(), []
    for i, k in enumerate(keys.tolist()):
        b = oracle.locate(k, buckets)[0]
        if b not in seen:
            seen.add(b)
            keep.append(i)
    return keys[np.array(keep)]


def test_customized_scores_that_go_down(oracle):
    """Customized: a key that is found gets the caller's score, which may be far below the one it
    had, through insert_or_assign, find_or_insert and assign_scores; a key that goes into a free slot
    may bring any score.  The bounds must follow, or the next evictions take the wrong keys."""
    cap, dim, bs = 1 << 13, 4, 2048
    t, o = make(cap, dim, EvictStrategy.kCustomized)
    ot = oracle.OracleTable(o)
    vb = dim * 4
    seed, pos, batch = 640, 0, 10
    while pos < cap + 4 * bs:  # past load factor 1.0 with growing scores
        k = w.unique_keys(seed, pos, bs)
        upsert(t, ot, k, w.values_from_keys(k, dim), w.monotone_scores(batch, bs, seed=64))
        pos += bs
        batch += 1
    assert_same_table(t, ot, vb)
    ok, bad, n_tight = bounds_hold(t)
    assert ok and n_tight > cap // 16 // 4, (bad, n_tight)

    def residents_by_score():
        k, _, sc = ot.export_all()
        return k[np.argsort(sc)]

    # the best-scored residents get the lowest scores of the table (hits only: nothing is evicted)
    top = residents_by_score()[-1500:]
    a, b_, c = top[:500], top[500:1000], top[1000:]
    upsert(t, ot, a, w.values_from_keys(a, dim) + 1, np.arange(1, 501, dtype=np.uint64))
    assert bounds_hold(t)[0]
    t.assign_scores(len(b_), dev(b_), dev(np.arange(501, 1001, dtype=np.uint64)))
    ot.assign_scores(b_, np.arange(501, 1001, dtype=np.uint64))
    assert bounds_hold(t)[0]
    v = w.values_from_keys(c, dim)
    dv = dev(v)
    t.find_or_insert(len(c), dev(c), dv, dev(np.arange(1001, 1501, dtype=np.uint64)))
    ov = bytes_of(v).copy()
    ot.find_or_insert(c, ov, np.arange(1001, 1501, dtype=np.uint64))
    assert bounds_hold(t)[0]
    assert_same_table(t, ot, vb)
    # free slots taken with scores below everything else (one key per bucket: two such keys in a
    # full bucket would evict each other in an order that nothing fixes)
    gone = residents_by_score()[2000:2600]
    t.erase(len(gone), dev(gone))
    ot.erase(gone)
    k = one_per_bucket(oracle, w.unique_keys(seed + 1, 0, 400), cap // 128)
    upsert(t, ot, k, w.values_from_keys(k, dim), np.arange(2001, 2001 + len(k), dtype=np.uint64))
    assert bounds_hold(t)[0]
    assert_same_table(t, ot, vb)
    # new keys with high scores: the low ones go first, through all three inserting calls
    for rep in range(4):
        k = w.unique_keys(seed + 2, rep * 900, 900)
        v = w.values_from_keys(k, dim)
        sc = w.monotone_scores(batch, len(k), seed=64)
        batch += 1
        if rep % 2 == 0:
            ek = torch.zeros(len(k), dtype=torch.int64, device=DEV)
            ev = torch.zeros(len(k), dim, dtype=torch.float32, device=DEV)
            es = torch.zeros(len(k), dtype=torch.int64, device=DEV)
            cnt = t.insert_and_evict(len(k), dev(k), dev(v), dev(sc), ek, ev, es)
            oek, _, oes = ot.insert_and_evict(k, bytes_of(v), sc)
            assert cnt == len(oek)
            got = sorted(zip(ek[:cnt].cpu().numpy().view(np.uint64).tolist(),
                             es[:cnt].cpu().numpy().view(np.uint64).tolist()))
            assert got == sorted(zip(oek.tolist(), oes.tolist()))
        else:
            upsert(t, ot, k, v, sc)
        ok, bad, _ = bounds_hold(t)
        assert ok, (rep, bad)
        assert_same_table(t, ot, vb)
    # a batch whose own scores are below the last batches': its bounds may not go above them
    k = w.unique_keys(seed + 3, 0, 900)
    upsert(t, ot, k, w.values_from_keys(k, dim), w.monotone_scores(5, len(k), seed=64))  # all refused or low
    assert bounds_hold(t)[0]
    assert_same_table(t, ot, vb)
    k = w.unique_keys(seed + 4, 0, 900)
    upsert(t, ot, k, w.values_from_keys(k, dim), w.monotone_scores(batch, len(k), seed=64))
    assert bounds_hold(t)[0]
    assert_same_table(t, ot, vb)
    t.close()


@pytest.mark.parametrize("row_bytes", [16, 36, 40])
def test_customized_calls_without_scores(oracle, row_bytes):
    """A full Customized table, ignore_evict_strategy and no scores: every key of the call counts as 0.
    New keys are refused where every score is above 0 and take the place of a key with score 0
    otherwise; a key that is found keeps its place with score 0 and is the next one to go.  (Under
    Customized only rows of 16-byte multiples use the bounds.)"""
    cap, bs, dim = 1 << 13, 2048, row_bytes // 4
    buckets = cap // 128
    t, o = make(cap, dim, EvictStrategy.kCustomized)
    ot = oracle.OracleTable(o)
    pos, batch = 0, 10
    while pos < cap + 4 * bs:
        k = w.unique_keys(660, pos, bs)
        upsert(t, ot, k, w.values_from_keys(k, dim), w.monotone_scores(batch, bs, seed=66))
        pos += bs
        batch += 1
    assert_same_table(t, ot, row_bytes)
    bounded = row_bytes % 16 == 0
    assert bounds_hold(t)[2] > 0 or not bounded
    at = 0
    for step in range(12):
        # one key of the call per bucket: two would evict each other in an order that nothing fixes
        fresh = one_per_bucket(oracle, w.unique_keys(661, at, 400), buckets)
        at += 400
        if step % 3 == 0:
            k = fresh  # refused at first (no score is 0 yet)
        else:
            # (a key with score 0 before any other of its bucket, so that no bucket gets two of them: which
            # of two goes first depends on where they are)
            resident, _, score = ot.export_all()
            order = np.random.default_rng(step).permutation(len(resident))
            found = one_per_bucket(oracle, resident[order][np.argsort(score[order] > 0, kind="stable")], buckets)
            k = found if step % 3 == 1 else one_per_bucket(oracle, np.concatenate([found[:20], fresh]), buckets)
        v = w.values_from_keys(k, dim) + step
        n, zeros = len(k), np.zeros(len(k), np.uint64)
        op = ("insert_or_assign", "accum_or_assign", "find_or_insert", "insert_and_evict")[(step // 3 + step % 3) % 4]
        if op == "insert_or_assign":
            t.insert_or_assign(n, dev(k), dev(v), None, ignore_evict_strategy=True)
            ot.insert_or_assign(k, bytes_of(v), zeros, ignore=True)
        elif op == "accum_or_assign":
            there = ot.contains(k)
            t.accum_or_assign(n, dev(k), dev(v), dev(there), None, ignore_evict_strategy=True)
            ot.accum_or_assign(k, bytes_of(v), there.astype(np.uint8), zeros, ignore=True)
        elif op == "find_or_insert":
            dv, ov = dev(v), bytes_of(v).copy()
            t.find_or_insert(n, dev(k), dv, None, ignore_evict_strategy=True)
            ot.find_or_insert(k, ov, zeros, ignore=True)
            assert (dv.cpu().numpy().view(np.uint8).reshape(n, -1) == ov).all(), step
        else:
            ek = torch.zeros(n, dtype=torch.int64, device=DEV)
            ev = torch.zeros(n, dim, dtype=torch.float32, device=DEV)
            es = torch.zeros(n, dtype=torch.int64, device=DEV)
            gone = t.insert_and_evict(n, dev(k), dev(v), None, ek, ev, es, ignore_evict_strategy=True)
            oek, _, oes = ot.insert_and_evict(k, bytes_of(v), zeros, ignore=True)
            got = zip(ek[:gone].cpu().numpy().view(np.uint64).tolist(), es[:gone].cpu().numpy().view(np.uint64).tolist())
            assert sorted(got) == sorted(zip(oek.tolist(), oes.tolist())), step
        assert_same_table(t, ot, row_bytes)
    # keys with scores again: the ones with score 0 go first, and the bounds are right
    assert (ot.export_all()[2] == 0).sum() > buckets // 2
    for rep in range(2):
        k = w.unique_keys(662, rep * 900, 900)
        upsert(t, ot, k, w.values_from_keys(k, dim), w.monotone_scores(batch + rep, len(k), seed=66))
        ok, bad, n_tight = bounds_hold(t)
        assert (ok and n_tight > 0) or not bounded, (rep, bad)
        assert_same_table(t, ot, row_bytes)
    t.close()


@pytest.mark.parametrize("row_bytes", [8, 36])
def test_customized_scores_that_stop_growing(oracle, row_bytes):
    """Rows of no multiple of 16 bytes: searches through the bounds while the lowest score of a call is above the ones
    before, full scans after some calls where it is not, and bounds again once the table has been cleared."""
    cap, bs, dim = 1 << 13, 2048, row_bytes // 4
    t, o = make(cap, dim, EvictStrategy.kCustomized)
    for again in range(2):
        ot = oracle.OracleTable(o)
        pos, batch = 0, 10
        while pos < cap + 4 * bs:
            k = w.unique_keys(670 + again, pos, bs)
            upsert(t, ot, k, w.values_from_keys(k, dim), w.monotone_scores(batch, bs, seed=67))
            pos += bs
            batch += 1
        ok, bad, n_tight = bounds_hold(t)
        assert ok and n_tight > 0, (again, bad)
        assert_same_table(t, ot, row_bytes)
        for step in range(12):
            k = one_per_bucket(oracle, w.unique_keys(680 + again, step * 400, 400), cap // 128)
            low = batch - step if step % 4 else batch + step  # falling, with a rise now and then
            upsert(t, ot, k, w.values_from_keys(k, dim), w.monotone_scores(low, len(k), seed=67))
            torch.cuda.synchronize()
            assert_same_table(t, ot, row_bytes)
        t.clear()
        assert t.size() == 0
    t.close()


@pytest.mark.parametrize("strategy", [EvictStrategy.kLfu, EvictStrategy.kEpochLfu])
def test_frequency_scores_and_bounds(oracle, strategy):
    """LFU / EpochLFU: a new key comes in with the caller's count, which under LFU may be below
    everything in its bucket (LFU never refuses); a key that is found only gains.  EpochLFU scores
    go down when the epoch is set back."""
    cap, dim, bs = 1 << 13, 4, 2048
    t, o = make(cap, dim, strategy)
    ot = oracle.OracleTable(o)
    vb = dim * 4
    epoch_lfu = strategy == EvictStrategy.kEpochLfu
    if epoch_lfu:
        t.set_global_epoch(3)
        ot.set_global_epoch(3)

    def distinct(b, n):
        return (np.uint64(b + 1) << np.uint64(20)) + np.random.Generator(np.random.PCG64(b)).permutation(n).astype(np.uint64)
    seed, pos, batch = 650, 0, 0
    while pos < cap + 4 * bs:
        k = w.unique_keys(seed, pos, bs)
        upsert(t, ot, k, w.values_from_keys(k, dim), distinct(batch, bs))
        pos += bs
        batch += 1
    assert_same_table(t, ot, vb)
    ok, bad, n_tight = bounds_hold(t)
    assert ok and n_tight > cap // 16 // 4, (bad, n_tight)
    # hits only: counts go up
    k = w.unique_keys(seed, pos - bs, bs)
    present = ot.contains(k)
    k = k[present]
    upsert(t, ot, k, w.values_from_keys(k, dim) + 2, distinct(40, len(k)))
    assert bounds_hold(t)[0]
    assert_same_table(t, ot, vb)
    if epoch_lfu:
        t.set_global_epoch(2)  # back: whatever is written now is below the rest
        ot.set_global_epoch(2)
    # new keys with counts below everything, one per bucket
    k = one_per_bucket(oracle, w.unique_keys(seed + 1, 0, 300), cap // 128)
    upsert(t, ot, k, w.values_from_keys(k, dim), np.arange(1, len(k) + 1, dtype=np.uint64))
    assert_same_table(t, ot, vb)
    if epoch_lfu:
        t.set_global_epoch(5)
        ot.set_global_epoch(5)
    # and new keys with high counts: under LFU the low ones above are what goes
    for rep in range(3):
        k = w.unique_keys(seed + 2, rep * 900, 900)
        upsert(t, ot, k, w.values_from_keys(k, dim), distinct(50 + rep, len(k)))
        ok, bad, _ = bounds_hold(t)
        assert ok, (rep, bad)
        assert_same_table(t, ot, vb)
    t.close()


def test_epoch_lru_bounds(oracle):
    """EpochLRU scores are (epoch << 32) | low half of clock >> 20: they grow while the epoch does
    not go back and the low half does not wrap.  Both are made to happen."""
    cap, dim, bs = 1 << 13, 4, 2048
    t, o = make(cap, dim, EvictStrategy.kEpochLru)
    ot = oracle.OracleTable(o)
    vb = dim * 4
    base = 1 << 44
    t.set_clock(1, base)
    ot.set_clock(1, base)
    seed, pos = 660, 0

    def epoch(e):
        t.set_global_epoch(e)
        ot.set_global_epoch(e)

    def step(n=bs, both=False):
        nonlocal pos
        k = w.unique_keys(seed, pos, n)
        if both:  # half from the latest batch, half new
            k = np.concatenate([w.unique_keys(seed, pos - n // 2, n // 2), k[: n - n // 2]])
        pos += n
        upsert(t, ot, k, w.values_from_keys(k, dim), None)

    epoch(1)
    while pos < cap + 3 * bs:
        step()
    assert_same_table(t, ot, vb)
    ok, bad, n_tight = bounds_hold(t)
    assert ok and n_tight > cap // 16 // 4, (bad, n_tight)
    epoch(2)
    for _ in range(3):
        step(both=True)
        assert bounds_hold(t)[0]
    assert_same_table(t, ot, vb)
    epoch(1)  # back: new scores below the old ones
    for _ in range(2):
        step()
        assert bounds_hold(t)[0]
        assert_same_table(t, ot, vb)
    epoch(3)
    step()  # (the latest batch holds low scores now: not what a batch should look for and evict at once)
    step(both=True)
    assert bounds_hold(t)[0]
    assert_same_table(t, ot, vb)
    # the low half of the clock wraps inside a call, and between calls
    wrap = (0xFFFFFFFF - 1000) << 20
    t.set_clock(1, wrap)
    ot.set_clock(1, wrap)
    for _ in range(2):  # the deterministic clock moves on by 2^40 ns = 2^20 units per call
        step()
        assert_same_table(t, ot, vb)
    epoch(4)  # above everything again, on the new side of the wrap
    step()
    assert bounds_hold(t)[0]
    step(both=True)
    assert bounds_hold(t)[0]
    assert_same_table(t, ot, vb)
    t.close()


@pytest.mark.parametrize("strategy,search", [(EvictStrategy.kLru, "bounds"), (EvictStrategy.kEpochLru, "bounds"),
                                             (EvictStrategy.kCustomized, "bounds"), (EvictStrategy.kLfu, "bounds"),
                                             (EvictStrategy.kEpochLfu, "bounds"), (EvictStrategy.kLru, "scan"),
                                             (EvictStrategy.kCustomized, "scan")])
def test_bounds_hold_under_arbitrary_scores(strategy, search, monkeypatch):
    """No oracle here (with scores that go up and down inside a batch the outcome depends on the order
    of its keys): 32 buckets and up to 1500 keys per call, i.e. some 47 keys of a call in every
    bucket; random scores from a small range (ties included), hits and new keys mixed, every call
    that writes scores, epochs that go back and forth; LRU and EpochLRU on the hardware clock.
    After every upsert: no bound is above a score of its line, no key is in the table twice, the
    table holds nothing but keys it held before and keys of the call, insert_and_evict accounts for
    every key that left, and every key that is found carries the row that was last written for it.
    "scan": the same with the score bounds switched off (the kernels that read all 128 scores)."""
    from gpu_util import export_table, host_u64
    if search == "scan":
        monkeypatch.setenv("HKV_SCORE_BOUNDS", "0")
    cap, dim = 1 << 12, 4
    t, o = make(cap, dim, strategy)
    rng = np.random.default_rng(1234 + int(strategy))
    universe = w.unique_keys(670, 0, 3 * cap)
    from_clock = strategy in (EvictStrategy.kLru, EvictStrategy.kEpochLru)
    epochs = strategy in (EvictStrategy.kEpochLfu, EvictStrategy.kEpochLru)
    if epochs:
        t.set_global_epoch(5)
    latest = {}
    used = 0
    resident = set()
    for step in range(80):
        n = int(rng.choice([17, 300, 1500]))
        keys = rng.choice(universe, size=n, replace=False)
        vals = rng.random((n, dim), dtype=np.float32)
        sc = rng.integers(1, 1 << int(rng.choice([4, 20, 40])), size=n, dtype=np.uint64)
        if epochs and step % 7 == 3:
            t.set_global_epoch(int(rng.integers(1, 9)))
        op = rng.choice(["insert_or_assign", "find_or_insert", "insert_and_evict", "accum_or_assign",
                         "assign", "assign_scores", "erase", "noalloc", "find_or_insert_ptr", "lock_unlock"],
                        p=[0.3, 0.08, 0.15, 0.1, 0.08, 0.07, 0.1, 0.04, 0.04, 0.04])
        dk, dv, ds = dev(keys), dev(vals), (None if from_clock else dev(sc))
        upsert_call = True
        evicted = None
        if op == "insert_or_assign":
            t.insert_or_assign(n, dk, dv, ds)
        elif op == "noalloc":
            try:
                t.insert_or_assign_noalloc(n, dk, dv, ds)
            except NotImplementedError:
                # after lock_keys the entry point that cannot wait refuses until an ordinary upsert
                # has read the count of locked slots back
                t.insert_or_assign(n, dk, dv, ds)
        elif op == "find_or_insert_ptr":
            ptrs = torch.zeros(n, dtype=torch.int64, device=DEV)
            founds = torch.zeros(n, dtype=torch.bool, device=DEV)
            t.find_or_insert_ptr(n, dk, ptrs, founds, ds)
        elif op == "lock_unlock":
            ptrs = torch.zeros(n, dtype=torch.int64, device=DEV)
            t.lock_keys(n, dk, ptrs, None, None, ds)
            t.unlock_keys(n, ptrs, dk)
            upsert_call = False
        elif op == "find_or_insert":
            t.find_or_insert(n, dk, dv, ds)
        elif op == "insert_and_evict":
            ek = torch.zeros(n, dtype=torch.int64, device=DEV)
            ev = torch.zeros(n, dim, dtype=torch.float32, device=DEV)
            es = torch.zeros(n, dtype=torch.int64, device=DEV)
            cnt = t.insert_and_evict(n, dk, dv, ds, ek, ev, es)
            evicted = host_u64(ek[:cnt]).tolist()
        elif op == "accum_or_assign":
            flags = torch.from_numpy(rng.random(n) < 0.5).to(DEV)
            t.accum_or_assign(n, dk, dv, flags, ds)
        elif op == "assign":
            t.assign(n, dk, dv, ds)
            upsert_call = False
        elif op == "assign_scores":
            t.assign_scores(n, dk, ds)
            upsert_call = False
        else:
            t.erase(n, dk)
            upsert_call = False
        used += n if upsert_call else 0
        if op in ("insert_or_assign", "insert_and_evict", "assign", "noalloc"):
            for k, v in zip(keys.tolist(), vals):
                latest[k] = v
        elif op in ("find_or_insert", "accum_or_assign", "erase", "find_or_insert_ptr"):
            for k in keys.tolist():
                latest.pop(k, None)  # (the row depends on whether the key was there: not tracked)
        gk, gv, _ = export_table(t, dim * 4)
        now = set(gk.tolist())
        batch = set(keys.tolist())
        assert len(now) == len(gk) == t.size() <= cap, (step, op)
        if op == "erase":
            assert now == resident - batch, (step, op)
        elif not upsert_call:
            assert now == resident, (step, op)
        else:
            assert now <= resident | batch, (step, op)
            if op == "accum_or_assign":
                pass  # which of its keys come in depends on their flags
            elif strategy == EvictStrategy.kLru:
                assert batch <= now, (step, op)  # the scores of the call are the highest: none is refused or evicted
        if evicted is not None:
            # Keys of other calls: the ones that left are exactly the ones handed back, once each.
            # Keys of this call (one may be evicted by another and come in again, or be refused):
            # one that is not there afterwards has been handed back.
            left = [k for k in evicted if k not in batch]
            assert len(set(left)) == len(left) and set(left) <= resident, (step, op)
            assert now - batch == (resident - batch) - set(left), (step, op)
            assert batch - now <= set(evicted), (step, op)
        resident = now
        rows = gv.view(np.float32).reshape(len(gk), dim)
        for k, row in zip(gk.tolist(), rows):
            if k in latest:
                assert np.array_equal(row, latest[k]), (step, op, k)
        # (made, and checked here, once upserts use them; the entry point that allocates nothing runs
        # another path, which leaves them to be made again by the next upsert)
        if search == "bounds" and upsert_call and used >= cap and op != "noalloc":
            ok, bad, _ = bounds_hold(t)
            assert ok, (step, op, bad)
    t.close()
