"""What insert_and_evict hands out on a full table: every key comes with its own row, a key that was refused with the
caller's, either with its score, and nothing is lost.  Rows on both sides of the sizes up to which a trip keeps all its rows in registers (512
bytes with one key per tile, 256 with two), batches on both sides of the sizes for one, two and eight keys per tile."""
import pytest
import torch

from gpu_util import DEV
from hierarchicalkv_amd import EvictStrategy, HashTable, Predicate, default_options

pytestmark = pytest.mark.gpu
CAPACITY = 1 << 17


def keys_of(lo, hi):
    return torch.arange(lo, hi, dtype=torch.int64, device=DEV) * 0x9E3779B97F4A7C1 + 3


def rows_of(keys, row_bytes):
    col = torch.arange(row_bytes, dtype=torch.int64, device=DEV)
    return ((keys[:, None] >> (col % 48)) + col * 37).to(torch.uint8)


def score_in(keys, scores, wanted):
    """The scores of the wanted keys, -1 for those that are not among the keys."""
    if keys.numel() == 0:
        return torch.full_like(wanted, -1)
    keys, order = torch.sort(keys)
    at = torch.searchsorted(keys, wanted).clamp_(max=keys.numel() - 1)
    return torch.where(keys[at] == wanted, scores[order][at], -1)


@pytest.mark.parametrize("row_bytes", [3, 12, 128, 129, 256, 260, 512, 516])
def test_rows_that_leave(row_bytes):
    t = HashTable()
    t.init(default_options(init_capacity=CAPACITY, max_capacity=CAPACITY, max_hbm_for_vectors=1 << 32, dim=row_bytes,
                           value_kind=0, value_size=1, evict_strategy=EvictStrategy.kCustomized))
    at = 0
    held = torch.empty(0, dtype=torch.int64, device=DEV)
    held_scores = torch.empty(0, dtype=torch.int64, device=DEV)
    gen = torch.Generator(device=DEV)
    gen.manual_seed(row_bytes)
    for step, n in enumerate((100000, 100000, 1001, (1 << 15) - 3, (1 << 15) + 5, 50021, 1 << 17, (1 << 18) + 7)):
        new = keys_of(at, at + n - n // 4)
        at += n - n // 4
        old = held[torch.randperm(held.numel(), device=DEV, generator=gen)[:n // 4]]
        keys = torch.cat([new, old])
        keys = keys[torch.randperm(keys.numel(), device=DEV, generator=gen)]
        n = keys.numel()
        scores = torch.randint(1, 1 << 20, (n,), device=DEV, generator=gen) + (step << 30)
        scores[torch.rand(n, device=DEV, generator=gen) < 0.05] = 0  # refused where their bucket is full
        ek = torch.full((n + 1,), -1, dtype=torch.int64, device=DEV)
        ev = torch.full((n + 1, row_bytes), 0xA5, dtype=torch.uint8, device=DEV)
        es = torch.full((n + 1,), -1, dtype=torch.int64, device=DEV)
        gone = t.insert_and_evict(n, keys, rows_of(keys, row_bytes), scores, ek, ev, es)
        assert bool((ek[gone:] == -1).all()) and bool((ev[gone:] == 0xA5).all()) and bool((es[gone:] == -1).all())
        assert torch.equal(ev[:gone], rows_of(ek[:gone], row_bytes))
        # evicted: the score it had before the call; refused, or evicted again after the call put it in: the caller's
        had, given, left = score_in(held, held_scores, ek[:gone]), score_in(keys, scores, ek[:gone]), es[:gone]
        assert bool(((left >= 0) & ((left == had) | (left == given))).all())
        count = torch.zeros(1, dtype=torch.int64, device=DEV)
        ok = torch.zeros(CAPACITY, dtype=torch.int64, device=DEV)
        ov = torch.zeros(CAPACITY, row_bytes, dtype=torch.uint8, device=DEV)
        os_ = torch.zeros(CAPACITY, dtype=torch.int64, device=DEV)
        t.export_batch_if(Predicate.kAlways, 0, 0, CAPACITY, 0, count, ok, ov, os_)
        m = int(count.item())
        assert torch.equal(ov[:m], rows_of(ok[:m], row_bytes))
        # (a key that was found, evicted and inserted again in one call comes out as often)
        everything = torch.unique(torch.cat([held, keys]))
        # what was not in the batch still has its score
        now, before, given = os_[:m], score_in(held, held_scores, ok[:m]), score_in(keys, scores, ok[:m])
        assert torch.equal(now, torch.where(given >= 0, given, before))
        held, held_scores = ok[:m], now
        assert held.unique().numel() == m
        assert torch.equal(torch.unique(torch.cat([held, ek[:gone]])), everything)
    assert gone > 0 and held.numel() > CAPACITY * 0.99
