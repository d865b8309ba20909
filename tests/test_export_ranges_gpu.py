"""export_batch_if over ranges on both sides of the size from which a workgroup takes a larger part of them (2^20 slots),
with ends that are no multiple of either part, against the same slots exported in small pieces without a condition."""
import pytest
import torch

from gpu_util import DEV
from hierarchicalkv_amd import EvictStrategy, HashTable, Predicate, default_options

pytestmark = pytest.mark.gpu
CAPACITY = 1 << 21
PIECE = 1 << 18


def export(t, dim, n, offset, threshold=None, scores=True):
    count = torch.full((1,), 77, dtype=torch.int64, device=DEV)
    room = min(n, CAPACITY - offset) + 1  # one more than can match: it has to stay as it is
    keys = torch.full((room,), -5, dtype=torch.int64, device=DEV)
    rows = torch.full((room, dim), -5.0, dtype=torch.float32, device=DEV)
    out = torch.full((room,), -5, dtype=torch.int64, device=DEV) if scores else None
    if threshold is None:
        t.export_batch(n, offset, count, keys, rows, out)
    else:
        t.export_batch_if(Predicate.kScoreGe, 0, threshold, n, offset, count, keys, rows, out)
    m = int(count.item())
    assert bool((keys[m:] == -5).all()) and bool((rows[m:] == -5).all())
    order = torch.argsort(keys[:m])
    return keys[:m][order], rows[:m][order], out[:m][order] if scores else None


# (rows of more than 512 bytes keep the smaller part)
@pytest.mark.parametrize("dim", [16, 3, 65, 128, 129])
def test_export_ranges(dim):
    t = HashTable()
    t.init(default_options(init_capacity=CAPACITY, max_capacity=CAPACITY, max_hbm_for_vectors=1 << 34, dim=dim,
                           evict_strategy=EvictStrategy.kCustomized))
    for at in range(0, CAPACITY * 3 // 4, PIECE):
        keys = torch.arange(at, at + PIECE, dtype=torch.int64, device=DEV) * 2654435761 + 1
        rows = (keys % 8191)[:, None].float() + torch.arange(dim, device=DEV)
        t.insert_or_assign(PIECE, keys, rows, scores=keys % 1000)
    for offset, n in ((0, CAPACITY), (0, (1 << 20) - 1), (0, 1 << 20), (0, (1 << 20) + 1), (1, CAPACITY),
                      (4097, (1 << 20) + 2047), (777, (1 << 20) + 4095), (CAPACITY - (1 << 20) - 3, 1 << 21)):
        end = min(CAPACITY, offset + n)
        pieces = [export(t, dim, min(PIECE, end - a), a) for a in range(offset, end, PIECE)]
        keys, rows, scores = (torch.cat(x) for x in zip(*pieces))
        order = torch.argsort(keys)
        keys, rows, scores = keys[order], rows[order], scores[order]
        for threshold in (0, 500, 990, 1000):
            match = scores >= threshold
            got = export(t, dim, n, offset, threshold, scores=threshold != 500)
            assert torch.equal(got[0], keys[match]) and torch.equal(got[1], rows[match])
            assert got[2] is None or torch.equal(got[2], scores[match])
