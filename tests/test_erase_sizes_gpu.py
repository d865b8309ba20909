"""erase at the batch sizes where its kernel changes (keys of a tile and of a wavefront, 2^14, 2^17):
exactly the keys of the batch are gone, a key that is named twice or is absent harms nobody."""
import numpy as np
import pytest
import torch

import workloads as w
from gpu_util import DEV, dev
from hierarchicalkv_amd import HashTable, default_options

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("api_lock", [1, 0])
@pytest.mark.parametrize("n", [1, 7, 8, 9, 16, 17, 65, 1 << 14, (1 << 14) + 1, (1 << 17) - 1, 1 << 17])
def test_exactly_the_batch_is_gone(n, api_lock):
    cap = 1 << 19
    t = HashTable()
    t.init(default_options(init_capacity=cap, max_capacity=cap, max_hbm_for_vectors=1 << 30, dim=4, api_lock=api_lock))
    keys = w.unique_keys(97, 0, 200000)
    t.insert_or_assign(len(keys), dev(keys), torch.zeros(len(keys), 4, device=DEV))
    assert t.size() == len(keys)
    rng = np.random.default_rng(n)
    gone = rng.choice(len(keys), n, replace=False)
    batch = keys[gone]
    if n >= 9:
        batch[1] = batch[0]  # in one tile
        batch[n - 1] = w.unique_keys(98, 0, 1)[0]  # not in the table
        gone = np.delete(gone, [1, n - 1])
    t.erase(n, dev(batch))
    present = torch.zeros(len(keys), dtype=torch.bool, device=DEV)
    t.contains(len(keys), dev(keys), present)
    want = np.ones(len(keys), bool)
    want[gone] = False
    assert (present.cpu().numpy() == want).all()
    assert t.size() == want.sum()
    t.close()
