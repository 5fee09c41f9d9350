"""The ordering of up to one block's pairs (`moe_order`), which takes its histogram from the wavefronts' counts: a lone pair and a lone
expert, wavefronts that are whole or not, experts around a wavefront's 64 lanes, ids beyond the experts, the first size of two chunks."""
import numpy as np
import pytest
import torch

import nuvec_amd as nv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pairs,experts", [(1, 1), (1024, 1), (63, 2), (65, 64), (1023, 65), (1024, 300), (1024, 900), (1025, 33), (2048, 129)])
@pytest.mark.parametrize("kind", ["spread", "one", "beyond"])
def test_order_of_one_chunk(pairs, experts, kind):
    rng = np.random.default_rng(pairs + experts)
    ids = rng.integers(0, experts, size=pairs).astype(np.int32)
    if kind == "one":
        ids[:] = experts - 1
    elif kind == "beyond":  # (clamped to the last expert)
        ids[::3] = experts + 5
    order, restore, sorted_ids, offsets = nv.moe_order(torch.from_numpy(ids).cuda(), experts)
    ids = np.minimum(ids, experts - 1)
    want = np.argsort(ids, kind="stable")
    inverse = np.empty(pairs, dtype=np.int64)
    inverse[want] = np.arange(pairs)
    assert np.array_equal(order.cpu().numpy(), want)
    assert np.array_equal(restore.cpu().numpy(), inverse)
    assert np.array_equal(sorted_ids.cpu().numpy(), ids[want])
    assert np.array_equal(offsets.cpu().numpy(), np.searchsorted(ids[want], np.arange(experts), side="left"))
