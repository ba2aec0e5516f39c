"""Rows side by side in the wave that draws their neighbours: fanouts at which they fill it, leave lanes over or take the
groups of sixteen, and row counts around a block's and a tile's (1024 rows)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("fanout", ([1], [2], [3, 5], [7], [16], [21, 2], [32], [33], [64], [100]))
@pytest.mark.parametrize("seeds", (1, 47, 1023, 1025, 2100))
def test_rows_side_by_side(orc, fanout, seeds):
    from hiscache import NeighborSampler
    rng = np.random.default_rng(seeds + fanout[0])
    nodes = 3000
    deg = np.minimum(rng.zipf(1.6, nodes), 400)
    deg[rng.random(nodes) < 0.1] = 0
    indptr = np.zeros(nodes + 1, np.int64)
    np.cumsum(deg, out=indptr[1:])
    indices = rng.integers(0, nodes, int(indptr[-1]))
    ids = rng.permutation(nodes)[:seeds].astype(np.int64)
    sampler = NeighborSampler(indptr, indices, fanout, seed=3, device=DEV)
    batch = sampler.sample(torch.from_numpy(ids).to(DEV))
    want = orc.sample_layers(indptr, indices, ids, fanout, sampler.batch_seed(0))
    np.testing.assert_array_equal(batch.ptr.cpu().numpy(), want["ptr"])
    np.testing.assert_array_equal(batch.idx.cpu().numpy(), want["idx"])
    np.testing.assert_array_equal(batch.sub_to_full.cpu().numpy(), want["sub_to_full"])
