"""The sampler's tiles of 1024 rows and edge slots: hops that end at, before and behind a tile's end, hops of many
tiles, and capacities of more than 4096 tiles (whose sums are scanned by a launch of their own).  Bit for bit against
the sequential statement."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def graph(rng, nodes, deg, used):
    """``deg`` neighbours, among all nodes, for each of the first ``used`` nodes; the others have none."""
    indptr = np.minimum(np.arange(nodes + 1, dtype=np.int64), used) * deg
    return indptr, rng.integers(0, nodes, size=int(indptr[-1]), dtype=np.int64)


@pytest.mark.parametrize("nodes,deg,used,seeds,fanout", [
    (20_000, 8, 20_000, 128, [8, 4]),              # 1024 edges in the first hop
    (20_000, 8, 20_000, 127, [8, 1]),              # 1016
    (20_000, 9, 20_000, 129, [8, 9]),              # 1032, the rows of the second hop around a tile
    (60_000, 17, 60_000, 1025, [15, 10, 5]),       # several tiles of rows and many of edges
    (20_000, 30, 20_000, 300, [100, 500]),         # capacity of 10 M edge slots in the second hop
    (8_600_000, 40, 3_000, 3000, [2900, 2]),       # capacity of 8.6 M rows in the second hop
    (100, 3, 1, 7, [3, 3]),                        # all but one row empty
])
def test_tiles_of_every_shape(orc, nodes, deg, used, seeds, fanout):
    from hiscache import NeighborSampler
    rng = np.random.default_rng(seeds)
    indptr, indices = graph(rng, nodes, deg, used)
    sampler = NeighborSampler(indptr, indices, fanout, seed=3, device=DEV)
    for it in range(2):                            # the second batch finds the node map clean
        ids = rng.choice(max(used, seeds), size=seeds, replace=False).astype(np.int64)
        print("sampler tiles", nodes, seeds, fanout, it, flush=True)
        batch = sampler.sample(torch.from_numpy(ids).to(DEV))
        want = orc.sample_layers(indptr, indices, ids, fanout, sampler.batch_seed(it))
        np.testing.assert_array_equal(batch.ptr.cpu().numpy(), want["ptr"])
        np.testing.assert_array_equal(batch.idx.cpu().numpy(), want["idx"])
        np.testing.assert_array_equal(batch.sub_to_full.cpu().numpy(), want["sub_to_full"])
        np.testing.assert_array_equal(batch.num_node_in_layer.numpy(), want["num_node_in_layer"])
    assert int((sampler.node_map != 0x7fffffff).sum()) == 0
