"""Buckets of sources that hold more edges than a compute unit gets on average, sorted in parts: one id per bucket (a part
cannot be split), fewer ids than parts, many; popular sources next to each other, at the front, in the middle and at the end
of the ids, one source with almost all edges; so many heavy
buckets that there are fewer parts than they ask for, down to one; bit-exact against NumPy's stable sort."""
import numpy as np
import pytest
import torch

from test_gpu_view_sort import T, be, stable_view  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,where,share", [(20, 0, 0.0), (3_000, 0, 0.5), (6_000, 2_999, 0.9), (40_000, 20_000, 0.3),
                                           (250_003, 0, 0.2), (1_000_003, 1_000_000, 0.1), (9_000_000, 4_000_000, 0.5)])
@pytest.mark.parametrize("spread", (1, 3, 200))
@pytest.mark.parametrize("want_edges", (False, True))
def test_heavy_buckets(be, N, where, share, spread, want_edges):
    rng = np.random.default_rng(N + spread)
    R = 40_000
    deg = rng.poisson(32, size=R).astype(np.int64)
    ptr = np.zeros(R + 1, np.int64)
    np.cumsum(deg, out=ptr[1:])
    E = int(ptr[-1])
    idx = rng.integers(0, N, size=E, dtype=np.int64)
    popular = rng.random(E) < share
    idx[popular] = np.minimum(where + rng.integers(0, spread, size=int(popular.sum())), N - 1)
    check(be, rng, ptr, idx, R, N, want_edges)


@pytest.mark.parametrize("N", (250_003, 1_000_003, 9_000_000))
@pytest.mark.parametrize("hubs,share", ((20, 0.5), (60, 0.8), (90, 0.95)))
@pytest.mark.parametrize("want_edges", (False, True))
def test_many_heavy_buckets(be, N, hubs, share, want_edges):
    # 900 000 live slots, 156 blocks for parts: 20 buckets of 23 000 pairs ask for 320, 60 of 12 000 for 480, 90 of 9 500 for 720
    rng = np.random.default_rng(N + hubs)
    R = 40_000
    deg = rng.poisson(32, size=R).astype(np.int64)
    ptr = np.zeros(R + 1, np.int64)
    np.cumsum(deg, out=ptr[1:])
    idx = rng.integers(0, N, size=int(ptr[-1]), dtype=np.int64)
    popular = rng.random(len(idx)) < share
    where = np.arange(hubs) * (N // hubs) + rng.integers(0, N // hubs, size=hubs)
    idx[popular] = where[rng.integers(0, hubs, size=int(popular.sum()))]
    check(be, rng, ptr, idx, R, N, want_edges)


def check(be, rng, ptr, idx, R, N, want_edges):
    E = len(idx)
    hrow = np.where(rng.random(R) < 0.3, 1, -1).astype(np.int64)
    ptrT, rowT, edgeT = be.build_transpose(T(ptr), T(idx), T(hrow), R, N, num_edge=E, want_edges=want_edges)
    want_ptr, want_edge, want_row = stable_view(ptr, idx, R, N, E, hrow)
    live = len(want_edge)
    np.testing.assert_array_equal(ptrT.cpu().numpy(), want_ptr)
    np.testing.assert_array_equal(rowT.cpu().numpy()[:live], want_row)
    if want_edges:
        np.testing.assert_array_equal(edgeT.cpu().numpy()[:live], want_edge)
