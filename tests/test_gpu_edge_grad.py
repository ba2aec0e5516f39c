"""The gradient of the edge weights at every division of the lanes among heads and columns, against fp64.  Bound: a
sum of F products in any order differs from the exact one by at most (F + 2) ulp/2 of the sum of their magnitudes."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("F,H", [(1, 1), (16, 1), (47, 1), (64, 1), (100, 1), (256, 1), (602, 1), (1030, 1), (32, 4), (16, 3),
                                 (47, 2), (100, 5), (1, 70), (8, 8), (256, 2), (3, 64)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_against_fp64(F, H, dtype):
    import hiscache_backend as be
    rng = np.random.default_rng(F + 100 * H)
    R, N, slack = 700, 300, 37
    deg = rng.integers(0, 9, size=R)
    deg[[0, 5, R - 1]] = [130, 700, 64]
    deg[20:60] = 0
    ptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int64)
    E = int(ptr[-1])
    idx = rng.integers(0, N, size=E + slack, dtype=np.int64)           # slots behind the last row get 0
    hmap = np.where(rng.random(R) < 0.2, 1, -1).astype(np.int64)
    x = torch.from_numpy(rng.standard_normal((N, H, F)).astype(np.float32)).to(dtype)
    g = rng.standard_normal((R, H, F)).astype(np.float32)
    ev = rng.standard_normal((E + slack, H)).astype(np.float32)
    T = lambda a: (torch.from_numpy(a) if isinstance(a, np.ndarray) else a).to(DEV).contiguous()
    multi = H > 1
    xt, gt, et = T(x if multi else x[:, 0]), T(g if multi else g[:, 0]), T(ev if multi else ev[:, 0])
    tr = be.build_transpose(T(ptr), T(idx), T(hmap), R, N)
    _, _, eg = be._aggr_bwd(T(ptr), T(idx), tr, gt, T(hmap), et, xt, True, (R, F * H), F * H, R, N, want_hist_grad=False)
    row = np.repeat(np.arange(R), deg)
    prod = g[row].astype(np.float64) * x.float().numpy()[idx[:E]].astype(np.float64)
    prod[hmap[row] != -1] = 0.0
    want, bound = prod.sum(2), (F + 2) * 2.0 ** -24 * np.abs(prod).sum(2)
    got = eg.cpu().numpy().reshape(E + slack, H).astype(np.float64)
    assert (np.abs(got[:E] - want) <= bound).all()
    assert (got[E:] == 0).all() and (got[:E][hmap[row] != -1] == 0).all()
