"""Rows that share a load (two or four of them per wave access): widths at the edges of a half and a quarter wave, row counts
at the edges of a wave's sixteen, masked rows, ids without a row, rows left to the other tier."""
import pytest
import torch

import hiscache_backend as be

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("F", (4, 60, 64, 68, 100, 124, 128, 132, 66))
@pytest.mark.parametrize("n", (1, 15, 16, 17, 1003))
@pytest.mark.parametrize("dtype", (torch.float32, torch.float16, torch.bfloat16))
def test_narrow_rows(F, n, dtype):
    gen = torch.Generator().manual_seed(F * 1000 + n)
    nodes, held = 500, 200
    x = torch.randn(nodes, F, generator=gen).to(dtype)
    ids = torch.randint(0, nodes, (n,), generator=gen)
    ids[n // 2] = nodes                                       # no such row: cleared
    ids[0] = -1                                               # counts from the end
    mask = torch.rand(n, generator=gen) < 0.7
    known = mask & (ids < nodes)
    at = ids.clamp(max=nodes - 1) % nodes
    want = torch.where(known[:, None], x.float()[at], torch.zeros(()))
    got = be.gather_rows(x.to(DEV), ids.to(DEV), mask.to(DEV))
    assert torch.equal(got.cpu(), want)
    slot = torch.full((nodes,), -1, dtype=torch.int32)
    owners = torch.randperm(nodes, generator=gen)[:held]
    slot[owners] = torch.arange(held, dtype=torch.int32)
    out = torch.full((n, F), 3.0, device=DEV, dtype=dtype)
    _, cold = be.gather_rows_hot(x[owners].to(DEV), slot.to(DEV), ids.to(DEV), mask.to(DEV), out=out)
    left = known & (slot[at] < 0)
    assert torch.equal(cold.cpu().bool(), left)
    assert torch.equal(out.cpu(), torch.where(left[:, None], torch.full((), 3.0), want).to(dtype))
