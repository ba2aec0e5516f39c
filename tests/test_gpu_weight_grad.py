"""hc_weight_grad at the edges of its pieces (32 rows), matrix instructions (4 rows) and slabs (64 rows), with operands off
16-byte boundaries, and the relational layer's weight gradient through it."""
import pytest
import torch

import hiscache_backend as be
from hiscache import history_model as hm

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _close(got, g, x, n):
    # n products and their additions in fp32, each off by at most half a unit of the sum of magnitudes
    bound = 1.01 * (n + 1) * 2.0 ** -24 * (g.double().abs().t() @ x.double().abs())
    assert bool(((got.double() - g.double().t() @ x.double()).abs() <= bound).all())


@pytest.mark.parametrize("n", (1, 3, 4, 5, 31, 32, 33, 63, 65, 96, 127, 129, 1025, 16_390))
@pytest.mark.parametrize("H,F", ((64, 64), (128, 192)))
def test_weight_grad_at_the_edges_of_pieces_and_slabs(n, H, F):
    gen = torch.Generator(device=DEV).manual_seed(n + H)
    g, x0, x1 = (torch.randn(n, c, device=DEV, generator=gen) for c in (H, F, F))
    both = be.weight_grad(g, x0, x1)
    for got, x in zip(both, (x0, x1)):
        _close(got, g, x, n)
    shifted = torch.empty(n * H + 1, device=DEV)[1:].view(n, H).copy_(g)
    assert all(torch.equal(a, b) for a, b in zip(be.weight_grad(shifted, x0, x1), both))


@pytest.mark.parametrize("n,K,F,H", ((1, 5, 64, 64), (301, 5, 128, 64), (4_200, 5, 768, 256), (90, 3, 20, 64), (2_100, 5, 64, 10)))
def test_relational_weight_gradient(n, K, F, H):
    gen = torch.Generator(device=DEV).manual_seed(n + F)
    agg, g = torch.randn(n, K, F, device=DEV, generator=gen), torch.randn(n, H, device=DEV, generator=gen)
    with torch.no_grad():
        got = hm._rel_weight_grad(agg, g)
    assert tuple(got.shape) == (K, F, H)
    _close(got.view(K * F, H), agg.view(n, K * F), g, n)


@pytest.mark.parametrize("n,KF,H,own", ((1000, 1280, 256, False), (2047, 640, 64, False), (2048, 640, 64, True), (2047, 1280, 256, False),
                                        (2048, 1280, 256, True), (3000, 1920, 256, False), (4200, 1920, 256, True),
                                        (4200, 3840, 64, True), (4200, 3840, 256, False), (30_000, 3840, 256, False)))
def test_relational_weight_gradient_by_the_faster_of_the_two(n, KF, H, own, monkeypatch):
    calls = []
    real = be.weight_grad
    monkeypatch.setattr(be, "weight_grad", lambda *a: (calls.append(1), real(*a))[1])
    agg, g = torch.randn(n, 5, KF // 5, device=DEV), torch.randn(n, H, device=DEV)
    with torch.no_grad():
        got = hm._rel_weight_grad(agg, g)
    assert bool(calls) == own
    _close(got.view(KF, H), agg.view(n, KF), g, n)


@pytest.mark.parametrize("n", (1, 5, 33, 64, 1000, 4097))
@pytest.mark.parametrize("H,F", ((1, 64), (10, 128), (47, 64), (63, 64), (65, 128), (153, 256), (172, 256), (256, 64)))
def test_linear_grad_for_any_number_of_outputs(n, H, F):
    gen = torch.Generator(device=DEV).manual_seed(n + H)
    g, x0, x1 = (torch.randn(n, c, device=DEV, generator=gen) for c in (H, F, F))
    d0, d1, db = be.linear_grad(g, x0, x1, True)
    _close(d0, g, x0, n)
    _close(d1, g, x1, n)
    assert db.shape == (H,)
    _close(db.view(H, 1), g, torch.ones(n, 1, device=DEV), n)
    e0, e1, none = be.linear_grad(torch.empty(n * H + 1, device=DEV)[1:].view(n, H).copy_(g), x0, x1, False)
    assert none is None and torch.equal(e0, d0) and torch.equal(e1, d1)      # the order depends on nothing else


def test_linear_grad_refuses_what_does_not_fit():
    g, x = torch.randn(9, 10, device=DEV), torch.randn(9, 64, device=DEV)
    for call in (lambda: be.linear_grad(g, x, x[:8], True), lambda: be.linear_grad(g, x[:8], x[:8], True),
                 lambda: be.linear_grad(g.half(), x, x, True), lambda: be.linear_grad(g, x[:, :32].contiguous(), x[:, :32].contiguous(), True)):
        with pytest.raises(ValueError):
            call()


@pytest.mark.parametrize("H,F", ((1024, 1024), (2048, 512)))
def test_long_slabs_are_summed_in_short_chains(H, F):
    # 256 tiles of dW leave four slabs of 2 048 rows.  2^27 in the first row: what is added to it four rows at a time is less
    # than half a unit (16) and lost, which must not be more than the first chain's 256 rows; chains' sums are added exactly
    n = 8192
    g, x = torch.ones(n, H, device=DEV), torch.ones(n, F, device=DEV)
    g[0] = 2.0 ** 27
    err = (be.weight_grad(g, x).double() - (2.0 ** 27 + n - 1)).abs()
    assert float(err.max()) <= 256


@pytest.mark.parametrize("n", (1, 65, 1000, 4097, 16_390))
@pytest.mark.parametrize("H,F", ((64, 64), (47, 128), (172, 64)))
def test_whole_numbers_are_summed_exactly(n, H, F):
    """Odd numbers up to 4 095, which half-precision types do not hold, and few enough of them that every partial sum is exact:
    a row left out, taken twice or rounded shows."""
    gen = torch.Generator(device=DEV).manual_seed(n + H)

    def odd(c):
        return 2.0 * torch.randint(-2048, 2048, (n, c), device=DEV, generator=gen) + 1.0

    def few(c):
        share = min(1.0, 2.0 ** 23 / (4095 * n))
        return torch.randint(0, 2, (n, c), device=DEV, generator=gen).mul(2).sub(1) * (
            torch.rand(n, c, device=DEV, generator=gen) < share).float()

    for g, x0, x1 in ((odd(H), few(F), few(F)), (few(H), odd(F), odd(F))):
        d0, d1, db = be.linear_grad(g, x0, x1, True)
        for got, x in ((d0, x0), (d1, x1), (db.view(H, 1), torch.ones(n, 1, device=DEV))):
            assert torch.equal(got.double(), g.double().t() @ x.double())
        if H % 64 == 0:
            assert torch.equal(be.weight_grad(g, x0), d0)
