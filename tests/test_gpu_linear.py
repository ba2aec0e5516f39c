"""hc_linear against the product in float64: edges of the tiles and of the pieces of the inner dimension, both layouts of
the weight, one and two products, bias, accumulation, misaligned operands."""
import pytest
import torch

import hiscache_backend as be

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

# M, N, K: results up to 2^19 go in tiles of 32 x 32 with pieces of 128 columns, more in tiles of 64 x 64 with pieces of 32
SIZES = [(1, 1, 1), (31, 33, 3), (32, 32, 128), (33, 31, 129), (65, 47, 132), (1000, 172, 256), (513, 10, 100),
         (2049, 256, 31), (2049, 256, 32), (4161, 129, 33), (8200, 65, 100), (2500, 255, 256), (11200, 47, 7)]


@pytest.mark.parametrize("M,N,K", SIZES)
@pytest.mark.parametrize("transposed", (False, True))
def test_linear_matches_the_float64_product(M, N, K, transposed):
    gen = torch.Generator().manual_seed(M * 1000 + N * 10 + K)

    def rnd(*shape):
        return torch.randn(*shape, generator=gen)

    ws = (K, N) if transposed else (N, K)
    a0, a1, w0, w1, bias, base = rnd(M, K), rnd(M, K), rnd(*ws), rnd(*ws), rnd(N), rnd(M, N)
    # operands that start 4 bytes behind a 16-byte boundary
    shifted = torch.empty(M * K + 1, device=DEV)[1:].view(M, K).copy_(a0)
    dev = [t.to(DEV) for t in (a0, w0, a1, w1, bias, base)]
    op = (lambda w: w.double()) if transposed else (lambda w: w.double().t())
    one, two = a0.double() @ op(w0), a1.double() @ op(w1)
    size = a0.double().abs() @ op(w0).abs(), a1.double().abs() @ op(w1).abs()
    # a sum of K products, each rounded once with its addition, is off by at most K half units of the sum of the
    # magnitudes, and each of the up to three additions behind it by half a unit of what is added
    unit = 2.0 ** -24

    def close(got, want, bound):
        assert bool(((got.cpu().double() - want).abs() <= 1.01 * bound * unit).all())

    got = be.linear(dev[0], dev[1], transposed=transposed)
    close(got, one, K * size[0])
    assert torch.equal(be.linear(shifted, dev[1], transposed=transposed), got)       # the order depends on nothing else
    assert torch.equal(be.linear(dev[0][: (M + 1) // 2], dev[1], transposed=transposed), got[: (M + 1) // 2])
    got = be.linear(dev[0], dev[1], dev[2], dev[3], dev[4], transposed=transposed)
    close(got, one + two + bias.double(), (K + 2) * (size[0] + size[1]) + bias.double().abs())
    res = be.linear(dev[0], dev[1], transposed=transposed, out=dev[5])
    assert res.data_ptr() == dev[5].data_ptr()
    close(res, base.double() + one, (K + 1) * size[0] + base.double().abs())


def test_linear_leaves_what_lies_behind_the_result():
    M, N, K = 65, 33, 10
    room = torch.full((M * N + 64,), 7.0, device=DEV)
    be.linear(torch.ones(M, K, device=DEV), torch.ones(N, K, device=DEV), out=room[: M * N].view(M, N))
    assert bool((room[: M * N] == 17.0).all()) and bool((room[M * N:] == 7.0).all())


def test_linear_refuses_what_does_not_fit():
    a, w = torch.ones(5, 8, device=DEV), torch.ones(3, 8, device=DEV)
    for call in (lambda: be.linear(a, w, transposed=True), lambda: be.linear(a, w, a), lambda: be.linear(a.half(), w),
                 lambda: be.linear(a, w, a[:4], w), lambda: be.linear(a, w, bias=torch.ones(2, device=DEV)),
                 lambda: be.linear(a, w, out=torch.ones(5, 4, device=DEV)), lambda: be.linear(a, w.t().contiguous().t())):
        with pytest.raises(ValueError):
            call()
    assert be.linear(a[:0], w).shape == (0, 3)


@pytest.mark.parametrize("watch", ("autocast", "dispatch"))
def test_a_layer_under_autocast_or_a_dispatch_mode_keeps_its_operators(watch):
    from torch.utils._python_dispatch import TorchDispatchMode

    from hiscache.history_model import MySageConvHistory

    class Seen(TorchDispatchMode):
        def __init__(self):
            super().__init__()
            self.names = []

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.names.append(str(func))
            return func(*args, **(kwargs or {}))

    conv = MySageConvHistory(8, 4, need_grad=False, root_weight=watch != "autocast").to(DEV)
    x, ptr, idx = torch.randn(4, 8, device=DEV), torch.tensor([0, 1, 3], device=DEV), torch.tensor([2, 3, 1], device=DEV)
    none = torch.empty(0, device=DEV)
    if watch == "autocast":
        with torch.autocast("cuda", dtype=torch.float16):
            assert conv(x, ptr, idx, none, none, 0, 2)[0].dtype == torch.float16
    else:
        with Seen() as seen:
            conv(x, ptr, idx, none, none, 0, 2)
        assert any("mm" in n for n in seen.names)


@pytest.mark.parametrize("M,N,K", ((300, 64, 47), (300, 47, 64), (9000, 64, 47), (9000, 68, 64), (700, 32, 65), (17_000, 32, 129),
                                   (40_001, 4, 63), (65, 1, 64), (2100, 256, 10)))
@pytest.mark.parametrize("transposed", (False, True))
def test_every_operand_off_its_boundary_by_itself(M, N, K, transposed):
    """Loads of either operand and stores are 16 bytes wide or not, each by its own width and address: the same bits."""
    gen = torch.Generator(device=DEV).manual_seed(M + N + K)

    def rnd(*shape):
        return torch.randn(*shape, device=DEV, generator=gen)

    def off(t):
        return torch.empty(t.numel() + 1, device=DEV)[1:].view(t.shape).copy_(t)

    ws = (K, N) if transposed else (N, K)
    a, w, b, c, bias, base = rnd(M, K), rnd(*ws), rnd(M, K), rnd(*ws), rnd(N), rnd(M, N)
    kw = dict(transposed=transposed)
    want, added = be.linear(a, w, b, c, bias, **kw), be.linear(a, w, out=base.clone(), **kw)
    op = (lambda t: t.double()) if transposed else (lambda t: t.double().t())
    size = a.double().abs() @ op(w).abs() + b.double().abs() @ op(c).abs() + bias.double().abs()
    exact = a.double() @ op(w) + b.double() @ op(c) + bias.double()
    assert bool(((want.double() - exact).abs() <= 1.01 * (K + 2) * 2.0 ** -24 * size).all())
    for i in range(5):
        ops = [off(t) if i == k else t for k, t in enumerate((a, w, b, c, bias))]
        assert torch.equal(be.linear(*ops, **kw), want)
    assert torch.equal(be.linear(a, w, out=off(base), **kw), added)


def test_tall_products_of_odd_widths_stay_with_the_library():
    def takes(M, N, K, transposed):
        with torch.no_grad():
            return be.linear_supported(torch.empty(M, K, device=DEV), torch.empty((K, N) if transposed else (N, K), device=DEV),
                                       transposed=transposed)

    assert takes(1000, 172, 256, False) and takes(1000, 256, 47, True) and takes(20_000, 256, 129, False)
    assert not takes(100_000, 256, 99, False) and not takes(100_000, 256, 47, True) and not takes(100_000, 99, 256, True)
    assert takes(100_000, 99, 256, False) and takes(200_000, 256, 100, True) and not takes(1000, 64, 602 + 1, False)
    # W [K, N] of an odd N and a long inner size, and few columns of a long inner size
    assert takes(300, 255, 512, True) and takes(2000, 602, 252, True) and not takes(2000, 602, 256, True)
    assert takes(1000, 602, 256, True) and not takes(1000, 602, 512, True) and takes(2000, 602, 256, False)
    assert takes(5000, 47, 768, False) and not takes(20_000, 47, 768, False) and not takes(20_000, 64, 516, False)
    assert takes(20_000, 32, 768, False) and takes(20_000, 65, 768, False) and takes(20_000, 47, 512, False)


@pytest.mark.parametrize("M", (40, 9000))
@pytest.mark.parametrize("transposed", (False, True))
def test_a_product_by_itself_is_two_chains(M, transposed):
    # 2^27 in the first column: what is added to it four columns at a time is less than half a unit (16) and lost, but only
    # in the chain that holds it, 128 of 256 columns; the other chain is exact
    K, N = 256, 64
    a = torch.ones(M, K, device=DEV)
    a[:, 0] = 2.0 ** 27
    got = be.linear(a, torch.ones((K, N) if transposed else (N, K), device=DEV), transposed=transposed)
    assert float((got.double() - (2.0 ** 27 + K - 1)).abs().max()) <= 128


@pytest.mark.parametrize("N", (4, 64))
@pytest.mark.parametrize("transposed", (False, True))
def test_rows_behind_2_to_the_31_elements(N, transposed):
    """Both operands' rows and, with 64 columns, the result's: the bits of the same rows by themselves."""
    K, M = 64, (1 << 25) + 70
    a = torch.randn(M, K, device=DEV)
    w, c = (torch.randn(*((K, N) if transposed else (N, K)), device=DEV) for _ in range(2))
    one, two = be.linear(a, w, transposed=transposed), be.linear(a, w, a, c, transposed=transposed)
    for rows in (slice(0, 200), slice((1 << 25) - 130, M)):
        part = a[rows].contiguous()
        assert torch.equal(one[rows], be.linear(part, w, transposed=transposed))
        assert torch.equal(two[rows], be.linear(part, w, part, c, transposed=transposed))
