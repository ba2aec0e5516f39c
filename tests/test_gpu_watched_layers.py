"""Weight gradients of a first layer where something stands between the operators and the memory: batched gradients, a lazily
negated one, a recorded backward (``create_graph``), a dispatch mode; on both sides of 2 048 rows, from which on the library's
kernel was once taken whatever was watching."""
import numpy as np
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from hiscache.history_model import MyRGCNConvHistory2, MySageConvHistory

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
ROWS = (300, 2100)
F, H, K = 64, 64, 3


def layer(kind, rows, seed=0):
    """A layer over features and what its forward pass gives; its only gradients are its parameters'."""
    rng = np.random.default_rng(rows + seed)
    torch.manual_seed(rows)
    deg = rng.integers(0, 6, rows)
    ptr = torch.from_numpy(np.concatenate([[0], np.cumsum(deg)])).to(DEV)
    idx = torch.from_numpy(rng.integers(0, rows, int(deg.sum()))).to(DEV)
    x = torch.from_numpy(rng.standard_normal((rows, F)).astype(np.float32)).to(DEV)
    none = torch.empty(0, device=DEV)
    if kind == "sage":
        conv = MySageConvHistory(F, H, need_grad=False).to(DEV)
        return conv, list(conv.parameters()), lambda: conv(x, ptr, idx, none, none, 0, rows)[0]
    conv = MyRGCNConvHistory2(F, H, K, need_grad=False).to(DEV)
    types = torch.from_numpy(rng.integers(0, K, len(idx))).to(DEV)
    return conv, [conv.linear], lambda: conv(x, ptr, idx, types, None, None, None, None, 0, rows)[0]


def close(got, want, rows):
    # two sums of n products in different orders, each off by at most n half units of the sum of the magnitudes; for
    # zero-mean operands of unit size that sum is at most n times an entry's root mean square over sqrt(n)
    for a, b in zip(got, want):
        assert a.shape == b.shape
        assert float((a - b).norm()) <= rows ** 1.5 * 2.0 ** -23 * float(b.norm())


@pytest.mark.parametrize("rows", ROWS)
@pytest.mark.parametrize("kind", ("sage", "rgcn"))
def test_batched_gradients(kind, rows):
    _, params, run = layer(kind, rows)
    out = run()
    v = torch.randn(3, rows, H, device=DEV, generator=torch.Generator(device=DEV).manual_seed(1))
    got = torch.autograd.grad(out, params, v, is_grads_batched=True, retain_graph=True)
    for i in range(3):
        close([t[i] for t in got], torch.autograd.grad(out, params, v[i], retain_graph=True), rows)


@pytest.mark.parametrize("rows", ROWS)
@pytest.mark.parametrize("kind", ("sage", "rgcn"))
def test_a_negated_gradient(kind, rows):
    _, params, run = layer(kind, rows)
    out = run()
    v = torch.randn(rows, H, device=DEV, generator=torch.Generator(device=DEV).manual_seed(1))
    want = torch.autograd.grad(out, params, -v, retain_graph=True)
    close(torch.autograd.grad(out, params, torch._neg_view(v)), want, rows)


@pytest.mark.parametrize("rows", ROWS)
def test_a_recorded_backward(rows):
    conv, params, run = layer("sage", rows)
    second = {}
    for conv.fused in (True, False):                         # one node, and operator by operator
        first = torch.autograd.grad(run().square().sum(), params, create_graph=True)
        assert all(t.requires_grad for t in first)
        second[conv.fused] = torch.autograd.grad(sum(t.square().mean() for t in first), params)
    close(second[True], second[False], rows)


@pytest.mark.parametrize("rows", ROWS)
@pytest.mark.parametrize("kind", ("sage", "rgcn"))
def test_a_dispatch_mode_sees_the_products(kind, rows):
    class Seen(TorchDispatchMode):
        names = []

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.names.append(str(func))
            return func(*args, **(kwargs or {}))

    _, params, run = layer(kind, rows)
    out = run()
    Seen.names = []
    with Seen():
        torch.autograd.grad(out, params, torch.ones_like(out))
    assert any("mm" in n for n in Seen.names)


def test_what_lies_in_memory():
    import hiscache_backend as be
    x = torch.randn(4, 3, device=DEV)
    assert be.in_memory(x, None, x)
    assert not be.in_memory(torch._neg_view(x))
    assert not be.in_memory(x, torch._efficientzerotensor((4, 3), device=DEV))
    seen = []
    torch.func.vmap(lambda t: (seen.append(be.in_memory(x[0], t)), t)[1])(x)
    assert seen == [False]
