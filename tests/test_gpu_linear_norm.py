"""A layer's dense half with the evaluation's batch normalisation behind it: the bits of the two calls, and the model's use
of it."""
from types import SimpleNamespace

import numpy as np
import pytest
import torch

import hiscache_backend as be

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("M,N,K", ((1, 4, 1), (33, 36, 129), (1000, 256, 100), (2050, 256, 33), (8200, 68, 100), (300, 47, 64),
                                   (12_000, 47, 20)))
@pytest.mark.parametrize("two,affine,bias", ((True, True, True), (False, False, False), (True, False, True)))
def test_norm_behind_the_product(M, N, K, two, affine, bias):
    gen = torch.Generator(device=DEV).manual_seed(M + N + K)

    def rnd(*shape):
        return torch.randn(*shape, device=DEV, generator=gen)

    a = rnd(M, K), rnd(N, K), rnd(M, K) if two else None, rnd(N, K) if two else None
    b, mean, var = rnd(N) if bias else None, rnd(N), torch.rand(N, device=DEV, generator=gen) + 0.1
    gamma, beta = (rnd(N), rnd(N)) if affine else (None, None)
    a[0][0, 0] = float("nan")
    a[0][M - 1, K - 1] = float("inf") if M > 1 else float("nan")
    got = be.linear(*a, b, norm=(gamma, beta, mean, var, 1e-5))
    x = be.linear(*a)
    if N % 4 == 0:
        want = be.bias_bn_relu_eval(x, b, gamma, beta, mean, var, 1e-5)
    else:                                        # the same steps, one rounding each, in fp32
        want = (x if b is None else x + b) - mean
        want = want * (1.0 / torch.sqrt(var + 1e-5))
        want = want * gamma + beta if affine else want * 1.0 + 0.0
        want = torch.where(want < 0, torch.zeros_like(want), want)
    assert torch.equal(got.nan_to_num(nan=-1.0), want.nan_to_num(nan=-1.0))


def test_norm_refuses_what_does_not_fit():
    a, w, v = torch.ones(5, 8, device=DEV), torch.ones(3, 8, device=DEV), torch.ones(3, device=DEV)
    for kw in (dict(norm=(v[:2], v, v, v, 1e-5)), dict(norm=(v, v, v, v.double(), 1e-5)),
               dict(norm=(v, v, v, v, 1e-5), out=torch.ones(5, 3, device=DEV))):
        with pytest.raises(ValueError):
            be.linear(a, w, **kw)


@pytest.mark.parametrize("bias", (True, False))
def test_evaluation_normalises_on_the_way_out(bias, monkeypatch):
    from hiscache import HistorySAGE, make_config
    from hiscache.synthetic import direct_power_law_batch, make_batch
    n, width, hidden, classes, layers = 20_000, 100, 64, 8, 3
    rng = np.random.default_rng(5)
    smp = direct_power_law_batch(n, 100, [5, 4, 3], 2.0, 9, degree_scale=2.0)
    torch.manual_seed(6)
    model = HistorySAGE(width, hidden, classes, layers, 0.0, "CSR_Layer", make_config(width, classes, hidden, layers, device=DEV),
                        SimpleNamespace(method=""), bias=bias).to(DEV).eval()
    for bn in model.bns:
        bn.running_mean.normal_()
        bn.running_var.uniform_(0.5, 2.0)
    b = make_batch(smp, rng.integers(0, classes, size=n), DEV)
    b.x = torch.from_numpy(rng.standard_normal((len(smp["sub_to_full"]), width)).astype(np.float32)).to(DEV)
    norms = []
    real = be.linear
    monkeypatch.setattr(be, "linear", lambda *a, **k: (norms.append("norm" in k), real(*a, **k))[1])
    with torch.no_grad():
        got = model(b)
        assert norms == [True, True, False]
        monkeypatch.setattr(HistorySAGE, "_evaluated", lambda *a: None)
        assert torch.equal(model(b), got)
