"""The backward aggregation's division of the sources among the waves: long sources (by column slices, in chunks or
strictly in order), runs of sources cut by their edges, and the plain runs of a call without scratch memory.  Bit for
bit against the oracle's summation order, at widths that need every vector width and column tile, and with the
gradient stored in each element type (one rounding of the fp32 sum)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.fixture(scope="module")
def be():
    import hiscache_backend
    hiscache_backend.load_library()
    return hiscache_backend


def T(a, dtype=None):
    t = torch.from_numpy(np.ascontiguousarray(a)).to(DEV)
    return t if dtype is None else t.to(dtype)


# in-degrees around every threshold: 64 edges of a stage, 128 (long), 512 (chunk), four chunks of a block's waves,
# 4096 (several blocks) and its multiples
DEGREES = {0: 1700, 1: 513, 2: 512, 3: 129, 4: 128, 5: 127, 6: 65, 7: 0, 8: 64, 9: 2048, 10: 2049, 300: 640,
           301: 4096, 302: 4097, 303: 8192, 304: 23456, -3: 9000, -1: 2600, -2: 1}


def block(rng, R, N, extra=4):
    """A block of R rows over N sources whose first, last and some inner sources have DEGREES edges."""
    count = rng.integers(0, 2 * extra + 1, size=N)
    count[200:260] = 0                                    # a stretch of sources without edges
    for s, d in DEGREES.items():
        count[s] = d
    idx = np.repeat(np.arange(N, dtype=np.int64), count)
    rng.shuffle(idx)
    cut = np.sort(rng.integers(0, len(idx) + 1, size=R - 1))
    return np.concatenate([[0], cut, [len(idx)]]).astype(np.int64), idx


def maps(rng, R, F):
    hmap = np.where(rng.random(R) < 0.2, 3, -1).astype(np.int64)
    return hmap, rng.standard_normal((R, F)).astype(np.float32)


def special(rng, R, F):
    """Gradient rows of ordinary values, with infinities, NaN, the largest and tiny values among them."""
    g = rng.standard_normal((R, F)).astype(np.float32)
    at = rng.integers(0, R, size=6)
    for r, v in zip(at, (np.inf, -np.inf, np.nan, 3.0e38, -0.0, 1e-30)):
        g[r, rng.integers(0, F)] = v
    return g


@pytest.mark.parametrize("F", [1, 16, 31, 47, 64, 100, 128, 130, 256, 300, 602, 1030])
@pytest.mark.parametrize("R,N", [(3000, 900), (20000, 30000)])
def test_mean(be, orc, F, R, N):
    rng = np.random.default_rng(F + R)
    ptr, idx = block(rng, R, N)
    hmap, _ = maps(rng, R, 1)
    g = special(rng, R, F)
    chunk = be.bwd_chunk_edges(F)
    view = be.build_batch_view(T(ptr), T(idx), R, N)
    ref_view, ref_h = orc.bwd_mean_row_batch_view(ptr, idx, g, hmap, N, R, hbuf_shape=(R, F), chunk=chunk)
    gx, gh = be._aggr_bwd_batch_view(T(ptr), view, T(g), T(hmap), (R, F), F, R, N)
    np.testing.assert_array_equal(gx.cpu().numpy(), ref_view)
    np.testing.assert_array_equal(gh.cpu().numpy(), ref_h)
    tr = be.build_transpose(T(ptr), T(idx), T(hmap), R, N, want_edges=False)
    ref, _ = orc.bwd_mean_row(ptr, idx, g, hmap, N, hbuf_shape=(R, F), chunk=chunk)
    out, _, _ = be._aggr_bwd(T(ptr), T(idx), tr, T(g), T(hmap), None, None, False, (R, F), F, R, N)
    np.testing.assert_array_equal(out.cpu().numpy(), ref)
    for dtype in (torch.float16, torch.bfloat16):
        half, _, _ = be._aggr_bwd(T(ptr), T(idx), tr, T(g), T(hmap), None, None, False, (R, F), F, R, N, dtype=dtype)
        want = torch.from_numpy(ref).to(dtype)
        assert torch.equal(torch.nan_to_num(half.cpu().float()), torch.nan_to_num(want.float()))
        assert torch.equal(half.cpu().isnan(), want.isnan())
        other, _ = be._aggr_bwd_batch_view(T(ptr), view, T(g), T(hmap), (R, F), F, R, N, dtype=dtype)
        assert torch.equal(torch.nan_to_num(other.cpu().float()),
                           torch.nan_to_num(torch.from_numpy(ref_view).to(dtype).float()))


@pytest.mark.parametrize("F", [47, 128])
@pytest.mark.parametrize("room", ["none", "lists"])
def test_scratch_of_each_size(be, orc, F, room):
    """Without scratch every source is summed strictly in order; with the lists alone the runs are of equal length."""
    rng = np.random.default_rng(F)
    R, N = 4000, 900
    ptr, idx = block(rng, R, N)
    g = rng.standard_normal((R, F)).astype(np.float32)
    tp, tg = T(ptr), T(g)
    ptrT, rowT, _ = be.build_transpose(tp, T(idx), None, R, N, want_edges=False)
    lib = be.load_library()
    nbytes = lib.hc_aggr_bwd_workspace_bytes(rowT.numel(), F)
    assert 0 < nbytes < lib.hc_aggr_bwd_workspace_bytes_for(rowT.numel(), F, N)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=DEV)
    out = torch.full((N, F), float("nan"), device=DEV)
    rc = lib.hc_aggr_bwd(tp.data_ptr(), None, ptrT.data_ptr(), rowT.data_ptr(), None, tg.data_ptr(), None, None, None, 0,
                         1, out.data_ptr(), None, 0, None, rowT.numel(), R, F, N,
                         None if room == "none" else ws.data_ptr(), 0 if room == "none" else nbytes,
                         torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    ref, _ = orc.bwd_mean_row(ptr, idx, g, None, N, chunk=0 if room == "none" else be.bwd_chunk_edges(F))
    np.testing.assert_array_equal(out.cpu().numpy(), ref)


@pytest.mark.parametrize("F,H", [(32, 4), (16, 3), (47, 2), (100, 5), (64, 1), (100, 1), (3, 1), (1, 70)])
def test_weighted(be, orc, F, H):
    """Weighted sums keep the order of the rows whatever a source's length; slices inside a head and across heads."""
    rng = np.random.default_rng(F + H)
    R, N = 3000, 900
    ptr, idx = block(rng, R, N)
    multi = H > 1
    x = rng.standard_normal((N, H, F) if multi else (N, F)).astype(np.float32)
    ev = rng.standard_normal((len(idx), H) if multi else (len(idx),)).astype(np.float32)
    g = rng.standard_normal((R, H, F) if multi else (R, F)).astype(np.float32)
    hmap = np.where(rng.random(R) < 0.2, 3, -1).astype(np.int64)
    tr = be.build_transpose(T(ptr), T(idx), T(hmap), R, N)
    gx, gh, eg = be._aggr_bwd(T(ptr), T(idx), tr, T(g), T(hmap), T(ev), T(x), True, (R, F * H), F * H, R, N)
    ref, ref_h, ref_e = orc.bwd_edge_value(ptr, idx, ev, g, hmap, x, N, hsize=F * H, want_edge_grad=True)
    np.testing.assert_array_equal(gx.cpu().numpy(), ref)
    np.testing.assert_array_equal(gh.cpu().numpy().reshape(ref_h.shape), ref_h)
    # (F products in any order against the oracle's: each within (F + 2) ulp/2 of the sum of their magnitudes)
    row = np.repeat(np.arange(R), np.diff(ptr))
    size = np.abs(g.reshape(R, H, F)[row].astype(np.float64) * x.reshape(N, H, F)[idx]).sum(2)
    size[hmap[row] != -1] = 0.0
    far = np.abs(eg.cpu().numpy().reshape(-1, H).astype(np.float64) - ref_e.reshape(-1, H))
    assert (far <= 2 * (F + 2) * 2.0 ** -24 * size).all()


def test_unaligned_gradient(be, orc):
    """An upstream gradient that starts at an odd element: narrower loads, the same bits."""
    rng = np.random.default_rng(11)
    R, N, F = 3000, 900, 128
    ptr, idx = block(rng, R, N)
    flat = T(rng.standard_normal(R * F + 3).astype(np.float32))
    g = flat[3:].view(R, F)
    tr = be.build_transpose(T(ptr), T(idx), None, R, N, want_edges=False)
    gx, _, _ = be._aggr_bwd(T(ptr), T(idx), tr, g, None, None, None, False, None, 0, R, N)
    np.testing.assert_array_equal(gx.cpu().numpy(), orc.bwd_mean_row(ptr, idx, g.cpu().numpy(), None, N,
                                                                     chunk=be.bwd_chunk_edges(F))[0])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_half_precision_features_through_autograd(be, orc, dtype):
    rng = np.random.default_rng(12)
    R, N, F = 3000, 900, 100
    ptr, idx = block(rng, R, N)
    x = T(rng.standard_normal((N, F)).astype(np.float32), dtype).requires_grad_(True)
    g = rng.standard_normal((R, F)).astype(np.float32)
    be.aggr_forward_history(x, T(ptr), T(idx), torch.empty(0, device=DEV), torch.empty(0, device=DEV), 0, R).backward(T(g))
    assert x.grad.dtype == dtype
    ref, _ = orc.bwd_mean_row(ptr, idx, g, None, N, chunk=be.bwd_chunk_edges(F))
    assert torch.equal(x.grad.cpu(), torch.from_numpy(ref).to(dtype))


@pytest.mark.parametrize("F", [64, 100])
def test_layer_without_rows_over_a_view_of_long_sources(be, F):
    """Every edge of the view is stepped over and there is no gradient row: zeros, whatever the sources' lengths."""
    rng = np.random.default_rng(13)
    R, N = 3000, 900
    ptr, idx = block(rng, R, N)
    tp, ti = T(ptr), T(idx)
    view = be.build_batch_view(tp, ti, R, N)
    lib = be.load_library()
    ws = torch.empty(lib.hc_aggr_bwd_workspace_bytes_for(len(idx), F, N), dtype=torch.uint8, device=DEV)
    out = torch.full((N, F), float("nan"), device=DEV)
    rc = lib.hc_aggr_bwd_batch_view(tp.data_ptr(), view.ptrT.data_ptr(), view.rowT.data_ptr(), None, None, out.data_ptr(),
                                    None, 0, len(idx), 0, F, N, ws.data_ptr(), ws.numel(),
                                    torch.cuda.current_stream().cuda_stream)
    assert rc == 0 and not out.any()
    none = torch.empty(0, device=DEV)
    x = T(rng.standard_normal((N, F)).astype(np.float32)).requires_grad_(True)
    y = be.aggr_forward_history(x, tp[:1], ti, none, none, 0, 0, view=view)
    assert y.shape == (0, F)
    y.sum().backward()
    assert x.grad.shape == (N, F) and not x.grad.any()


@pytest.mark.parametrize("F", [47, 128])
@pytest.mark.parametrize("runs", [False, True])
@pytest.mark.parametrize("announced", [200, 5000])
def test_view_of_more_entries_than_announced(be, orc, F, runs, announced):
    """The lists and runs are sized by the caller's number of entries; a view that holds more is summed without them,
    strictly in order, with nothing left out and nothing written behind the scratch."""
    rng = np.random.default_rng(F)
    R, N = 4000, 9000
    ptr, idx = block(rng, R, N)
    g = rng.standard_normal((R, F)).astype(np.float32)
    tp, tg = T(ptr), T(g)
    view = be.build_batch_view(tp, T(idx), R, N)
    lib = be.load_library()
    need = (lib.hc_aggr_bwd_workspace_bytes_for(announced, F, N) if runs else lib.hc_aggr_bwd_workspace_bytes(announced, F))
    ws = torch.full((need + 4096,), 0x5a, dtype=torch.uint8, device=DEV)
    want, _ = orc.bwd_mean_row(ptr, idx, g, None, N, chunk=0)
    st = torch.cuda.current_stream().cuda_stream
    for masked in (False, True):
        out = torch.full((N, F), float("nan"), device=DEV)
        if masked:
            rc = lib.hc_aggr_bwd_batch_view(tp.data_ptr(), view.ptrT.data_ptr(), view.rowT.data_ptr(), tg.data_ptr(), None,
                                            out.data_ptr(), None, 0, announced, R, F, N, ws.data_ptr(), need, st)
        else:
            rc = lib.hc_aggr_bwd(tp.data_ptr(), None, view.ptrT.data_ptr(), view.rowT.data_ptr(), None, tg.data_ptr(), None,
                                 None, None, 0, 1, out.data_ptr(), None, 0, None, announced, R, F, N, ws.data_ptr(), need, st)
        assert rc == 0
        np.testing.assert_array_equal(out.cpu().numpy(), want)
        assert (ws[need:] == 0x5a).all()


@pytest.mark.parametrize("F", [64, 100])
def test_underflowing_gradient(be, orc, F):
    """Gradients around and below the smallest normal number.  A subnormal quotient is one of the two numbers next to
    the exact one, and sums of subnormals are exact: a source of n edges lies within n * 2^-149 of the divisions' sum.
    Above, the quotients are the divisions' and the sums have the same bits."""
    rng = np.random.default_rng(14)
    R, N = 3000, 900
    ptr, idx = block(rng, R, N)
    count = np.bincount(idx, minlength=N)[:, None]
    tr = be.build_transpose(T(ptr), T(idx), None, R, N, want_edges=False)
    longest = int(np.diff(ptr).max())
    for low, high in ((0, 40), (0, 1 << 13), (longest << 23, longest << 25)):      # in units of 2^-149
        g = np.ldexp(rng.integers(low, high, size=(R, F)).astype(np.float32), -149)
        gx, _, _ = be._aggr_bwd(T(ptr), T(idx), tr, T(g), None, None, None, False, None, 0, R, N)
        ref, _ = orc.bwd_mean_row(ptr, idx, g, None, N, chunk=be.bwd_chunk_edges(F))
        if low == 0:
            assert np.abs(ref).max() < 2.0 ** -125              # (up to there the sums are exact)
            assert (np.abs(gx.cpu().numpy().astype(np.float64) - ref) <= count * 2.0 ** -149).all()
        else:
            np.testing.assert_array_equal(gx.cpu().numpy(), ref)


@pytest.mark.parametrize("F", [64, 100, 256])
@pytest.mark.parametrize("rows", [1, 40, 700, 2999, 3000])
def test_inner_layer_over_a_view_of_long_sources(be, orc, F, rows):
    """A layer that owns a few of the view's rows: stretches of hundreds of positions without a live edge, stages put
    together from several of them, and (all rows) stages taken as they come."""
    rng = np.random.default_rng(rows + F)
    R, N = 3000, 900
    ptr, idx = block(rng, R, N)
    hmap = np.where(rng.random(rows) < 0.2, 3, -1).astype(np.int64)
    g = special(rng, rows, F)
    view = be.build_batch_view(T(ptr), T(idx), R, N)
    want, _ = orc.bwd_mean_row_batch_view(ptr, idx, g, hmap, N, R, hbuf_shape=(rows, F), chunk=be.bwd_chunk_edges(F))
    for m in (hmap, None):
        if m is None:
            want, _ = orc.bwd_mean_row_batch_view(ptr, idx, g, m, N, R, chunk=be.bwd_chunk_edges(F))
        gx, _ = be._aggr_bwd_batch_view(T(ptr), view, T(g), None if m is None else T(m), None, 0, rows, N,
                                        want_hist_grad=False)
        np.testing.assert_array_equal(gx.cpu().numpy(), want)


def test_gradient_rows_behind_four_gigabytes(be):
    """A gradient of more than 4 GiB, whose rows the slices address in 64 bits: the bits of the same call over its last
    rows alone, which are addressed in 32."""
    rng = np.random.default_rng(15)
    few, N, F = 2000, 900, 64
    ptr, idx = block(rng, few, N)
    R = (1 << 24) + 4321
    skip = R - few
    wide = torch.cat([torch.zeros(skip, dtype=torch.int64, device=DEV), T(ptr)])
    g = torch.empty(R, F, device=DEV)
    g[skip:] = torch.randn(few, F, device=DEV)
    ti, E = T(idx), len(idx)
    for H in (0, 1, 4):
        ev = T(rng.random((E, H) if H > 1 else E).astype(np.float32)) if H else None
        out = []
        for p, gr, n in ((wide, g, R), (T(ptr), g[skip:], few)):
            gr = gr.view(n, H, F // H) if H > 1 else gr
            tr = be.build_transpose(p, ti, None, n, N, want_edges=H > 0)
            out.append(be._aggr_bwd(p, ti, tr, gr, None, ev, None, False, None, 0, n, N)[0])
        assert torch.equal(*out), H
    views = [be.build_batch_view(p, ti, n, N) for p, n in ((wide, R), (T(ptr), few))]
    out = [be._aggr_bwd_batch_view(p, v, gr, None, None, 0, n, N)[0]
           for p, v, gr, n in ((wide, views[0], g, R), (T(ptr), views[1], g[skip:], few))]
    assert torch.equal(*out)
