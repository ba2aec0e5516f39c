"""Long rows of the forward aggregation, every way they can be shared out: looked up by the front blocks
themselves (few rows), listed and sliced, listed whole (large blocks: rows between 256 edges and 1/8192 of the
block), summed by the row's own block (no workspace).  Bit for bit against the oracle's statement of the
summation order, at widths whose rows need every vector width and column tile."""
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


def none():
    return torch.empty(0, device=DEV)


def block(rng, R, N, lengths, mean=4):
    """R rows of up to 2 * mean edges with rows of ``lengths`` edges planted at the ends and in between."""
    deg = rng.integers(0, 2 * mean + 1, size=R)
    at = np.concatenate([[0, R - 1], rng.choice(np.arange(1, R - 1), size=len(lengths) - 2, replace=False)])
    deg[at] = lengths
    ptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int64)
    return ptr, rng.integers(0, N, size=int(ptr[-1]), dtype=np.int64)


LENGTHS = [257, 1000, 255, 256, 64, 63, 65, 128, 129, 5000, 1024, 271]


@pytest.mark.parametrize("F,dtype", [(1, torch.float32), (31, torch.float32), (33, torch.bfloat16), (47, torch.float16),
                                     (64, torch.bfloat16), (100, torch.float32), (100, torch.float16),
                                     (130, torch.float32), (256, torch.float32), (258, torch.bfloat16),
                                     (602, torch.float32), (1030, torch.float32), (2056, torch.float16)])
@pytest.mark.parametrize("R", [300, 5000])
def test_mean_rows(be, orc, F, dtype, R):
    rng = np.random.default_rng(F + R)
    N = 700
    ptr, idx = block(rng, R, N, LENGTHS)
    x = T(rng.standard_normal((N, F)).astype(np.float32), dtype)
    hmap = np.where(rng.random(R) < 0.2, 3, -1).astype(np.int64)
    hmap[0], hmap[R - 1] = -1, 5                       # a long row that is summed, one that takes its history row
    hbuf = rng.standard_normal((R, F)).astype(np.float32)
    out = be._aggr_fwd(be.SUBST_ROW, T(ptr), T(idx), x, T(hmap), T(hbuf), F, None, R)
    x32 = x.float().cpu().numpy()
    ref = orc.fwd_mean_row(ptr, idx, x32, hmap, hbuf, split_above=be.long_row_edges(F, dtype))
    np.testing.assert_array_equal(out.cpu().numpy(), ref)
    # no scratch at all: the same bits from the rows' own blocks
    lib = be.load_library()
    out2 = torch.full((R, F), float("nan"), device=DEV)
    th, tb, tp, ti = T(hmap), T(hbuf), T(ptr), T(idx)
    rc = lib.hc_aggr_fwd(0, tp.data_ptr(), ti.data_ptr(), x.data_ptr(), be._DTYPES[dtype], th.data_ptr(), tb.data_ptr(), 0, F,
                         None, 1, out2.data_ptr(), R, F, N, None, 0, torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    assert torch.equal(out, out2)


@pytest.mark.parametrize("F", [24, 100])
def test_large_block_uses_both_lists(be, orc, F):
    """More than 2 M edges: rows up to 1/8192 of them are listed whole, longer ones sliced."""
    rng = np.random.default_rng(F)
    R, N = 90_000, 3000
    ptr, idx = block(rng, R, N, [300, 290, 257, 256, 9000, 2000, 280, 281, 282, 283], mean=27)
    total = int(ptr[-1])
    far = max(256, total // 8192)
    assert far > 270
    deg = np.diff(ptr)
    deg[[7, 8]] = [far, far + 1]
    ptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int64)
    idx = rng.integers(0, N, size=int(ptr[-1]), dtype=np.int64)
    x = rng.standard_normal((N, F)).astype(np.float32)
    out = be._aggr_fwd(be.SUBST_ROW, T(ptr), T(idx), T(x), None, None, 0, None, R)
    np.testing.assert_array_equal(out.cpu().numpy(), orc.fwd_mean_row(ptr, idx, x, None, None, split_above=256))


@pytest.mark.parametrize("F,H", [(32, 4), (16, 3), (47, 2), (100, 5), (64, 1), (100, 1), (3, 1)])
@pytest.mark.parametrize("R", [300, 5000])
def test_weighted_rows(be, orc, F, H, R):
    """Heads: rows above 128 edges sliced, never split (slices inside one head and across heads); a single head
    follows the quarter rule."""
    rng = np.random.default_rng(F + H + R)
    N = 500
    ptr, idx = block(rng, R, N, LENGTHS)
    E = len(idx)
    multi = H > 1
    x = rng.standard_normal((N, H, F) if multi else (N, F)).astype(np.float32)
    ev = rng.standard_normal((E, H) if multi else (E,)).astype(np.float32)
    out = be._aggr_fwd(be.SUBST_ROW, T(ptr), T(idx), T(x), None, None, 0, T(ev), R)
    ref = orc.fwd_edge_value(ptr, idx, ev, x, None, None, split_above=0 if multi else be.long_row_edges(F))
    np.testing.assert_array_equal(out.cpu().numpy(), ref)


@pytest.mark.parametrize("F,table", [(256, torch.float32), (100, torch.float16), (47, torch.bfloat16), (130, torch.float32)])
@pytest.mark.parametrize("R", [300, 5000])
def test_source_substitution_rows(be, orc, F, table, R):
    rng = np.random.default_rng(F + R)
    N, Hn = 900, 200
    ptr, idx = block(rng, R, N, LENGTHS)
    x = rng.standard_normal((N, F)).astype(np.float32)
    hist = T(rng.standard_normal((Hn, F)).astype(np.float32), table)
    hmap = np.where(rng.random(N) < 0.4, rng.integers(0, Hn, size=N), -1).astype(np.int64)
    out = be.aggr_forward_source_history(T(x), T(ptr), T(idx), T(hmap), hist)
    ref = orc.fwd_mean_src(ptr, idx, x, hmap, hist.float().cpu().numpy(), split_above=be.long_row_edges(F))
    np.testing.assert_array_equal(out.cpu().numpy(), ref)


def test_bounded_degree_is_one_launch_with_the_same_bits(be, orc):
    rng = np.random.default_rng(9)
    R, N, F = 6000, 800, 100
    ptr, idx = block(rng, R, N, [128, 127, 1, 100])
    x = T(rng.standard_normal((N, F)).astype(np.float32))
    free = be._aggr_fwd(be.SUBST_ROW, T(ptr), T(idx), x, None, None, 0, None, R)
    bound = be._aggr_fwd(be.SUBST_ROW, T(ptr), T(idx), x, None, None, 0, None, R, max_degree=128)
    assert torch.equal(free, bound)
    np.testing.assert_array_equal(free.cpu().numpy(), orc.fwd_mean_row(ptr, idx, x.cpu().numpy(), None, None))


def test_unaligned_rows(be, orc):
    """A feature matrix that starts at an odd element: narrower loads, the same bits."""
    rng = np.random.default_rng(10)
    R, N, F = 400, 300, 128
    ptr, idx = block(rng, R, N, LENGTHS)
    for dtype in (torch.float32, torch.float16):
        flat = T(rng.standard_normal(N * F + 3).astype(np.float32), dtype)
        x = flat[3:].view(N, F)
        out = be._aggr_fwd(be.SUBST_ROW, T(ptr), T(idx), x, None, None, 0, None, R)
        ref = orc.fwd_mean_row(ptr, idx, x.float().cpu().numpy(), None, None, split_above=256)
        np.testing.assert_array_equal(out.cpu().numpy(), ref)


@pytest.mark.parametrize("F,dtype", [(64, torch.float32), (128, torch.float32), (256, torch.float32), (1024, torch.float32),
                                     (512, torch.bfloat16), (47, torch.float16)])
def test_rows_of_every_short_length(be, orc, F, dtype):
    """0 to 70 edges: every remainder of a batch of 16, 8 and 4 rows in flight, plain and weighted, a head and two."""
    rng = np.random.default_rng(F)
    N = 300
    deg = rng.permutation(np.repeat(np.arange(71), 3))
    ptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int64)
    R, E = len(deg), int(ptr[-1])
    idx = rng.integers(0, N, size=E, dtype=np.int64)
    x = T(rng.standard_normal((N, F)).astype(np.float32), dtype)
    x32 = x.float().cpu().numpy()
    out = be._aggr_fwd(be.SUBST_ROW, T(ptr), T(idx), x, None, None, 0, None, R)
    np.testing.assert_array_equal(out.cpu().numpy(), orc.fwd_mean_row(ptr, idx, x32, None, None))
    hist = T(rng.standard_normal((40, F)).astype(np.float32), dtype)
    hmap = np.where(rng.random(N) < 0.4, rng.integers(0, 40, size=N), -1).astype(np.int64)
    out = be.aggr_forward_source_history(x, T(ptr), T(idx), T(hmap), hist)
    np.testing.assert_array_equal(out.cpu().numpy(), orc.fwd_mean_src(ptr, idx, x32, hmap, hist.float().cpu().numpy()))
    for H in ((1,) if F % 2 else (1, 2)):
        ev = rng.standard_normal((E, H) if H > 1 else (E,)).astype(np.float32)
        shape = (N, H, F // H) if H > 1 else (N, F)
        out = be._aggr_fwd(be.SUBST_ROW, T(ptr), T(idx), x.view(shape), None, None, 0, T(ev), R)
        np.testing.assert_array_equal(out.cpu().numpy(), orc.fwd_edge_value(ptr, idx, ev, x32.reshape(shape), None, None))


def test_rows_behind_four_gigabytes(be):
    """Features of more than 4 GiB, whose rows the slices address in 64 bits: the bits of the same call over the matrix's
    last rows alone, which are addressed in 32."""
    rng = np.random.default_rng(11)
    N, few, R, F = (1 << 24) + 777, 500, 300, 64
    ptr, idx = block(rng, R, few, LENGTHS)
    x = torch.empty(N, F, device=DEV)
    x[N - few:] = torch.randn(few, F, device=DEV)
    tp, far, near = T(ptr), T(idx + (N - few)), T(idx)
    for H in (0, 1, 4):
        ev = T(rng.random((len(idx), H) if H > 1 else len(idx)).astype(np.float32)) if H else None
        out = [be._aggr_fwd(be.SUBST_ROW, tp, ids, m.view(-1, H, F // H) if H > 1 else m, None, None, 0, ev, R)
               for ids, m in ((far, x), (near, x[N - few:]))]
        assert torch.equal(*out), H
