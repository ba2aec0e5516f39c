"""Rows of several heads so long that their source rows are copied side by side before they are summed: bit for bit
against the oracle's sums in edge order, at lengths around the copies' units and the thresholds, in every element type,
with copies that do not all find room, and beside history rows."""
import numpy as np
import pytest
import torch

from test_gpu_long_rows import DEV, T, block

pytestmark = pytest.mark.gpu

# (at 300 000 edges rows above 2 048 edges are copied, above 2 432 with 128 columns and more, 64 edges at a time; the first two
# lie at the block's ends)
LENGTHS = [2049, 40_000, 2048, 2047, 2080, 2081, 2303, 2304, 2305, 100_001, 119_999, 5000, 3000, 129]
EDGE_LENGTHS = [2433, 40_000, 2432, 2431, 2495, 2496, 2497, 2559, 2560, 2561, 100_001, 119_999, 5000, 3000, 129]


@pytest.fixture(scope="module")
def be():
    import hiscache_backend
    hiscache_backend.load_library()
    return hiscache_backend


def check(be, orc, F, H, lengths, dtype=torch.float32, history=False, shift=0, R=5000):
    rng = np.random.default_rng(F * 10 + H)
    N = 700
    ptr, idx = block(rng, R, N, lengths)
    assert len(idx) >= 1 << 18                          # smaller blocks are never copied
    flat = torch.empty(N * H * F + shift, device=DEV, dtype=dtype)
    x = flat[shift:].view(N, H, F)
    x.copy_(T(rng.standard_normal((N, H, F)).astype(np.float32), dtype))
    ev = rng.standard_normal((len(idx), H)).astype(np.float32)
    hmap = hbuf = None
    if history:
        hmap = np.where(rng.random(R) < 0.3, 1, -1).astype(np.int64)
        hmap[0], hmap[R - 1] = -1, 1                    # one of the longest rows is served from the history
        hbuf = rng.standard_normal((R, H * F)).astype(np.float32)
    out = be._aggr_fwd(be.SUBST_ROW, T(ptr), T(idx), x, None if hmap is None else T(hmap),
                       None if hbuf is None else T(hbuf), H * F if history else 0, T(ev), R)
    ref = orc.fwd_edge_value(ptr, idx, ev, x.float().cpu().numpy(), hmap, hbuf, split_above=0)
    np.testing.assert_array_equal(out.cpu().numpy(), ref)


@pytest.mark.parametrize("F,H,dtype,shift", [(32, 4, torch.float32, 0), (8, 2, torch.float32, 0), (40, 3, torch.float32, 1),
                                             (32, 4, torch.float16, 0), (24, 2, torch.bfloat16, 3), (12, 4, torch.float32, 0)])
@pytest.mark.parametrize("lengths", (LENGTHS, EDGE_LENGTHS))
def test_staged_rows(be, orc, F, H, dtype, shift, lengths):
    check(be, orc, F, H, lengths, dtype, shift=shift)


def test_staged_rows_beside_history_rows(be, orc):
    check(be, orc, 32, 4, LENGTHS, history=True)


@pytest.mark.parametrize("lengths", ([9000, 40_000, 120_000, 100_001, 30_000, 9001], [120_000, 9000, 40_000, 100_001],
                                     [8100 + 137 * (i * 7 % 29) for i in range(30)],      # the four longest
                                     [8100 + 60 * (i * 7 % 27) for i in range(26)] + [13_000, 10_000, 12_500, 12_000]))      # the longest again
def test_copies_without_room(be, orc, lengths):
    """512 columns: 96 MB hold 48 000 edges, so that some of these rows, or all but the longest, are summed from the matrix."""
    check(be, orc, 64, 8, lengths)


def test_a_smaller_workspace_gives_the_same_bits(be):
    """hc_aggr_fwd_bounded and its workspace know nothing of copies."""
    rng = np.random.default_rng(3)
    R, N, F, H = 5000, 700, 32, 4
    ptr, idx = block(rng, R, N, LENGTHS)
    x, ev = T(rng.standard_normal((N, H, F)).astype(np.float32)), T(rng.standard_normal((len(idx), H)).astype(np.float32))
    lib, tp, ti = be.load_library(), T(ptr), T(idx)
    want = be._aggr_fwd(be.SUBST_ROW, tp, ti, x, None, None, 0, ev, R)
    size = lib.hc_aggr_fwd_workspace_bytes(be.SUBST_ROW, R, len(idx), N)
    ws = torch.empty(size, dtype=torch.uint8, device=DEV)
    for call, extra in ((lib.hc_aggr_fwd_bounded, ()), (lib.hc_aggr_fwd_for, (len(idx),))):
        out = torch.empty_like(want)
        assert call(be.SUBST_ROW, tp.data_ptr(), ti.data_ptr(), x.data_ptr(), 0, None, None, 0, 0, ev.data_ptr(), H,
                    out.data_ptr(), R, F, N, *extra, -1, ws.data_ptr(), size, be._stream()) == 0
        assert torch.equal(out, want)
