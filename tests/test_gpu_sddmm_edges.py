"""The edge-list SDDMM at the sizes where its shapes meet: chunks that end inside a 128-bit word, heads side by side and in
blocks, edge counts around a batch and around what a wavefront stages, results placed through edge_pos, operands that
start on any float, 32-bit and 64-bit row offsets, non-finite rows next to the words a lane drops."""
import ctypes

import numpy as np
import pytest

from helpers import assert_sum_close

pytestmark = pytest.mark.gpu

# (heads, head length): lanes per head 2 / 4 / 8 / 16 / 32 (see lanes_per_head), whole and ragged chunks, one and several of
# them; blocks of heads (3, 5, 6, 12 heads, more heads than a wavefront has groups, more than it stages); 1 .. 3 floats
SHAPES = [(1, 1), (1, 3), (1, 4), (1, 5), (1, 8), (1, 9), (1, 16), (1, 17), (1, 31), (1, 32), (1, 33), (1, 48), (1, 64), (1, 65), (1, 96),
          (1, 100), (1, 127), (1, 130), (1, 160), (1, 239), (1, 338), (2, 8), (8, 8), (3, 16), (6, 20), (5, 32), (16, 48), (32, 8), (64, 4), (300, 4), (3, 2)]


@pytest.mark.parametrize("H,D", SHAPES)
@pytest.mark.parametrize("n_edges", [1, 33, 255, 257, 3001])
def test_edges_match_float64(H, D, n_edges):
    import torch
    from featgraph_amd import _lib
    rng = np.random.default_rng(100 * H + D + n_edges)
    n_src, n_dst = 37, 23
    row, col = rng.integers(0, n_dst, n_edges), rng.integers(0, n_src, n_edges)
    row[: n_edges // 2] = np.sort(row[: n_edges // 2])          # half of the batches with repeated destination rows
    row[: n_edges // 4] = 3
    perm = rng.permutation(n_edges)
    src = rng.standard_normal((n_src, H, D)).astype(np.float32)
    dst = rng.standard_normal((n_dst, H, D)).astype(np.float32)
    src[5, :, -1] = np.nan
    dst[7, :, 0] = np.inf
    with np.errstate(invalid="ignore"):
        want = np.einsum("ehd,ehd->eh", src[col].astype("f8"), dst[row].astype("f8"))
    mass = np.einsum("ehd,ehd->eh", np.abs(src[col]).astype("f8"), np.abs(dst[row]).astype("f8"))
    finite = np.isfinite(want)

    def on_device(a, dtype):
        return torch.from_numpy(np.ascontiguousarray(a)).to("cuda", dtype)
    # operands one float past a 128-bit boundary
    buf_s, buf_d = torch.zeros(src.size + 1, device="cuda"), torch.zeros(dst.size + 1, device="cuda")
    buf_s[1:] = on_device(src.ravel(), torch.float32)
    buf_d[1:] = on_device(dst.ravel(), torch.float32)
    aligned = (on_device(src, torch.float32), on_device(dst, torch.float32))
    r, c, p = (on_device(a, torch.int32) for a in (row, col, perm))
    ptr, stream = _lib.dev_ptr, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for s, d, pos, extents in ((aligned[0], aligned[1], None, (n_src, n_dst)), (aligned[0], aligned[1], p, (n_src, n_dst)),
                               (buf_s[1:], buf_d[1:], p, (0, 0)), (buf_s[1:], buf_d[1:], None, (n_src, n_dst))):
        out = torch.full((n_edges, H), float("nan"), device="cuda")
        _lib.check(_lib.lib().fg_sddmm_edges_f32(ptr(r), ptr(c), ptr(pos), n_edges, extents[0], extents[1], ptr(s), ptr(d), ptr(out),
                                                 H, D, stream))
        got = out.cpu().numpy()
        if pos is not None:
            got = got[perm]
        what = "H=%d D=%d %d edges" % (H, D, n_edges)
        assert np.array_equal(np.isnan(got), np.isnan(want)), what
        assert np.array_equal(got[~finite & ~np.isnan(want)], want[~finite & ~np.isnan(want)].astype(np.float32)), what
        assert_sum_close(got[finite], want[finite], mass[finite], what)


@pytest.mark.parametrize("H,D", [(1, 3), (1, 5), (1, 16), (1, 31), (1, 64), (1, 100), (1, 127), (1, 338), (1, 512), (2, 8), (3, 16), (6, 20), (5, 32), (300, 4)])
def test_rows_addressed_with_64_bits_give_the_same_results(H, D):
    """Without the operands' row counts (and for operands of 4 GiB or more) rows are addressed with 64 bits and walked half a batch at a time; every dot
    product adds up in the same order."""
    import torch
    from featgraph_amd import _lib
    rng = np.random.default_rng(D)
    ptr, stream = _lib.dev_ptr, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for n_edges in (1, 255, 3001):
        row, col = rng.integers(0, 23, n_edges), rng.integers(0, 37, n_edges)
        row[: n_edges // 2] = np.sort(row[: n_edges // 2])
        r, c = (torch.from_numpy(a.astype(np.int32)).cuda() for a in (row, col))
        src, dst = (torch.from_numpy(rng.standard_normal((n, H, D), dtype=np.float32)).cuda() for n in (37, 23))
        narrow, wide = (torch.full((n_edges, H), float("nan"), device="cuda") for _ in range(2))
        _lib.check(_lib.lib().fg_sddmm_edges_f32(ptr(r), ptr(c), None, n_edges, 37, 23, ptr(src), ptr(dst), ptr(narrow), H, D, stream))
        _lib.check(_lib.lib().fg_sddmm_coo_f32(ptr(r), ptr(c), n_edges, ptr(src), ptr(dst), ptr(wide), H, D, stream))
        assert torch.equal(narrow, wide)
