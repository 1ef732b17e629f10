"""How finely a plan cuts its rows follows the graph's size (fg_spmm_plan_create): pieces of 128, 256, 512 or 1024
elements and items of 16 to 256.  Graphs on both sides of every line but the last (2^25), with rows one element below, at and
above the piece lengths, against float64; the plan's own account of its cut on both sides of all of them; and the entry point with a fixed scratch array on a plan cut finer than its limit counts."""
import ctypes

import numpy as np
import pytest
import scipy.sparse as sp

from helpers import assert_sum_close, spmm_mass

pytestmark = pytest.mark.gpu

EDGE_LENS = [0, 1, 15, 16, 17, 127, 128, 129, 191, 192, 255, 256, 257, 511, 512, 513, 1023, 1024, 1025, 1100]


def _graph(nnz, seed):
    """Rows of the lengths at which a cut can go wrong, then rows of 24 elements until the matrix holds nnz."""
    n_src = 1200
    rng = np.random.default_rng(seed)
    lens = [l for l in EDGE_LENS if l <= nnz // 3]
    rest = nnz - sum(lens)
    assert rest >= 0
    lens += [24] * (rest // 24) + ([rest % 24] if rest % 24 else [])
    indptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    start = rng.integers(0, n_src, size=len(lens))
    cols = (np.arange(nnz) - np.repeat(indptr[:-1], lens) + np.repeat(start, lens)) % n_src      # consecutive columns: no duplicates
    adj = sp.csr_matrix((rng.standard_normal(nnz).astype("float32"), cols.astype(np.int32), indptr), shape=(len(lens), n_src))
    adj.sort_indices()
    return adj


@pytest.mark.parametrize("nnz", [40, 65535, 65536, 131071, 131072, (1 << 20) - 1, 1 << 20, (1 << 23) - 1, 1 << 23])
def test_rows_of_every_cut_are_summed_whole(nnz):
    import torch
    from featgraph_amd.module import EdgeSoftmaxhip, VanillaSpMMhip, placeholder
    adj = _graph(nnz, nnz % 97)
    F = 8 if nnz > (1 << 20) else 36
    rng = np.random.default_rng(5)
    x = rng.standard_normal((adj.shape[1], F)).astype("float32")
    m = VanillaSpMMhip(adj)
    m.build([placeholder(x.shape)], {}, {})
    m.out_tvm.fill_(float("nan"))
    out = m.run([torch.from_numpy(x).cuda()]).cpu().numpy()
    assert_sum_close(out, adj.astype(np.float64).dot(x.astype(np.float64)), spmm_mass(adj, x), "nnz=%d" % nnz)
    s = EdgeSoftmaxhip(adj)
    s.build([placeholder((nnz, 2))])
    scores = torch.from_numpy(rng.standard_normal((nnz, 2)).astype("float32")).cuda()
    a = s.run([scores]).double()
    rows = torch.repeat_interleave(torch.arange(adj.shape[0], device="cuda"), torch.from_numpy(np.diff(adj.indptr)).cuda().long())
    e = scores.double().exp()
    ref = e / torch.zeros((adj.shape[0], 2), dtype=torch.float64, device="cuda").index_add_(0, rows, e)[rows]
    assert ((a - ref).abs() <= 1e-5 * ref).all()


@pytest.mark.parametrize("feat_len,tiles", [(2048, 0), (2048, 8), (1400, 0), (1027, 0)])
def test_fixed_scratch_takes_a_finer_cut_in_column_ranges(feat_len, tiles):
    """300,000 elements in rows of 1000: about 2,400 pieces of 128, none of 1024; 2,400 * F exceeds the fixed array."""
    import torch
    from featgraph_amd import _lib
    L = _lib.lib()
    rng = np.random.default_rng(6)
    n, n_src = 300, 1200
    indptr = (np.arange(n + 1) * 1000).astype(np.int32)
    cols = np.sort((np.arange(1000)[None, :] + rng.integers(0, n_src, size=n)[:, None]) % n_src, axis=1).astype(np.int32).reshape(-1)
    vals = torch.from_numpy(rng.standard_normal(cols.size).astype("float32")).cuda()
    x = torch.from_numpy(rng.standard_normal((n_src, feat_len)).astype("float32")).cuda()
    ip, ix = torch.from_numpy(indptr).cuda(), torch.from_numpy(cols).cuda()
    plan = ctypes.c_void_p()
    assert L.fg_spmm_plan_create(_lib.host_ptr(indptr), n, n_src, 1, None, ctypes.byref(plan)) == 0
    try:
        p, s = _lib.dev_ptr, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        ref = torch.full((n, feat_len), float("nan"), device="cuda")
        got = torch.full((n, feat_len), float("nan"), device="cuda")
        assert L.fg_spmm_csr_f32(plan, p(ip), p(ix), p(vals), p(x), p(ref), feat_len, tiles, s) == 0
        assert L.fg_spmm_csr_noalloc_f32(plan, p(ip), p(ix), p(vals), p(x), p(got), feat_len, tiles, s) == 0
        torch.cuda.synchronize()
        assert torch.isfinite(ref).all() and torch.equal(ref, got)
    finally:
        L.fg_spmm_plan_destroy(plan)


def _plan(indptr, n_src):
    from featgraph_amd import _lib
    L, plan = _lib.lib(), ctypes.c_void_p()
    assert L.fg_spmm_plan_create(_lib.host_ptr(indptr), len(indptr) - 1, n_src, 1, None, ctypes.byref(plan)) == 0
    return plan


def test_as_many_pieces_as_a_finer_cut_may_make():
    """4,091 rows of 129 elements, two pieces each, and one of 1200, ten: 8192 pieces are the most that a finer cut makes and
    with tiles of 512 columns fill the fixed array to its last float."""
    import torch
    from featgraph_amd import _lib
    L, n_src, F = _lib.lib(), 1200, 1024
    lens = np.concatenate([np.full(4091, 129), [1200]])
    indptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    rng = np.random.default_rng(7)
    nnz = int(indptr[-1])
    start = rng.integers(0, n_src, size=len(lens))
    cols = ((np.arange(nnz) - np.repeat(indptr[:-1], lens) + np.repeat(start, lens)) % n_src).astype(np.int32)
    vals = torch.from_numpy(rng.standard_normal(nnz).astype("float32")).cuda()
    x = torch.from_numpy(rng.standard_normal((n_src, F)).astype("float32")).cuda()
    ip, ix = torch.from_numpy(indptr).cuda(), torch.from_numpy(cols).cuda()
    plan = _plan(indptr, n_src)
    try:
        p, s = _lib.dev_ptr, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        ref, got = (torch.full((len(lens), F), float("nan"), device="cuda") for _ in range(2))
        assert L.fg_spmm_csr_f32(plan, p(ip), p(ix), p(vals), p(x), p(ref), F, 0, s) == 0
        assert L.fg_spmm_csr_noalloc_f32(plan, p(ip), p(ix), p(vals), p(x), p(got), F, 0, s) == 0
        torch.cuda.synchronize()
        assert torch.isfinite(ref).all() and torch.equal(ref, got)
        row = torch.repeat_interleave(torch.arange(len(lens)), torch.from_numpy(lens)).cuda()
        want = torch.zeros((len(lens), 8), dtype=torch.float64, device="cuda").index_add(0, row, (vals[:, None] * x[:, -8:][ix.long()].double()))
        mass = torch.zeros_like(want).index_add(0, row, (vals[:, None] * x[:, -8:][ix.long()].double()).abs())
        assert bool(((got[:, -8:] - want).abs() <= 64 * 6e-8 * mass).all())
    finally:
        L.fg_spmm_plan_destroy(plan)


def _cut(lens):
    """A default plan's description."""
    from featgraph_amd import _lib
    plan = _plan(np.concatenate([[0], np.cumsum(lens)]).astype(np.int32), int(max(lens)))
    try:
        text = ctypes.create_string_buffer(4096)
        assert _lib.lib().fg_spmm_plan_describe(plan, 0, 0, text, 4096) >= 0
        return text.value.decode()
    finally:
        _lib.lib().fg_spmm_plan_destroy(plan)


@pytest.mark.parametrize("lens,split,item", [
    ([256] * 4, 1024, 16), ([257] * 4, 128, 16),                                    # rows left whole up to 256
    ([512] * 1700, 1024, 256), ([512] * 1699, 128, 128), ([513] * 1700, 256, 256),  # ... up to 512 with 1,700 times as much
    ([4] * 32767, 1024, 16), ([4] * 32768, 1024, 256),                              # 4 elements per row on average
    ([5] * 10879, 1024, 16), ([5] * 10880, 1024, 32),                               # 16 * 2 * 1700 elements
    ([2000] + [16] * 65410, 128, 128), ([2000] + [16] * 65411, 256, 256),           # 2^20
    ([2000] + [16] * 524162, 256, 256), ([2000] + [16] * 524163, 512, 256),         # 2^23
    ([3000] + [64] * 524241, 512, 256), ([3000] + [64] * 524242, 1024, 256),        # 2^25
    ([600] * 1638, 128, 128), ([600] * 1639, 256, 256),                             # 8192 pieces: five of a row
])
def test_where_the_cut_changes(lens, split, item):
    text = _cut(lens)
    assert "split threshold  : %d elements" % split in text and "(<= %d elements)" % item in text, text
