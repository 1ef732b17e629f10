"""Edge softmax at the row lengths where its kernels change: what a chunk, a wavefront's and a workgroup's registers
hold, what one workgroup takes at all; split and unsplit rows; arrays that are only 4-byte aligned.  Float64 is the
reference (the snapshot has no such operator: parity unpinned by it)."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu
EPS = float(np.finfo(np.float32).eps)


def _lengths(H):
    ch = 12 if H in (3, 6) else 4
    marks = [ch // H if ch > H else 1, 512 // H, 1024 // H]
    for chunks in (1, 2, 4, 8):                      # chunks per lane of a wavefront and of a workgroup of four
        marks += [64 * ch * chunks // H, 256 * ch * chunks // H]
    marks.append((1 << 17) // H)                     # longest row of one workgroup
    around = sorted({max(1, m + d) for m in marks for d in (-1, 0, 1, 2)})
    return [0, 1, 2, 3] + around + [0, 5] + [1] * 70 + [9] * 40 + [40] * 9


@pytest.mark.parametrize("split", [0, 100_000])      # 0: the plan's own pieces; 100,000: every row but the longest in one item
@pytest.mark.parametrize("H", [1, 2, 3, 4, 6, 8, 16, 64])
def test_every_row_length_class(monkeypatch, H, split):
    import torch
    from featgraph_amd import _lib
    from featgraph_amd.module import EdgeSoftmaxhip, placeholder
    if split:
        monkeypatch.setattr(_lib, "plan_opts", _lib.FgPlanOpts(split_threshold=split))
    rng = np.random.default_rng(H)
    lens = np.array(_lengths(H))
    rng.shuffle(lens)
    indptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    nnz = int(indptr[-1])
    indices = np.concatenate([np.arange(n) for n in lens]).astype(np.int32)
    m = EdgeSoftmaxhip(sp.csr_matrix((np.ones(nnz, np.float32), indices, indptr), shape=(len(lens), max(lens))))
    shape = (nnz, H)
    m.build([placeholder(shape)])
    gen = torch.Generator(device="cuda").manual_seed(H)
    # views one float into their storage: aligned like a float and no better
    x = torch.randn(nnz * H + 1, generator=gen, device="cuda")[1:].view(shape) * 1.0
    flat = torch.empty(nnz * H + 1, device="cuda")
    flat[1:] = x.reshape(-1) * 3
    x = flat[1:].view(shape)
    g = torch.randn(nnz * H + 1, generator=gen, device="cuda")[1:].view(shape)
    m.out_tvm.fill_(float("nan"))
    a = m.run([x])
    row = torch.repeat_interleave(torch.arange(len(lens), device="cuda"), torch.from_numpy(lens).cuda())
    x64 = x.double()
    top = torch.full((len(lens), H), -float("inf"), dtype=torch.float64, device="cuda").scatter_reduce(0, row[:, None].expand(-1, H), x64, "amax")
    ex = torch.exp(x64 - top[row])
    ref = ex / torch.zeros_like(top).index_add_(0, row, ex)[row]
    # relative: the exponent's rounding, |x - max| * log2(e) * eps, and about 16 roundings of sums and products
    tol = ref * EPS * (16 + 4 * (top[row] - x64))
    assert bool(((a.double() - ref).abs() <= tol).all()), float(((a.double() - ref).abs() / ref).max())
    assert torch.equal(a, m.run([x]))

    a = a.clone()
    dx = m.backward(a, g).double()
    ag = a.double() * g.double()
    zero = torch.zeros_like(top)
    ref = a.double() * (g.double() - zero.index_add(0, row, ag)[row])
    mass = a.double() * (g.double().abs() + zero.index_add(0, row, ag.abs())[row])
    # a lane adds up to some hundred terms one after the other, then a tree; about 64 roundings of the absolute mass
    assert bool(((dx - ref).abs() <= 64 * EPS * mass).all()), float(((dx - ref).abs() / mass.clamp_min(1e-30)).max())


@pytest.mark.parametrize("H", [1, 3, 4, 8])
def test_special_values_stay_in_their_row(H):
    """NaN, an infinity or nothing but -inf in one row: that row and head only, in every row class."""
    import torch
    from featgraph_amd.module import EdgeSoftmaxhip, placeholder
    lens = np.array([3, 700, 5, 3000, 20, 40_000, 8, 33, 33])
    indptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    nnz = int(indptr[-1])
    indices = np.concatenate([np.arange(n) for n in lens]).astype(np.int32)
    m = EdgeSoftmaxhip(sp.csr_matrix((np.ones(nnz, np.float32), indices, indptr), shape=(len(lens), max(lens))))
    m.build([placeholder((nnz, H))])
    for r in range(len(lens)):
        for value in (float("nan"), float("inf"), -float("inf")):
            x = torch.randn(nnz, H, generator=torch.Generator(device="cuda").manual_seed(r), device="cuda")
            x[indptr[r], 0] = value
            if value == -float("inf"):
                x[indptr[r]:indptr[r + 1], 0] = value
            bad = torch.isnan(m.run([x]))
            inside = bad[indptr[r]:indptr[r + 1], 0]
            if value == float("inf"):
                assert bool(inside[0])                   # inf / inf
            else:
                assert bool(inside.all())
            assert int(bad.sum()) == int(inside.sum())


@pytest.mark.parametrize("H", [1, 2, 3, 4, 5, 8, 12, 64])
def test_nan_anywhere_reaches_its_whole_row(H):
    """A NaN score at the first, a middle or the last element of a row, alone or among scores of -inf, makes the row's every
    value NaN, also where a lane sees nothing but that NaN: short last pieces (1, 5 and 64 elements) of rows that are
    swept in pieces, and a row longer than a workgroup takes at every head count."""
    import torch
    from featgraph_amd.module import EdgeSoftmaxhip, placeholder
    lens = np.array([3, 700, 5, 2565, 20, 1025, 40_000, 8, 33, 140_000, 4, 33])
    indptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    nnz = int(indptr[-1])
    indices = np.concatenate([np.arange(n) for n in lens]).astype(np.int32)
    m = EdgeSoftmaxhip(sp.csr_matrix((np.ones(nnz, np.float32), indices, indptr), shape=(len(lens), max(lens))))
    m.build([placeholder((nnz, H))])
    x0 = torch.randn(nnz, H, generator=torch.Generator(device="cuda").manual_seed(H), device="cuda")
    for r in range(len(lens)):
        b, e = int(indptr[r]), int(indptr[r + 1])
        for at in sorted({b, (b + e) // 2, e - 1}):
            for masked in (False, True):
                x = x0.clone()
                if masked:
                    x[b:e, 0] = -float("inf")
                    x[b if at != b else e - 1, 0] = 0.5         # the row's one number
                x[at, 0] = float("nan")
                bad = torch.isnan(m.run([x]))
                assert bool(bad[b:e, 0].all()), (r, at - b, masked)
                assert int(bad.sum()) == e - b


@pytest.mark.parametrize("H", [1, 3, 4, 5, 12, 64, 65, 100])
def test_a_piece_of_masked_scores_leaves_its_row_finite(H):
    """Scores of -inf throughout the first, a middle or the last piece of a row that is swept in pieces (128 elements each
    here): zeros there, and the softmax of the rest elsewhere, against float64."""
    import torch
    from featgraph_amd.module import EdgeSoftmaxhip, placeholder
    lens = np.array([300, 3, 700, 129, 20, 2100])
    indptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    nnz = int(indptr[-1])
    indices = np.concatenate([np.arange(n) for n in lens]).astype(np.int32)
    m = EdgeSoftmaxhip(sp.csr_matrix((np.ones(nnz, np.float32), indices, indptr), shape=(len(lens), max(lens))))
    m.build([placeholder((nnz, H))])
    x = torch.randn(nnz, H, generator=torch.Generator(device="cuda").manual_seed(H), device="cuda")
    for b, e in zip(indptr[:-1].tolist(), indptr[1:].tolist()):
        if e - b == 700:
            x[b + 120:b + 400, ::2] = -float("inf")
        elif e - b == 2100:
            x[b + 1000:e, 1::2] = -float("inf")
        else:
            x[b:b + (e - b) // 2 + 1, :] = -float("inf")
    got = m.run([x]).double()
    for b, e in zip(indptr[:-1].tolist(), indptr[1:].tolist()):
        ref = torch.softmax(x[b:e].double(), 0)
        # as in test_every_row_length_class, with differences of at most 10 between finite scores of a row
        assert bool(((got[b:e] - ref).abs() <= ref * EPS * (16 + 4 * 10)).all()), (b, e)


@pytest.mark.parametrize("many", [False, True])
@pytest.mark.parametrize("H", [1, 3, 4, 16])
def test_longest_row_of_a_workgroup(H, many):
    """Rows around the most floats that one workgroup takes: 2^15, or a 128th of all there are (many: 160 rows of 40,000 and
    more, which workgroups take there and pieces take on the small graph); the merge of many pieces' statistics."""
    import torch
    from featgraph_amd.module import EdgeSoftmaxhip, placeholder
    at = (1 << 15) // H
    lens = np.array([at - 1, 7, at, at + 1, 3, 40_000 // H, 60_000 // H] + [40_000 // H] * (160 if many else 0) + [140_000 // H])
    indptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    nnz = int(indptr[-1])
    indices = np.concatenate([np.arange(n) for n in lens]).astype(np.int32)
    m = EdgeSoftmaxhip(sp.csr_matrix((np.ones(nnz, np.float32), indices, indptr), shape=(len(lens), max(lens))))
    m.build([placeholder((nnz, H))])
    gen = torch.Generator(device="cuda").manual_seed(H)
    x, g = torch.randn(nnz, H, generator=gen, device="cuda"), torch.randn(nnz, H, generator=gen, device="cuda")
    a = m.run([x]).clone()
    dx = m.backward(a, g)
    for b, e in zip(indptr[:8].tolist() + [int(indptr[-2])], indptr[1:9].tolist() + [nnz]):
        ref = torch.softmax(x[b:e].double(), 0)
        # the exponent's rounding (differences of at most 10) and up to 128 terms per lane, added up with few roundings to one side
        assert bool(((a[b:e].double() - ref).abs() <= ref * EPS * (64 + 4 * 10)).all()), (b, e)
        ag = a[b:e].double() * g[b:e].double()
        ref = ag - a[b:e].double() * ag.sum(0)
        mass = ag.abs() + a[b:e].double() * ag.abs().sum(0)
        assert bool(((dx[b:e].double() - ref).abs() <= 64 * EPS * mass).all()), (b, e)
