"""The two gradients of a weighted sum from one sweep over the transposed graph (fg_spmm_dot_f32), against float64: sources
with no, one, a few, 255 .. 257 and thousands of out-edges (whole rows, lane groups on rows of their own, pieces of split
rows), one and several partitions, one and several feature tiles, one and several heads per tile, padded lengths."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


def _graph(kind, rng):
    n_dst, n_src = 4000, 150
    lengths = {"few": [0, 1, 2, 3, 5], "long": [0, 1, 255, 256, 257, 1500, 3900], "mixed": [0, 2, 40, 300]}[kind]
    rows, cols = [], []
    for c in range(n_src):
        k = lengths[rng.integers(len(lengths))]
        rows += list(rng.choice(n_dst, size=k, replace=False))
        cols += [c] * k
    adj = sp.csr_matrix((np.ones(len(rows), np.float32), (rows, cols)), shape=(n_dst, n_src))
    adj.sort_indices()
    return adj


@pytest.mark.parametrize("kind", ["few", "long", "mixed"])
@pytest.mark.parametrize("tail,parts,tiles", [((16,), 1, 0), ((16,), 3, 0), ((100,), 1, 0), ((128,), 2, 1), ((128,), 1, 2), ((256,), 1, 1),
                                              ((602,), 3, 10), ((2, 32), 1, 0), ((4, 16), 2, 0), ((4, 8), 1, 0), ((3, 64), 3, 0),
                                              ((8, 64), 1, 0), ((2, 20), 1, 0), ((2, 128), 1, 0), ((1, 64), 1, 0)])
def test_gradients_match_float64(monkeypatch, kind, tail, parts, tiles):
    import torch
    from featgraph_amd import autograd, tuning
    monkeypatch.setattr(tuning, "PAD_MIN_GATHERED", 0)
    monkeypatch.setattr(tuning, "choose_spmm", lambda *a, **k: (parts, tiles))
    # two sweeps: heads cut into tiles (their parts are not added up), and one head as an axis (the broadcasting kernel)
    fused = tail not in ((2, 128), (1, 64))
    if fused:
        monkeypatch.setattr(autograd.Graph, "_sddmm_raw", lambda *a: pytest.fail("the gradients took two sweeps"))
    adj = _graph(kind, np.random.default_rng(sum(tail) + parts))
    g = autograd.Graph(adj)
    gen = torch.Generator(device="cuda").manual_seed(2)
    normal = lambda *shape: torch.randn(shape, generator=gen, device="cuda")
    x = normal(adj.shape[1], *tail).requires_grad_()
    w = normal(adj.nnz, *tail[:-1]).requires_grad_()
    dy = normal(adj.shape[0], *tail)
    for _ in range(2):                      # the second step reuses the plan's scratch
        dx, dw = torch.autograd.grad(g.spmm(x, w), (x, w), dy)
    row = torch.from_numpy(np.repeat(np.arange(adj.shape[0]), np.diff(adj.indptr))).cuda()
    col = torch.from_numpy(adj.indices).long().cuda()
    terms = x.detach().double()[col] * dy.double()[row]
    # eps32 / 2 per rounding; a dot product of D terms and the adds across lanes and tiles round each partial sum of |terms|
    bound = 2.0 ** -24 * 16 * terms.abs().sum(-1) + 1e-30
    assert bool(((dw.double() - terms.sum(-1)).abs() <= bound).all())
    parts_of = w.detach().double()[..., None] * dy.double()[row]
    zero = torch.zeros(x.shape, dtype=torch.float64, device="cuda")
    ref, size = zero.index_add(0, col, parts_of), zero.index_add(0, col, parts_of.abs())
    assert bool(((dx.double() - ref).abs() <= 2.0 ** -24 * 64 * size + 1e-30).all())
    # one gradient at a time: the plain operators, the same sums
    monkeypatch.undo()
    only, = torch.autograd.grad(g.spmm(x, w.detach()), (x,), dy)
    assert torch.equal(only, dx)


def test_non_finite_rows_stay_where_they_belong():
    import torch
    from featgraph_amd.autograd import Graph
    adj = _graph("mixed", np.random.default_rng(1))
    g = Graph(adj)
    x = torch.ones(adj.shape[1], 64, device="cuda", requires_grad=True)
    w = torch.ones(adj.nnz, device="cuda", requires_grad=True)
    row = np.repeat(np.arange(adj.shape[0]), np.diff(adj.indptr))
    bad = int(np.argmax(np.diff(adj.indptr)))
    dy = torch.ones(adj.shape[0], 64, device="cuda")
    dy[bad] = float("inf")
    dx, dw = torch.autograd.grad(g.spmm(x, w), (x, w), dy)
    hit = np.zeros(adj.shape[1], bool)
    hit[adj.indices[row == bad]] = True
    assert np.array_equal(~np.isfinite(dx.cpu().numpy()).all(1), hit)
    assert np.array_equal(~np.isfinite(dw.cpu().numpy()), row == bad)


@pytest.mark.parametrize("tail,outputs", [((64,), 1), ((2, 128), 1)])
def test_one_output_is_allocated_whichever_way_is_taken(monkeypatch, tail, outputs):
    import torch
    from featgraph_amd.autograd import Graph
    adj = _graph("mixed", np.random.default_rng(1))
    g = Graph(adj)
    x = torch.ones((adj.shape[1],) + tail, device="cuda", requires_grad=True)
    w = torch.ones((adj.nnz,) + tail[:-1], device="cuda", requires_grad=True)
    dy = torch.ones((adj.shape[0],) + tail, device="cuda")
    torch.autograd.grad(g.spmm(x, w), (x, w), dy)              # builds what it needs
    taken, empty = [], torch.empty
    y = g.spmm(x, w)
    monkeypatch.setattr(torch, "empty", lambda *a, **k: taken.append(a[0]) or empty(*a, **k))
    torch.autograd.grad(y, (x, w), dy)
    assert taken.count(tuple(x.shape)) == outputs


@pytest.mark.parametrize("tail", [(16,), (64,), (4, 16), (2, 32), (4, 8)])
@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_non_finite_rows_stay_where_they_belong_on_short_rows(tail, value):
    """Rows of a few elements, which lane groups walk on their own: the slots past a row's end hold other groups' elements, whose
    weights may have given way to dot products already."""
    import torch
    from featgraph_amd.autograd import Graph
    adj = _graph("few", np.random.default_rng(2))
    out_degree = np.bincount(adj.indices, minlength=adj.shape[1])
    assert out_degree.max() <= 5 and (out_degree > 0).sum() >= 64      # whole rows of the transposed graph, many to an item
    row = np.repeat(np.arange(adj.shape[0]), np.diff(adj.indptr))
    bad = row[::37]                                                      # destinations of every 37th edge
    w = torch.rand((adj.nnz,) + tail[:-1], device="cuda").add_(0.5).requires_grad_()
    x = torch.ones((adj.shape[1],) + tail, device="cuda", requires_grad=True)
    clean = torch.ones((adj.shape[0],) + tail, device="cuda")
    dy = clean.clone()
    dy[torch.from_numpy(bad).cuda()] = value
    g = Graph(adj)
    y = g.spmm(x, w)
    want = torch.autograd.grad(y, (x, w), clean, retain_graph=True)
    dx, dw = torch.autograd.grad(y, (x, w), dy)
    hit_w = np.isin(row, bad)
    hit_x = np.isin(np.arange(adj.shape[1]), adj.indices[hit_w])
    for got, ref, hit in ((dx, want[0], hit_x), (dw, want[1], hit_w)):
        hit = torch.from_numpy(hit).cuda()
        assert not bool(torch.isfinite(got[hit]).any())
        assert torch.equal(got[~hit], ref[~hit])
