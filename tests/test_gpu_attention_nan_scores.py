"""A row that holds a NaN score, or one of +inf, is NaN for that head -- out and every gradient that the row takes part in -- as the
softmax, the weighted sum and their gradients put together give it, and nothing else is.  Rows of no, one, a few, 64, 256, 257
and more elements, NaN alone or among other scores, one and several partitions, passes in buffers of their own and in place.
A row whose scores are all -inf counts as one without edges: 0."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu

H, D, SLOPE = 4, 32, 0.2


def _graph(kind, rng):
    n_dst, n_src = 300, 700
    lengths = {"few": [0, 1, 2, 3, 5, 8, 9], "edges": [1, 63, 64, 65, 255, 256, 257, 600]}[kind]
    rows, cols = [], []
    for r in range(n_dst):
        k = lengths[r % len(lengths)]
        rows += [r] * k
        cols += list(rng.choice(n_src, size=k, replace=False))
    adj = sp.csr_matrix((np.ones(len(rows), np.float32), (rows, cols)), shape=(n_dst, n_src))
    adj.sort_indices()
    return adj


def _float64(adj, scores, v, dout, leaves):
    """Softmax and weighted sum over the rows' edges and their gradients, in float64; a row's maximum is NaN if a score is."""
    import torch
    row = torch.from_numpy(np.repeat(np.arange(adj.shape[0]), np.diff(adj.indptr))).cuda()
    col = torch.from_numpy(adj.indices).long().cuda()
    s = scores(row, col)
    top = torch.full((adj.shape[0], H), -float("inf"), dtype=torch.float64, device="cuda")
    top = top.scatter_reduce(0, row[:, None].expand_as(s), s.detach(), "amax")
    p = (s - top[row]).exp()
    a = p / torch.zeros_like(top).index_add(0, row, p)[row]
    out = torch.zeros((adj.shape[0], H, D), dtype=torch.float64, device="cuda").index_add(0, row, a[:, :, None] * v[col])
    return (out,) + torch.autograd.grad(out, leaves, dout.double())


def _same(names, got, ref):
    import torch
    for name, x, y in zip(names, got, ref):
        assert torch.equal(torch.isnan(x), torch.isnan(y)), name
        ok = ~torch.isnan(y)
        # sums of up to 700 terms and softmax values of scores of a few units: as in the tests of finite inputs, entry by entry
        assert bool(((x.double() - y)[ok].abs() <= 1e-4 * (1 + y[ok].abs())).all()), name


def _setup(monkeypatch, parts, pass_buffers):
    from featgraph_amd import _lib, tuning
    monkeypatch.setattr(tuning, "_partitions", lambda *a, **k: parts)
    monkeypatch.setattr(_lib, "plan_opts", _lib.FgPlanOpts(pass_buffers=pass_buffers))


WAYS = pytest.mark.parametrize("parts,pass_buffers", [(1, 0), (3, 0), (3, 2)])


@pytest.mark.parametrize("kind", ["few", "edges"])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
@WAYS
def test_additive(monkeypatch, kind, value, parts, pass_buffers):
    import torch
    from featgraph_amd.autograd import Graph
    _setup(monkeypatch, parts, pass_buffers)
    adj = _graph(kind, np.random.default_rng(3))
    gen = torch.Generator(device="cuda").manual_seed(3)
    normal = lambda *s: torch.randn(s, generator=gen, device="cuda")
    er, el, v, dout = normal(adj.shape[0], H), normal(adj.shape[1], H), normal(adj.shape[1], H, D), normal(adj.shape[0], H, D)
    lens = np.diff(adj.indptr)
    for i, n in enumerate(np.unique(lens)):                        # every score of one row of each length, in one head
        er[int(np.flatnonzero(lens == n)[3]), i % H] = value
    el[int(np.bincount(adj.indices).argmin()), 1] = value          # one score of the few rows that reference this source
    leaves = [t.clone().requires_grad_() for t in (er, el, v)]
    out = Graph(adj).gat_attention(*leaves, negative_slope=SLOPE)
    got = (out.detach(),) + torch.autograd.grad(out, leaves, dout)
    e, l, w = (t.detach().double().requires_grad_() for t in (er, el, v))
    ref = _float64(adj, lambda row, col: torch.nn.functional.leaky_relu(l[col] + e[row], SLOPE), w, dout, (e, l, w))
    assert int(torch.isnan(ref[0]).any(2).sum()) >= 6 and not bool(torch.isnan(ref[0]).all())
    _same(("out", "dEr", "dEl", "dV"), got, ref)
    with torch.no_grad():
        plain = Graph(adj).gat_attention(er, el, v, negative_slope=SLOPE)
    assert torch.equal(torch.nan_to_num(plain, nan=7.0), torch.nan_to_num(got[0], nan=7.0))


@pytest.mark.parametrize("kind", ["few", "edges"])
@pytest.mark.parametrize("kept", [True, False])
@WAYS
def test_dot(monkeypatch, kind, kept, parts, pass_buffers):
    import torch
    from featgraph_amd import tuning
    from featgraph_amd.autograd import Graph
    _setup(monkeypatch, parts, pass_buffers)
    monkeypatch.setattr(tuning, "attention_keeps_score_gradients", lambda *a: kept)
    adj = _graph(kind, np.random.default_rng(3))
    gen = torch.Generator(device="cuda").manual_seed(3)
    normal = lambda n: torch.randn((n, H, D), generator=gen, device="cuda")
    q, k, v, dout = normal(adj.shape[0]), normal(adj.shape[1]), normal(adj.shape[1]), normal(adj.shape[0])
    lens = np.diff(adj.indptr)
    for i, n in enumerate(np.unique(lens)):
        q[int(np.flatnonzero(lens == n)[3]), i % H, 5] = float("nan")
    k[int(np.bincount(adj.indices).argmin()), 1, 0] = float("nan")
    leaves = [t.clone().requires_grad_() for t in (q, k, v)]
    out = Graph(adj).attention(*leaves, scale=0.2)
    got = (out.detach(),) + torch.autograd.grad(out, leaves, dout)
    a, b, w = (t.detach().double().requires_grad_() for t in (q, k, v))
    ref = _float64(adj, lambda row, col: 0.2 * (b[col] * a[row]).sum(-1), w, dout, (a, b, w))
    assert int(torch.isnan(ref[0]).any(2).sum()) >= 6 and not bool(torch.isnan(ref[0]).all())
    _same(("out", "dQ", "dK", "dV"), got, ref)


@WAYS
def test_rows_of_minus_infinity_count_as_empty(monkeypatch, parts, pass_buffers):
    import torch
    from featgraph_amd.autograd import Graph
    _setup(monkeypatch, parts, pass_buffers)
    adj = _graph("edges", np.random.default_rng(3))
    er, el = torch.zeros((adj.shape[0], H), device="cuda"), torch.zeros((adj.shape[1], H), device="cuda")
    v = torch.ones((adj.shape[1], H, D), device="cuda")
    er[5, 2] = -float("inf")
    leaves = [t.requires_grad_() for t in (er, el, v)]
    out = Graph(adj).gat_attention(*leaves)
    der, del_, dv = torch.autograd.grad(out, leaves, torch.ones_like(out))
    assert bool((out[5, 2] == 0).all()) and bool(torch.isfinite(out).all()) and bool(torch.isfinite(dv).all())
    assert bool(torch.isfinite(der).all()) and bool(torch.isfinite(del_).all())
