"""Additive attention with gradients in two sweeps: the forward pass keeps the sums over the edges with a positive score,
from which dEr follows without a sweep of its own.  Against float64 torch autograd, at the sizes where the sweeps change
their path: rows of no, one, a few, 64, 256, 257 and more elements, one and several source partitions, every pass into a
buffer of its own and passes that merge in place, and scores that are all positive or all negative (dEr is then 0)."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


def _graph(kind, rng):
    n_dst, n_src = 300, 700
    lengths = {"few": [0, 1, 2, 3, 5, 8, 9], "edges": [0, 1, 63, 64, 65, 255, 256, 257, 600], "mixed": [0, 1, 4, 30, 90, 300]}[kind]
    rows, cols = [], []
    for r in range(n_dst):
        k = lengths[rng.integers(len(lengths))]
        rows += [r] * k
        cols += list(rng.choice(n_src, size=k, replace=False))
    return sp.csr_matrix((np.ones(len(rows), np.float32), (rows, cols)), shape=(n_dst, n_src))


def _float64(adj, er, el, v, dout, slope):
    import torch
    er, el, v = (t.detach().double().requires_grad_() for t in (er, el, v))
    row = torch.from_numpy(np.repeat(np.arange(adj.shape[0]), np.diff(adj.indptr))).cuda()
    col = torch.from_numpy(adj.indices).long().cuda()
    s = torch.nn.functional.leaky_relu(el[col] + er[row], slope)
    top = torch.full((adj.shape[0], s.shape[1]), -1e300, dtype=torch.float64, device="cuda")
    top = top.scatter_reduce(0, row[:, None].expand_as(s), s.detach(), "amax")
    p = (s - top[row]).exp()
    a = p / torch.zeros_like(top).index_add(0, row, p)[row]
    out = torch.zeros((adj.shape[0],) + tuple(v.shape[1:]), dtype=torch.float64, device="cuda").index_add(0, row, a[:, :, None] * v[col])
    return (out,) + torch.autograd.grad(out, (er, el, v), dout.double())


@pytest.mark.parametrize("kind", ["few", "edges", "mixed"])
@pytest.mark.parametrize("heads,head_len", [(1, 64), (3, 32), (4, 16), (16, 16)])
@pytest.mark.parametrize("parts,pass_buffers", [(1, 0), (3, 0), (3, 2)])
def test_step_matches_float64(monkeypatch, kind, heads, head_len, parts, pass_buffers):
    import torch
    from featgraph_amd import _lib, tuning
    from featgraph_amd.autograd import Graph
    monkeypatch.setattr(tuning, "_partitions", lambda *a, **k: parts)
    monkeypatch.setattr(_lib, "plan_opts", _lib.FgPlanOpts(pass_buffers=pass_buffers))
    adj = _graph(kind, np.random.default_rng(heads * 100 + head_len + parts))
    adj.sort_indices()
    gen = torch.Generator(device="cuda").manual_seed(3)
    normal = lambda *shape: torch.randn(shape, generator=gen, device="cuda")
    n_dst, n_src = adj.shape
    g = Graph(adj)
    dout = normal(n_dst, heads, head_len)
    for shift, slope in ((0.0, 0.2), (50.0, 0.2), (-50.0, 0.01)):
        er, el, v = normal(n_dst, heads) + shift, normal(n_src, heads), normal(n_src, heads, head_len)
        leaves = [t.clone().requires_grad_() for t in (er, el, v)]
        out = g.gat_attention(*leaves, negative_slope=slope)
        got = (out.detach(),) + torch.autograd.grad(out, leaves, dout)
        ref = _float64(adj, er, el, v, dout, slope)
        for name, x, y in zip(("out", "dEr", "dEl", "dV"), got, ref):
            if shift and name == "dEr":
                # one slope over the whole row: mathematically 0; what is left is rounding, 2^-24 of the sums' terms
                # (sqrt(head_len) * up to a few standard deviations) times a row's worth of additions
                assert float(x.abs().max()) <= 1e-4
                continue
            # fp32 sums of at most 700 terms and softmax values of scores up to 50 (c1 = m + log l rounds to 50 * 2^-24 = 3e-6
            # there, to 3e-7 around 0); what is seen is a sixth of these
            bound = 2e-5 if shift else 2e-6
            assert float((x.double() - y).norm()) <= bound * float(y.norm()), (name, shift)
        with torch.no_grad():
            assert torch.equal(g.gat_attention(er, el, v, negative_slope=slope), got[0])


@pytest.mark.parametrize("kind", ["few", "edges"])
@pytest.mark.parametrize("heads,head_len", [(1, 64), (4, 16)])
@pytest.mark.parametrize("parts,pass_buffers", [(1, 0), (3, 0), (3, 2)])
def test_non_finite_rows_stay_where_they_belong(monkeypatch, kind, heads, head_len, parts, pass_buffers):
    """A source with an infinite row of V, a destination with an infinite row of dout: only what the formulas give them."""
    import torch
    from featgraph_amd import _lib, tuning
    from featgraph_amd.autograd import Graph
    monkeypatch.setattr(tuning, "_partitions", lambda *a, **k: parts)
    monkeypatch.setattr(_lib, "plan_opts", _lib.FgPlanOpts(pass_buffers=pass_buffers))
    adj = _graph(kind, np.random.default_rng(heads + parts))
    adj.sort_indices()
    n_dst, n_src = adj.shape
    row = np.repeat(np.arange(n_dst), np.diff(adj.indptr))
    gen = torch.Generator(device="cuda").manual_seed(3)
    normal = lambda *shape: torch.randn(shape, generator=gen, device="cuda")
    er, el, v, dout = normal(n_dst, heads), normal(n_src, heads), normal(n_src, heads, head_len), normal(n_dst, heads, head_len)
    g = Graph(adj)

    def step(v, dout):
        leaves = [t.clone().requires_grad_() for t in (er, el, v)]
        out = g.gat_attention(*leaves)
        return (out.detach(),) + torch.autograd.grad(out, leaves, dout)

    clean = step(v, dout)
    degree = np.bincount(adj.indices, minlength=n_src)
    c = int(np.flatnonzero(degree > 0)[degree[degree > 0].argmin()])      # referenced by few rows
    r = int(np.flatnonzero(np.diff(adj.indptr) > 0)[0])
    rows_of_c = np.isin(np.arange(n_dst), row[adj.indices == c])
    cols_of = lambda rows: np.isin(np.arange(n_src), adj.indices[np.isin(row, np.flatnonzero(rows))])
    only_r = np.arange(n_dst) == r
    vb, db = v.clone(), dout.clone()
    vb[c] = float("inf")
    db[r] = float("inf")
    none_r, none_c = np.zeros(n_dst, bool), np.zeros(n_src, bool)
    for got, hits in ((step(vb, dout), (rows_of_c, rows_of_c, cols_of(rows_of_c), none_c)),
                      (step(v, db), (none_r, only_r, cols_of(only_r), cols_of(only_r)))):
        for name, x, y, hit in zip(("out", "dEr", "dEl", "dV"), got, clean, hits):
            hit = torch.from_numpy(hit).cuda()
            assert not bool(torch.isfinite(x[hit]).any()), name
            assert torch.equal(x[~hit], y[~hit]), name
