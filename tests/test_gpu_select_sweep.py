"""The gradient of a max / min aggregation by sweeps over the edges: the tiles' edges and partly filled words, rows without
elements, short rows by a lane group each, rows of one item and rows cut into pieces, both operands and every operator, and infinite
gradients that must reach the selected edge alone."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


def _graph(rng):
    a = sp.random(300, 260, density=0.02, format="lil", random_state=rng)
    a[:, 7] = 1                                   # one source with 300 edges: a row of its own in the transposed layout
    a[11, :] = 1                                  # one long row
    a[[0, 150, 299], :] = 0
    a[:, [0, 100, 259]] = 0
    a = a.tocsr()
    a.eliminate_zeros()
    a.sort_indices()
    return a


@pytest.mark.parametrize("F", [4, 5, 15, 16, 17, 63, 64, 65, 100, 127, 128, 130, 257])
@pytest.mark.parametrize("op", ["copy", "add", "sub", "mul", "div"])
@pytest.mark.parametrize("split", [0, 16])
def test_sweeps_match_the_selected_edges(monkeypatch, F, op, split):
    import torch
    from featgraph_amd import _lib, ops, tuning
    from featgraph_amd.autograd import Graph
    rng = np.random.default_rng(F)
    adj = _graph(rng)
    if split:                                     # the long rows become pieces
        monkeypatch.setattr(_lib, "plan_opts", _lib.FgPlanOpts(split_threshold=split, item_edges=split))
    calls = []
    monkeypatch.setattr(tuning, "select_by_sweep", lambda *a: calls.append(a) or True)
    g = Graph(adj)
    row, col = np.repeat(np.arange(300), np.diff(adj.indptr)), adj.indices
    x = rng.standard_normal((260, F)).astype(np.float32)
    dout = rng.standard_normal((300, F)).astype(np.float32)
    dout[5, F // 2] = np.inf
    for e_len in ([0] if op == "copy" else [1, F]):
        w = (1.5 + rng.random((adj.nnz, max(1, e_len)))).astype(np.float32)
        xt, wt, dt = torch.from_numpy(x).cuda().requires_grad_(), torch.from_numpy(w).cuda().requires_grad_(), torch.from_numpy(dout).cuda()
        leaves = [xt] if op == "copy" else [xt, wt]
        out = g.aggregate(xt, "max") if op == "copy" else ops.gspmm(g, op, "max", xt, wt)
        got = [t.cpu().numpy() for t in torch.autograd.grad(out, leaves, dt)]
        # in float64: every result's selected edge (the first of the largest messages, formed in float32 as the kernel does)
        m = x[col] if op == "copy" else {"add": np.add, "sub": np.subtract, "mul": np.multiply, "div": np.divide}[op](x[col], w)
        dx, dw = np.zeros((260, F)), np.zeros((adj.nnz, F))
        mass = np.zeros((260, F))
        with np.errstate(invalid="ignore"):
            for v in range(300):
                b, e = adj.indptr[v], adj.indptr[v + 1]
                if b == e:
                    continue
                at = b + np.argmax(m[b:e], axis=0)
                f = np.arange(F)
                d, xs, ws = dout[v].astype("f8"), x[col[at], f].astype("f8"), w[at, f if e_len == F else 0].astype("f8")
                to_x = {"copy": d, "add": d, "sub": d, "mul": d * ws, "div": d / ws}[op]
                np.add.at(dx, (col[at], f), to_x)
                np.add.at(mass, (col[at], f), np.abs(to_x))
                dw[at, f] = {"copy": d, "add": d, "sub": -d, "mul": d * xs, "div": -d * xs / ws ** 2}[op]
        def check(a, want, mass, what):
            # sums of float32 in some order: (terms + 2) roundings of the summed mass at most
            assert np.array_equal(np.isfinite(a), np.isfinite(want)), what
            ok = np.isfinite(want)
            assert (np.abs(a[ok] - want[ok]) <= 310 * np.finfo(np.float32).eps * mass[ok]).all(), what
        check(got[0], dx, mass, "%s dx, %d edge features" % (op, e_len))
        if op != "copy":
            with np.errstate(invalid="ignore"):
                check(got[1], dw if e_len == F else dw.sum(1, keepdims=True), np.abs(dw) if e_len == F else np.abs(dw).sum(1, keepdims=True),
                      "%s dw, %d edge features" % (op, e_len))
    assert len(calls) >= (1 if op == "copy" else 2)


@pytest.mark.parametrize("msg", ["%s_%s_%s" % (a, op, b) for op in ("add", "sub", "mul", "div") for a in "ue" for b in "ue"])
@pytest.mark.parametrize("lens", [(8, 8), (1, 8), (8, 1)])
def test_operands_on_every_target(monkeypatch, msg, lens):
    """Messages of one target twice, and of the targets the other way round, against the gradients from torch's operators."""
    import torch
    from featgraph_amd import tuning
    from featgraph_amd.autograd import Graph, _GSpMMExtreme
    monkeypatch.setattr(tuning, "select_by_sweep", lambda *a: True)
    rng = np.random.default_rng(3)
    adj = _graph(rng)
    g = Graph(adj)
    leaves = [torch.from_numpy((1.5 + rng.random((260 if t == "u" else adj.nnz, n))).astype(np.float32)).cuda().requires_grad_()
              for t, n in zip((msg[0], msg[-1]), lens)]
    dout = torch.from_numpy(rng.standard_normal((300, 8)).astype(np.float32)).cuda()
    out = _GSpMMExtreme.apply(g, msg, "max", *leaves)
    got = torch.autograd.grad(out, leaves, dout, retain_graph=True)
    want = torch.autograd.grad(out, leaves, dout, create_graph=True)
    for a, b in zip(got, want):
        # up to 300 * 8 terms of at most 4 * 2.5 / 1.5 ** 2 in float32, in two orders
        assert torch.allclose(a, b, rtol=1e-5, atol=1e-4), msg
