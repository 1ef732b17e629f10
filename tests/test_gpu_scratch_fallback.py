"""Gradients whose faster way needs memory that is not there take the way that needs less: the library or torch reporting that an
allocation failed (forced from the host, no device is exhausted) must not end a training step that the other way can finish."""
import ctypes

import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu

FG_ERR_NOMEM = -5


def _graph(n_dst=400, n_src=300, density=0.05):
    adj = sp.random(n_dst, n_src, density=density, format="csr", random_state=np.random.default_rng(4)).astype("float32")
    adj.sort_indices()
    return adj


def _failing(calls):
    def fail(*args):
        calls.append(1)
        return FG_ERR_NOMEM
    return fail


@pytest.mark.parametrize("tail", [(64,), (4, 32)])
def test_weighted_sum_gradients_without_memory_for_the_dots(monkeypatch, tail):
    import torch
    from featgraph_amd import _lib
    from featgraph_amd.autograd import Graph
    adj = _graph()
    gen = torch.Generator(device="cuda").manual_seed(1)
    normal = lambda *s: torch.randn(s, generator=gen, device="cuda")
    x, w, dy = normal(adj.shape[1], *tail).requires_grad_(), normal(adj.nnz, *tail[:-1]).requires_grad_(), normal(adj.shape[0], *tail)
    g = Graph(adj)
    ref = torch.autograd.grad(g.spmm(x, w), (x, w), dy)
    calls = []
    monkeypatch.setattr(_lib.lib(), "fg_spmm_dot_f32", _failing(calls))
    for _ in range(2):
        got = torch.autograd.grad(g.spmm(x, w), (x, w), dy)
        assert torch.equal(got[0], ref[0])
        # the dots in another order: 64 products each, 2^-24 per rounding of the sum of |terms| (standard normal: below 64)
        assert float((got[1] - ref[1]).abs().max()) <= 64 * 2.0 ** -24 * 64
    assert len(calls) == 1                      # a step does not try again what did not fit


def test_dots_that_would_take_more_than_the_cap_are_refused():
    """One array of nnz dot products per tile or head, 8 GiB of them at most.  (Plans alone: nothing is launched.)"""
    from featgraph_amd import _lib
    L = _lib.lib()
    rows, per_row = 1 << 20, 1 << 10            # 2^30 elements: 4 GiB per array
    pos = np.arange(0, rows * per_row + 1, per_row, dtype=np.int32)
    plan = ctypes.c_void_p()
    _lib.check(L.fg_spmm_plan_create(_lib.host_ptr(pos), rows, 4096, 1, None, ctypes.byref(plan)))
    try:
        for F, heads, tiles, takes in ((64, 1, 1, 1), (128, 1, 2, 1), (192, 1, 3, 0), (128, 2, 0, 1), (256, 4, 0, 0)):
            assert L.fg_spmm_dot_takes(plan, F, heads, tiles) == takes, (F, heads, tiles)
    finally:
        L.fg_spmm_plan_destroy(plan)


@pytest.mark.parametrize("where", ["sweep", "sum", "positions", "arrays"])
@pytest.mark.parametrize("shared", [True, False])
def test_attention_gradients_without_memory_for_the_scores_gradients(monkeypatch, where, shared):
    """The two arrays, the weighted sum they are for, its positions or the sweep's own scratch do not fit: the second sweep."""
    import torch
    from featgraph_amd import _lib, tuning
    from featgraph_amd.autograd import Graph
    from featgraph_amd.module import GraphAttentionhip, GSpMMhip, placeholder
    adj = _graph()
    H, D = 4, 32
    gen = torch.Generator(device="cuda").manual_seed(1)
    normal = lambda n: torch.randn((n, H, D), generator=gen, device="cuda")
    q, k, v, dout = normal(adj.shape[0]), normal(adj.shape[1]), normal(adj.shape[1]), normal(adj.shape[0])

    def step():
        if shared:
            leaves = [t.clone().requires_grad_() for t in (q, k, v)]
            return torch.autograd.grad(g.attention(*leaves, scale=0.2), leaves, dout)
        out = m.run([q, k, v])
        return m.backward(q, k, v, out, m.state_tvm, dout)

    def build():
        m = GraphAttentionhip(adj)
        m.build([placeholder(q.shape), placeholder(k.shape), placeholder(v.shape)], {'scale': 0.2})
        return m

    monkeypatch.setattr(tuning, "attention_keeps_score_gradients", lambda *a: False)
    g, m = (Graph(adj), None) if shared else (None, build())
    ref = step()
    g, m = (Graph(adj), None) if shared else (None, build())
    monkeypatch.setattr(tuning, "attention_keeps_score_gradients", lambda *a: True)
    calls = []
    if where == "sweep":
        monkeypatch.setattr(_lib.lib(), "fg_graph_attention_backward_kv_ds_f32", _failing(calls))
    elif where == "sum":
        def no_plan(self, *a):
            calls.append(1)
            raise MemoryError("cannot allocate the plan's scratch buffer")
        monkeypatch.setattr(GSpMMhip, "build", no_plan)
    elif where == "positions":
        def no_positions(self):
            calls.append(1)
            raise torch.cuda.OutOfMemoryError("positions")
        monkeypatch.setattr(GSpMMhip, "layout_positions", no_positions)
    else:
        real = torch.empty

        def no_arrays(*a, **kw):
            if a and a[0] == (2, H, adj.nnz):
                calls.append(1)
                raise torch.cuda.OutOfMemoryError("arrays")
            return real(*a, **kw)
        monkeypatch.setattr(torch, "empty", no_arrays)
    for _ in range(2):
        got = step()
        assert all(torch.equal(a, b) for a, b in zip(got, ref))
    assert len(calls) == 1


@pytest.mark.parametrize("where", ["scratch", "arrays"])
def test_additive_attention_without_memory_for_the_kept_sums(monkeypatch, where):
    """The training pass's buffers, or the array it keeps, do not fit: the plain forward pass and a sweep of its own for dEr."""
    import torch
    from featgraph_amd import _lib
    from featgraph_amd.autograd import Graph
    from featgraph_amd.module import GraphAttentionhip
    adj = _graph()
    H, D = 4, 32
    gen = torch.Generator(device="cuda").manual_seed(1)
    leaves = [torch.randn(s, generator=gen, device="cuda").requires_grad_() for s in ((adj.shape[0], H), (adj.shape[1], H), (adj.shape[1], H, D))]
    dout = torch.randn((adj.shape[0], H, D), generator=gen, device="cuda")

    def step(g):
        out = g.gat_attention(*leaves)
        return (out.detach(),) + torch.autograd.grad(out, leaves, dout)

    ref = step(Graph(adj))
    calls = []
    if where == "scratch":
        monkeypatch.setattr(_lib.lib(), "fg_graph_attention_additive_train_f32", _failing(calls))
    else:
        def no_arrays(self, *a):
            calls.append(1)
            raise torch.cuda.OutOfMemoryError("plus")
        monkeypatch.setattr(GraphAttentionhip, "train_forward", no_arrays)
    g = Graph(adj)
    for _ in range(2):
        got = step(g)
        assert torch.equal(got[0], ref[0])
        for a, b in zip(got[1:], ref[1:]):
            # either way within 2e-6 of float64 on such rows
            assert float((a - b).norm()) <= 4e-6 * float(b.norm())
    assert len(calls) == 1


@pytest.mark.parametrize("where", ["positions", "layout", "scratch", "call"])
@pytest.mark.parametrize("op", ["copy", "mul"])
def test_max_gradients_without_memory_for_the_sweeps(monkeypatch, where, op):
    """The sweep's layout, its positions, its scratch or the library's own buffers do not fit: the gradient result by result, from then on
    without another attempt, and nothing of the attempt stays."""
    import torch
    from featgraph_amd import _lib, ops, tuning
    from featgraph_amd.autograd import Graph
    from featgraph_amd.module import GSpMMhip, common
    adj = _graph()
    gen = torch.Generator(device="cuda").manual_seed(1)
    normal = lambda *s: torch.randn(s, generator=gen, device="cuda")
    leaves = [normal(adj.shape[1], 64).requires_grad_()] + ([normal(adj.nnz, 64).requires_grad_()] if op == "mul" else [])
    dy = normal(adj.shape[0], 64)
    g = Graph(adj)

    def step():
        out = g.aggregate(leaves[0], "max") if op == "copy" else ops.gspmm(g, "mul", "max", *leaves)
        return torch.autograd.grad(out, leaves, dy)

    monkeypatch.setattr(tuning, "select_by_sweep", lambda *a: False)
    ref = step()
    monkeypatch.setattr(tuning, "select_by_sweep", lambda *a: True)
    calls = []

    def no(error):
        def fail(*a, **kw):
            calls.append(1)
            raise error
        return fail
    if where == "positions":
        monkeypatch.setattr(GSpMMhip, "set_weight_order", no(torch.cuda.OutOfMemoryError("positions")))
    elif where == "layout":
        monkeypatch.setattr(GSpMMhip, "_layout", no(torch.cuda.OutOfMemoryError("layout")))
    elif where == "scratch":
        monkeypatch.setattr(common, "reserve", no(MemoryError("scratch")))
    else:
        monkeypatch.setattr(_lib.lib(), "fg_select_sources_f32", _failing(calls))
        monkeypatch.setattr(_lib.lib(), "fg_select_edges_f32", _failing(calls))
    for _ in range(2):
        for a, b in zip(step(), ref):
            # float sums of up to 400 results in two orders
            assert float((a - b).norm()) <= 400 * 2.0 ** -24 * float(b.norm())
    assert len(calls) == (1 if op == "copy" or where == "scratch" else 2)          # each operand's sweep (the edges' has no scratch), once
    if where == "scratch":
        assert 1 not in getattr(g._layout_owner.get(True), "_layouts", {})
