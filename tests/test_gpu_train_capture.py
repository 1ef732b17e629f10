"""Additive attention's training pass recorded into a HIP graph: its scratch is sized for the shape that is built, not once per
module, and never grown while a stream is being captured."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


def test_scratch_is_reserved_per_build_and_never_grown_under_capture():
    import torch
    from featgraph_amd import _lib
    from featgraph_amd.module import GraphAttentionhip, placeholder
    n_dst, n_src = 500, 400
    adj = sp.random(n_dst, n_src, density=0.05, format="csr", random_state=np.random.default_rng(6)).astype("float32")
    gen = torch.Generator(device="cuda").manual_seed(1)
    m = GraphAttentionhip(adj)

    def inputs(H, D):
        return [torch.randn(s, generator=gen, device="cuda") for s in ((n_dst, H), (n_src, H), (n_src, H, D))]

    def build(H, D):
        m.build([placeholder(s) for s in ((n_dst, H), (n_src, H), (n_src, H, D))], {'scores': 'additive'},
                {'num_src_partitions': 3, 'num_dst_partitions': 2})

    def plan_bytes():
        return _lib.lib().fg_spmm_plan_bytes(m._active['plan'])

    build(1, 16)                                    # the kernels are loaded (head lengths 16 and 32)
    m.train_forward(*inputs(1, 16))
    build(1, 32)
    m.train_forward(*inputs(1, 32))
    for H, D in ((2, 32), (8, 32)):                 # the second build needs more than the first one left
        x = inputs(H, D)
        build(H, D)
        torch.cuda.synchronize()
        refused = torch.cuda.CUDAGraph()
        with torch.cuda.graph(refused):
            with pytest.raises(ValueError, match="fg_spmm_plan_reserve"):
                m.train_forward(*x)
        m.reserve_train()
        held = plan_bytes()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out, saved = m.train_forward(*x)
        assert plan_bytes() == held
        for _ in range(3):
            for t in x:
                t.copy_(torch.randn(t.shape, generator=gen, device="cuda"))
            want, kept = m.train_forward(*x)
            for t in (out,) + saved:
                t.fill_(float("nan"))
            graph.replay()
            torch.cuda.synchronize()
            assert all(torch.equal(a, b) for a, b in zip((out,) + saved, (want,) + kept))


@pytest.mark.parametrize("tail,parts", [((64,), 1), ((4, 16), 2)])
def test_sum_with_dots_scratch_can_be_reserved(monkeypatch, tail, parts):
    import torch
    from featgraph_amd import _lib, tuning
    from featgraph_amd.module import GSpMMhip, placeholder
    monkeypatch.setattr(tuning, "choose_spmm", lambda *a, **k: (parts, 0))
    n_dst, n_src = 500, 3000
    adj = sp.random(n_dst, n_src, density=0.05, format="csr", random_state=np.random.default_rng(6)).astype("float32").tolil()
    adj[7, :] = 1.0                                 # a row in pieces
    adj = adj.tocsr().astype("float32")
    gen = torch.Generator(device="cuda").manual_seed(1)
    normal = lambda *s: torch.randn(s, generator=gen, device="cuda")
    x, w, own = normal(n_src, *tail), normal(adj.nnz, *tail[:-1]), normal(n_dst, *tail)

    def build():
        m = GSpMMhip(adj)
        m.build([placeholder(x.shape), placeholder(w.shape)], {}, {})
        assert m._active['P'] == parts
        m.set_weight_order(np.arange(adj.nnz)[::-1].copy())
        return m

    warm, m = build(), build()
    warm.run_with_dots(x, w, own)                   # the kernels are loaded
    torch.cuda.synchronize()
    m.run([x, w])                                   # lays the weights' buffer out
    refused = torch.cuda.CUDAGraph()
    with torch.cuda.graph(refused):
        with pytest.raises(ValueError, match="fg_spmm_plan_reserve"):
            m.run_with_dots(x, w, own)
    m.reserve_dots()
    held = _lib.lib().fg_spmm_plan_bytes(m._active['plan'])
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out, dots = m.run_with_dots(x, w, own)
    assert _lib.lib().fg_spmm_plan_bytes(m._active['plan']) == held
    for _ in range(3):
        for t in (x, w, own):
            t.copy_(torch.randn(t.shape, generator=gen, device="cuda"))
        want = warm.run_with_dots(x, w, own)
        out.fill_(float("nan"))
        dots.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want[0]) and torch.equal(dots, want[1])
    for heads, head_len in ((2, 128), (1, 20)):     # a head cut into tiles; a tile that is not whole
        with pytest.raises(ValueError):
            _lib.check(_lib.lib().fg_spmm_plan_reserve(m._active['plan'], 9, heads, head_len, 0))
