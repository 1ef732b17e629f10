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
