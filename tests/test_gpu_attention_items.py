"""The plan that attention walks: rows above one staging round lead each partition, longest first, and runs of short rows
are as short as the graph is small.  Forward and gradients against float64, with long rows in no order of length, empty
rows between them and rows at the edges of a round."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu

LENS = [1, 0, 257, 16, 17, 0, 255, 256, 900, 3, 512, 513, 0] + [2] * 130 + [300, 40, 700, 0, 258]


@pytest.mark.parametrize("kind,heads,head_len", [("dot", 3, 16), ("dot", 1, 64), ("gat", 2, 32), ("gat", 9, 16)])
@pytest.mark.parametrize("repeat", [1, 20])
def test_attention_matches_float64(kind, heads, head_len, repeat):
    import torch
    from featgraph_amd.autograd import Graph
    rng = np.random.default_rng(heads)
    lens, n_src = LENS * repeat, 1000
    cols = [np.sort(rng.choice(n_src, size=l, replace=False)) for l in lens]
    indptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    adj = sp.csr_matrix((np.ones(indptr[-1], np.float32), np.concatenate(cols).astype(np.int32), indptr), shape=(len(lens), n_src))
    g, n = Graph(adj), len(lens)
    t = lambda *s: torch.from_numpy(rng.standard_normal(s).astype(np.float32)).cuda().requires_grad_()
    v, dout = t(n_src, heads, head_len), t(n, heads, head_len).detach()
    a, b = (t(n, heads, head_len), t(n_src, heads, head_len)) if kind == "dot" else (t(n, heads), t(n_src, heads))
    out = g.attention(a, b, v) if kind == "dot" else g.gat_attention(a, b, v)
    got = (out,) + torch.autograd.grad(out, [a, b, v], dout)

    a64, b64, v64 = (x.detach().double().requires_grad_() for x in (a, b, v))
    row = torch.repeat_interleave(torch.arange(n), torch.from_numpy(np.diff(indptr)).long()).cuda()
    col = torch.from_numpy(adj.indices).cuda().long()
    s = (a64[row] * b64[col]).sum(-1) / head_len ** 0.5 if kind == "dot" else torch.nn.functional.leaky_relu(a64[row] + b64[col], 0.2)
    top = torch.full((n, heads), -np.inf, dtype=torch.float64, device="cuda").index_reduce(0, row, s.detach(), "amax")
    p = torch.exp(s - top[row])
    p = p / torch.zeros((n, heads), dtype=torch.float64, device="cuda").index_add(0, row, p)[row]
    ref = torch.zeros((n, heads, head_len), dtype=torch.float64, device="cuda").index_add(0, row, p[..., None] * v64[col])
    for x, y in zip(got, (ref,) + torch.autograd.grad(ref, [a64, b64, v64], dout.double())):
        # sums of up to 900 (gradients: 60 * repeat * a few) fp32 products, and an exponential good to 2 ulp of its argument
        assert float((x.detach().double() - y.detach()).norm() / y.detach().norm()) <= 1e-5


@pytest.mark.parametrize("head_len,degree", [(64, 1), (64, 23), (64, 24), (32, 19), (32, 20), (16, 11), (16, 12)])
def test_head_by_head_copy_changes_no_bit(monkeypatch, head_len, degree):
    """On both sides of the line from which the gathered operands are copied (24, 20 or 12 elements per source, 64 MB)."""
    import torch
    from featgraph_amd import _lib
    from featgraph_amd.autograd import Graph
    n, heads = 33000, 512 // head_len
    cols = np.sort((np.arange(n)[:, None] * 7 + np.arange(degree)[None, :] * 613) % n, axis=1)
    adj = sp.csr_matrix((np.ones(n * degree, np.float32), cols.ravel().astype(np.int32),
                         (np.arange(n + 1) * degree).astype(np.int32)), shape=(n, n))
    gen = torch.Generator(device="cuda").manual_seed(degree)
    q, k, v, dout = (torch.randn(n, heads, head_len, generator=gen, device="cuda").requires_grad_() for _ in range(4))
    results = []
    for tile_major in (0, 1, 2):
        monkeypatch.setattr(_lib, "plan_opts", _lib.FgPlanOpts(tile_major=tile_major) if tile_major else None)
        out = Graph(adj).attention(q, k, v)
        results.append((out.detach(),) + torch.autograd.grad(out, [q, k, v], dout.detach()))
    for other in results[1:]:
        assert all(torch.equal(a, b) for a, b in zip(results[0], other))
