"""dQ of dot-product attention as a weighted sum with the scores' gradients that the sweep for dK and dV leaves, against
float64 torch autograd and against the sweep of its own: rows (both ways round) of no, one, a few, 64, 256, 257 and more
elements, one and several partitions on either side, and edge counts that are no multiple of four."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


def _graph(kind, rng):
    n_dst, n_src = 700, 500
    lengths = {"few": [0, 1, 2, 3, 5, 8, 9], "edges": [0, 1, 63, 64, 65, 255, 256, 257, 490], "mixed": [0, 1, 4, 30, 90, 300]}[kind]
    rows, cols = [], []
    for r in range(n_dst):
        k = lengths[rng.integers(len(lengths))]
        rows += [r] * k
        cols += list(rng.choice(n_src, size=k, replace=False))
    for r in range(0, n_dst, 2):                        # a column of more than 256 elements, and one of none
        if 7 not in cols[-k:]:
            rows.append(r)
            cols.append(7)
    adj = sp.csr_matrix((np.ones(len(rows), np.float32), (rows, cols)), shape=(n_dst, n_src + 1))
    adj.sum_duplicates()
    return adj


def _float64(adj, q, k, v, dout, scale):
    import torch
    q, k, v = (t.detach().double().requires_grad_() for t in (q, k, v))
    row = torch.from_numpy(np.repeat(np.arange(adj.shape[0]), np.diff(adj.indptr))).cuda()
    col = torch.from_numpy(adj.indices).long().cuda()
    s = scale * (k[col] * q[row]).sum(-1)
    top = torch.full((adj.shape[0], s.shape[1]), -1e300, dtype=torch.float64, device="cuda")
    top = top.scatter_reduce(0, row[:, None].expand_as(s), s.detach(), "amax")
    p = (s - top[row]).exp()
    a = p / torch.zeros_like(top).index_add(0, row, p)[row]
    out = torch.zeros_like(q).index_add(0, row, a[:, :, None] * v[col])
    return torch.autograd.grad(out, (q, k, v), dout.double())


@pytest.mark.parametrize("kind", ["few", "edges", "mixed"])
@pytest.mark.parametrize("heads,head_len", [(1, 64), (1, 16), (3, 32), (4, 16), (16, 32)])
@pytest.mark.parametrize("parts", [1, 3])
def test_both_ways_match_float64(monkeypatch, kind, heads, head_len, parts):
    import torch
    from featgraph_amd import tuning
    from featgraph_amd.autograd import Graph
    monkeypatch.setattr(tuning, "_partitions", lambda *a, **k: parts)
    adj = _graph(kind, np.random.default_rng(heads * 100 + head_len))
    gen = torch.Generator(device="cuda").manual_seed(4)
    normal = lambda n: torch.randn((n, heads, head_len), generator=gen, device="cuda")
    q, k, v, dout = normal(adj.shape[0]), normal(adj.shape[1]), normal(adj.shape[1]), normal(adj.shape[0])
    ref = _float64(adj, q, k, v, dout, 0.3)
    got = {}
    for kept in (True, False):
        monkeypatch.setattr(tuning, "attention_keeps_score_gradients", lambda *a, kept=kept: kept)
        leaves = [t.clone().requires_grad_() for t in (q, k, v)]
        got[kept] = torch.autograd.grad(Graph(adj).attention(*leaves, scale=0.3), leaves, dout)
        for name, x, y in zip(("dQ", "dK", "dV"), got[kept], ref):
            # fp32 sums of at most 700 terms, dot products of 64 and an exponential good to 2 ulp of its argument (scores up to
            # about 10: 10 * 2^-24 = 6e-7 relative)
            assert float((x.double() - y).norm()) <= 2e-6 * float(y.norm()), (name, kept)
    assert torch.equal(got[True][1], got[False][1]) and torch.equal(got[True][2], got[False][2])


def test_host_positions_are_let_go_and_made_again(monkeypatch):
    """The elements' CSR positions (4 bytes per edge) stay on the host only until the device has the positions made of them, not at
    all where nothing will be, and a second build() makes its own."""
    import torch
    from featgraph_amd import tuning
    from featgraph_amd.module import GraphAttentionhip, placeholder
    adj = _graph("mixed", np.random.default_rng(1))
    monkeypatch.setattr(tuning, "attention_keeps_score_gradients", lambda *a: True)
    gen = torch.Generator(device="cuda").manual_seed(4)
    m = GraphAttentionhip(adj)
    for heads, head_len in ((4, 16), (1, 64)):
        q, k, v, dout = (torch.randn((n, heads, head_len), generator=gen, device="cuda") for n in adj.shape[:1] + adj.shape[1:] * 2 + adj.shape[:1])
        m.build([placeholder(q.shape), placeholder(k.shape), placeholder(v.shape)], {'scale': 0.3}, {'num_dst_partitions': 2})
        out = m.run([q, k, v])
        got = m.backward(q, k, v, out, m.state_tvm, dout)
        for x, y in zip(got, _float64(adj, q, k, v, dout, 0.3)):
            assert float((x.double() - y).norm()) <= 2e-6 * float(y.norm())      # as above
        assert [lay for lay in m._layouts.values() if 'csr_pos_host' in lay] == []
        assert len([lay for lay in m._layouts.values() if 'sum_position' in lay]) == 1
    m = GraphAttentionhip(adj)
    er, el, v = (torch.randn(s, generator=gen, device="cuda") for s in ((adj.shape[0], 2), (adj.shape[1], 2), (adj.shape[1], 2, 32)))
    m.build([placeholder(t.shape) for t in (er, el, v)], {'scores': 'additive'})
    out, saved = m.train_forward(er, el, v)
    m.train_backward(er, el, v, out, saved, torch.ones_like(out))
    assert [lay for lay in m._layouts.values() if 'csr_pos_host' in lay] == []


@pytest.mark.parametrize("kind", ["few", "edges"])
@pytest.mark.parametrize("heads,head_len", [(8, 16), (8, 64), (12, 16)])
def test_relayout_of_eight_and_of_twelve_heads(monkeypatch, kind, heads, head_len):
    """The scores' gradients of 8 heads go through a relayout kernel of their own, those of 12 through the one for any count."""
    test_both_ways_match_float64(monkeypatch, kind, heads, head_len, 3)
