"""Items of several rows in dot-product attention and its gradients: rows on one lane group, on some and on all of a wavefront's, empty rows and
uneven ones among them, against float64."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mean", [1, 4, 9, 20, 45, 110])
@pytest.mark.parametrize("heads,head_len", [(1, 16), (3, 16), (2, 32), (1, 64)])
def test_rows_of_every_length(mean, heads, head_len):
    import torch
    from featgraph_amd.autograd import Graph
    rng = np.random.default_rng(mean)
    n, m = 211, 260
    deg = np.minimum(np.where(rng.random(n) < 0.15, 0, rng.geometric(1.0 / mean, n)), m)
    indptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    idx = np.concatenate([np.sort(rng.choice(m, d, replace=False)) for d in deg] + [np.zeros(0, int)]).astype(np.int32)
    adj = sp.csr_matrix((np.ones(len(idx), np.float32), idx, indptr), shape=(n, m))
    row, col = torch.from_numpy(np.repeat(np.arange(n), deg)), torch.from_numpy(idx.astype(np.int64))
    values = [torch.from_numpy(rng.standard_normal((k, heads, head_len)).astype(np.float32)) for k in (n, m, m)]
    dout = torch.from_numpy(rng.standard_normal((n, heads, head_len)).astype(np.float32))
    leaves = [v.cuda().requires_grad_() for v in values]
    out = Graph(adj).attention(*leaves)
    got = (out,) + torch.autograd.grad(out, leaves, dout.cuda())
    q, k, v = exact = [t.double().requires_grad_() for t in values]
    s = (q[row] * k[col]).sum(-1) / head_len ** 0.5
    top = torch.full((n, heads), -np.inf, dtype=torch.float64).scatter_reduce(0, row[:, None].expand(-1, heads), s.detach(), "amax")
    p = torch.exp(s - top[row])
    a = p / torch.zeros(n, heads, dtype=torch.float64).index_add(0, row, p)[row]
    want = torch.zeros(n, heads, head_len, dtype=torch.float64).index_add(0, row, a.unsqueeze(-1) * v[col])
    want = (want,) + torch.autograd.grad(want, exact, dout.double())
    for name, x, y in zip(("out", "dq", "dk", "dv"), got, want):
        # scores of up to about 5 with an error of head_len roundings, through the exponential, and sums of up to a row
        assert float((x.double().cpu() - y).norm()) <= 4e-6 * float(y.norm()), name
