"""Items of several rows in the weighted sum: from one row to 64 of a wavefront, each on one lane group, on some and on all of them, with
empty rows among them, remainders of every size and a non-finite source row that must reach its own destinations alone."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mean", [1, 3, 6, 12, 25, 50, 110])
@pytest.mark.parametrize("shape", [(4,), (8,), (16,), (24,), (32,), (64,), (128,), (4, 8), (4, 16), (2, 32)])
@pytest.mark.parametrize("parts", [None, 2])
def test_rows_of_every_length(mean, shape, parts):
    import torch
    from featgraph_amd.module import GSpMMhip, placeholder
    rng = np.random.default_rng(mean)
    n, m, heads = 257, 300, shape[0] if len(shape) == 2 else 1
    deg = np.minimum(rng.integers(0, 2 * mean + 1, n), m)
    indptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    idx = np.concatenate([np.sort(rng.choice(m, d, replace=False)) for d in deg] + [np.zeros(0, int)]).astype(np.int32)
    adj = sp.csr_matrix((np.ones(len(idx), np.float32), idx, indptr), shape=(n, m))
    x = rng.standard_normal((m,) + shape).astype(np.float32)
    x[7] = np.inf
    own = rng.standard_normal((n,) + shape).astype(np.float32)
    w = (0.5 + rng.random((adj.nnz, heads))).astype(np.float32)
    row, flat = np.repeat(np.arange(n), deg), x.reshape(m, heads, -1).astype(np.float64)
    terms = w[:, :, None].astype(np.float64) * flat[idx]
    want, mass = np.zeros((n,) + flat.shape[1:]), np.zeros((n,) + flat.shape[1:])
    np.add.at(want, row, terms)
    np.add.at(mass, row, np.abs(terms))
    g = GSpMMhip(adj)
    ws = (adj.nnz,) if heads == 1 else w.shape
    g.build([placeholder(x.shape), placeholder(ws)], {}, {"num_src_partitions": parts})
    wt, xt = torch.from_numpy(w).cuda().reshape(ws), torch.from_numpy(x).cuda()

    def check(got, want, mass, terms):
        ok = np.isfinite(want)
        got = got.cpu().numpy().astype(np.float64).reshape(want.shape)
        assert np.array_equal(np.isfinite(got), ok)
        # one rounding per term and per addition
        assert (np.abs(got[ok] - want[ok]) <= (terms + 2) * np.finfo(np.float32).eps * mass[ok]).all()

    g.out_tvm.fill_(float("nan"))
    check(g.run([xt, wt]), want, mass, 2 * mean)
    g.set_weight_order(np.arange(adj.nnz))
    both = g.run_with_dots(xt, wt, torch.from_numpy(own).cuda())
    if both is not None:
        check(both[0], want, mass, 2 * mean)
        with np.errstate(invalid="ignore"):
            prod = own.reshape(n, heads, -1).astype(np.float64)[row] * flat[idx]
            check(both[1], prod.sum(-1), np.abs(prod).sum(-1), flat.shape[-1])
