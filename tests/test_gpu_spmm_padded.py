"""Weighted sums over rows of a length that suits no tile, computed on a zero-padded copy and stored short: every remainder of a
16-byte word, one tile and several, masked tiles, passes with buffers of their own and passes that add, split rows, 64-bit offsets,
several heads, inputs at 4-byte alignment, and the sum with dots."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


def _graph(rng):
    a = sp.random(330, 410, density=0.03, format="lil", random_state=rng)
    a[17, :] = 1
    a[200, :300] = 1
    a[[0, 150, 329], :] = 0
    a = a.tocsr()
    a.data[:] = rng.standard_normal(a.nnz)
    a.eliminate_zeros()
    a.sort_indices()
    return a.astype(np.float32)


OPTS = [dict(), dict(split_threshold=64, item_edges=64), dict(wide_offsets=1), dict(tile_major=1, item_edges=16)]


@pytest.mark.parametrize("shape", [(9,), (30,), (31,), (41,), (63,), (65,), (79,), (97,), (98,), (130,), (239,), (602,), (3, 13), (2, 20), (4, 6), (4, 13), (2, 70)])
@pytest.mark.parametrize("opts", range(len(OPTS)))
@pytest.mark.parametrize("parts,buffers", [(None, 0), (3, 1), (3, 2)])
def test_short_rows(monkeypatch, shape, opts, parts, buffers):
    import torch
    from featgraph_amd import _lib, tuning
    from featgraph_amd.module import GSpMMhip, VanillaSpMMhip, placeholder
    monkeypatch.setattr(_lib, "plan_opts", _lib.FgPlanOpts(pass_buffers=buffers, **OPTS[opts]))
    monkeypatch.setattr(tuning, "PAD_MIN_GATHERED", 0)
    rng = np.random.default_rng(len(shape) * 1000 + shape[0])
    adj = _graph(rng)
    n, m = adj.shape
    heads = shape[0] if len(shape) == 2 else 1
    x = rng.standard_normal((m,) + shape).astype(np.float32)
    w = rng.standard_normal((adj.nnz, heads)).astype(np.float32)
    own = rng.standard_normal((n,) + shape).astype(np.float32)
    row, col = np.repeat(np.arange(n), np.diff(adj.indptr)), adj.indices
    flat, f64 = x.reshape(m, heads, -1), np.float64

    def summed(weights):
        out, mass = np.zeros((n,) + flat.shape[1:]), np.zeros((n,) + flat.shape[1:])
        terms = weights.astype(f64)[:, :, None] * flat.astype(f64)[col]
        np.add.at(out, row, terms)
        np.add.at(mass, row, np.abs(terms))
        return out.reshape((n,) + shape), mass.reshape((n,) + shape)

    def check(got, want, mass, terms):
        got = got.cpu().numpy()
        assert got.shape == want.shape and (np.abs(got - want) <= (terms + 4) * np.finfo(np.float32).eps * mass).all()

    store = torch.empty(x.size + 1, dtype=torch.float32, device="cuda")
    xt = store[1:].view(x.shape)                        # 4-byte aligned
    xt.copy_(torch.from_numpy(x))
    sched = {"num_src_partitions": parts}
    if heads == 1:
        v = VanillaSpMMhip(adj)
        v.build([placeholder(x.shape)], {}, sched)
        assert v._pad_from == shape[0]
        v.out_tvm.fill_(float("nan"))
        check(v.run([xt]), *summed(adj.data[:, None]), 410)
    g = GSpMMhip(adj)
    ws = (adj.nnz,) if heads == 1 else w.shape
    g.build([placeholder(x.shape), placeholder(ws)], {}, sched)
    assert g._pad_from == shape[-1]
    g.out_tvm.fill_(float("nan"))
    wt = torch.from_numpy(w).cuda().reshape(ws)
    check(g.run([xt, wt]), *summed(w), 410)
    g.set_weight_order(np.arange(adj.nnz))
    both = g.run_with_dots(torch.from_numpy(x).cuda(), wt, torch.from_numpy(own).cuda())
    if both is None:
        assert not _lib.lib().fg_spmm_dot_takes(g._active["plan"], g._feat_len, heads, g._num_feat_partitions)
        return
    check(both[0], *summed(w), 410)
    prod = own.reshape(n, heads, -1).astype(f64)[row] * flat.astype(f64)[col]
    check(both[1], prod.sum(-1).reshape(ws), np.abs(prod).sum(-1).reshape(ws), shape[-1])
