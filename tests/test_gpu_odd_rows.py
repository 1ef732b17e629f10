"""Broadcast messages over rows of every remainder of a 16-byte word, at 4-byte alignment, on rows that one lane group, a few of them or
all of a wavefront's share: aggregated with and without positions, in one source partition and several, and per edge."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu
BIN = {"add": np.add, "sub": np.subtract, "mul": np.multiply, "div": np.divide}


def _graph(rng, kind):
    n, m = 190, 230
    if kind == "short":
        a = sp.random(n, m, density=0.015, format="lil", random_state=rng)
    else:
        a = sp.lil_matrix((n, m))
        for v in range(n):                       # items of 1, 2, 3, .. rows
            k = int(rng.integers(0, 200)) if v % 7 == 0 else int(rng.integers(0, 24))
            a[v, rng.choice(m, k, replace=False)] = 1
    a[[0, 100, 189], :] = 0
    a = a.tocsr()
    a.eliminate_zeros()
    a.sort_indices()
    return a.astype(np.float32)


def _odd(x):
    import torch
    store = torch.empty(x.size + 1, dtype=torch.float32, device="cuda")
    t = store[1:].view(x.shape)
    t.copy_(torch.from_numpy(x))
    return t


@pytest.mark.parametrize("F", [1, 3, 4, 5, 6, 7, 8, 9, 13, 16, 17, 31, 33, 63, 65, 130, 259])
@pytest.mark.parametrize("kind", ["short", "mixed"])
@pytest.mark.parametrize("parts", [None, 3])
def test_aggregated(F, kind, parts):
    import torch
    from featgraph_amd.module import GSpMMhip, placeholder
    rng = np.random.default_rng(F)
    adj = _graph(rng, kind)
    n, m = adj.shape
    row, col = np.repeat(np.arange(n), np.diff(adj.indptr)), adj.indices
    x = rng.standard_normal((m, F)).astype(np.float32)
    for op, e_len, reduce in [("mul", F, "sum"), ("add", 1, "sum"), ("sub", F, "max"), ("mul", 1, "min"), ("div", F, "mean"), ("copy", 0, "max")]:
        if op == "copy":
            msg, args = x[col], [_odd(x)]
            name, phs = "copy_u", [placeholder(x.shape)]
        else:
            w = (1.5 + rng.random((adj.nnz, e_len))).astype(np.float32)
            msg, args = BIN[op](x[col], w), [_odd(x), _odd(w)]
            name, phs = "u_%s_e" % op, [placeholder(x.shape), placeholder(w.shape)]
        extreme = reduce in ("max", "min")
        g = GSpMMhip(adj)
        g.build(phs, {"msg": name, "reduce": reduce, "broadcast": True, "return_arg": extreme}, {"num_src_partitions": parts})
        g.out_tvm.fill_(float("nan"))
        got = g.run(args).cpu().numpy().reshape(n, F)
        want, at, mass = np.zeros((n, F)), np.full((n, F), -1), np.zeros((n, F))
        for v in range(n):
            b, e = adj.indptr[v], adj.indptr[v + 1]
            if e > b:
                seg = msg[b:e].astype(np.float64)
                want[v] = seg.sum(0) if reduce == "sum" else seg.mean(0) if reduce == "mean" else seg.max(0) if reduce == "max" else seg.min(0)
                mass[v] = np.abs(seg).sum(0) if not extreme else 0
                if extreme:
                    at[v] = b + (np.argmax(msg[b:e], 0) if reduce == "max" else np.argmin(msg[b:e], 0))
        what = "%s %s F=%d, %d edge features" % (name, reduce, F, e_len)
        # one rounding per term of the sum, two of the message and the scale
        assert (np.abs(got - want) <= 240 * np.finfo(np.float32).eps * mass).all(), what
        if extreme:
            assert np.array_equal(g.arg_tvm.cpu().numpy().reshape(n, F), at), what


@pytest.mark.parametrize("F", [1, 3, 4, 5, 7, 8, 9, 18, 31, 65, 131])
def test_per_edge(F):
    import torch
    from featgraph_amd import ops
    from featgraph_amd.autograd import Graph
    rng = np.random.default_rng(F)
    adj = _graph(rng, "mixed")
    n, m = adj.shape
    g = Graph(adj)
    row, col = np.repeat(np.arange(n), np.diff(adj.indptr)), adj.indices
    values = {"u": rng.standard_normal((m, F)), "v": rng.standard_normal((n, F)), "e": 1.5 + rng.random((adj.nnz, F)), "1": 1.5 + rng.random((adj.nnz, 1))}
    values = {k: v.astype(np.float32) for k, v in values.items()}
    at = {"u": col, "v": row, "e": slice(None), "1": slice(None)}
    for op, lhs, rhs in [("add", "u", "v"), ("sub", "v", "e"), ("mul", "u", "1"), ("div", "u", "e"), ("mul", "1", "v")]:
        got = ops.gsddmm(g, op, _odd(values[lhs]), _odd(values[rhs]), lhs.replace("1", "e"), rhs.replace("1", "e")).cpu().numpy()
        want = BIN[op](values[lhs][at[lhs]], values[rhs][at[rhs]])
        assert np.array_equal(got, want) if op != "div" else np.allclose(got, want, rtol=3e-7, atol=0), (op, lhs, rhs)


@pytest.mark.parametrize("F", [5, 32, 33, 65, 257])
@pytest.mark.parametrize("targets", [("e", "v"), ("u", "e"), ("e", "e")])
def test_per_edge_over_an_operand_of_its_own(F, targets):
    """Results written over the edge operand they are formed from."""
    import torch
    from featgraph_amd.module import GSDDMMhip, placeholder
    rng = np.random.default_rng(F)
    adj = _graph(rng, "mixed")
    n, m = adj.shape
    at = {"u": adj.indices, "v": np.repeat(np.arange(n), np.diff(adj.indptr)), "e": slice(None)}
    x, y = (rng.standard_normal(({"u": m, "v": n, "e": adj.nnz}[t], F), dtype=np.float32) for t in targets)
    mod = GSDDMMhip(adj)
    mod.build([placeholder(x.shape), placeholder(y.shape)], {"op": "sub", "lhs_target": targets[0], "rhs_target": targets[1]}, {})
    own = 0 if targets[0] == "e" else 1
    mod.out_tvm.copy_(torch.from_numpy((x, y)[own]))
    args = [torch.from_numpy(a).cuda() for a in (x, y)]
    args[own] = mod.out_tvm
    assert np.array_equal(mod.run(args).cpu().numpy(), x[at[targets[0]]] - y[at[targets[1]]])
