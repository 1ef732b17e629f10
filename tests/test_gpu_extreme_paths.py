"""max / min with positions: the kernel finds them by one comparison per message and falls back to the full rule (first
of the best, NaN above everything, the first message always enters) where that may differ -- NaN messages, rows of -inf,
edge positions in another order.  Values and positions exactly as the oracle's, with ties, signed zeros and split rows,
at feature lengths with one to sixteen lane groups per wavefront; and the gradient that follows the positions."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


def _graph(rng, lens, n_src=700):
    cols = [np.sort(rng.choice(n_src, size=l, replace=False)) for l in lens]
    indptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    return sp.csr_matrix((np.ones(indptr[-1], np.float32), np.concatenate(cols).astype(np.int32), indptr), shape=(len(lens), n_src))


LENS = [1, 2, 3, 0, 17, 64, 65, 127, 128, 129, 300, 600] + [2] * 70 + [40] * 6


@pytest.mark.parametrize("special", ["ties", "nan", "minus_inf"])
@pytest.mark.parametrize("reduce", ["max", "min"])
@pytest.mark.parametrize("feat_len", [7, 16, 36, 100, 260])
def test_positions_match_the_oracle(oracle, special, reduce, feat_len):
    import torch
    from featgraph_amd.module import GSpMMhip, placeholder
    rng = np.random.default_rng(feat_len)
    adj = _graph(rng, LENS)
    x = rng.integers(-1, 2, size=(700, feat_len)).astype(np.float32)         # -1, 0, 1: ties everywhere
    x[x == 0] *= np.where(rng.random((x == 0).sum()) < 0.5, -1, 1)           # zeros of both signs tie as well
    if special == "nan":
        x[rng.random(x.shape) < 0.01] = np.nan
    if special == "minus_inf":
        x[rng.random(x.shape) < 0.7] = -np.inf if reduce == "max" else np.inf
    e = np.zeros((adj.nnz, 1), np.float32)
    for msg, arrays, o in (("copy_u", [x], ("copy_lhs", x, None, "u", "e")), ("u_add_e", [x, e], ("add", x, e, "u", "e"))):
        ref, ref_arg = oracle.gspmm_bcast(adj.indptr, adj.indices, o[0], reduce, o[1], o[2], o[3], o[4])
        for P in (None, 3):
            m = GSpMMhip(adj)
            m.build([placeholder(a.shape) for a in arrays], {'msg': msg, 'reduce': reduce, 'return_arg': True, 'broadcast': True},
                    {'num_src_partitions': P})
            out = m.run([torch.from_numpy(a).cuda() for a in arrays]).cpu().numpy()
            assert np.array_equal(out, ref, equal_nan=True), (msg, P)
            assert np.array_equal(m.arg_tvm.cpu().numpy(), ref_arg), (msg, P)
    # edge operands in another order: the first of a tie is the first in that order
    where = rng.permutation(adj.nnz).astype(np.int32)
    m = GSpMMhip(adj)
    m.build([placeholder(x.shape), placeholder(e.shape)], {'msg': 'u_add_e', 'reduce': reduce, 'return_arg': True, 'broadcast': True}, {})
    m.set_weight_order(where)
    out = m.run([torch.from_numpy(x).cuda(), torch.from_numpy(e).cuda()]).cpu().numpy()
    assert np.array_equal(out, ref, equal_nan=True)
    arg = m.arg_tvm.cpu().numpy()
    for v in np.flatnonzero(np.diff(adj.indptr)):
        a, b = adj.indptr[v], adj.indptr[v + 1]
        seg = x[adj.indices[a:b]]
        best = (seg == ref[v]) | (np.isnan(seg) & np.isnan(ref[v]))
        want = np.where(best, where[a:b, None], np.iinfo(np.int32).max).min(0)
        assert np.array_equal(arg[v], want), v


@pytest.mark.parametrize("op,e_len", [("add", 1), ("sub", 5), ("mul", 5), ("mul", 1), ("div", 5)])
def test_gradient_goes_to_the_selected_edge(op, e_len):
    import torch
    from featgraph_amd import ops
    from featgraph_amd.autograd import Graph
    rng = np.random.default_rng(3)
    adj = _graph(rng, LENS)
    g = Graph(adj)
    x = torch.from_numpy(rng.standard_normal((700, 5)).astype(np.float32)).cuda().requires_grad_()
    e = torch.from_numpy((rng.random((adj.nnz, e_len)) + 0.5).astype(np.float32)).cuda().requires_grad_()
    dout = torch.from_numpy(rng.standard_normal((len(LENS), 5)).astype(np.float32)).cuda()
    got = torch.autograd.grad(ops.gspmm(g, op, "max", x, e), [x, e], dout)
    x64, e64 = x.detach().double().requires_grad_(), e.detach().double().requires_grad_()
    row = torch.repeat_interleave(torch.arange(len(LENS)), torch.from_numpy(np.diff(adj.indptr)).long()).cuda()
    xs = x64[torch.from_numpy(adj.indices).cuda().long()]
    m = xs + e64 if op == "add" else xs - e64 if op == "sub" else xs * e64 if op == "mul" else xs / e64
    out = torch.zeros((len(LENS), 5), dtype=torch.float64, device="cuda").scatter_reduce(
        0, row[:, None].expand_as(m), m, "amax", include_self=False)
    for a, b in zip(got, torch.autograd.grad(out, [x64, e64], dout.double())):
        # one product of three fp32 factors per term, at most 5 * 83 terms per sum
        assert ((a.double() - b).abs() <= 1e-5 + 1e-4 * b.abs()).all()


@pytest.mark.parametrize("msg", ["copy", "mul"])
def test_gradient_can_be_differentiated_again(msg):
    """create_graph: d/d(dout) and d/d(operand) of a max gradient, against the same chain in float64."""
    import torch
    from featgraph_amd import ops
    from featgraph_amd.autograd import Graph
    rng = np.random.default_rng(5)
    adj = _graph(rng, LENS)
    g = Graph(adj)
    x = torch.from_numpy(rng.standard_normal((5, 700)).astype(np.float32)).cuda().t().requires_grad_()      # not contiguous
    e = torch.from_numpy((rng.random((adj.nnz, 5)) + 0.5).astype(np.float32)).cuda().requires_grad_()
    dout = torch.from_numpy(rng.standard_normal((len(LENS), 5)).astype(np.float32)).cuda().requires_grad_()
    row = torch.repeat_interleave(torch.arange(len(LENS)), torch.from_numpy(np.diff(adj.indptr)).long()).cuda()
    col = torch.from_numpy(adj.indices).cuda().long()

    def second(forward, x, e, dout):
        dx = torch.autograd.grad(forward(x, e), x, dout, create_graph=True)[0]
        return torch.autograd.grad((dx * dx).sum(), [dout, e] if msg == "mul" else [dout])

    def wide(x, e):
        m = x[col] * e if msg == "mul" else x[col]
        return torch.zeros((len(LENS), 5), dtype=torch.float64, device="cuda").scatter_reduce(
            0, row[:, None].expand_as(m), m, "amax", include_self=False)

    got = second((lambda x, e: ops.gspmm(g, "mul", "max", x, e)) if msg == "mul" else (lambda x, e: g.aggregate(x, "max")), x, e, dout)
    want = second(wide, *[t.detach().double().requires_grad_() for t in (x, e, dout)])
    for a, b in zip(got, want):      # as above: products of a few fp32 factors, at most 5 * 83 terms per sum
        assert ((a.double() - b).abs() <= 1e-5 + 1e-4 * b.abs()).all()


def test_input_may_change_before_the_gradient():
    """A max aggregation's gradient needs the positions alone: overwriting its input in between is allowed."""
    import torch
    from featgraph_amd.autograd import Graph
    rng = np.random.default_rng(6)
    g = Graph(_graph(rng, LENS))
    leaf = torch.from_numpy(rng.standard_normal((700, 5)).astype(np.float32)).cuda().requires_grad_()
    x = leaf * 1
    out = g.aggregate(x, "max")
    before = torch.autograd.grad(out.sum(), leaf, retain_graph=True)[0]
    x.mul_(2)
    assert torch.equal(before, torch.autograd.grad(out.sum(), leaf)[0])


@pytest.mark.parametrize("reduce", ["max", "min"])
@pytest.mark.parametrize("feat_len", [7, 36, 100, 260])
def test_masked_messages_and_nan_together(oracle, reduce, feat_len):
    """Features that are masked in most sources, in all, or not at all, with NaN among them: the first of a row's masked
    messages where there is nothing else, the first NaN where there is one, whatever the other features hold."""
    import torch
    from featgraph_amd.module import GSpMMhip, placeholder
    rng = np.random.default_rng(feat_len)
    adj = _graph(rng, LENS)
    x = rng.integers(-1, 2, size=(700, feat_len)).astype(np.float32)
    x[rng.random(x.shape) < rng.choice([0, 0.9, 1], size=feat_len)] = -np.inf if reduce == "max" else np.inf
    x[rng.random(x.shape) < rng.choice([0, 0.01], size=feat_len)] = np.nan
    ref, ref_arg = oracle.gspmm_bcast(adj.indptr, adj.indices, "copy_lhs", reduce, x, None, "u", "e")
    for P in (None, 3):
        m = GSpMMhip(adj)
        m.build([placeholder(x.shape)], {'msg': 'copy_u', 'reduce': reduce, 'return_arg': True}, {'num_src_partitions': P})
        out = m.run([torch.from_numpy(x).cuda()]).cpu().numpy()
        assert np.array_equal(out, ref, equal_nan=True), P
        assert np.array_equal(m.arg_tvm.cpu().numpy(), ref_arg), P


@pytest.mark.parametrize("feat_len", [64, 100])
def test_masked_messages_cost_no_second_walk(feat_len):
    """max with positions over features that are -inf in most sources takes what it takes without them (1.0 measured; with
    every such row walked a second time, by the full rule, 3.0)."""
    import torch
    from featgraph_amd.module import GSpMMhip, placeholder
    n, degree = 20000, 100
    rng = np.random.default_rng(4)
    cols = np.sort(rng.integers(0, n // degree, size=(n, degree)) + np.arange(degree) * (n // degree), axis=1).astype(np.int32)
    adj = sp.csr_matrix((np.ones(n * degree, np.float32), cols.reshape(-1), (np.arange(n + 1) * degree).astype(np.int32)), shape=(n, n))
    m = GSpMMhip(adj)
    m.build([placeholder((n, feat_len))], {'msg': 'copy_u', 'reduce': 'max', 'return_arg': True}, {})
    gen = torch.Generator(device="cuda").manual_seed(1)
    plain = torch.randn(n, feat_len, generator=gen, device="cuda")
    masked = plain.masked_fill(torch.rand(n, feat_len, generator=gen, device="cuda") < 0.98, -float("inf"))
    best = {}
    for _ in range(6):
        for name, x in (("plain", plain), ("masked", masked)):
            m.run([x])
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(5):
                m.run([x])
            b.record()
            torch.cuda.synchronize()
            best[name] = min(best.get(name, 1e9), a.elapsed_time(b))
    assert best["masked"] < 1.6 * best["plain"], best


@pytest.mark.parametrize("what", ["aggregate", "gspmm"])
def test_fixed_order_on_request(monkeypatch, what):
    """Under use_deterministic_algorithms the gradient comes from torch's operators: the same bits twice, close to float64, and
    without the kernel that adds by atomics."""
    import torch
    from featgraph_amd.autograd import Graph
    from featgraph_amd.module.general import BroadcastOp
    rng = np.random.default_rng(11)
    adj = _graph(rng, LENS)
    g = Graph(adj)
    t = lambda *s: torch.from_numpy(rng.standard_normal(s).astype(np.float32)).cuda().requires_grad_()
    x, e, d = t(700, 36), t(adj.nnz, 36), t(adj.shape[0], 36).detach()
    operands = [x] if what == "aggregate" else [x, e]
    step = lambda: torch.autograd.grad(g.aggregate(x, "max") if what == "aggregate" else g.gspmm("u_mul_e", x, e, "max"), operands, d)
    free = step()

    def never(*args, **kwargs):
        raise AssertionError("the kernel with atomics was called")
    monkeypatch.setattr(BroadcastOp, "select_backward", never)
    before = torch.are_deterministic_algorithms_enabled()
    torch.use_deterministic_algorithms(True)
    try:
        first, second = step(), step()
    finally:
        torch.use_deterministic_algorithms(before)
    assert all(torch.equal(a, b) for a, b in zip(first, second))
    # float64 by the selected elements: a row's messages, the first largest
    x64, e64 = x.detach().cpu().double().numpy(), e.detach().cpu().double().numpy()
    ref = [np.zeros_like(x64), np.zeros_like(e64)]
    for v in np.flatnonzero(np.diff(adj.indptr)):
        a, b = adj.indptr[v], adj.indptr[v + 1]
        u = adj.indices[a:b]
        m = x64[u] if what == "aggregate" else (x.detach().cpu().numpy()[u] * e.detach().cpu().numpy()[a:b])
        at, f, dv = m.argmax(0), np.arange(36), d[v].cpu().double().numpy()
        np.add.at(ref[0], (u[at], f), dv if what == "aggregate" else dv * e64[a + at, f])
        ref[1][a + at, f] += dv * x64[u[at], f]
    for got in (first, free):
        for i, r in enumerate(got):
            # sums of up to about 100 fp32 products
            assert np.linalg.norm(r.cpu().double().numpy() - ref[i]) <= 1e-6 * np.linalg.norm(ref[i])


@pytest.mark.parametrize("feat_len", [1, 3, 36, 257])
@pytest.mark.parametrize("degree", [1, 4, 5])
def test_gradients_of_rows_of_a_few_elements(feat_len, degree):
    """Both sides of the line from which results that meet are combined first, with operands that broadcast and that do not."""
    import torch
    from featgraph_amd.autograd import Graph
    n, rng = 700, np.random.default_rng(degree)
    adj = _graph(rng, [degree] * n)
    g = Graph(adj)
    t = lambda *s: torch.from_numpy(rng.standard_normal(s).astype(np.float32)).cuda().requires_grad_()
    x, d = t(n, 2, feat_len), t(n, 2, feat_len).detach()
    for e in (t(adj.nnz, 2, feat_len), t(adj.nnz, 2, 1)):
        for msg in ("u_mul_e", "u_sub_e"):
            got = torch.autograd.grad(g.gspmm(msg, x, e, "max"), [x, e], d)
            xs, es = x.detach().double().requires_grad_(), e.detach().double().requires_grad_()
            gathered = xs[torch.from_numpy(adj.indices).cuda().long()]
            m = gathered * es if msg == "u_mul_e" else gathered - es
            ref = torch.autograd.grad(m.view(n, degree, 2, feat_len).amax(1), [xs, es], d.double())
            for a, b in zip(got, ref):
                # sums of at most a few hundred fp32 products
                assert float((a.double() - b).norm()) <= 1e-5 * float(b.norm())


@pytest.mark.parametrize("special", ["ties", "nan", "minus_inf"])
@pytest.mark.parametrize("reduce", ["max", "min"])
@pytest.mark.parametrize("feat_len", [128, 192, 320])
def test_positions_in_feature_tiles(oracle, special, reduce, feat_len):
    """Feature lengths that the launch cuts into tiles of 64: exactly the oracle's values and positions, in every tile."""
    import torch
    from featgraph_amd.module import GSpMMhip, placeholder
    rng = np.random.default_rng(feat_len)
    adj = _graph(rng, LENS)
    x = rng.integers(-1, 2, size=(700, feat_len)).astype(np.float32)
    if special == "nan":
        x[rng.random(x.shape) < 0.01] = np.nan
    if special == "minus_inf":
        x[rng.random(x.shape) < 0.7] = -np.inf if reduce == "max" else np.inf
    e = rng.integers(0, 2, size=(adj.nnz, 1)).astype(np.float32)
    for msg, arrays, o in (("copy_u", [x], ("copy_lhs", x, None, "u", "e")), ("u_add_e", [x, e], ("add", x, e, "u", "e"))):
        ref, ref_arg = oracle.gspmm_bcast(adj.indptr, adj.indices, o[0], reduce, o[1], o[2], o[3], o[4])
        for P in (None, 3):
            m = GSpMMhip(adj)
            m.build([placeholder(a.shape) for a in arrays], {'msg': msg, 'reduce': reduce, 'return_arg': True, 'broadcast': True},
                    {'num_src_partitions': P})
            assert m._bop.feature_tiles(True) == (feat_len // 64 if msg == "copy_u" else 1)
            out = m.run([torch.from_numpy(a).cuda() for a in arrays]).cpu().numpy()
            assert np.array_equal(out, ref, equal_nan=True), (msg, P)
            assert np.array_equal(m.arg_tvm.cpu().numpy(), ref_arg), (msg, P)


@pytest.mark.parametrize("degree,feat_len,tiles", [(64, 128, 2), (64, 256, 4), (64, 192, 1), (20, 128, 1), (20, 256, 1)])
@pytest.mark.parametrize("reduce", ["max", "min"])
def test_positions_on_either_side_of_the_tiling_rule(oracle, degree, feat_len, tiles, reduce):
    """From 2^15 edges on the feature axis is cut for positions where the degree and the number of tiles make it pay; values and
    positions are the oracle's either way, over one and several partitions."""
    import torch
    from featgraph_amd.module import GSpMMhip, placeholder
    rng = np.random.default_rng(degree + feat_len)
    adj = _graph(rng, [degree] * ((1 << 15) // degree + 1))
    x = rng.integers(-1, 2, size=(700, feat_len)).astype(np.float32)
    ref, ref_arg = oracle.gspmm_bcast(adj.indptr, adj.indices, "copy_lhs", reduce, x, None, "u", "e")
    for P in (None, 3):
        m = GSpMMhip(adj)
        m.build([placeholder(x.shape)], {'msg': 'copy_u', 'reduce': reduce, 'return_arg': True}, {'num_src_partitions': P})
        assert m._bop.feature_tiles(True) == tiles
        out = m.run([torch.from_numpy(x).cuda()]).cpu().numpy()
        assert np.array_equal(out, ref) and np.array_equal(m.arg_tvm.cpu().numpy(), ref_arg), P
