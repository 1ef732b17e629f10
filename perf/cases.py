"""The work a user of this package has it do, as cases that can be timed and compared.

Every family below is one way the package is used, through its public entry points:

  pair       weighted CSR SpMM, then SDDMM over the same edges: the operator pair of bench.py (module classes)
  heads      multi-head SDDMM, one score per edge and head (module class)
  shuffled   SDDMM over edges that are stored in no order, results in the stored order (module class)
  softmax    edge softmax and its gradient (module class)
  sum_step   weighted neighbour sum with gradients for the features and for the edge weights (autograd.Graph)
  pool_step  neighbour maximum / mean / sum with its gradient (autograd.Graph)
  dot_step   dot-product attention over the edges with its gradients (autograd.Graph)
  gat_step   additive-score attention over the edges with its gradients (autograd.Graph)
  msg_step   sum / mean / max of u-op-e messages with vector edge features, with gradients (ops)
  chain_step an attention layer put together from single operators, with gradients (ops): what a layer
             definition looks like before anybody has fused it, on the small graphs where launches count

Graphs are power-law (both ends of an edge drawn by Chung-Lu weights) or uniform, without duplicates and with
self-loops, with weights in [0, 1) and standard normal features; all of it comes from the seed.
"""
import functools
import math

import numpy as np
import scipy.sparse
import torch

from featgraph_amd import ops
from featgraph_amd.autograd import Graph
from featgraph_amd.module import (EdgeSoftmaxhip, MultiHeadSDDMMhip, VanillaSDDMMhip, VanillaSpMMhip, placeholder)


def listed():
    reddit_like = dict(nodes=232965, edges=114_766_039, exponent=2.1, max_degree=26500)
    ordinary = dict(nodes=58000, edges=12_500_000, exponent=2.1, max_degree=6600)
    return [
        # one call on a small graph: launches and host work (the 10,000-node benchmark graph)
        dict(name="pair_10k_f32", family="pair", nodes=10000, edges=169_867, exponent=0.0, max_degree=0, feat=32),
        # the headline benchmark: dense power-law graph, long features
        dict(name="pair_233k_f512", family="pair", feat=512, **reddit_like),
        # many nodes of low degree: the 2.45M-node benchmark graph
        dict(name="pair_2450k_f128", family="pair", nodes=2_450_000, edges=61_903_880, exponent=2.5, max_degree=17600, feat=128),
        # attention scores of 8 heads on the headline graph
        dict(name="heads_233k_8x32", family="heads", heads=8, head_len=32, **reddit_like),
        # an edge list as it comes out of a file or a sampler
        dict(name="shuffled_58k_f128", family="shuffled", feat=128, **ordinary),
        # the normalisation between the two halves of an attention layer, forward and backward
        dict(name="softmax_233k_h4", family="softmax", heads=4, **reddit_like),
        # first layer of a node classifier with learned edge weights: raw features of the length real data has
        dict(name="sum_step_58k_f602", family="sum_step", feat=602, **ordinary),
        # neighbourhood max-pooling, a feature length that suits no tile
        dict(name="pool_step_58k_f100", family="pool_step", reduce="max", feat=100, **ordinary),
        # transformer-style attention layer, forward and backward
        dict(name="dot_step_58k_8x64", family="dot_step", heads=8, head_len=64, **ordinary),
        # additive attention layer, forward and backward
        dict(name="gat_step_58k_4x32", family="gat_step", heads=4, head_len=32, **ordinary),
        # edge-conditioned convolution: one feature vector per edge
        dict(name="msg_step_58k_f64", family="msg_step", op="mul", reduce="sum", feat=64, edge_feat=64, **ordinary),
        # a training step on a citation-sized graph: many short launches
        dict(name="chain_step_3k_8x8", family="chain_step", heads=8, head_len=8, nodes=2700, edges=10500, exponent=2.6, max_degree=170),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_graph(rng, nodes_lo, nodes_hi, edges_hi, degree_lo=4, degree_hi=500):
    nodes = _log_int(rng, nodes_lo, nodes_hi)
    degree = math.exp(rng.uniform(math.log(degree_lo), math.log(min(degree_hi, nodes / 8, edges_hi / nodes))))
    edges = int(nodes * degree)
    if rng.random() < 0.2:
        return dict(nodes=nodes, edges=edges, exponent=0.0, max_degree=0)
    return dict(nodes=nodes, edges=edges, exponent=round(rng.uniform(2.05, 2.7), 2),
                max_degree=int(min(nodes / 8, degree * rng.uniform(15, 60))) + 1)


def draw(rng):
    family = rng.choice(["pair", "pair", "heads", "shuffled", "softmax", "sum_step", "pool_step", "dot_step", "gat_step",
                         "msg_step", "chain_step"])
    # feature lengths: half of them the usual powers of two, half anything
    feat = rng.choice([16, 32, 64, 128, 256, 512]) if rng.random() < 0.5 else _log_int(rng, 8, 602)
    if family == "pair":
        return dict(family=family, feat=feat, **_draw_graph(rng, 2000, 400_000, 30_000_000))
    if family == "heads":
        return dict(family=family, heads=rng.choice([2, 3, 4, 8, 16]), head_len=rng.choice([8, 16, 20, 32, 48, 64]),
                    **_draw_graph(rng, 2000, 200_000, 12_000_000))
    if family == "shuffled":
        return dict(family=family, feat=feat, **_draw_graph(rng, 2000, 200_000, 20_000_000))
    if family == "softmax":
        return dict(family=family, heads=rng.choice([1, 2, 3, 4, 6, 8, 16]), **_draw_graph(rng, 2000, 400_000, 40_000_000))
    if family == "sum_step":
        return dict(family=family, feat=feat, **_draw_graph(rng, 2000, 200_000, 12_000_000))
    if family == "pool_step":
        return dict(family=family, reduce=rng.choice(["max", "max", "min", "mean", "sum"]), feat=min(feat, 256),
                    **_draw_graph(rng, 2000, 200_000, 12_000_000))
    if family == "dot_step":
        return dict(family=family, heads=rng.choice([1, 2, 4, 8]), head_len=rng.choice([16, 32, 64]),
                    **_draw_graph(rng, 2000, 200_000, 12_000_000))
    if family == "gat_step":
        return dict(family=family, heads=rng.choice([1, 2, 4, 8]), head_len=rng.choice([16, 32, 64]),
                    **_draw_graph(rng, 2000, 200_000, 12_000_000))
    if family == "msg_step":
        feat = min(feat, 128)
        op, reduce = rng.choice([("mul", "sum"), ("mul", "sum"), ("mul", "mean"), ("add", "sum"), ("add", "max"), ("sub", "max"), ("mul", "max")])
        return dict(family=family, op=op, reduce=reduce, feat=feat, edge_feat=rng.choice([1, feat, feat]),
                    **_draw_graph(rng, 2000, 100_000, 8_000_000))
    return dict(family=family, heads=rng.choice([1, 2, 4, 8]), head_len=rng.choice([8, 16, 32, 64]),
                **_draw_graph(rng, 500, 20_000, 400_000, degree_hi=40))


# ---- graphs ---------------------------------------------------------------------------------------------

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) & 0x7FFFFFFF)


def _powerlaw_weights(nodes, total, exponent, max_degree):
    """max_degree * ((i + i0) / i0) ** (-1 / (exponent - 1)) with i0 such that the weights add up to `total`."""
    i = torch.arange(nodes, dtype=torch.float64, device="cuda")

    def weights(i0):
        return max_degree * ((i + i0) / i0) ** (-1.0 / (exponent - 1.0))

    lo, hi = 1e-3, nodes * 1e3
    for _ in range(60):
        mid = math.sqrt(lo * hi)
        if float(weights(mid).sum()) < total:
            lo = mid
        else:
            hi = mid
    return weights(hi)


def _adjacency(case, gen):
    """Seeded square adjacency with exactly case["edges"] stored elements, rows = destinations, no duplicates, a self-loop
    per node, column ids sorted inside a row, weights in [0, 1).  Degrees follow the same weights in both directions."""
    n, edges = case["nodes"], case["edges"]
    if case["exponent"] > 0:
        cdf = torch.cumsum(_powerlaw_weights(n, edges, case["exponent"], case["max_degree"]), 0)
        id_of_rank = torch.randperm(n, generator=gen, device="cuda")

        def pick(k):
            at = torch.rand(k, generator=gen, dtype=torch.float64, device="cuda") * cdf[-1]
            return id_of_rank[torch.searchsorted(cdf, at).clamp_(max=n - 1)]
    else:
        def pick(k):
            return torch.randint(n, (k,), generator=gen, device="cuda")
    key = torch.empty(0, dtype=torch.int64, device="cuda")    # row * n + column
    while key.numel() < edges - n:
        k = int(1.06 * (edges - n - key.numel())) + 64
        rows, cols = pick(k), pick(k)
        key = torch.unique(torch.cat([key, (rows * n + cols)[rows != cols]]))
    spare = key.numel() - (edges - n)
    keep = torch.ones(key.numel(), dtype=torch.bool, device="cuda")
    keep[torch.randperm(key.numel(), generator=gen, device="cuda")[:spare]] = False
    key = torch.sort(torch.cat([key[keep], torch.arange(n, device="cuda") * (n + 1)]))[0]
    indptr = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    torch.cumsum(torch.bincount(key // n, minlength=n), 0, out=indptr[1:])
    vals = torch.rand(edges, generator=gen, device="cuda")
    adj = scipy.sparse.csr_matrix((vals.cpu().numpy(), (key % n).int().cpu().numpy(), indptr.int().cpu().numpy()), shape=(n, n))
    adj.has_sorted_indices = True
    return adj


# ---- states and passes ----------------------------------------------------------------------------------

def prepare(case, seed):
    gen = _generator(seed)
    adj = _adjacency(case, gen)
    n, nnz = case["nodes"], adj.nnz
    normal = functools.partial(torch.randn, generator=gen, device="cuda")
    family = case["family"]
    st = {"case": case}
    if family == "pair":
        F = case["feat"]
        st["x"], st["y"] = normal(n, F), normal(n, F)
        st["spmm"] = VanillaSpMMhip(adj)
        st["spmm"].build([placeholder((n, F))], {}, {})
        st["sddmm"] = VanillaSDDMMhip(adj)
        st["sddmm"].share_layouts(st["spmm"])
        st["sddmm"].build([placeholder((n, F)), placeholder((n, F))], {}, {})
        return st
    if family == "heads":
        shape = (n, case["heads"], case["head_len"])
        st["x"], st["y"] = normal(*shape), normal(*shape)
        st["sddmm"] = MultiHeadSDDMMhip(adj)
        st["sddmm"].build([placeholder(shape), placeholder(shape)], {}, {})
        return st
    if family == "shuffled":
        F = case["feat"]
        coo = adj.tocoo()
        order = torch.randperm(nnz, generator=gen, device="cuda").cpu().numpy()
        coo = scipy.sparse.coo_matrix((coo.data[order], (coo.row[order], coo.col[order])), shape=coo.shape)
        st["x"], st["y"] = normal(n, F), normal(n, F)
        st["sddmm"] = VanillaSDDMMhip(coo)
        st["sddmm"].build([placeholder((n, F)), placeholder((n, F))], {}, {})
        return st
    if family == "softmax":
        st["x"], st["dy"] = normal(nnz, case["heads"]), normal(nnz, case["heads"])
        st["softmax"] = EdgeSoftmaxhip(adj)
        st["softmax"].build([placeholder((nnz, case["heads"]))])
        return st
    # training steps: leaves that collect gradients, and the gradient that arrives from the layer above
    st["graph"] = Graph(adj)
    if family == "sum_step":
        leaves = [normal(n, case["feat"]), torch.from_numpy(adj.data).cuda()]
        st["dout"] = normal(n, case["feat"])
    elif family == "pool_step":
        leaves = [normal(n, case["feat"])]
        st["dout"] = normal(n, case["feat"])
    elif family == "dot_step":
        shape = (n, case["heads"], case["head_len"])
        leaves = [normal(*shape), normal(*shape), normal(*shape)]
        st["dout"] = normal(*shape)
    elif family in ("gat_step", "chain_step"):
        H, D = case["heads"], case["head_len"]
        leaves = [normal(n, H), normal(n, H), normal(n, H, D)]
        st["dout"] = normal(n, H, D)
    elif family == "msg_step":
        leaves = [normal(n, case["feat"]), normal(nnz, case["edge_feat"])]
        st["dout"] = normal(n, case["feat"])
    else:
        raise ValueError("unknown family %r" % (family,))
    st["leaves"] = [t.requires_grad_() for t in leaves]
    run(st)                     # a Graph lays out what its operators need at their first use
    return st


def run(state):
    case = state["case"]
    family = case["family"]
    if family == "pair":
        return state["spmm"].run([state["x"]]), state["sddmm"].run([state["x"], state["y"]])
    if family in ("heads", "shuffled"):
        return state["sddmm"].run([state["x"], state["y"]])
    if family == "softmax":
        a = state["softmax"].run([state["x"]])
        return a, state["softmax"].backward(a, state["dy"])
    g, leaves = state["graph"], state["leaves"]
    if family == "sum_step":
        out = g.spmm(*leaves)
    elif family == "pool_step":
        out = g.aggregate(leaves[0], case["reduce"])
    elif family == "dot_step":
        out = g.attention(*leaves)
    elif family == "gat_step":
        out = g.gat_attention(*leaves)
    elif family == "msg_step":
        out = ops.gspmm(g, case["op"], case["reduce"], *leaves)
    else:
        er, el, v = leaves
        scores = torch.nn.functional.leaky_relu(ops.gsddmm(g, "add", el, er), 0.2)
        out = ops.gspmm(g, "mul", "sum", v, ops.edge_softmax(g, scores).unsqueeze(-1))
    return (out.detach(),) + torch.autograd.grad(out, leaves, state["dout"])


# ---- what a pass cannot do without ----------------------------------------------------------------------

def work(case):
    """Each input read once (structure included: 4 bytes per row and per edge), each output written once; flops of
    the products and sums that the result is made of."""
    n, e = case["nodes"], case["edges"]
    family = case["family"]
    graph = 4 * (n + 1) + 4 * e
    if family == "pair":
        F = case["feat"]
        return {"bytes": 2 * graph + 4 * e + 8 * n * F + 8 * n * F + 4 * e, "flops": 4 * e * F}
    if family == "heads":
        H, F = case["heads"], case["heads"] * case["head_len"]
        return {"bytes": graph + 8 * n * F + 4 * e * H, "flops": 2 * e * F}
    if family == "shuffled":
        F = case["feat"]
        return {"bytes": 8 * e + 8 * n * F + 4 * e, "flops": 2 * e * F}
    if family == "softmax":
        # scores in, softmax out; softmax and its gradient in, gradient of the scores out
        return {"bytes": 8 * (n + 1) + 20 * e * case["heads"], "flops": 9 * e * case["heads"]}
    if family == "sum_step":
        F = case["feat"]
        # forward: x, w -> out; backward: dout, w, x -> dx, dw
        return {"bytes": 3 * graph + 12 * e + 5 * 4 * n * F, "flops": 6 * e * F}
    if family == "pool_step":
        F = case["feat"]
        return {"bytes": graph + 4 * 4 * n * F, "flops": 2 * e * F if case["reduce"] in ("sum", "mean") else e * F + n * F}
    if family == "dot_step":
        F = case["heads"] * case["head_len"]
        # forward: q . k and a * v per edge; backward: q . k and dout . v again, then three sums
        return {"bytes": 2 * graph + 4 * n * F * (4 + 5 + 3), "flops": (4 + 10) * e * F}
    if family in ("gat_step", "chain_step"):
        H, F = case["heads"], case["heads"] * case["head_len"]
        return {"bytes": 2 * graph + 4 * n * F * (2 + 4) + 4 * n * H * 6, "flops": 6 * e * F + 20 * e * H}
    F, Fe = case["feat"], case["edge_feat"]
    return {"bytes": 2 * graph + 4 * n * F * (2 + 3) + 4 * e * Fe * 3, "flops": 6 * e * F}


def tolerance(case):
    """fp32 sums in another order (measured against the same operators in float64); attention and softmax values also
    pass through the hardware's exponential."""
    return {"rel": {"pair": 1e-6, "heads": 1e-6, "shuffled": 1e-6, "softmax": 1e-6, "sum_step": 1e-6, "pool_step": 1e-6,
                    "dot_step": 1.5e-6, "gat_step": 3e-6, "msg_step": 1e-6, "chain_step": 3e-6}[case["family"]]}
