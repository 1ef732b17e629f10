"""Per-edge operators at the feature lengths and edge counts where the lane assignment of their kernel changes: rows of
one vector, rows that no power of two of lanes fits, scalar lanes, a last wavefront with one edge, broadcast operands."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nnz", [1, 63, 64, 65, 4097])
@pytest.mark.parametrize("feat_len", [1, 3, 4, 7, 12, 64, 100, 257, 260, 1028])
def test_messages_equal_the_gathered_operands(nnz, feat_len):
    import torch
    from featgraph_amd.module import GSDDMMhip, placeholder
    rng = np.random.default_rng(nnz * 1000 + feat_len)
    row = np.sort(rng.integers(0, 90, nnz))
    col = rng.integers(0, 70, nnz)
    coo = sp.coo_matrix((np.ones(nnz, "float32"), (row, col)), shape=(90, 70))
    gen = torch.Generator(device="cuda").manual_seed(feat_len)
    u = torch.randn(70, feat_len, generator=gen, device="cuda")
    v = torch.randn(90, feat_len, generator=gen, device="cuda")
    e = torch.randn(nnz, feat_len, generator=gen, device="cuda")
    one = torch.randn(90, 1, generator=gen, device="cuda")
    r, c = torch.from_numpy(row).cuda(), torch.from_numpy(col).cuda()
    for op, lt, rt, a, b, want in (("mul", "u", "v", u, v, u[c] * v[r]), ("sub", "v", "e", v, e, v[r] - e),
                                   ("add", "u", "v", u, one, u[c] + one[r]), ("copy_lhs", "u", None, u, None, u[c]),
                                   ("div", "e", "u", e, u, e / u[c])):
        m = GSDDMMhip(coo)
        args = {"op": op, "lhs_target": lt}
        if rt:
            args["rhs_target"] = rt
        ins = [t for t in (a, b) if t is not None]
        m.build([placeholder(tuple(t.shape)) for t in ins], args, {})
        m.out_tvm.fill_(float("nan"))
        got = m.run(ins)
        if op == "div":         # one correctly rounded division in each, or one within a unit in the last place
            assert torch.allclose(got, want, rtol=2.5e-7, atol=0)
        else:                   # one rounded operation each: the same bits
            assert torch.equal(got, want), (op, lt, rt)
