"""Schedules of the SDDMM modules that name a part of the tiled traversal's shape: the rest is completed to a shape that the kernel takes."""
import numpy as np
import pytest
import scipy.sparse as sp

from helpers import assert_sum_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,deg,shape", [(60000, 8, (8, 64)), (60000, 8, (16, 32)), (140000, 16, (320,)), (40000, 9, (8, 48)), (3000, 5, (4, 16)), (3000, 5, (512,)),
                                         (3000, 5, (64,))])
@pytest.mark.parametrize("schedule", [{"order": "tiled"}, {"num_src_partitions": 2}, {"order": "tiled", "num_src_partitions": 3}])
def test_partial_schedules_are_completed(n, deg, shape, schedule):
    import torch
    from featgraph_amd.module import MultiHeadSDDMMhip, VanillaSDDMMhip, placeholder
    rng = np.random.default_rng(n + len(shape))
    row = np.repeat(np.arange(n), deg)
    col = np.sort(rng.integers(0, n, (n, deg)), axis=1).ravel()
    keep = np.r_[True, (row[1:] != row[:-1]) | (col[1:] != col[:-1])]
    adj = sp.csr_matrix((np.ones(int(keep.sum()), np.float32), (row[keep], col[keep])), shape=(n, n))
    adj.sort_indices()
    row, col = np.repeat(np.arange(n), np.diff(adj.indptr)), adj.indices
    x, y = (rng.standard_normal((n,) + shape, dtype=np.float32) for _ in range(2))
    m = (MultiHeadSDDMMhip if len(shape) == 2 else VanillaSDDMMhip)(adj)
    m.build([placeholder(x.shape)] * 2, {}, dict(schedule))
    assert m._tiled is not None and m._tiled[0]["P"] == schedule.get("num_src_partitions", m._tiled[0]["P"])
    m.out_tvm.fill_(float("nan"))
    got = m.run([torch.from_numpy(x).cuda(), torch.from_numpy(y).cuda()]).cpu().numpy()
    at = rng.choice(len(col), 2000)                 # (all of them in float64 would take minutes)
    assert np.isfinite(got).all()
    prod = (x[col[at]].astype("f8") * y[row[at]]).reshape((2000,) + (shape if len(shape) == 2 else (1,) + shape))
    want, mass = prod.sum(-1), np.abs(prod).sum(-1)
    assert_sum_close(got[at].reshape(want.shape), want, mass, str((n, shape, schedule)))


@pytest.mark.parametrize("shapes", [((100,), (512,)), ((8, 48), (8, 64)), ((512,), (100,))])
def test_descriptions_do_not_depend_on_what_was_built_before(shapes):
    """lower_to_ir() describes what build() would take for its own arguments, padded rows included, whatever the module was built for."""
    from featgraph_amd.module import MultiHeadSDDMMhip, VanillaSDDMMhip, placeholder
    rng = np.random.default_rng(1)
    n, deg = 60000, 40
    col = rng.integers(0, n, (n, deg)).ravel()
    adj = sp.coo_matrix((np.ones(n * deg, np.float32), (np.repeat(np.arange(n), deg), col)), shape=(n, n)).tocsr()
    adj.sort_indices()
    make = MultiHeadSDDMMhip if len(shapes[0]) == 2 else VanillaSDDMMhip
    phs = [[placeholder((n,) + s)] * 2 for s in shapes]
    m = make(adj)
    m.build(phs[0], {}, {})
    assert m.lower_to_ir(phs[1], {}, {}) == make(adj).lower_to_ir(phs[1], {}, {})
    text = m.lower_to_ir(phs[0], {}, {})
    assert ("sddmm_tiled_kernel" in text) == (m._tiled is not None) and ("zero-padded" in text) == (m._src_pad is not None)
    if m._tiled is not None:
        assert "%d source-column partition(s) x %d feature tile(s)" % (m._tiled[0]["P"], m._tiled[1]) in text


def test_several_heads_on_a_rectangular_adjacency_are_chosen_for_its_own_column_counts():
    """Far fewer sources than destinations: every column is referenced far more often than a row is long."""
    from featgraph_amd import tuning
    from featgraph_amd.module import MultiHeadSDDMMhip, placeholder
    rng = np.random.default_rng(2)
    rows, cols, deg = 300000, 20000, 20
    col = np.sort(rng.integers(0, cols, (rows, deg)), axis=1)
    adj = sp.csr_matrix((np.ones(rows * deg, np.float32), col.ravel(), np.arange(0, rows * deg + 1, deg)), shape=(rows, cols))
    adj.sum_duplicates()
    m = MultiHeadSDDMMhip(adj)
    m.build([placeholder((cols, 8, 32)), placeholder((rows, 8, 32))], {}, {})
    want = tuning.choose_sddmm(rows, cols, adj.nnz, 8, 32, tuning.GraphStats.from_csr(adj.indptr, adj.indices, cols))
    assert want is not None and m._tiled is not None and (m._tiled[0]["P"], m._tiled[1]) == want
