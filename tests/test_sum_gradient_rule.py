"""Which weighted sums take both gradients from one sweep: the shapes on either side of the rule's lines, as they were measured."""
import pytest

from featgraph_amd import tuning


@pytest.mark.parametrize("heads,head_len,nnz,degree,one", [
    (1, 16, 400_000, 8, True), (1, 16, 4_000_000, 30, False), (1, 16, 13_000_000, 120, False), (1, 64, 13_000_000, 120, True),
    (1, 32, 4_000_000, 20, False), (1, 32, 12_500_000, 215, True), (1, 24, 4_000_000, 20, True), (1, 602, 4_000_000, 20, True),
    (2, 16, 100_000, 8, True), (2, 16, 400_000, 8, False), (2, 16, 12_500_000, 215, False),
    (4, 16, 13_000_000, 8, True), (4, 16, 12_500_000, 215, False), (12, 16, 12_500_000, 215, True),
    (4, 8, 1_000_000, 30, True), (4, 8, 4_000_000, 30, False), (8, 8, 4_000_000, 200, False), (2, 32, 4_000_000, 120, False),
    (16, 8, 4_000_000, 30, True), (16, 8, 4_000_000, 120, False),
    (3, 32, 13_000_000, 120, False), (6, 32, 13_000_000, 120, False), (6, 32, 4_000_000, 8, True),
    (4, 32, 12_500_000, 215, True), (8, 64, 12_500_000, 215, True), (8, 16, 12_500_000, 215, True),
    # shapes that the SDDMM has no tile for on these graphs
    (3, 16, 4_000_000, 120, True), (6, 32, 2_000_000, 120, True), (12, 8, 4_000_000, 120, True)])
def test_rule(heads, head_len, nnz, degree, one):
    nodes = int(nnz / degree)
    assert tuning.sum_gradients_in_one_sweep(nodes, nodes, nnz, heads, head_len) is one
