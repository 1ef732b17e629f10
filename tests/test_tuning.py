"""Rules of the default tilings that hold for every graph."""
from featgraph_amd import tuning


def test_scattered_edges_take_the_tiled_walk_sooner():
    """Edges in no order of their rows: the edge-list kernel gathers both operands, so whatever row-ordered edges are tiled for, scattered ones
    of more than a few per row are tiled for as well; every choice is one that the kernel takes."""
    for n in (5000, 30000, 140000):
        for deg in (16, 40, 160):
            for F, given in ((64, None), (128, None), (256, 222), (512, None)):
                if n * deg > 2e7:
                    continue
                args = (n, n, n * deg, 1, F, None, given)
                ordered, scattered = tuning.choose_sddmm(*args), tuning.choose_sddmm(*args, scattered=True)
                assert scattered is not None or ordered is None or n == 5000
                if scattered is not None:
                    tile = F // scattered[1]
                    assert F % scattered[1] == 0 and 16 <= tile <= 256 and tile & (tile - 1) == 0
    assert tuning.choose_sddmm(140000, 140000, 5_600_000, 1, 256, None, 222, scattered=True) is not None
    assert tuning.choose_sddmm(30000, 30000, 240_000, 1, 32, None, None, scattered=True) is None


def test_heads_on_small_graphs_get_tiles_that_the_kernel_takes():
    for n, deg in ((6000, 6), (6000, 90), (40000, 25), (150000, 90)):
        for heads in (2, 3, 4, 6, 8, 12, 16):
            for head_len in (8, 16, 32, 64):
                got = tuning.choose_sddmm(n, n, n * deg, heads, head_len)
                if got is not None:
                    tile = heads * head_len // got[1]
                    assert heads * head_len % got[1] == 0 and 16 <= tile <= 256 and tile & (tile - 1) == 0
                    assert tile % head_len == 0 or head_len % tile == 0 and heads == 1
    assert tuning.choose_sddmm(150000, 150000, 900_000, 8, 64) is None          # degree 6: the edge list
    assert tuning.choose_sddmm(40000, 40000, 3_600_000, 4, 32) is not None


def test_scattered_edges_of_several_heads_take_the_tiled_walk_sooner():
    for n in (5000, 30000, 140000, 1_000_000):
        for deg in (6, 16, 40, 160):
            if n * deg > 6.5e7:
                continue
            for heads, head_len, given in ((2, 16, None), (8, 8, None), (4, 32, None), (8, 32, None), (2, 64, None), (8, 64, None), (8, 64, 48), (2, 32, 20)):
                args = (n, n, n * deg, heads, head_len, None, given)
                ordered, scattered = tuning.choose_sddmm(*args), tuning.choose_sddmm(*args, scattered=True)
                assert scattered is not None or ordered is None, args
                if scattered is not None:
                    tile = heads * head_len // scattered[1]
                    assert heads * head_len % scattered[1] == 0 and 16 <= tile <= 256 and tile & (tile - 1) == 0 and tile % head_len == 0
    # where the edge list, which gathers both operands, takes 1.2 to 2.1 times as long
    for n, deg, heads, head_len in ((140000, 40, 8, 16), (140000, 40, 2, 64), (60000, 20, 4, 16), (60000, 20, 8, 8), (36608, 11, 4, 32), (150000, 6, 8, 32),
                                    (200000, 16, 8, 64), (1_000_000, 60, 8, 32)):
        assert tuning.choose_sddmm(n, n, n * deg, heads, head_len, scattered=True) is not None
    assert tuning.choose_sddmm(40000, 40000, 1_000_000, 8, 64, given_len=48, scattered=True) is not None
    assert tuning.choose_sddmm(6000, 6000, 120_000, 2, 16, scattered=True) is None              # everything in the caches


def test_a_tiled_traversal_that_is_asked_for_gets_tiles_that_the_kernel_takes():
    for n, nnz in ((1000, 5000), (60000, 480000), (140000, 2240000), (2_000_000, 40_000_000)):
        for heads, head_len in ((8, 64), (16, 32), (1, 320), (8, 48 + 16), (12, 16), (1, 512), (1, 2048), (1, 64), (2, 8), (3, 8 * 4)):
            p, t = tuning.complete_tiled_sddmm(n, n, nnz, heads, head_len)
            tile = heads * head_len // t
            assert p >= 1 and heads * head_len % t == 0 and 16 <= tile <= 256 and tile & (tile - 1) == 0 and (heads == 1 or tile % head_len == 0)
    assert tuning.complete_tiled_sddmm(1000, 1000, 5000, 3, 20) == (1, 1)            # nothing fits: the kernel refuses, as ever


def test_choices_on_small_graphs_that_were_measured():
    """Where the fitted model is known to be wrong by more than the measurements' noise, on both sides of the rules that say so (uniform degrees)."""
    def sddmm(n, deg, feat_len, **kw):
        return tuning.choose_sddmm(n, n, n * deg, 1, feat_len, **kw)
    # partitions with one tile: results in pieces of a few elements (40,000 nodes of degree 20 and the like: 1.3 to 1.5 times the edge list's time)
    for n, deg, feat_len in ((25000, 20, 128), (15000, 12, 256), (40000, 12, 64), (200000, 32, 128)):
        got = sddmm(n, deg, feat_len)
        assert got is None or got[1] > 1 or got[0] == 1, (n, deg, feat_len)
    assert sddmm(150000, 62, 32) == (4, 1) and sddmm(140000, 62, 16)[1] == 1
    # from 200,000 sources on the second set of coefficients has to see more of a gain
    for n, deg, feat_len in ((250000, 50, 128), (400000, 62, 128), (250000, 40, 256)):
        assert tuning.choose_spmm(n, n, n * deg, feat_len) == (4, feat_len // 32), (n, deg, feat_len)
    assert tuning.choose_spmm(320000, 320000, 320000 * 32, 64)[0] == 1
