"""Default tiling / partitioning choices for gfx950 (MI355X), from a cost model in hardware terms.

What the two knobs do on this part.  The 8 XCDs have 4 MB of L2 each and are dealt workgroups
round-robin, so a feature-tile index that varies fastest with the workgroup id gives every XCD one
slice of the feature axis: T tiles of `tile` floats make a gathered row slice `4 * tile` bytes.
P source-column partitions (the reference's DDS format) bound the source rows one pass touches.
Together they set how many slices an XCD's gathers range over, n_src / P, against how many its L2
holds, L2 / (4 * tile).  The price: every tile re-reads the edge list (T edge visits per edge), every
partition cuts each row into a segment with its own start-up, read of the destination row / earlier
sums and write, and with 4 or more tiles the gathered matrix is first copied tile by tile.

The model adds those terms up for every (P, T) and takes the cheapest:

    gathered bytes  nnz * F * 4, a share h at the L1/L2-hit rate and 1 - h at the miss rate;
        h = hit rate of an LRU cache of (L2 / slice bytes) entries under the graph's own column
        reference counts (Che's approximation), over the columns of one partition;
        misses slow down with the span of memory an XCD's gathers range over;
    row segments    (non-empty (row, partition) pairs, from the degree histogram) * T * seconds each;
    edge visits     nnz * T * seconds each  (index / weight words, staging);
    streamed bytes  the output re-read and re-written per pass (SpMM); destination rows per segment
        and the per-tile partial sums (SDDMM); the tile-by-tile copy of the gathered matrix.

The coefficients are rates of this part -- bytes per second through the L1/L2-hit path, the miss path
and the streaming path, seconds per segment and per edge visit -- fitted to sweeps of P x T on five
graphs (232,965-node and 2.45M-node power-law graphs, a 1M-node uniform graph of degree 64, a 1M-node
power-law graph of degree 100, a 100k x 1M non-square graph; feature lengths 32..512).  On those
sweeps the model's choice is within 7.5 % of the best point (SpMM at F = 512 on the uniform graph:
15 %), 1-2.5 % on average; `autotune` (see the module classes' schedule argument 'tune') times the
model's best few candidates on the graph itself and keeps the fastest.
"""
import math

import numpy as np

N_XCD = 8
L2_BYTES = 4 << 20               # per XCD
COPY_BYTES_PER_S = 6.5e12        # tile_major_kernel: 477 MB read and written in 0.147 ms
MAX_PARTITIONS = 32
MIN_TILE_FLOATS = 32             # 16-float tiles cost 1.6-2x everywhere they were measured
TIE = 0.03                       # predicted times closer than this are equal: fewer tiles / partitions win

# cache: effective L2 capacity as a multiple of L2_BYTES under the independent-reference estimate (the
# gather stream has more locality than independent references, so the 4 MB behave like ~2x);
# hit / miss / stream: bytes per second; span: slow-down of misses per doubling of the gathered span beyond
# 128 MB; seg / edge: seconds per row segment and per edge visit.
SPMM_COEF = dict(cache=2.12, hit=24.0e12, miss=7.07e12, span=0.011, seg=1.64e-11, edge=1.04e-12, stream=4.15e12)
SDDMM_COEF = dict(cache=2.26, hit=23.5e12, miss=6.58e12, span=0.0, seg=3.82e-11, edge=0.0, stream=3.86e12)

# Below this many stored elements the launches, the sums that follow them and the caches' real size weigh more.  A second set of
# coefficients, fitted to sweeps of P (1 .. 16) x T on 23 graphs, overrules the first where it sees 15 % (SpMM) or 5 % (SDDMM) less time for its own
# choice; from more than 200,000 sources on 30 % and 10 %, where the first set is the nearer one.  Held against 276 other graphs (4,000 to 400,000
# nodes, degrees 6 to 260, uniform and power-law, feature lengths 16 .. 512, P 1 .. 8 with every T): the choice's time against the first set's, mean / worst,
# SpMM 0.972 / 1.17 (beyond 200,000 sources 0.999 / 1.00), SDDMM 0.935 / 1.17 (0.996 / 1.07); against the best of the sweep SpMM 1.031 (first set 1.061), SDDMM
# 1.038 (1.110).  With 15 % and 5 % everywhere the worst beyond 200,000 sources are 1.23 (250,000 of degree 50, uniform, F=128, SpMM 719 -> 886 us) and
# 1.21 (280,000 of 32, power-law, F=256, SDDMM 1053 -> 1278); without the second set there, uniform, SpMM 320,000 of 32, F=64 365 -> 408, SDDMM 250,000 of 20, F=32 99 -> 125.
# The largest, us: 17,600 nodes of degree 266, uniform, F=512: SpMM 723 -> 360, SDDMM 1128 -> 400; 12,000 of degree 200, F=512: 232 -> 190, 473 -> 195.
SMALL_NNZ = 1 << 25
MANY_SOURCES = 200_000
# pass / sum: seconds that a second pass over the graph (SpMM) and the sum of the tiles' scores (SDDMM) cost whatever their size;
# seg_tiled: per row segment and tile where there are several; edges_dst: the edge-list kernel's reads of destination rows, as
# a share of the gathered bytes at the hit rate.
SPMM_SMALL_COEF = dict(cache=0.99, hit=29.95e12, miss=6.55e12, span=0.041, seg=2.86e-11, seg_tiled=6.2e-11, edge=1.37e-12, stream=3.93e12,
                       **{'pass': 7.0e-6})
SDDMM_SMALL_COEF = dict(cache=1.32, hit=24.7e12, miss=8.49e12, span=0.006, seg=2.85e-11, edge=0.21e-12, stream=3.85e12, sum=9.7e-6,
                        edges_dst=0.26)


def _is_small(stats):
    return stats.nnz < SMALL_NNZ


# legacy names (attention module): per-XCD slice that two L2s' worth of slices add up to
SPMM_SLICE_BYTES = 7.5e6
SDDMM_SLICE_BYTES = 7.5e6
TILE_FLOATS = 64


class GraphStats(object):
    """What the model needs to know about an adjacency: sizes, how often each source column is
    referenced (as a histogram: `count_vals[i]` references occur for `count_mult[i]` columns) and the
    row degrees (same form)."""

    def __init__(self, n_dst, n_src, nnz, count_vals=None, count_mult=None, deg_vals=None, deg_mult=None):
        self.n_dst, self.n_src, self.nnz = int(n_dst), int(n_src), int(nnz)
        if count_vals is None:          # nothing known: every column referenced equally often
            count_vals, count_mult = [self.nnz / max(1, self.n_src)], [self.n_src]
        if deg_vals is None:
            deg_vals, deg_mult = [self.nnz / max(1, self.n_dst)], [self.n_dst]
        self.count_vals = np.asarray(count_vals, dtype=np.float64)
        self.count_mult = np.asarray(count_mult, dtype=np.float64)
        self.deg_vals = np.asarray(deg_vals, dtype=np.float64)
        self.deg_mult = np.asarray(deg_mult, dtype=np.float64)
        keep = self.count_vals > 0
        self.count_vals, self.count_mult = self.count_vals[keep], self.count_mult[keep]
        self._hits = {}

    @classmethod
    def from_csr(cls, indptr, indices, n_src):
        indptr = np.asarray(indptr)
        nnz = int(indptr[-1]) if len(indptr) else 0
        counts = np.bincount(np.asarray(indices), minlength=int(n_src)) if nnz else np.zeros(int(n_src), np.int64)
        cv, cm = np.unique(counts, return_counts=True)
        dv, dm = np.unique(np.diff(indptr), return_counts=True)
        return cls(len(indptr) - 1, n_src, nnz, cv, cm, dv, dm)

    def segments(self, P):
        """Expected number of non-empty (row, partition) pairs: a row of degree d spreads its elements
        over P equally likely partitions."""
        if P == 1:
            return float((self.deg_mult * (self.deg_vals > 0)).sum())
        return float((self.deg_mult * P * (1.0 - (1.0 - 1.0 / P) ** self.deg_vals)).sum())

    def hit_rate(self, entries):
        """Hit rate of an LRU cache of `entries` column slices under independent references with
        these columns' rates (Che's approximation: a slice stays for a characteristic time t with
        sum_c (1 - exp(-rate_c t)) = entries)."""
        total = float((self.count_vals * self.count_mult).sum())
        if total <= 0:
            return 0.0
        key = round(math.log2(max(entries, 1e-9)), 3)
        if key in self._hits:
            return self._hits[key]
        v, m = self.count_vals, self.count_mult
        if entries >= m.sum():
            h = 1.0 - m.sum() / total                     # only first references miss
        else:
            occupied = lambda t: float((m * -np.expm1(-v * t)).sum())
            lo, hi = 0.0, 1.0 / max(v.max(), 1e-30)
            while occupied(hi) < entries:
                hi *= 2.0
            for _ in range(50):
                mid = 0.5 * (lo + hi)
                if occupied(mid) < entries:
                    lo = mid
                else:
                    hi = mid
            h = float((v * m * -np.expm1(-v * hi)).sum() / total)
        self._hits[key] = h
        return h


def _pow2_floor(v):
    p = 1
    while p * 2 <= v:
        p *= 2
    return p


def feature_tiles(feat_len):
    """Number of feature tiles: tiles of TILE_FLOATS floats when that divides feat_len."""
    if feat_len % TILE_FLOATS == 0:
        return feat_len // TILE_FLOATS
    return 1


def padded_feature_len(feat_len):
    """The feature length the kernels should run at for rows of `feat_len` floats: the same, when it is a multiple of
    32 (tiles of 32 or 64 floats cover it) or too short to matter; else the next length that is -- a power of two up to
    64, a multiple of 32 up to 128, a multiple of 64 beyond.  Rows of any other length leave the kernels one tile and
    scalar accesses (232,965-node graph, SpMM / SDDMM in ms: F=30 1.69 / 2.69 against 0.97 / 1.11 at 32; F=100 4.18 / 6.69
    against 3.17 / 3.58 at 128; F=300 19.8 / 19.1 against 7.67 / 8.41 at 320; F=602 40.8 / 75.9 against 14.7 / 16.6 at 640);
    zero columns change neither the sums nor the dot products."""
    F = int(feat_len)
    if F < 9 or F % 32 == 0:
        return F
    if F <= 64:
        p = 16
        while p < F:
            p *= 2
        return p
    if F <= 128:
        return (F + 31) // 32 * 32
    return (F + 63) // 64 * 64


def padded_head_len(head_len):
    """The head length the multi-head kernels should run at: a power of two up to 64 or a multiple of 64 (a head then
    fills whole lane groups and tiles); other lengths are zero-padded to the next such length (232,965-node graph,
    multi-head SDDMM: 3 heads of 20 floats 26.5 ms, 8 heads of 48 floats 69 ms on the kernel that takes any shape)."""
    D = int(head_len)
    if D % 64 == 0 or (D & (D - 1)) == 0:
        return D
    if D < 64:
        p = 4
        while p < D:
            p *= 2
        return p
    return (D + 63) // 64 * 64


# Padding costs two or three passes over the feature matrices; below this many gathered floats it is not attempted.
PAD_MIN_GATHERED = 1 << 24


def copies_tile_major(n_src, feat_len, n_tiles):
    """The library's rule for gathering from a tile-by-tile copy (fg_plan_opts.tile_major = 0)."""
    xbytes = 4 * n_src * feat_len
    return n_tiles >= 4 and (64 << 20) <= xbytes < (1 << 32)


def _gather_seconds(stats, feat_len, P, T, c):
    tile_bytes = 4.0 * feat_len / T
    h = stats.hit_rate(c['cache'] * L2_BYTES / tile_bytes * P)       # entries counted over all partitions' columns
    tiled = copies_tile_major(stats.n_src, feat_len, T)
    span = stats.n_src * tile_bytes if tiled else 4.0 * stats.n_src * feat_len
    slow = 1.0 + c['span'] * max(0.0, math.log2(span / (128.0 * (1 << 20))))
    gathered = 4.0 * stats.nnz * feat_len
    t = gathered * (h / c['hit'] + (1.0 - h) * slow / c['miss'])
    t += stats.segments(P) * T * (c.get('seg_tiled', c['seg']) if T > 1 else c['seg']) + stats.nnz * T * c['edge']
    if tiled:
        t += 2.0 * 4.0 * stats.n_src * feat_len / COPY_BYTES_PER_S
    return t


def predict_spmm(stats, feat_len, P, T, coef=SPMM_COEF):
    """Modelled seconds of one SpMM with P source-column partitions and T feature tiles."""
    t = _gather_seconds(stats, feat_len, P, T, coef) + (coef.get('pass', 0.0) if P > 1 else 0.0)
    # out: one buffer written per pass and read back once by the sum (fitted as (2P - 1) when later passes re-read `out`)
    return t + 4.0 * stats.n_dst * feat_len * (2 * P - 1) / coef['stream']


def predict_sddmm(stats, feat_len, P, T, coef=SDDMM_COEF):
    """Modelled seconds of one single-head SDDMM over the tiled traversal ((1, 1): the row-order kernel)."""
    t = _gather_seconds(stats, feat_len, P, T, coef) + (coef.get('sum', 0.0) if T > 1 else 0.0)
    t += stats.segments(P) * 4.0 * feat_len / coef['stream']                    # destination rows: once per segment
    if (P, T) == (1, 1) and 'edges_dst' in coef:
        t += 4.0 * stats.nnz * feat_len * coef['edges_dst'] / coef['hit']
    # per-tile partial sums: written, read, scattered; results of several partitions go through a position
    out_bytes = 4.0 * stats.nnz * ((2 * T + 2) if T > 1 else (2 if P > 1 and 'edges_dst' in coef else 1))
    return t + out_bytes / coef['stream']


def _candidates(feat_len, max_tile=256):
    tiles = sorted({feat_len // w for w in (32, 64, 128, 256) if feat_len % w == 0 and w <= max_tile and feat_len // w >= 1} | {1})
    tiles = [t for t in tiles if t == 1 or feat_len // t >= MIN_TILE_FLOATS]
    parts = [p for p in (1, 2, 4, 8, 16, 32) if p <= MAX_PARTITIONS]
    return [(p, t) for p in parts for t in tiles]


def _rank(stats, feat_len, predict, cands, tie_key, coef):
    timed = sorted(((predict(stats, feat_len, p, t, coef), p, t) for p, t in cands))
    if not timed:
        return []
    best = timed[0][0]
    near = sorted(((s, p, t) for s, p, t in timed if s <= best * (1.0 + TIE)), key=lambda e: tie_key(e[1], e[2]) + (e[0],))
    rest = [(s, p, t) for s, p, t in timed if s > best * (1.0 + TIE)]
    return [(p, t) for s, p, t in near] + [(p, t) for s, p, t in rest]


def _overrule(stats, feat_len, predict, ranked, cands, coef, margin):
    """On a small graph: the candidates in the order of the coefficients fitted to such graphs, behind the first choice `ranked[0]` of
    the others unless these see `margin` less time for their own."""
    order = [c for _, c in sorted((predict(stats, feat_len, p, t, coef), (p, t)) for p, t in cands)]
    first = ranked[0]
    if predict(stats, feat_len, *first, coef) > (1.0 + margin) * predict(stats, feat_len, *order[0], coef):
        return order
    return [first] + [c for c in order if c != first]


# predicted times within TIE of the best: SpMM takes fewer tiles (fewer passes over the edge list), SDDMM fewer
# partitions (fewer reads of the destination rows)
_spmm_tie = lambda p, t: (t, p)
_sddmm_tie = lambda p, t: (p, t)


def rank_spmm(stats, feat_len):
    """(num_col_partitions, num_feat_partitions) candidates, most promising first."""
    cands = [(p, t) for p, t in _candidates(feat_len) if p <= max(1, stats.n_src)]
    if feat_len > 256:
        cands = [(p, t) for p, t in cands if t > 1]          # rows wider than 256 floats are always tiled
    ranked = _rank(stats, feat_len, predict_spmm, cands, _spmm_tie, SPMM_COEF)
    if not ranked or not _is_small(stats):
        return ranked
    if feat_len % 64 == 0 and stats.nnz < 36 * stats.n_dst:
        # short rows: 32-float tiles, which the model likes for their hit rate, are behind (30,000 nodes of degree 30, us with tiles of 64 / 32
        # floats: F=64 25 / 28, F=256 65 / 78, F=512 116 / 150; 60,000 of degree 40, F=512 385 / 333)
        cands = [(p, t) for p, t in cands if feat_len // t >= 64]
    return _overrule(stats, feat_len, predict_spmm, ranked, cands, SPMM_SMALL_COEF, 0.15 if stats.n_src <= MANY_SOURCES else 0.3)


def rank_sddmm(stats, feat_len, pieces=None):
    """(num_src_partitions, num_feat_tiles) candidates of the tiled traversal, most promising first;
    (1, 1) stands for the edge-list kernel.  pieces: see below."""
    cands = [(p, t) for p, t in _candidates(feat_len) if not (t == 1 and p > 1 and feat_len > 256)]
    ranked = _rank(stats, feat_len, predict_sddmm, cands, _sddmm_tie, SDDMM_COEF)
    if not ranked or not _is_small(stats):
        return ranked
    takes = [(p, t) for p, t in cands if (p, t) == (1, 1) or feat_len // t <= 256 and _is_pow2(feat_len // t) and feat_len // t >= 16]
    ranked = [c for c in ranked if c in takes]
    if 4.0 * stats.n_src * feat_len <= N_XCD * L2_BYTES / 4 or ranked[0][0] == 1:
        ranked = [(1, 1)]
    # Several partitions and one tile write each row's results in pieces, 4 bytes at a time where a row has few elements per partition, which the model does
    # not price: only from `pieces` of them on, or where the first set is for it too (edge list / 2 x 1: 40,000 nodes of degree 20, power-law, F=128
    # 45 / 66, F=64 24 / 32; 25,000 of 32 37 / 54; 15,000 of 12, uniform, F=256 22 / 31; 200,000 of 32, uniform, F=128 2 x 4 460, 2 x 1 570; 40,000 of
    # 32, uniform, F=64 39 / 37).  Over the 276 graphs 93 of 1539 choices are more than 5 % behind the first set's and 34 more than 15 % without this line,
    # 22 and 1 with it.
    if pieces is None:
        pieces = 20 if feat_len <= 64 else 32
    if not (ranked[0][0] > 1 and ranked[0][1] == 1):
        takes = [(p, t) for p, t in takes if p == 1 or t > 1 or stats.nnz >= pieces * p * stats.n_dst]
    return _overrule(stats, feat_len, predict_sddmm, ranked, takes, SDDMM_SMALL_COEF, 0.05 if stats.n_src <= MANY_SOURCES else 0.1)


def choose_spmm(n_dst, n_src, nnz, feat_len, stats=None):
    """(num_col_partitions, num_feat_partitions) for an SpMM of this size (num_feat_partitions 0:
    the kernel's own single tile).  `stats`: GraphStats of the adjacency; without them every column
    counts as equally referenced and every row as of average degree."""
    if nnz == 0 or n_dst == 0:
        return 1, 0
    if stats is None:
        stats = GraphStats(n_dst, n_src, nnz)
    if feat_len >= 2048 and feat_len % 128 == 0:
        # rows of 8 KB and more: 128-float tiles (measured at F=2048: 57.0 ms against 68.7 ms with 64-float tiles)
        cands = [(p, feat_len // 128) for p in (1, 2, 4, 8, 16, 32)]
        p, t = _rank(stats, feat_len, predict_spmm, cands, _spmm_tie, SPMM_COEF)[0]
        return p, t
    ranked = rank_spmm(stats, feat_len)
    if not ranked:
        return 1, 0
    p, t = ranked[0]
    if p == 1 and t == 1:
        return 1, 1
    return p, (t if t > 1 else 0)


# The broadcasting kernel reduces one row segment after the other, all lane groups on the same segment, where the
# weighted-sum kernel gives short segments a lane group each: a segment costs it a few tenths of a nanosecond of
# machine time more.  With this coefficient the choice was the fastest or within 3 % of it on the 233k-node graph
# (u_add_e with one weight per edge, ms at 1 / 2 / 4 / 8 / 16 partitions: F=32 1.30 / 1.20 / 1.22 / 1.38 / 1.98,
# F=64 3.02 / - / 2.14 / 2.20 / 2.56, F=128 6.58 / 5.95 / 4.99 / 4.14 / 4.38, F=256 15.7 / 14.1 / 12.3 / 10.2 / 8.87;
# u_mul_e with [nnz, F] edge features: F=64 6.87 / - / 6.19 / 6.66 / 7.23, F=128 14.4 / 13.7 / 12.7 / 13.1 / 14.1).
BCAST_COEF = dict(SPMM_COEF, seg=4.5e-10)
# ... and per tile when the feature axis is tiled (u_add_e, F=256 in 4 tiles: 12.8 / 11.2 / 9.21 / 7.83 / 9.54 ms at 1 / 2 / 4 / 8 / 16
# partitions; F=128 in 2 tiles: 6.03 / 5.16 / 4.04 / 4.08 / 4.93)
BCAST_TILED_COEF = dict(SPMM_COEF, seg=2.0e-10)


def choose_gather_partitions(n_dst, n_src, nnz, gathered_len, out_len, stats=None, tiles=1):
    """Source-column partitions for a generalised SpMM whose gathered operand has `gathered_len` floats per source
    node and whose result has `out_len` per destination, with the feature axis in `tiles` tiles (the library's own
    choice: 64-float tiles from 128 features on, when the 128-bit paths apply); every partition's results take a
    buffer of their own (8 GiB at most)."""
    if nnz == 0 or n_dst == 0 or gathered_len < 1:
        return 1
    if stats is None:
        stats = GraphStats(n_dst, n_src, nnz)
    tiles = max(1, int(tiles))
    cands = [(p, tiles) for p in (1, 2, 4, 8, 16, 32)
             if p <= min(MAX_PARTITIONS, max(1, n_src)) and (p == 1 or 4.0 * p * n_dst * out_len <= float(8 << 30))]
    coef = BCAST_TILED_COEF if tiles > 1 else BCAST_COEF
    return _rank(stats, gathered_len, predict_spmm, cands, _spmm_tie, coef)[0][0]


# What a row that starts inside a 128-byte line costs the edge-list kernel, in floats (us at F=64 / 71 / 100 / 128: 120,000 nodes of degree
# 100 394 / 598 / 785 / 820, 12,000 of degree 200 37 / 61 / 66 / 69).
EDGES_MISALIGNED = 16


def _choose_sddmm_scattered(stats, feat_len, given_len):
    """A small graph whose edges are stored in no order: the edge-list kernel gathers both operands and meets no row twice in a row, the
    tiled traversal scatters its results.  us, edge list / tiled, uniform graphs unless said: 30,000 nodes of degree 8, F=128 33 / 30
    (power-law 28 / 37), F=512 125 / 74; of degree 40, F=64 66 / 41, F=222 333 / 127; of degree 160, F=16 52 / 71, F=37 194 / 137;
    140,000 of degree 8, F=37 79 / 93, F=64 79 / 74, F=128 157 / 119, F=256 330 / 213; of degree 40, F=222 1642 / 763."""
    # (partitions with one tile: from 12 elements per row on -- 30,000 nodes of degree 8, power-law, F=256 edge list 52, 2 x 1 63 --, and above 64 floats only
    # where nothing else is ahead of the edge list: 40,000 of 16, power-law, F=128 1 x 2 43, 2 x 1 62; 20,000 of 16, F=128 edge list 42, 2 x 1 27; 40,000 of
    # 16, F=64 41, 32)
    coef, edges_len, more = SDDMM_SMALL_COEF, feat_len, 12e-6 + 7e-12 * stats.nnz
    if given_len is not None and given_len != feat_len:
        edges_len = given_len + EDGES_MISALIGNED
        more += _padding_seconds(stats, given_len, feat_len)
    edges = 1.15 * (predict_sddmm(stats, edges_len, 1, 1, coef) + _gather_seconds(stats, edges_len, 1, 1, coef))
    for pieces in (0,) if feat_len <= 64 else (32, 0):
        takes = [(p, t) for p, t in rank_sddmm(stats, feat_len, pieces) if (p, t) != (1, 1) and (t > 1 or stats.nnz >= 12 * stats.n_dst)]
        if takes and predict_sddmm(stats, feat_len, *takes[0], coef) + more < edges:
            return takes[0]
    return None


def _padding_seconds(stats, given_len, feat_len):
    """Padded copies of both operands."""
    return 2 * 4e-6 + 8.0 * max(stats.n_dst, stats.n_src) * (given_len + feat_len) / SDDMM_SMALL_COEF['stream']


def choose_sddmm(n_rows, n_cols, nnz, heads, head_len, stats=None, given_len=None, scattered=False):
    """(num_src_partitions, num_feat_tiles) for the tiled traversal, or None when the plain
    kernels should be used (small feature matrices, or a shape the tiled kernel does not take).  given_len: the rows' length where
    head_len is what the tiled traversal would pad them to.  scattered: the edges are stored in no order of their rows.
    stats: GraphStats, or a function that returns them, called where they are read."""
    feat_len = heads * head_len
    if heads == 1:
        if nnz == 0 or feat_len % 4 != 0:
            return None
        if stats is None:
            stats = GraphStats(n_rows, n_cols, nnz)
        elif callable(stats):
            stats = stats()
        if _is_small(stats) and scattered:
            return _choose_sddmm_scattered(stats, feat_len, given_len)
        if _is_small(stats):
            ranked = rank_sddmm(stats, feat_len)
            if given_len is not None and given_len != feat_len:
                # unpadded on the edge-list kernel, or padded copies of both operands and the tiled traversal
                tiled = [c for c in ranked if c != (1, 1)]
                if not tiled:
                    return None
                copies = _padding_seconds(stats, given_len, feat_len)
                edges = predict_sddmm(stats, given_len + EDGES_MISALIGNED, 1, 1, SDDMM_SMALL_COEF)
                return tiled[0] if copies + predict_sddmm(stats, feat_len, *tiled[0], SDDMM_SMALL_COEF) < edges else None
            return None if not ranked or ranked[0] == (1, 1) else ranked[0]
        if 4.0 * n_cols * feat_len <= N_XCD * L2_BYTES / 4:
            return None                                # the whole operand sits in every L2: nothing to tile
        ranked = [(p, t) for p, t in rank_sddmm(stats, feat_len)
                  if feat_len // t <= 256 and _is_pow2(feat_len // t) and feat_len // t >= 16]
        if not ranked or ranked[0][0] == 1:
            # No source partitions: the stored-order kernels.  Without partitions the traversal has no slice to keep in
            # the L2s and still pays for its partial sums and the scatter to the stored order (measured: 2-8 % behind at
            # 1 x 1; 2.45M-node graph at F = 512: 1 x 2 tiles 22.5 ms, stored order 20.1 ms; uniform 1M-node graph: 23.3 / 22.7 ms).
            return None
        return ranked[0]
    first = _choose_sddmm_heads(n_rows, n_cols, nnz, heads, head_len, scattered)
    padded = given_len is not None and given_len != head_len
    if 0 < nnz < SMALL_NNZ and (scattered or not padded) and 8 <= head_len <= 64 and _is_pow2(head_len):
        stats = GraphStats(n_rows, n_cols, nnz) if stats is None else stats() if callable(stats) else stats
        return _choose_sddmm_heads_small(stats, heads, head_len, first, given_len if padded else None, scattered)
    if padded and not scattered and first is not None and first[0] == 1:
        # padded heads without source partitions: the edge-list kernel reads them unpadded (40,000 nodes of degree 4, 8 x 48:
        # 131 -> 44 us; 193,000 of degree 17 1289 -> 706; 172,000 of degree 16, 2 x 20 141 -> 81)
        return None
    return first


def complete_tiled_sddmm(n_rows, n_cols, nnz, heads, head_len, stats=None):
    """(num_src_partitions, num_feat_tiles) for a caller who asks for the tiled traversal, or for one of the two numbers, where choose_sddmm
    would take an edge-list kernel: tiles that the kernel takes, (1, 1) where there are none."""
    feat_len = heads * head_len
    takes = lambda tile: 16 <= tile <= 256 and _is_pow2(tile) and (heads == 1 or tile % head_len == 0 and head_len % 4 == 0 and head_len >= 8)
    if heads == 1:
        if takes(feat_len) or nnz == 0 or feat_len % 4 != 0:
            return 1, 1
        if stats is None:
            stats = GraphStats(n_rows, n_cols, nnz)
        cands = [(p, t) for p, t in _candidates(feat_len) if feat_len % t == 0 and takes(feat_len // t)]
        ranked = _rank(stats, feat_len, predict_sddmm, cands, _sddmm_tie, SDDMM_COEF)
        return ranked[0] if ranked else (1, 1)
    first = _choose_sddmm_heads(n_rows, n_cols, nnz, heads, head_len, scattered=True)
    if first is not None:
        return first
    return 1, next((feat_len // tile for tile in (256, 128, 64, 32, 16) if feat_len % tile == 0 and takes(tile)), 1)


def _is_pow2(v):
    return v > 0 and (v & (v - 1)) == 0


def _partitions(n_src, row_bytes, nnz, n_rows, slice_bytes, min_segment):
    """Partitions that bring an XCD's slice of the gathered rows down to `slice_bytes` while row
    segments keep `min_segment` elements on average (the rule the multi-head and attention operators use)."""
    want = (n_src * row_bytes) / slice_bytes
    if want <= 1.0:
        return 1
    p = _pow2_floor(int(want + 0.5)) if want >= 2 else 2
    avg_deg = nnz / max(1, n_rows)
    while p > 1 and avg_deg / p < min_segment:
        p //= 2
    return max(1, min(64, p))


# Several heads on a small graph: seconds of the edge list (factor on the model's time of it, launch) and of the tiled walk (the same, per byte of results that
# are staged, per byte of those that are scattered, a last kernel, per row segment and tile).  Fitted to 336 graphs and shapes (6,000 to
# 150,000 nodes, degrees 6 to 90, uniform and power-law, 2 to 16 heads of 8 to 64 floats): 4 % behind the best of edge list and 1 to 8 partitions on average, where
# the rule for large graphs below is 12 %.  us, that rule's choice / this: 40,000 nodes of degree 90, 8 x 32 493 / 325, 4 x 32 217 / 116, 2 x 64 213 / 111; of degree
# 25, 16 x 32 316 / 196; 150,000 of degree 6, 3 x 16 89 / 38, 8 x 64 461 / 303.
_HEADS_SMALL = dict(edges=1.527, edges_launch=1.2e-6, tiled=1.718, staged=0.177e-12, scattered=0.145e-12, launch=3.6e-6, last=4.3e-6, segment=0.023e-10)


# The same where the edges are stored in no order: the edge list gathers both operands (shares of the model's time for row-ordered edges and of one
# operand's gather), the tiled walk's results go to random places (more per byte).  Fitted to 294 graphs and shapes (6,000 to 500,000 nodes, degrees 6 to
# 200, 2 to 16 heads of 8 to 128 floats), 5 % behind the best of edge list and 1 to 8 partitions on average; the rule for large graphs is 13 % behind, and the
# numbers above, which know nothing of the second gather, 16 %.  us, edge list / (1, 1) / this: 140,000 nodes of degree 40, 8 x 16 811 / 456 / 456, 4 x 32 767 /
# 433 / 368, 8 x 64 3037 / - / 1624; 60,000 of 20, 8 x 8 85 / 60 / 60; 200,000 of 16, power-law, 8 x 64 1749 / - / 1102; 150,000 of 6, power-law, 2 x 16 34 / 48 / 34.
_HEADS_SCATTERED = dict(ordered=0.5, gather=1.4, staged=0.5e-12, scattered=0.25e-12)


def _choose_sddmm_heads_small(stats, heads, head_len, first, given_len=None, scattered=False):
    """The choice of this model, or `first` where that is a candidate and the model sees less than 5 % (10 % for scattered edges, whose times
    it knows less well) more time for it.  given_len (scattered edges): the heads' length where head_len is what the tiled walk would pad them to."""
    feat_len, out_bytes, c = heads * head_len, 4.0 * stats.nnz * heads, _HEADS_SMALL
    more = _HEADS_SCATTERED if scattered else dict(staged=0.0, scattered=0.0)
    copies = 0.0 if given_len is None else _padding_seconds(stats, heads * given_len, feat_len)

    def tiled(p, t):
        tile = feat_len // t
        per_tile, segments = tile // head_len, stats.segments(p)
        s = c['tiled'] * (_gather_seconds(stats, feat_len, p, t, SDDMM_SMALL_COEF) + segments * 4.0 * feat_len / SDDMM_SMALL_COEF['stream'])
        s += c['launch'] + segments * t * c['segment'] + copies
        if per_tile == 1 and heads >= 4 and t > 1:
            return s + out_bytes * (c['staged'] + more['staged']) + c['last']
        return s + out_bytes * (c['scattered'] + more['scattered']) * max(1.0, 8.0 / per_tile)

    def edge_list():
        length = feat_len if given_len is None else heads * given_len + (EDGES_MISALIGNED if heads * given_len % 32 else 0)
        s = predict_sddmm(stats, length, 1, 1, SDDMM_SMALL_COEF)
        if scattered:
            s = more['ordered'] * s + more['gather'] * _gather_seconds(stats, length, 1, 1, SDDMM_SMALL_COEF)
        # (unpadded against padded: 90,000 nodes of degree 30, power-law, edge list / tiled: 2 x 20 144 / 126, 3 x 20 217 / 228, 8 x 48 1072 / 740; 100,000 of 12
        # 70 / 85, 105 / 150, 532 / 529; 500,000 of 8 281 / 367, 389 / 707, 1928 / 2602)
        return (1.0 if given_len is None else 1.1) * c['edges'] * s + c['edges_launch']

    cands = [(p, feat_len // w) for w in (32, 64, 128, 256) if feat_len % w == 0 and w % head_len == 0 for p in (1, 2, 4, 8) if p <= max(1, stats.n_src)]
    costs = {c: tiled(*c) for c in cands}
    costs[None] = edge_list()
    best = min(costs, key=costs.get)
    margin = 0.1 if scattered and given_len is None else 0.05
    return first if first in costs and costs[best] > (1.0 - margin) * costs[first] else best


def _choose_sddmm_heads(n_rows, n_cols, nnz, heads, head_len, scattered=False):
    """Several heads per edge.  What an (edge, tile) pair writes decides the tile: the memory system writes whole 32-byte
    sectors, so a tile that holds fewer than 8 heads and scatters them to `out` pays a sector for its 8 or 16 bytes
    (232,965-node graph, counted at the fabric: 8.0 GB written for 3.67 GB of results at H=8, D=32 with 128-float tiles,
    16.2 GB at H=8, D=64).  Hence
      * heads of up to 32 floats, 8 or more of them: 256-float tiles (8 or more heads, 32 bytes or more per edge and
        tile, written where they belong) -- H=8, D=32: 8.64 -> 7.71 ms with one tile x 32 partitions;
      * longer heads: one head per tile, each tile's results kept in traversal order (whole runs) and every edge's H
        results written as one run by a last kernel -- H=8, D=64: 15.2 -> 13.4 ms with 8 tiles x 8 partitions;
      * fewer than 8 short heads: 64-float tiles as before (H=4, D=32: one 128-float tile is no faster).
    Partitions: two L2s' worth of slices per XCD, segments of 24 elements or more (12 for the 256-float tiles, whose
    slices need four times the partitions: 7.7 ms at 32 partitions against 8.4 at 16)."""
    feat_len = heads * head_len
    if head_len % 4 != 0 or head_len < 8 or (head_len & (head_len - 1)) != 0:
        return None
    min_segment = 24
    if head_len <= 32 and heads >= 8 and feat_len % 256 == 0:
        tile, min_segment = 256, 12
    elif head_len in (64, 128) and feat_len >= 256:
        tile = head_len
    else:
        tile = None
        for cand in (64, 128, 256, 32, 16):
            if feat_len % cand == 0 and (cand % head_len == 0 or head_len == cand):
                tile = cand
                break
        if tile is None:
            return None
    t = feat_len // tile
    row_bytes = 4 * feat_len / t          # more than 8 tiles are launched 8 at a time: one tile's slice per XCD
    if n_cols * row_bytes <= SDDMM_SLICE_BYTES:
        return None
    p = _partitions(n_cols, row_bytes, nnz, n_rows, SDDMM_SLICE_BYTES, min_segment=min_segment)
    if p > 1 and t < 8 and 8 % t == 0 and p < 8 // t:
        # at least one partition per XCD (a single launch covers them all) -- unless that leaves the segments too short
        p = 8 // t if nnz / max(1, n_rows) / (8 // t) >= min_segment else 1
    if p == 1 and (t == 1 or feat_len <= 256 and _is_pow2(feat_len)):
        # Row-ordered edges: the edge-list kernel, which needs no positions (36,608 nodes of degree 11, 8x32 69 -> 61 us; 124,691 of degree 67, 8x8
        # 322 -> 315; 2,450,000 of degree 25, power-law, 8x32 11672 -> 10827; 1,000,000 of 60, 8x16 4435 -> 4522).  Scattered ones: one tile, which gathers
        # one operand and reads a destination row once per segment, where the edge list gathers both (edge list / one tile: 1,000,000 of 60, 8x32 20831
        # / 12795, 4x16 4257 / 3932; 700,000 of 50, power-law, 8x32 9642 / 5475, 2x16 1259 / 1084) -- unless rows are short and few edges share
        # one (2,450,000 of 25, power-law, 8x32 20995 / 13765, but 4x16 4371 / 4814, 2x16 2322 / 3062).
        if scattered and 16 <= feat_len <= 256 and _is_pow2(feat_len) and (feat_len > 64 or nnz >= 32 * n_rows or nnz < SMALL_NNZ):
            return 1, 1
        return None
    return p, t


# What attention's gradients may take for two [nnz, H] arrays while a call lasts.
ATTENTION_EDGE_BYTES = 16 << 30


def attention_keeps_score_gradients(nnz, num_rows, heads, head_len):
    """Whether the gradients of dot-product attention keep the scores' gradients and take dQ from a weighted sum that
    gathers K alone, instead of a second sweep that gathers K and V.  Saved per edge and head: a gather of head_len floats and
    the score's second evaluation; paid: the values written, brought into the other order (in fours of heads at about 1.5 times
    a copy's time, one to three heads a scattered 4-byte read each) and read.  Whole steps, second sweep -> kept, in us:
      58,000 nodes, 12.5 M edges: 8x64 8335 -> 7450, 1x64 1110 -> 1020, 8x32 5565 -> 5037, 8x16 4907 -> 4244, 4x16 2296 -> 2052,
        but 4x32 2185 -> 2219, 2x32 1003 -> 1075, 1x32 551 -> 598
      20,000 nodes, 4 M edges: 4x64 1335 -> 1160, 4x32 696 -> 643, 2x32 332 -> 348
      200,000 nodes, 4 M edges: 8x64 7345 -> 6221, 4x32 1857 -> 1651, 2x32 876 -> 835, 1x32 454 -> 432, 1x16 395 -> 392
      100,000 nodes, 8 M edges: 4x32 1956 -> 1842, 2x32 930 -> 935
      20,000 nodes, 200,000 edges (launches): 4x64 183 -> 165, 2x64 147 -> 157, 8x16 218 -> 206, 4x32 136 -> 163
      heads of 64, one / two / three / four of them: 200,000 nodes, 1.6 M edges 541 -> 468, 1054 -> 899, 1581 -> 1350, 2169 -> 1864; 400,000, 6 M
        1594 -> 1445, 3244 -> 2921, 4960 -> 4439, 7555 -> 6419; 100,000, 8 M 1586 -> 1294, 3200 -> 2728, 5323 -> 4576, 6388 -> 5344; 10,000, 3.9 M
        275 -> 263, 528 -> 496, 1422 -> 1148, 1119 -> 977; sources skewed, 20,000, 3.7 M 1024 -> 1017, 1205 -> 1181, 2087 -> 1842, 1677 -> 1552;
        sources skewed, 200,000, 6 M 4624 -> 4525, 6401 -> 6215, 7746 -> 7379, 9135 -> 8549"""
    if nnz * heads * head_len < 3 << 24 or 2 * 4 * nnz * heads > ATTENTION_EDGE_BYTES:
        return False
    if head_len == 64:
        return True
    if heads % 4:
        return nnz <= 32 * num_rows
    return head_len == 16 or heads % 8 == 0 or nnz <= 128 * num_rows


def sum_gradients_in_one_sweep(num_rows, num_cols, nnz, heads, head_len):
    """Whether the two gradients of a weighted sum come faster from one sweep over the transposed graph than from a sum and a
    separate SDDMM (heads of head_len floats).  The kernels with dots lose where a lane group is
    small -- tiles of one head of 16 floats, of several short heads -- and the SDDMM has whole tiles for the shape; they win
    many times over where it has not.  Whole steps, two sweeps -> one, in us:
      one head, 16 floats: 400,000 elements 69 -> 65 (degree 8); 4 M 179 -> 198 (30), 13 M 453 -> 492 (120); 32 floats: 2 M 161 -> 172 (8), 4 M 236 -> 240
        (20), 216 -> 219 (30), 12.5 M 455 -> 425 (215); 24, run as 32: 4 M 302 -> 285 (20); 64: 4 M 560 -> 496 (8), 370 -> 321 (30), 238 -> 206 (120)
      2x16: 100,000 74 -> 71, 400,000 93 -> 97, 4 M 528 -> 577 (8), 334 -> 415 (30), 212 -> 275 (120)
      4x16: 4 M 668 -> 582 (8), 300 -> 298 (120); 13 M 2106 -> 1876 (8), 1231 -> 1130 (120), but 945 -> 973 (215)
      4x8 / 8x8 / 2x32, 1 M: 155 -> 143 / 218 -> 194 / 178 -> 166 (8), 157 -> 150 / 161 -> 162 / 152 -> 147 (30); 4 M: 306 -> 325 / 552 -> 560 /
        464 -> 469 (30), 225 -> 244 / 402 -> 458 / 260 -> 299 (120)
      16x8: 4 M 1572 -> 1469 (8), 1112 -> 1039 (30), 825 -> 840 (120); 3x32, 6x32: 1020 -> 959, 1913 -> 1851 (8), 613 -> 643, 1442 -> 1449 (30);
        13 M 1397 -> 1593, 2991 -> 3407 (120)
      4x32, 8x32, 8x16: 4 M 852 -> 667, 1744 -> 1288, 933 -> 790 (30), 454 -> 391, 925 -> 781, 573 -> 555 (120)
      no tile of the SDDMM's: 3x16 1128 -> 423, 6x32 1092 -> 412, 12x8 3403 -> 975 (4 M, 2 M, 4 M; 120)"""
    feat_len = heads * head_len
    if heads == 1:
        return nnz < 1 << 20 or head_len > 16 and (head_len != 32 or nnz >= 24 * num_rows)
    if head_len >= 64 or not _is_pow2(feat_len) and _choose_sddmm_heads(num_rows, num_cols, nnz, heads, head_len) is None:
        return True
    if head_len == 16:
        if heads % 4:
            return nnz < 1 << 18
        return feat_len >= 128 or nnz < 1 << 22 or nnz <= 128 * num_rows
    if head_len == 32 and _is_pow2(feat_len) and feat_len >= 128:
        return True
    return nnz < 1 << 20 or (feat_len >= 128 and nnz <= (16 if head_len == 32 else 64) * num_rows)


def select_by_sweep(nnz, num_rows, feat_len, target, own_len, other_len):
    """Whether the gradient of a max / min aggregation for an operand on `target` comes from a sweep over the edges (own_len features, 1 where
    it was broadcast over feat_len; other_len features of the other operand of a product or quotient, 0 without one) instead of an
    atomic per result.  Whole gradient calls, atomics -> sweep, in us, uniform graphs / power-law ones:
      120,000 rows, sources, F=64, 4 / 8 / 16 / 32 elements per row: copies 106 -> 43, 344 -> 76, 348 -> 138, 331 -> 259 / 98 -> 45, 324 -> 75, 338 -> 135,
        318 -> 251; times F edge features 108 -> 63, 377 -> 119, 396 -> 215, 410 -> 405 / 101 -> 70, 362 -> 132, 396 -> 231, 406 -> 411; times one 362 -> 332 / 360 -> 327 (32)
      F=16: copies 104 -> 33, 105 -> 57, 104 -> 102 (8, 16, 32) / 104 -> 51, 104 -> 76, 103 -> 118; times F 112 -> 56, 118 -> 98 / 113 -> 87, 122 -> 133 (8, 16)
      20,000 rows of 32, F=128: copies 107 -> 78 / 112 -> 69; of 64 90 -> 137 / 93 -> 125
      edges, F features, no other operand: F=64 136 -> 96, 298 -> 161, 443 -> 253 / 122 -> 101, 257 -> 176, 398 -> 293 (8, 16, 32); 20,000 rows of 128 195 -> 153 / 189 ->
        158; F=16 41 -> 27 / 36 -> 43 (8), 96 -> 67 / 82 -> 101 (32); with a product F=64 161 -> 119 / 139 -> 156 (8), F=16 46 -> 38 / 40 -> 97
      edges, one value: F=64 264 -> 34, 333 -> 72 / 294 -> 51, 308 -> 117 (8, 32), F=16 79 -> 25 / 78 -> 35 (8), 102 -> 76 / 102 -> 100 (64); with a product F=64 79 -> 67,
        293 -> 65, 350 -> 160 / 83 -> 91, 307 -> 104, 327 -> 227 (4, 8, 32), 20,000 rows of 64 84 -> 50 / 90 -> 99; F=16 93 -> 30 / 90 -> 82 (8), 107 -> 73 / 105 -> 161 (32)"""
    wide, degree = feat_len >= 48, nnz / max(1, num_rows)
    if target == 'u':
        if other_len == 0:
            return degree <= (32 if wide else 24)
        return degree <= ((24 if other_len > 1 else 32) if wide else 12)
    if own_len == feat_len:
        return wide and other_len == 0 and degree <= 128
    if other_len == 0:
        return degree <= 64
    return wide and 6 <= degree <= 48
