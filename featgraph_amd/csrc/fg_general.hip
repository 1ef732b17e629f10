// Generalised SpMM / SDDMM with broadcasting, for gfx950: the two operands of the message may live on the
// source nodes (u: indexed by the element's column), the destination nodes (v: its row) or the stored
// elements themselves (e), and their feature shapes may differ as long as they broadcast against each
// other.  The caller describes the broadcast by two index arrays: output feature f takes operand feature
// lhs_off[f] and rhs_off[f] (a null array is the identity).
//
//   SpMM : out[v, f]  = reduce over the elements e of row v of  lhs[.., lhs_off[f]] op rhs[.., rhs_off[f]]
//   SDDMM: out[e, f]  = lhs[.., lhs_off[f]] op rhs[.., rhs_off[f]]           (element-wise operators)
//          out[e, f]  = sum_{i < R} lhs[.., lhs_off[f] * R + i] * rhs[.., rhs_off[f] * R + i]   (dot)
//
// No counterpart in the reference, whose operators are the weighted sum (python/featgraph/op/vanilla_spmm.py)
// and the dot product (python/featgraph/op/vanilla_sddmm.py); the message / reduce vocabulary is the one its
// README.md:9-11 names ("generalized SpMM and SDDMM").
//
// The SpMM kernel walks the plan's work items, one wavefront each, like the weighted-sum kernel.  A lane holds
// V output features (V = 4 with 128-bit accesses when the shapes allow it, else 1); a group of L lanes
// (L = the power of two that covers the F / V vectors, at most 64) takes one element at a time and the
// 64 / L groups take different elements of the row, several steps in flight (in an item of many short rows
// every group takes a row of its own instead); feature axes of 128 floats and more, in multiples of 64, are cut
// into 64-float tiles for different workgroups when an operand is gathered (each L2 then holds one tile's slice of
// the gathered rows); other long axes are walked 64 vectors at a time.  With one group (64 vectors or more, no
// tiles), and for rows that a group has to itself, a row's sum is formed in the stored element order.  The edge operand, when there is one, is the dominant stream ([nnz, len] floats read once,
// coalesced, past the caches); the node operand is gathered, through column words that the wavefront has staged
// in LDS for the whole item.
//
// Over a plan with several source-column partitions (fg_gspmm_bcast_dds_f32) one launch walks all partitions'
// items in partition order, so that the gathered operand's rows of the current partition stay in the L2s: a
// partition's row segments are reduced into a buffer of its own and a closing kernel combines the buffers in
// partition order.  The elements then come in the partitioned layout's order and reach the operands on the edges
// (and the reported positions) through the layout's element -> stored position array.
#include <hip/hip_runtime.h>

#include <climits>
#include <type_traits>

#include "fg_common.h"
#include "fg_device.h"

using fg::fail;
using fg::Fixup;
using fg::Item;
using fg::wave_lds_sync;

// Every message is one correctly rounded float32 operation and every sum adds the rounded messages one by
// one, so that max / min, the selected positions and (with one lane group per row) the sums in stored
// order can be compared bit for bit with a sequential float32 evaluation.  This file is therefore compiled
// with -ffp-contract=off (featgraph_amd/build.py); a pragma alone does not stop the back end from fusing
// when the command line says -ffp-contract=fast.

namespace {

constexpr int kWavesPerBlock = 4;
constexpr int kBlock = 64 * kWavesPerBlock;
constexpr int kStage = 256;             // elements whose index words a wavefront keeps in LDS at a time

struct GenArgs {
    const Item *items;
    int64_t n_items;
    const int32_t *indptr;
    const int32_t *indices;
    const uint16_t *indices16;   // the plan's 16-bit copy of `indices`, read instead of it (null: none)
    const float *lhs, *rhs;
    const int32_t *lhs_off, *rhs_off;
    int lhs_len, rhs_len;
    int lhs_target, rhs_target;
    float sign;                  // -1: the launch computes a minimum as the negated maximum of the negated messages; else 1
    const float *row_scale;      // out[v, :] *= row_scale[v] (null: 1), applied where a row is completed
    float *out;
    int32_t *arg;                // optional: stored position of the selected element (max / min)
    float *partial;              // pieces of split rows: [slot][F] values
    int32_t *partial_arg;        //                       [slot][F] positions
    int F, L;
    int spread;                  // a row of an item of n rows is shared by the fewest lane groups (a power of two) that are spread / n of all
    // PART: the elements are not addressed by their own positions -- several source-column partitions (indptr /
    // indices are the partitioned layout's position and local column arrays, item_off the plan's item ranges per
    // partition, out / arg the partitions' buffers; strides in elements, per partition), or edge operands that the
    // caller keeps in another order: edge_pos gives every element's row in the edge operands (and the position that
    // is reported for it).
    const int64_t *item_off;
    const int32_t *edge_pos;
    int n_parts;
    int n_tiles, tile_vecs;      // the feature axis in n_tiles tiles of tile_vecs vectors (V floats each), one per workgroup
    int ordered;                 // element positions ascend along every row (segment) of the walked layout
    int final;                   // the kernel's rows are results (one partition), not a partition's share of them
    int64_t pos_stride, col_width, out_stride, partial_stride;
    bool src32;                  // the left operand lies on the source nodes and spans less than 4 GiB
};

// The operand features of a lane's V outputs: V consecutive ones (CONTIG: one 128-bit load) or one value V times.
// NT: a non-temporal load, for an operand on the stored elements, which is read once from end to end and should not
// displace the gathered operand's rows from the L2.
// (At 4-byte alignment: one 128-bit load all the same.)
typedef float nt_f4 __attribute__((ext_vector_type(4), aligned(4)));
template <int V, bool CONTIG, bool NT = false>
__device__ __forceinline__ void load_operand(const float *p, float (&o)[V]) {
    if (V == 4 && CONTIG && NT) {
        const nt_f4 t = __builtin_nontemporal_load(reinterpret_cast<const nt_f4 *>(p));
        o[0] = t.x; o[1 % V] = t.y; o[2 % V] = t.z; o[3 % V] = t.w;
    } else if (V == 4 && CONTIG) {
        const nt_f4 t = *reinterpret_cast<const nt_f4 *>(p);
        o[0] = t.x; o[1 % V] = t.y; o[2 % V] = t.z; o[3 % V] = t.w;
    } else {
        const float s = *p;
#pragma unroll
        for (int i = 0; i < V; ++i) o[i] = s;
    }
}

// The row `row` of an operand whose rows are `row_bytes` long, from the lane's first feature on: one 64-bit multiply-add.
__device__ __forceinline__ const float *row_at(const char *lane_base, int row, uint32_t row_bytes) {
    return reinterpret_cast<const float *>(lane_base + (uint64_t)(uint32_t)row * row_bytes);
}

// The first of the V features that vector `i` of a row of F covers.  F need not be a multiple of V: the last vector then starts earlier and
// shares features with the one before it, and the two lanes form and store the same values.  One feature per
// lane -> so, us on 20,000 rows of 60 elements, F=65 / 145: copy_u max 90 -> 60 / 142 -> 91, u_mul_e sum 141 -> 118 / 304 -> 212, per edge u_mul_e 149 -> 139
// / 327 -> 307, with one value per edge 182 -> 88 / 385 -> 210; F=11 28 -> 21, 25 -> 16.
template <int V> __device__ __forceinline__ int first_feature(int i, int F) { return V == 1 ? i : min(i * V, F - V); }

template <int OP> __device__ __forceinline__ float binary(float l, float r) {
    return OP == FG_BIN_ADD ? l + r : OP == FG_BIN_SUB ? l - r : OP == FG_BIN_MUL ? l * r
         : OP == FG_BIN_DIV ? l / r : OP == FG_BIN_COPY_LHS ? l : r;
}
template <int OP> constexpr bool kUsesLhs = OP != FG_BIN_COPY_RHS;
template <int OP> constexpr bool kUsesRhs = OP != FG_BIN_COPY_LHS;

template <int RED> __device__ __forceinline__ float identity() {
    return RED == FG_REDUCE_SUM ? 0.f : RED == FG_REDUCE_MAX ? -INFINITY : INFINITY;
}
// Max / min treat a NaN message as beating every number, so that it reaches the row's result the way it does through
// a sum (what numpy's maximum / minimum reductions and argmax / argmin do): the running extreme of (acc, m).  The part's
// v_maximum3_f32 / v_minimum3_f32 do exactly that in one instruction (two messages of a step share one).
template <int RED> __device__ __forceinline__ float extreme(float acc, float m) {
    return RED == FG_REDUCE_MAX ? __builtin_elementwise_maximum(acc, m) : __builtin_elementwise_minimum(acc, m);
}
// Whether candidate (m, at element em) replaces (acc, at element ea): the better value (a NaN is better than any
// number), or the same value (two NaNs count as the same) at an earlier element; the first value always enters.
template <int RED> __device__ __forceinline__ bool replaces(float m, int em, float acc, int ea) {
    const bool m_nan = m != m, acc_nan = acc != acc;
    const bool better = m_nan ? !acc_nan : (!acc_nan && (RED == FG_REDUCE_MAX ? m > acc : m < acc));
    const bool same = m_nan ? acc_nan : m == acc;
    return em != INT_MAX && (ea == INT_MAX || better || (same && em < ea));
}

enum { kFirst, kFull, kNaNs };      // how a walk finds positions, see batch() below

// LC / RC (V == 4 only): the operand's 4 features are consecutive (one 128-bit load), else one value 4 times.
// No branch stands between the loads of a step: one around a load would make the wavefront wait for everything
// issued before it.
// PART: see GenArgs; with several partitions (a.final == 0) a row segment without elements keeps the reduction's
// identity and no row is scaled, both being the combining kernel's business.
// LNT / RNT: see load_operand.  RED: FG_REDUCE_SUM or FG_REDUCE_MAX; a minimum runs as the maximum of the negated
// messages (a.sign = -1; negation is exact, so values, ties and selected positions are those of the minimum).
// SRC32: the left operand lies on the source nodes and spans less than 4 GiB: its rows' byte offsets are formed once,
// where the columns are staged, and the gathers add them to a scalar base.  SIGN (not 0): the sign as a compile-time constant
// (GenArgs::sign is not read), which the comparison and the maximum take as an operand modifier.  Both for the selected
// copies in ascending order, the walk that vector instructions bound (26 of them per gathered 128 bits without, 17 with);
// registers still allow 4 wavefronts per SIMD, and forcing 6 spills (F=100 452 -> 530 us).  12.5M edges on 58,000 nodes, copy_u max,
// F=64 / 100 / 128: 289 / 474 / 575 -> 270 / 452 / 544 us.
template <int OP, int RED, bool ARG, int V, bool LC, bool RC, bool LNT, bool RNT, bool PART, bool SRC32 = false, int SIGN = 0>
__global__ __launch_bounds__(kBlock) void gspmm_bcast_kernel(const GenArgs a) {
    static_assert(RED == FG_REDUCE_SUM || RED == FG_REDUCE_MAX, "a minimum is a maximum with a.sign = -1");
    constexpr bool kLhs = kUsesLhs<OP>, kRhs = kUsesRhs<OP>;
    const float sign = RED == FG_REDUCE_SUM ? 1.f : SIGN ? (float)SIGN : a.sign;
    const bool final = !PART || a.final != 0;
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    // workgroup id = item block * n_tiles + tile: the XCDs, dealt workgroups in turn, work on different feature tiles
    // of the same items, so that each L2 holds one tile's slice of the gathered rows
    const int tile = (int)(blockIdx.x % (unsigned)a.n_tiles);
    const int64_t item_id = (int64_t)(blockIdx.x / (unsigned)a.n_tiles) * kWavesPerBlock + wave;
    if (item_id >= a.n_items) return;
    const Item it = a.items[item_id];
    const int L = a.L, G = 64 / L, g = lane / L, li = lane % L;
    const int F = a.F, FV = (F + V - 1) / V;
    const int fv_lo = tile * a.tile_vecs, fv_hi = min(FV, fv_lo + a.tile_vecs);
    int part = 0;
    if (PART) {
        const int64_t id = ((int64_t)__builtin_amdgcn_readfirstlane((int)(item_id >> 32)) << 32) |
                           (uint32_t)__builtin_amdgcn_readfirstlane((int)item_id);
        while (part + 1 < a.n_parts && id >= a.item_off[part + 1]) ++part;
    }
    const int32_t *const pos_p = a.indptr + (PART ? part * a.pos_stride : 0);
    const int64_t ubase = PART ? part * a.col_width : 0;       // the partition's first column
    float *const out_p = a.out + (PART ? part * a.out_stride : 0);
    int32_t *const arg_p = ARG ? a.arg + (PART ? part * a.out_stride : 0) : nullptr;
    float *const partial_p = a.partial + (PART ? part * a.partial_stride : 0);
    int32_t *const partial_arg_p = ARG ? a.partial_arg + (PART ? part * a.partial_stride : 0) : nullptr;
    const bool l_on_e = a.lhs_target == FG_TARGET_E, r_on_e = a.rhs_target == FG_TARGET_E;
    constexpr int U = V == 4 ? 4 : 8;     // elements in flight per lane group: the loads of a step are issued before their use

    // The column and the stored position of up to kStage consecutive elements, read once with coalesced loads: the
    // gathers of a step then wait for LDS, not for a load of their own index words.
    __shared__ int2 s_el[kWavesPerBlock][kStage];
    int2 *const el = s_el[wave];
    auto stage = [&](int64_t c0, int n) {
        for (int t = lane; t < n; t += 64) {
            const int col = a.indices16 ? (int)a.indices16[c0 + t] : a.indices[c0 + t];      // uniform choice
            const uint32_t src = (uint32_t)(col + (int)ubase);
            el[t] = make_int2((int)(SRC32 ? src * ((uint32_t)a.lhs_len * 4u) : src), PART ? a.edge_pos[c0 + t] : (int)(c0 + t));
        }
        wave_lds_sync();
    };

    // the elements [e0, e1) of output row v: reduce and store to (dst_v, dst_a); `done`: the row is complete.
    // staged_at >= 0: the range lies inside the elements staged from that position on; else it is staged here, kStage
    // elements at a time (a lane group keeps its elements and their order: kStage is a multiple of the groups).
    // own (a std::bool_constant): false = the wavefront's lane groups share the row, taking every G-th element each, and
    // their results are combined; true = every `share` (a power of two) neighbouring lane groups have a row of their own (e0,
    // e1, v and the destinations differ, `mine` says whether they have a row at all), of whose elements each takes every
    // share-th, and the first of them stores it -- for items of several rows, whose elements are all staged.
    auto reduce_range = [&](auto own, int share, bool mine, int64_t e0, int64_t e1, int64_t staged_at, int v, float *dst_v, int32_t *dst_a,
                            bool done) {
        constexpr bool OWN = decltype(own)::value;
        const int first = OWN ? g & (share - 1) : g, step = OWN ? share : G, lanes = OWN ? L * share : 64;
        for (int f0 = fv_lo; f0 < fv_hi; f0 += L) {
            const bool active = f0 + li < fv_hi;
            const int fc = first_feature<V>(active ? f0 + li : fv_hi - 1, F);       // the lane's first output feature
            const int fl = kLhs ? (a.lhs_off ? a.lhs_off[fc] : fc) : 0;
            const int fr = kRhs ? (a.rhs_off ? a.rhs_off[fc] : fc) : 0;
            const char *const lbase = reinterpret_cast<const char *>(kLhs ? a.lhs + fl : nullptr);
            const char *const rbase = reinterpret_cast<const char *>(kRhs ? a.rhs + fr : nullptr);
            const uint32_t lbytes = (uint32_t)a.lhs_len * 4u, rbytes = (uint32_t)a.rhs_len * 4u;
            float acc[V];
            int at[V];
            // One step of U elements (staged slots tb, tb + step, ...) into acc / at.  ALL: every slot lies below t1; else
            // a slot beyond re-reads the group's element tb, which a maximum does not notice and a sum discards by a select.
            // Positions (FIND): kFull, by the full rule of replaces(); kFirst, by "larger than all before" -- one comparison,
            // one maximum and one select per message where the rule takes a dozen instructions -- which agrees with it when
            // positions ascend along the walk, except for features with a NaN or with nothing above -inf (the caller
            // mends them); kNaNs, the earliest NaN's position only.  copy_u max with positions, 12.5M edges, F=100: 1130 us with
            // the rule on every message, 441 us by kFirst (11 TB/s of gathered rows); 114.8M edges, F=64: 4.1 -> 2.56 ms.
            auto batch = [&](auto all_tag, auto find_tag, int tb, int t1) {
                constexpr bool ALL = decltype(all_tag)::value;
                constexpr int FIND = decltype(find_tag)::value;
                float m[U][V];
                int stored[U];          // the element's position in the caller's edge order
#pragma unroll
                for (int k = 0; k < U; ++k) {
                    const int t = tb + k * step;
                    const int2 w = el[(ALL || t < t1) ? t : tb];
                    stored[k] = w.y;
                    float l[V], r[V];
                    if (SRC32)
                        load_operand<V, LC, LNT>(reinterpret_cast<const float *>(reinterpret_cast<const char *>(a.lhs) +
                                                                                 ((uint32_t)w.x + (uint32_t)fl * 4u)), l);
                    else if (kLhs) load_operand<V, LC, LNT>(row_at(lbase, l_on_e ? w.y : w.x, lbytes), l);
                    if (kRhs) load_operand<V, RC, RNT>(row_at(rbase, r_on_e ? w.y : w.x, rbytes), r);
#pragma unroll
                    for (int i = 0; i < V; ++i) {
                        m[k][i] = binary<OP>(kLhs ? l[i] : 0.f, kRhs ? r[i] : 0.f);
                        if (RED != FG_REDUCE_SUM) m[k][i] *= sign;
                    }
                }
#pragma unroll
                for (int k = 0; k < U; ++k) {
#pragma unroll
                    for (int i = 0; i < V; ++i) {
                        if (RED == FG_REDUCE_SUM) {
                            acc[i] += (ALL || tb + k * step < t1) ? m[k][i] : 0.f;
                        } else if (ARG && FIND == kNaNs) {
                            at[i] = m[k][i] != m[k][i] ? min(at[i], stored[k]) : at[i];
                        } else if (ARG && FIND == kFull) {
                            if (replaces<RED>(m[k][i], stored[k], acc[i], at[i])) { acc[i] = m[k][i]; at[i] = stored[k]; }
                        } else if (ARG) {
                            at[i] = !(m[k][i] <= acc[i]) ? stored[k] : at[i];
                            acc[i] = extreme<RED>(acc[i], m[k][i]);
                        } else {
                            acc[i] = extreme<RED>(acc[i], m[k][i]);
                        }
                    }
                }
            };
            auto walk = [&](auto find_tag) {
                if (decltype(find_tag)::value != kNaNs) {
#pragma unroll
                    for (int i = 0; i < V; ++i) { acc[i] = identity<RED>(); at[i] = INT_MAX; }
                }
                for (int64_t c0 = e0; c0 < e1; c0 += kStage) {
                    const int64_t c1 = min(c0 + kStage, e1);
                    int64_t base = staged_at;
                    if (!OWN && staged_at < 0) {
                        wave_lds_sync();          // the reads of what was staged before
                        stage(c0, (int)(c1 - c0));
                        base = c0;
                    }
                    const int t1 = (int)(c1 - base);       // positions in the staged window
                    int tb = (int)(c0 - base) + first;
                    // (a step of its own for the last slots costs registers, which the launches without positions
                    // and those of one feature per lane have no use for: 94 -> 106 and a wavefront per SIMD less, 600,000 edges on 300,000 nodes, F=64 u_mul_e
                    // 66 -> 89 us)
                    if constexpr (ARG && V == 4)
                        for (; tb + (U - 1) * step < t1; tb += step * U) batch(std::true_type{}, find_tag, tb, t1);
                    for (; tb < t1; tb += step * U) batch(std::false_type{}, find_tag, tb, t1);
                }
            };
            bool full_rule = ARG && !SRC32 && !a.ordered;      // whether the groups' results need it as well
            if constexpr (ARG) {
                if (full_rule) {
                    if constexpr (!SRC32) walk(std::integral_constant<int, kFull>{});
                } else {
                    walk(std::integral_constant<int, kFirst>{});
                    // Nothing above -inf though the group had elements: the first of them.  12.5M edges, F=64 / 100 / 256, 97 %
                    // of the messages -inf: 823 / 1277 / 2152 us with such rows walked again by the full rule, 281 / 451 /
                    // 1040 so (no -inf: 285 / 454 / 1032).
                    bool none = false, nan = false;
#pragma unroll
                    for (int i = 0; i < V; ++i) { none = none || at[i] == INT_MAX; nan = nan || acc[i] != acc[i]; }
                    if (none && e0 + first < e1) {
                        const int head = PART ? a.edge_pos[e0 + first] : (int)(e0 + first);
#pragma unroll
                        for (int i = 0; i < V; ++i) at[i] = at[i] == INT_MAX ? head : at[i];
                    }
                    // A NaN: its features' positions by a second walk.  1 % of the messages NaN, so that nearly every row has
                    // one: 826 / 1516 / 2814 us with the full rule, 460 / 806 / 1800 so (the full rule alone, as the only
                    // walk: 682 / 1296 / 2419; 1M edges on 200,000 nodes, F=256: 425, 327, 278).
                    full_rule = __any(nan);              // uniform over the wavefront
                    if (full_rule) {
#pragma unroll
                        for (int i = 0; i < V; ++i) at[i] = acc[i] != acc[i] ? INT_MAX : at[i];
                        walk(std::integral_constant<int, kNaNs>{});
                    }
                }
            } else {
                walk(std::integral_constant<int, kFirst>{});
            }
            if (ARG && !full_rule) {
                // no NaN anywhere: the groups' largest value first, then the earliest position that has it
                float best[V];
#pragma unroll
                for (int i = 0; i < V; ++i) best[i] = acc[i];
                for (int off = L; off < lanes; off <<= 1)
#pragma unroll
                    for (int i = 0; i < V; ++i) best[i] = extreme<RED>(best[i], __shfl_xor(best[i], off));
#pragma unroll
                for (int i = 0; i < V; ++i) { at[i] = acc[i] == best[i] ? at[i] : INT_MAX; acc[i] = best[i]; }
                for (int off = L; off < lanes; off <<= 1)
#pragma unroll
                    for (int i = 0; i < V; ++i) at[i] = min(at[i], __shfl_xor(at[i], off));
            } else
            for (int off = L; off < lanes; off <<= 1) {
#pragma unroll
                for (int i = 0; i < V; ++i) {
                    const float o = __shfl_xor(acc[i], off);
                    if (RED == FG_REDUCE_SUM) acc[i] += o;
                    else if (ARG) {
                        const int oa = __shfl_xor(at[i], off);
                        if (replaces<RED>(o, oa, acc[i], at[i])) { acc[i] = o; at[i] = oa; }
                    } else acc[i] = extreme<RED>(acc[i], o);
                }
            }
            if (mine && first == 0 && active) {
                const bool empty = e1 <= e0;
                const float scale = (done && a.row_scale) ? a.row_scale[v] : 1.f;
#pragma unroll
                for (int i = 0; i < V; ++i) {
                    if (RED != FG_REDUCE_SUM) acc[i] *= sign;
                    acc[i] = (RED != FG_REDUCE_SUM && empty && final) ? 0.f : acc[i];
                    if (done && a.row_scale) acc[i] *= scale;
                    if (ARG) at[i] = (at[i] == INT_MAX) ? -1 : at[i];
                }
                if (V == 4) {
                    *reinterpret_cast<fg::Words4<float> *>(dst_v + fc) = {{acc[0], acc[1 % V], acc[2 % V], acc[3 % V]}};
                    if (ARG) *reinterpret_cast<fg::Words4<int32_t> *>(dst_a + fc) = {{at[0], at[1 % V], at[2 % V], at[3 % V]}};
                } else {
                    dst_v[fc] = acc[0];
                    if (ARG) dst_a[fc] = at[0];
                }
            }
        }
    };

    if (it.info < 0) {
        const int nrows = -it.info;
        const bool fits = it.len <= kStage;       // always, for an item of several rows
        if (fits) stage(it.start, it.len);
        // as many rows at a time as there are, if the groups suffice
        int share = 1;
        while (share < G && share * nrows < a.spread * G) share *= 2;
        if (fits && share < G) {
            for (int q0 = 0; q0 < nrows; q0 += G / share) {
                const int q = q0 + g / share;
                const bool mine = q < nrows;
                const int v = it.row + min(q, nrows - 1);
                const int64_t e0 = pos_p[v], e1 = mine ? pos_p[v + 1] : e0;
                reduce_range(std::true_type{}, share, mine, e0, e1, it.start, v, out_p + (int64_t)v * F,
                             ARG ? arg_p + (int64_t)v * F : nullptr, final);
            }
            return;
        }
        for (int q = 0; q < nrows; ++q) {
            const int v = it.row + q;
            const int64_t e0 = pos_p[v], e1 = pos_p[v + 1];
            reduce_range(std::false_type{}, G, true, e0, e1, fits ? (int64_t)it.start : -1, v, out_p + (int64_t)v * F,
                         ARG ? arg_p + (int64_t)v * F : nullptr, final);
        }
        return;
    }
    reduce_range(std::false_type{}, G, true, it.start, (int64_t)it.start + it.len, -1, it.row, partial_p + (int64_t)it.info * F,
                 ARG ? partial_arg_p + (int64_t)it.info * F : nullptr, false);
}

// The pieces of a split row, combined in stored order.
// partial_stride / out_stride: per source partition (0 with one partition); the split segment's partition is fx.part.
template <int RED, bool ARG>
__global__ __launch_bounds__(256) void gspmm_bcast_fixup_kernel(const Fixup *fixups, int64_t n_fixups, const float *partial,
                                                                const int32_t *partial_arg, const float *row_scale,
                                                                float *out, int32_t *arg, int F, int64_t partial_stride,
                                                                int64_t out_stride) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n_fixups * F) return;
    const Fixup fx = fixups[t / F];
    const int f = (int)(t % F);
    const int64_t from = fx.part * partial_stride, to = fx.part * out_stride;
    float acc = identity<RED>();
    int at = INT_MAX;
    const int64_t first = from + (int64_t)fx.slot0 * F + f;
    struct Piece { float m; int at; };
    fg::each_piece(0, fx.n_pieces, [&](int p) { return Piece{partial[first + (int64_t)p * F], ARG ? partial_arg[first + (int64_t)p * F] : 0}; },
                   [&](int p, const Piece &c) {
        if (RED == FG_REDUCE_SUM) acc = p == 0 ? c.m : acc + c.m;
        else if (ARG) { if (c.at >= 0 && replaces<RED>(c.m, c.at, acc, at)) { acc = c.m; at = c.at; } }
        else acc = extreme<RED>(acc, c.m);
    });
    if (row_scale) acc *= row_scale[fx.row];
    out[to + (int64_t)fx.row * F + f] = acc;
    if (ARG) arg[to + (int64_t)fx.row * F + f] = (at == INT_MAX) ? -1 : at;
}

// out[v, f] = the partitions' results for row v combined in partition order (buf[p * buf_stride + v * F + f], positions abuf likewise, with -1
// for "none"); a row without elements in any partition gives 0 for max / min; rows are scaled here.
template <int RED, bool ARG>
__global__ __launch_bounds__(256) void gspmm_bcast_combine_kernel(const float *buf, const int32_t *abuf, const int32_t *pos,
                                                                  int n_parts, int64_t pos_stride, int64_t buf_stride,
                                                                  int64_t n_rows, int F, const float *row_scale, float *out,
                                                                  int32_t *arg) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n_rows * F) return;
    const int64_t v = t / F;
    float acc = identity<RED>();
    int at = INT_MAX;
    bool any = false;
    for (int p = 0; p < n_parts; ++p) {
        const float m = buf[p * buf_stride + t];
        if (RED == FG_REDUCE_SUM) acc = p == 0 ? m : acc + m;
        else {
            any = any || pos[p * pos_stride + v + 1] > pos[p * pos_stride + v];
            if (ARG) {
                const int am = abuf[p * buf_stride + t];
                if (am >= 0 && replaces<RED>(m, am, acc, at)) { acc = m; at = am; }
            } else acc = extreme<RED>(acc, m);
        }
    }
    if (RED != FG_REDUCE_SUM && !any) acc = 0.f;
    if (row_scale) acc *= row_scale[v];
    out[t] = acc;
    if (ARG) arg[t] = (at == INT_MAX) ? -1 : at;
}

// vec: 0 = one feature per lane; else 4 per lane with (lhs, rhs) read as 1 = (consecutive, consecutive),
// 2 = (consecutive, one value), 3 = (one value, consecutive); lnt / rnt: that operand streams from the stored elements
template <int OP, int RED, bool ARG, bool PART>
void launch_spmm_variant(int vec, bool lnt, bool rnt, dim3 grid, hipStream_t st, const GenArgs &a) {
    constexpr int USES = (kUsesLhs<OP> ? 1 : 0) | (kUsesRhs<OP> ? 2 : 0);
#define FG_GO(V, LC, RC, LNT, RNT) \
    hipLaunchKernelGGL((gspmm_bcast_kernel<OP, RED, ARG, V, LC, RC, LNT, RNT, PART>), grid, dim3(kBlock), 0, st, a)
    if (vec == 0) { FG_GO(1, true, true, false, false); return; }
    const bool lc = vec != 3, rc = vec != 2;
    lnt = lnt && lc; rnt = rnt && rc;
    if constexpr (OP == FG_BIN_COPY_LHS && ARG) {
        if (a.src32 && a.ordered && lc) {
            if (a.sign > 0) hipLaunchKernelGGL((gspmm_bcast_kernel<OP, RED, ARG, 4, true, true, false, false, PART, true, 1>), grid, dim3(kBlock), 0, st, a);
            else hipLaunchKernelGGL((gspmm_bcast_kernel<OP, RED, ARG, 4, true, true, false, false, PART, true, -1>), grid, dim3(kBlock), 0, st, a);
            return;
        }
    }
    if constexpr (USES == 1) {             // the right operand is not read: one instantiation stands for all its modes
        if (!lc) FG_GO(4, false, true, false, false);
        else if (lnt) FG_GO(4, true, true, true, false);
        else FG_GO(4, true, true, false, false);
    } else if constexpr (USES == 2) {
        if (!rc) FG_GO(4, true, false, false, false);
        else if (rnt) FG_GO(4, true, true, false, true);
        else FG_GO(4, true, true, false, false);
    } else {
        if (lc && rc) {
            if (lnt && rnt) FG_GO(4, true, true, true, true);
            else if (lnt) FG_GO(4, true, true, true, false);
            else if (rnt) FG_GO(4, true, true, false, true);
            else FG_GO(4, true, true, false, false);
        } else if (lc) {
            if (lnt) FG_GO(4, true, false, true, false);
            else FG_GO(4, true, false, false, false);
        } else {
            if (rnt) FG_GO(4, false, true, false, true);
            else FG_GO(4, false, true, false, false);
        }
    }
#undef FG_GO
}
template <int OP, int RED, bool ARG>
void launch_spmm_ora(int vec, bool lnt, bool rnt, dim3 grid, hipStream_t st, const GenArgs &a) {
    if (a.n_parts > 1 || a.edge_pos) launch_spmm_variant<OP, RED, ARG, true>(vec, lnt, rnt, grid, st, a);
    else launch_spmm_variant<OP, RED, ARG, false>(vec, lnt, rnt, grid, st, a);
}
template <int OP>
void launch_spmm_o(int reduce, bool with_arg, int vec, bool lnt, bool rnt, dim3 grid, hipStream_t st, const GenArgs &a) {
    if (reduce == FG_REDUCE_SUM) launch_spmm_ora<OP, FG_REDUCE_SUM, false>(vec, lnt, rnt, grid, st, a);
    else if (with_arg) launch_spmm_ora<OP, FG_REDUCE_MAX, true>(vec, lnt, rnt, grid, st, a);       // max, or min by a.sign
    else launch_spmm_ora<OP, FG_REDUCE_MAX, false>(vec, lnt, rnt, grid, st, a);
}
void launch_spmm(int op, int reduce, bool with_arg, int vec, bool lnt, bool rnt, dim3 grid, hipStream_t st, const GenArgs &a) {
    switch (op) {
        case FG_BIN_ADD: launch_spmm_o<FG_BIN_ADD>(reduce, with_arg, vec, lnt, rnt, grid, st, a); break;
        case FG_BIN_SUB: launch_spmm_o<FG_BIN_SUB>(reduce, with_arg, vec, lnt, rnt, grid, st, a); break;
        case FG_BIN_MUL: launch_spmm_o<FG_BIN_MUL>(reduce, with_arg, vec, lnt, rnt, grid, st, a); break;
        case FG_BIN_DIV: launch_spmm_o<FG_BIN_DIV>(reduce, with_arg, vec, lnt, rnt, grid, st, a); break;
        case FG_BIN_COPY_LHS: launch_spmm_o<FG_BIN_COPY_LHS>(reduce, with_arg, vec, lnt, rnt, grid, st, a); break;
        default: launch_spmm_o<FG_BIN_COPY_RHS>(reduce, with_arg, vec, lnt, rnt, grid, st, a); break;
    }
}

// How one operand can be read when a lane holds 4 consecutive output features: 1 = 4 consecutive features by one
// 128-bit load, 2 = one feature 4 times, 0 = neither (scalar kernel).  Without an offset array the operand has the
// output's layout, and an operand of one feature repeats it; with one, the caller's flags say which pattern every aligned group of 4
// follows, which holds for every lane's group where F is a multiple of 4.
int vector_mode(bool used, int len, const int32_t *off, int F, int flags, int vec_flag, int splat_flag) {
    if (!used || !off) return 1;
    if (len == 1) return 2;
    if (F % 4 != 0) return 0;
    return (flags & vec_flag) ? 1 : (flags & splat_flag) ? 2 : 0;
}
// The launchers' `vec` from the two operands' modes (0: scalar kernel).
int vector_variant(bool can_vec, int lmode, int rmode) {
    if (!can_vec || !lmode || !rmode) return 0;
    if (lmode == 1 && rmode == 1) return 1;
    if (lmode == 1 && rmode == 2) return 2;
    if (lmode == 2 && rmode == 1) return 3;
    return 0;       // both operands repeat one value over every group of 4: nothing to gain
}

int lanes_for(int F) {
    int L = 1;
    while (L < F && L < 64) L <<= 1;
    return L;
}

// rows: how many rows the operand has in this call (an operand without rows may be a null pointer)
int check_operand(const char *name, bool used, const float *p, int64_t rows, int len, int target, bool allow_v) {
    if (!used) return FG_OK;
    if (!p && rows > 0) return fail(FG_ERR_ARG, "%s is null", name);
    if (len < 1) return fail(FG_ERR_SHAPE, "%s feature length must be positive, got %d", name, len);
    if (!(target == FG_TARGET_U || target == FG_TARGET_E || (allow_v && target == FG_TARGET_V)))
        return fail(FG_ERR_ARG, "%s target %d is not valid here", name, target);
    return FG_OK;
}

// Scratch of one call, in floats: per partition the pieces of its split rows ([slot][F], rounded up to 16 bytes) and,
// with several partitions, a buffer of [n_dst][F] results; the selected positions, when wanted, take as much again.
struct BcastScratch {
    size_t pieces = 0;      // per partition
    size_t buffers = 0;     // per partition (0 with one partition)
    size_t half = 0;        // all partitions' values; the positions follow
    size_t total = 0;
};
BcastScratch bcast_scratch(const fg_spmm_plan *pl, int F, bool with_arg) {
    BcastScratch b;
    const size_t P = (size_t)pl->num_col_partitions;
    b.pieces = (((size_t)pl->max_slots_in_partition * (size_t)F) + 3) & ~(size_t)3;
    b.buffers = P > 1 ? (((size_t)pl->n_dst * (size_t)F) + 3) & ~(size_t)3 : 0;
    b.half = P * (b.pieces + b.buffers);
    b.total = with_arg ? 2 * b.half : b.half;
    return b;
}
constexpr size_t kMaxBufferBytes = (size_t)8 << 30;     // all partitions' result buffers together

// ---- gradient of a max / min aggregation ------------------------------------------------------------
//
// Every result out[v, f] is one message, the one at stored position arg[v, f] (-1: none), so its gradient goes to that
// element's two operands, one launch per operand.  What bounds the launch is not the 8 bytes per result that it reads but
// float atomics on scattered addresses (about 24 G a second, fewer where they meet: the source with a feature's largest
// value is selected by most of its neighbours).  A workgroup therefore takes kSelWidth features of up to kSelRows rows, adds
// up what goes to the same operand feature in a table in LDS, and only then adds to memory; what finds its slot taken
// by another address goes to memory at once.  Few features and many rows, because equal addresses share their feature.
// 58,000 nodes, F=100, normal features, 12.5M / 0.6M edges: 331 / 300 us with every result added to memory directly,
// 268 / 250 us with 16 features x 256 rows, 128 / 240 us with 4 x 8192 (2 x 8192: 152 / 246).
//
// Without the table (TABLE false: neighbouring lanes take neighbouring features of a row, and nothing is combined) where few
// results can meet: rows of up to kSelFewEdges elements on average with operands
// that are not broadcast, or UNIQUE, an operand on the edges without an offset array,
// whose every feature is one row's and is added to without atomics; a broadcast operand of such rows keeps the table, by whole
// rows.  Both gradients, with 4 x 8192 always -> now: 500,000 rows of 2, F=64 u_add_e 2116 -> 415 us, u_mul_e with 4 weights
// per edge 2105 -> 548; maximum of the sources alone 1065 -> 224 (5 elements per row, with the table 274).
constexpr int kSelWidth = 4, kSelRows = 8192, kSelLogSlots = 13, kSelSlots = 1 << kSelLogSlots, kSelThreads = 1024, kSelUnroll = 4;
constexpr int kSelFewEdges = 4;
enum { FG_SEL_PLUS, FG_SEL_MINUS, FG_SEL_TIMES_OTHER, FG_SEL_OVER_OTHER, FG_SEL_DENOMINATOR };
struct SelectArgs {
    const int32_t *arg, *col;
    int64_t n_dst;
    const float *own, *other, *dout;        // the operand whose gradient is formed, and the other one (values read as `kind` needs)
    const int32_t *own_off, *other_off;
    int own_len, other_len;
    int own_target, other_target;
    float *grad;
    int F, kind;
    int width, rows;                        // features and rows per workgroup
};
template <bool TABLE, bool UNIQUE>
__global__ __launch_bounds__(kSelThreads) void gspmm_select_backward_kernel(const SelectArgs a) {
    __shared__ uint32_t s_key[TABLE ? kSelSlots : 1];   // operand feature + 1; 0: free
    __shared__ float s_sum[TABLE ? kSelSlots : 1];
    if constexpr (TABLE) {
        for (int i = threadIdx.x; i < kSelSlots; i += kSelThreads) { s_key[i] = 0; s_sum[i] = 0.f; }
        __syncthreads();
    }
    const int f_tiles = (a.F + a.width - 1) / a.width;
    const int f = (int)(blockIdx.x % (unsigned)f_tiles) * a.width + (int)(threadIdx.x % (unsigned)a.width);
    const int64_t v0 = (int64_t)(blockIdx.x / (unsigned)f_tiles) * a.rows;
    const int64_t v1 = min(v0 + a.rows, a.n_dst);
    const int rows = kSelThreads / a.width;         // rows per step of the workgroup
    const bool on = f < a.F && (int)(threadIdx.x / (unsigned)a.width) < rows;
    const int fo = on ? (a.own_off ? a.own_off[f] : f) : 0;
    const int fx = on ? (a.other_off ? a.other_off[f] : f) : 0;
    const bool reads_other = a.kind >= FG_SEL_TIMES_OTHER;
    for (int64_t v = v0 + threadIdx.x / (unsigned)a.width; v < v1 && on; v += (int64_t)rows * kSelUnroll) {
        int e[kSelUnroll];
        float d[kSelUnroll];
        int64_t u[kSelUnroll];
#pragma unroll
        for (int k = 0; k < kSelUnroll; ++k) {
            const int64_t vk = v + (int64_t)rows * k;
            const int64_t t = min(vk, v1 - 1) * a.F + f;
            const int at = a.arg[t];
            e[k] = vk < v1 ? at : -1;
            d[k] = a.dout[t];
        }
#pragma unroll
        for (int k = 0; k < kSelUnroll; ++k) u[k] = a.col[max(e[k], 0)];
#pragma unroll
        for (int k = 0; k < kSelUnroll; ++k) {
            if (e[k] < 0) continue;
            const int64_t to = (a.own_target == FG_TARGET_U ? u[k] : (int64_t)e[k]) * a.own_len + fo;
            float g = a.kind == FG_SEL_MINUS ? -d[k] : d[k];
            if (reads_other) {
                const float x = a.other[(a.other_target == FG_TARGET_U ? u[k] : (int64_t)e[k]) * a.other_len + fx];
                if (a.kind == FG_SEL_TIMES_OTHER) g = d[k] * x;
                else if (a.kind == FG_SEL_OVER_OTHER) g = d[k] / x;
                else { const float r = a.own[to]; g = -d[k] * x / (r * r); }
            }
            if (UNIQUE) { a.grad[to] += g; continue; }
            if (!TABLE || (uint64_t)to >= 0xffffffffull) { unsafeAtomicAdd(a.grad + to, g); continue; }
            const uint32_t key = (uint32_t)to + 1u;
            const uint32_t slot = (key * 2654435761u) >> (32 - kSelLogSlots);
            const uint32_t was = atomicCAS(&s_key[slot], 0u, key);
            if (was == 0u || was == key) atomicAdd(&s_sum[slot], g);
            else unsafeAtomicAdd(a.grad + to, g);
        }
    }
    if constexpr (TABLE) {
        __syncthreads();
        for (int i = threadIdx.x; i < kSelSlots; i += kSelThreads)
            if (s_key[i]) unsafeAtomicAdd(a.grad + (s_key[i] - 1u), s_sum[i]);
    }
}

// ---- SDDMM ------------------------------------------------------------------------------------------

struct EdgeArgs {
    const int32_t *lhs_index, *rhs_index;   // per edge: the operand's row (col for u, row for v; any valid array for e)
    int64_t n_edges;
    const float *lhs, *rhs;
    const int32_t *lhs_off, *rhs_off;
    int lhs_len, rhs_len;
    int lhs_target, rhs_target;
    float *out;
    int F, L, R;
    uint32_t vec_magic;      // ceil(2^32 / vectors of an output row)
};

// 64 edges per wavefront, U steps of 64 lanes * V floats in flight, no branch between the loads of a step; the edges'
// index words come in by one coalesced load each and go to the lanes by shuffles, so no gather waits for a load of its
// own index.  Bound by the stream of results (and of an operand on the edges) to memory.
//   FLAT : no operand has an offset array: the wavefront's edges * F / V vectors are dealt to the lanes in order, whatever
//          F; a lane finds its edge by one high multiplication (64 * (F / V)^2 < 2^32).
//   else : a group of L lanes (the power of two not below F / V, at most 64) takes an edge.
// u_mul_v on 12.5 M edges, F = 64, within a step of 3 such sweeps: 951 -> 741 us (3.2 GB written, 4.3 TB/s).
template <int OP, int V, bool LC, bool RC, bool FLAT, int U>
__global__ __launch_bounds__(kBlock) void gsddmm_bcast_kernel(const EdgeArgs a) {
    const int lane = threadIdx.x & 63;
    const int64_t wave_id = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int L = a.L, G = 64 / L;
    const int FV = (a.F + V - 1) / V;
    const int64_t e0 = wave_id * 64;
    if (e0 >= a.n_edges) return;
    const int n = (int)min((int64_t)64, a.n_edges - e0);
    const bool l_on_e = a.lhs_target == FG_TARGET_E, r_on_e = a.rhs_target == FG_TARGET_E;
    const int il_all = kUsesLhs<OP> ? a.lhs_index[e0 + min(lane, n - 1)] : 0, ir_all = kUsesRhs<OP> ? a.rhs_index[e0 + min(lane, n - 1)] : 0;
    // U edges t[] (valid where ok[]) at the lane's output features fc[], operand features fl[] and fr[]
    auto step = [&](const int (&t)[U], const bool (&ok)[U], const int (&fc)[U], const int (&fl)[U], const int (&fr)[U]) {
        float m[U][V];
#pragma unroll
        for (int k = 0; k < U; ++k) {
            const int64_t ec = e0 + t[k];
            const int64_t il = kUsesLhs<OP> ? (int64_t)__shfl(il_all, t[k]) : 0, ir = kUsesRhs<OP> ? (int64_t)__shfl(ir_all, t[k]) : 0;
            const float *lp = a.lhs + (l_on_e ? ec : il) * a.lhs_len;
            const float *rp = a.rhs + (r_on_e ? ec : ir) * a.rhs_len;
            if (OP == FG_BIN_DOT) {
                const float *l = lp + (int64_t)fl[k] * a.R, *r = rp + (int64_t)fr[k] * a.R;
                float sum = 0.f;
                for (int i = 0; i < a.R; ++i) sum += l[i] * r[i];
                m[k][0] = sum;
            } else {
                float l[V], r[V];
                if (kUsesLhs<OP>) load_operand<V, LC>(lp + fl[k], l);
                if (kUsesRhs<OP>) load_operand<V, RC>(rp + fr[k], r);
#pragma unroll
                for (int i = 0; i < V; ++i) m[k][i] = binary<OP>(kUsesLhs<OP> ? l[i] : 0.f, kUsesRhs<OP> ? r[i] : 0.f);
            }
        }
#pragma unroll
        for (int k = 0; k < U; ++k) {
            if (!ok[k]) continue;
            float *o = a.out + (e0 + t[k]) * a.F + fc[k];
            if (V == 4) { nt_f4 t4; t4.x = m[k][0]; t4.y = m[k][1 % V]; t4.z = m[k][2 % V]; t4.w = m[k][3 % V]; __builtin_nontemporal_store(t4, reinterpret_cast<nt_f4 *>(o)); }
            else *o = m[k][0];
        }
    };
    int t[U], fc[U], fl[U], fr[U];
    bool ok[U];
    if constexpr (FLAT) {
        const int total = n * FV;
        for (int p0 = lane; p0 - lane < total; p0 += 64 * U) {
#pragma unroll
            for (int k = 0; k < U; ++k) {
                ok[k] = p0 + 64 * k < total;
                const uint32_t p = ok[k] ? p0 + 64 * k : total - 1;
                t[k] = FV == 1 ? (int)p : (int)__umulhi(p, a.vec_magic);
                fc[k] = fl[k] = fr[k] = first_feature<V>((int)p - t[k] * FV, a.F);
            }
            step(t, ok, fc, fl, fr);
        }
    } else {
        const int g = lane / L, li = lane % L;
        for (int f0 = 0; f0 < FV; f0 += L) {
            const bool in_row = f0 + li < FV;
            const int f = first_feature<V>(in_row ? f0 + li : FV - 1, a.F);
            const int l = kUsesLhs<OP> ? (a.lhs_off ? a.lhs_off[f] : f) : 0;
            const int r = kUsesRhs<OP> ? (a.rhs_off ? a.rhs_off[f] : f) : 0;
            for (int tb = 0; tb < n; tb += G * U) {
#pragma unroll
                for (int k = 0; k < U; ++k) {
                    const int at = tb + k * G + g;
                    ok[k] = in_row && at < n;
                    t[k] = min(at, n - 1);
                    fc[k] = f; fl[k] = l; fr[k] = r;
                }
                step(t, ok, fc, fl, fr);
            }
        }
    }
}

// Dot products over a contracted axis of R floats (R a multiple of 4, operands 16-byte aligned): a group of L lanes
// (4 L >= R up to 64 lanes) reads the two operands' R floats of one (edge, output feature) pair with 128-bit loads and
// adds its products up with shuffles; the 64 / L groups take different pairs of the wavefront's 64 edges, U pairs in
// flight each.  (gsddmm_bcast_kernel<FG_BIN_DOT> walks the axis lane by lane and serves every other shape.)
template <int L>
__global__ __launch_bounds__(kBlock) void gsddmm_dot_kernel(const EdgeArgs a) {
    constexpr int G = 64 / L, U = 4;
    const int lane = threadIdx.x & 63, g = lane / L, li = lane % L;
    const int64_t wave_id = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int64_t e0 = wave_id * 64;
    if (e0 >= a.n_edges) return;
    const int n_e = (int)min((int64_t)64, a.n_edges - e0);
    const int F = a.F, R = a.R;
    const int n_pairs = n_e * F;
    const bool l_on_e = a.lhs_target == FG_TARGET_E, r_on_e = a.rhs_target == FG_TARGET_E;
    for (int pb = g; pb < n_pairs; pb += G * U) {
        float s[U];
        bool ok[U];
#pragma unroll
        for (int k = 0; k < U; ++k) {
            const int p = pb + k * G;
            ok[k] = p < n_pairs;
            const int pc = ok[k] ? p : pb;
            const int64_t e = e0 + pc / F;
            const int f = pc % F;
            const int64_t il = a.lhs_index[e], ir = a.rhs_index[e];
            const int fl = a.lhs_off ? a.lhs_off[f] : f, fr = a.rhs_off ? a.rhs_off[f] : f;
            const float *lp = a.lhs + (l_on_e ? e : il) * a.lhs_len + (int64_t)fl * R;
            const float *rp = a.rhs + (r_on_e ? e : ir) * a.rhs_len + (int64_t)fr * R;
            float acc = 0.f;
            for (int c = li * 4; c < R; c += L * 4) {
                const float4 x = *reinterpret_cast<const float4 *>(lp + c), y = *reinterpret_cast<const float4 *>(rp + c);
                acc += (x.x * y.x + x.y * y.y) + (x.z * y.z + x.w * y.w);
            }
            s[k] = acc;
        }
#pragma unroll
        for (int k = 0; k < U; ++k) {
            for (int off = 1; off < L; off <<= 1) s[k] += __shfl_xor(s[k], off);
            const int p = pb + k * G;
            if (li == 0 && ok[k]) a.out[(e0 + p / F) * F + p % F] = s[k];
        }
    }
}

template <int OP>
void launch_sddmm(int vec, dim3 grid, hipStream_t st, EdgeArgs a) {
    const int FV = vec ? (a.F + 3) / 4 : a.F;
    a.vec_magic = FV > 1 ? (uint32_t)((0x100000000ull + FV - 1) / FV) : 0;
    const bool flat = !(kUsesLhs<OP> && a.lhs_off) && !(kUsesRhs<OP> && a.rhs_off) && FV < 8192;
    // a wavefront's 64 edges fill eight steps; 3 M edges, u_add_v with eight / four: F=4 35 / 25 us, F=8 38 / 29, F=16 49 / 43
    const bool wide = FV > 4;
#define FG_GO(V, LC, RC, FLAT) \
    do { \
        if (wide) hipLaunchKernelGGL((gsddmm_bcast_kernel<OP, V, LC, RC, FLAT, 8>), grid, dim3(kBlock), 0, st, a); \
        else hipLaunchKernelGGL((gsddmm_bcast_kernel<OP, V, LC, RC, FLAT, 4>), grid, dim3(kBlock), 0, st, a); \
    } while (0)
    if (vec == 1 && flat) FG_GO(4, true, true, true);
    else if (vec == 1) FG_GO(4, true, true, false);
    else if (vec == 2) FG_GO(4, true, false, false);
    else if (vec == 3) FG_GO(4, false, true, false);
    else if (flat) FG_GO(1, true, true, true);
    else hipLaunchKernelGGL((gsddmm_bcast_kernel<OP, 1, true, true, false, 4>), grid, dim3(kBlock), 0, st, a);
#undef FG_GO
}

}  // namespace

namespace fg {
int gspmm_bcast_scratch_need(const fg_spmm_plan *pl, int F, bool with_arg, ScratchNeed *need) {
    if (F < 1) return fail(FG_ERR_SHAPE, "feature length must be positive, got %d", F);
    const BcastScratch b = bcast_scratch(pl, F, with_arg);
    if ((size_t)pl->num_col_partitions * b.buffers * 4 * (with_arg ? 2 : 1) > kMaxBufferBytes)
        return fail(FG_ERR_SHAPE, "%d source partitions of [%lld, %d] results need more than 8 GiB of buffers; use fewer partitions",
                    pl->num_col_partitions, (long long)pl->n_dst, F);
    need->partial = b.total;
    need->tiled = 0;
    return FG_OK;
}
}  // namespace fg

namespace {

// pos / idx: indptr / indices of the CSR arrays with one partition, else the partitioned layout's position and local
// column arrays; edge_pos (required with several partitions): the row of each element in the edge operands.
int gspmm_bcast_run(fg_spmm_plan *pl, const int32_t *pos_dev, const int32_t *idx_dev, const int32_t *edge_pos_dev, int op,
                    int reduce, const float *lhs_dev, int lhs_target, int lhs_len, const int32_t *lhs_off_dev,
                    const float *rhs_dev, int rhs_target, int rhs_len, const int32_t *rhs_off_dev, int flags,
                    const float *row_scale_dev, float *out_dev, int32_t *arg_dev, int out_len, void *stream) {
    if (op < FG_BIN_ADD || op > FG_BIN_COPY_RHS) return fail(FG_ERR_ARG, "unknown message operator %d", op);
    if (reduce != FG_REDUCE_SUM && reduce != FG_REDUCE_MAX && reduce != FG_REDUCE_MIN)
        return fail(FG_ERR_ARG, "unknown reduce op %d", reduce);
    if (arg_dev && reduce == FG_REDUCE_SUM) return fail(FG_ERR_ARG, "positions of the selected elements exist for max / min only");
    fg::ScratchNeed need;
    if (int rc = fg::gspmm_bcast_scratch_need(pl, out_len, arg_dev != nullptr, &need)) return rc;
    const int P = pl->num_col_partitions;
    const bool uses_l = op != FG_BIN_COPY_RHS, uses_r = op != FG_BIN_COPY_LHS;
    if (int rc = check_operand("lhs", uses_l, lhs_dev, lhs_target == FG_TARGET_E ? pl->nnz : pl->n_src, lhs_len, lhs_target, false)) return rc;
    if (int rc = check_operand("rhs", uses_r, rhs_dev, rhs_target == FG_TARGET_E ? pl->nnz : pl->n_src, rhs_len, rhs_target, false)) return rc;
    if ((uses_l && !lhs_off_dev && lhs_len != out_len) || (uses_r && !rhs_off_dev && rhs_len != out_len))
        return fail(FG_ERR_SHAPE, "an operand without an offset array must have the output's feature length %d", out_len);
    if (pl->n_dst == 0) return FG_OK;
    if (!out_dev || !pos_dev || (pl->nnz > 0 && (!idx_dev || (P > 1 && !edge_pos_dev)))) return fail(FG_ERR_ARG, "null device pointer");
    if (int rc = fg::ensure_scratch(pl, need, stream)) return rc;
    hipStream_t st = (hipStream_t)stream;
    const BcastScratch b = bcast_scratch(pl, out_len, arg_dev != nullptr);
    const int lmode = vector_mode(uses_l, lhs_len, lhs_off_dev, out_len, flags, FG_BCAST_LHS_VEC4, FG_BCAST_LHS_SPLAT4);
    const int rmode = vector_mode(uses_r, rhs_len, rhs_off_dev, out_len, flags, FG_BCAST_RHS_VEC4, FG_BCAST_RHS_SPLAT4);
    const bool streams = (uses_l && lhs_target == FG_TARGET_E && lmode == 1) || (uses_r && rhs_target == FG_TARGET_E && rmode == 1);
    // An operand streamed from the edges in short rows of an odd length: one feature per lane, whose loads walk consecutive words (u_mul_e
    // sum, one / 4 features per lane, 20,000 rows of 200 elements F=9 / 13 / 17 52 / 67, 57 / 81, 99 / 98 us; 100,000 of 8 30 / 33, 31 / 37, 47 / 47).
    const bool short_odd = streams && out_len % 4 != 0 && out_len <= 16;
    const int vec = vector_variant(out_len >= 4 && !short_odd, lmode, rmode);
    const int V = vec ? 4 : 1;
    float *const values = pl->partial_dev;                                          // [P][pieces] then [P][buffers]
    int32_t *const positions = reinterpret_cast<int32_t *>(pl->partial_dev + b.half);
    float *const buf = values + (size_t)P * b.pieces;
    int32_t *const abuf = positions + (size_t)P * b.pieces;
    GenArgs a;
    a.items = pl->items_dev; a.n_items = pl->n_items;
    a.indptr = pos_dev; a.indices = idx_dev; a.indices16 = fg::narrow_indices(pl, idx_dev);
    a.lhs = lhs_dev; a.rhs = rhs_dev; a.lhs_off = lhs_off_dev; a.rhs_off = rhs_off_dev;
    a.lhs_len = lhs_len; a.rhs_len = rhs_len; a.lhs_target = lhs_target; a.rhs_target = rhs_target;
    a.sign = reduce == FG_REDUCE_MIN ? -1.f : 1.f;
    a.src32 = uses_l && lhs_target == FG_TARGET_U && (uint64_t)pl->n_src * (uint64_t)lhs_len * 4u < (1ull << 32);
    a.row_scale = P > 1 ? nullptr : row_scale_dev;
    a.out = P > 1 ? buf : out_dev;
    a.arg = P > 1 ? (arg_dev ? abuf : nullptr) : arg_dev;
    a.partial = values; a.partial_arg = positions;
    // Feature tiles of 64 floats over the workgroups (as for the weighted sum) when an operand is gathered from the
    // source nodes and the 128-bit paths apply: a partition's slice of a tile is what an L2 has to hold.
    // (Not with an operand streamed from the edges, which sets the time.  With positions of the selected elements for copies
    // only, in tiles that divide the 8 XCDs, from degree 32 on: below that a row's start and end cost each tile more than the
    // L2s gain.  copy_u max with its gradient, untiled -> tiled, F=128 / 256 / 512, 4M edges: degree 200 219 -> 210 / 415 -> 362 / 922 -> 682 us,
    // 80 384 -> 353 / 873 -> 724 / 1812 -> 1358, 40 (F=128 / 256) 723 -> 706 / 1491 -> 1394, 30 985 -> 974 / 1976 -> 1887 / 3919 -> 3780, 15 1857 -> 1859 / 3583 -> 3630 / 7087 -> 7231; 9M edges of
    // degree 15 4287 -> 4385 / 8284 -> 8528 / 16374 -> 16879; F=192 / 320 at degree 200 313 -> 338 / 605 -> 614.  Below 2^15 edges
    // launches are all there is, and either is the other's time.  u_add_e max, which instructions bound, 12.5M edges on 58,000 nodes 669 -> 683 / 1132 -> 1270 / 2573 -> 2403, 8M on 200,000 509 -> 549 / 1101 -> 1030 / 2320 -> 2198.)
    const bool gathers = (uses_l && lhs_target == FG_TARGET_U) || (uses_r && rhs_target == FG_TARGET_U);
    int T = (V == 4 && gathers && !streams && out_len >= 128 && out_len % 64 == 0) ? out_len / 64 : 1;
    if (arg_dev && !(op == FG_BIN_COPY_LHS && (T & (T - 1)) == 0 && pl->nnz >= 32 * pl->n_dst) && pl->nnz >= (1 << 15)) T = 1;
    a.n_tiles = T; a.tile_vecs = T > 1 ? 16 : (out_len + V - 1) / V;
    a.F = out_len; a.L = lanes_for(T > 1 ? 16 : (out_len + V - 1) / V);
    // Lane groups that hold several rows at once: see GenArgs.  Spread over as many groups as there are, rows take the fewest
    // steps; kept closer together, uneven rows leave fewer groups idle and streamed operands are read in longer runs.  1 / 2 / 4, us: copy_u max on 100,000 rows
    // of 40, F=4 44 / 58 / -, F=16 62 / 67 / -, F=32 87 / 82 / -; of 8, F=16 31 / 24 / -; u_mul_e sum with F edge features on rows of 8, F=8 34 / 28 / 30,
    // F=32 61 / 57 / 47, F=64 - / 79 / 76, of 16, F=16 64 / 52 / 55, F=32 89 / 79 / 72.  With a row either in one group or in all of them F=4 115, F=16 112 and 74,
    // F=32 115; u_mul_e F=8 98, F=16 91, F=32 56 and 79.
    a.spread = streams ? (out_len > 16 ? 4 : 2) : (out_len <= 8 ? 1 : 2);
    a.item_off = pl->item_off_dev; a.edge_pos = edge_pos_dev; a.n_parts = P; a.final = P == 1;
    a.ordered = !edge_pos_dev || (flags & FG_BCAST_EDGES_ASCEND) != 0;
    a.pos_stride = pl->n_dst + 1; a.col_width = (pl->n_src + P - 1) / P;
    a.out_stride = (int64_t)b.buffers; a.partial_stride = (int64_t)b.pieces;
    const int64_t blocks = ((pl->n_items + kWavesPerBlock - 1) / kWavesPerBlock) * T;
    if (blocks > 0x7fffffffLL) return fail(FG_ERR_SHAPE, "grid of %lld workgroups is too large", (long long)blocks);
    // an operand on the stored elements that is read with 128-bit loads streams past the caches
    const bool lnt = uses_l && lhs_target == FG_TARGET_E && lmode == 1, rnt = uses_r && rhs_target == FG_TARGET_E && rmode == 1;
    if (blocks > 0) launch_spmm(op, reduce, arg_dev != nullptr, vec, lnt, rnt, dim3((unsigned)blocks), st, a);
    const int which = reduce == FG_REDUCE_SUM ? 0 : (reduce == FG_REDUCE_MAX ? 1 : 3) + (arg_dev ? 1 : 0);
    if (pl->n_fixups > 0) {
        const int64_t threads = pl->n_fixups * (int64_t)out_len;
        const dim3 grid((unsigned)((threads + 255) / 256));
#define FG_FIXUP(RED, ARG) hipLaunchKernelGGL((gspmm_bcast_fixup_kernel<RED, ARG>), grid, dim3(256), 0, st, pl->fixups_dev, pl->n_fixups, \
                                              a.partial, a.partial_arg, a.row_scale, a.out, a.arg, out_len, a.partial_stride, a.out_stride)
        switch (which) {
            case 0: FG_FIXUP(FG_REDUCE_SUM, false); break;
            case 1: FG_FIXUP(FG_REDUCE_MAX, false); break;
            case 2: FG_FIXUP(FG_REDUCE_MAX, true); break;
            case 3: FG_FIXUP(FG_REDUCE_MIN, false); break;
            default: FG_FIXUP(FG_REDUCE_MIN, true); break;
        }
#undef FG_FIXUP
    }
    if (P > 1) {
        const int64_t threads = pl->n_dst * (int64_t)out_len;
        if ((threads + 255) / 256 > 0x7fffffffLL) return fail(FG_ERR_SHAPE, "output of %lld values is too large", (long long)threads);
        const dim3 grid((unsigned)((threads + 255) / 256));
#define FG_COMBINE(RED, ARG) hipLaunchKernelGGL((gspmm_bcast_combine_kernel<RED, ARG>), grid, dim3(256), 0, st, buf, abuf, pos_dev, P, \
                                                a.pos_stride, a.out_stride, pl->n_dst, out_len, row_scale_dev, out_dev, arg_dev)
        switch (which) {
            case 0: FG_COMBINE(FG_REDUCE_SUM, false); break;
            case 1: FG_COMBINE(FG_REDUCE_MAX, false); break;
            case 2: FG_COMBINE(FG_REDUCE_MAX, true); break;
            case 3: FG_COMBINE(FG_REDUCE_MIN, false); break;
            default: FG_COMBINE(FG_REDUCE_MIN, true); break;
        }
#undef FG_COMBINE
    }
    FG_HIP_TRY(hipGetLastError());
    return FG_OK;
}

}  // namespace

extern "C" int fg_gspmm_bcast_f32(fg_spmm_plan *pl, const int32_t *indptr_dev, const int32_t *indices_dev, int op,
                                  int reduce, const float *lhs_dev, int lhs_target, int lhs_len,
                                  const int32_t *lhs_off_dev, const float *rhs_dev, int rhs_target, int rhs_len,
                                  const int32_t *rhs_off_dev, int flags, const float *row_scale_dev, float *out_dev,
                                  int32_t *arg_dev, int out_len, void *stream) {
    if (!pl) return fail(FG_ERR_ARG, "plan is null");
    if (int drc = fg::check_device(pl)) return drc;
    if (pl->num_col_partitions != 1)
        return fail(FG_ERR_ARG, "fg_gspmm_bcast_f32 takes a plan with one column partition (fg_gspmm_bcast_dds_f32: several)");
    return gspmm_bcast_run(pl, indptr_dev, indices_dev, nullptr, op, reduce, lhs_dev, lhs_target, lhs_len, lhs_off_dev, rhs_dev,
                           rhs_target, rhs_len, rhs_off_dev, flags, row_scale_dev, out_dev, arg_dev, out_len, stream);
}

extern "C" int fg_gspmm_bcast_dds_f32(fg_spmm_plan *pl, const int32_t *s1_pos_dev, const int32_t *s1_idx_dev,
                                      const int32_t *edge_pos_dev, int op, int reduce, const float *lhs_dev, int lhs_target,
                                      int lhs_len, const int32_t *lhs_off_dev, const float *rhs_dev, int rhs_target,
                                      int rhs_len, const int32_t *rhs_off_dev, int flags, const float *row_scale_dev,
                                      float *out_dev, int32_t *arg_dev, int out_len, void *stream) {
    if (!pl) return fail(FG_ERR_ARG, "plan is null");
    if (int drc = fg::check_device(pl)) return drc;
    return gspmm_bcast_run(pl, s1_pos_dev, s1_idx_dev, edge_pos_dev, op, reduce, lhs_dev, lhs_target, lhs_len, lhs_off_dev, rhs_dev,
                           rhs_target, rhs_len, rhs_off_dev, flags, row_scale_dev, out_dev, arg_dev, out_len, stream);
}

extern "C" int fg_gspmm_select_backward_f32(const int32_t *arg_dev, const int32_t *col_dev, int64_t n_dst, int64_t n_edges, int op,
                                            const float *lhs_dev, int lhs_target, int lhs_len, const int32_t *lhs_off_dev,
                                            const float *rhs_dev, int rhs_target, int rhs_len, const int32_t *rhs_off_dev,
                                            const float *dout_dev, int out_len, float *dlhs_dev, float *drhs_dev, void *stream) {
    if (op < FG_BIN_ADD || op > FG_BIN_COPY_LHS) return fail(FG_ERR_ARG, "operator %d has no gradient here", op);
    if (n_dst < 0 || n_edges < 0) return fail(FG_ERR_ARG, "negative size");
    if (out_len < 1) return fail(FG_ERR_SHAPE, "feature length must be positive, got %d", out_len);
    const bool values = op == FG_BIN_MUL || op == FG_BIN_DIV, two = op != FG_BIN_COPY_LHS;
    if (!two && drhs_dev) return fail(FG_ERR_ARG, "a copy has one operand");
    if (lhs_len < 1 || (two && rhs_len < 1)) return fail(FG_ERR_SHAPE, "operand feature lengths must be positive");
    if ((!lhs_off_dev && lhs_len != out_len) || (two && !rhs_off_dev && rhs_len != out_len))
        return fail(FG_ERR_SHAPE, "an operand without an offset array must have the output's feature length %d", out_len);
    for (int target : {lhs_target, two ? rhs_target : lhs_target})
        if (target != FG_TARGET_U && target != FG_TARGET_E) return fail(FG_ERR_ARG, "operand target %d is not valid here", target);
    if (n_dst == 0 || n_edges == 0 || (!dlhs_dev && !drhs_dev)) return FG_OK;
    if (!arg_dev || !col_dev || !dout_dev || (values && (!lhs_dev || !rhs_dev))) return fail(FG_ERR_ARG, "null device pointer");
    SelectArgs a;
    a.arg = arg_dev; a.col = col_dev; a.n_dst = n_dst; a.dout = dout_dev; a.F = out_len;
    for (int side = 0; side < 2; ++side) {
        if (!(side ? drhs_dev : dlhs_dev)) continue;
        a.grad = side ? drhs_dev : dlhs_dev;
        a.own = side ? rhs_dev : lhs_dev; a.other = side ? lhs_dev : rhs_dev;
        a.own_off = side ? rhs_off_dev : lhs_off_dev; a.other_off = two ? (side ? lhs_off_dev : rhs_off_dev) : nullptr;
        a.own_len = side ? rhs_len : lhs_len; a.other_len = side ? lhs_len : rhs_len;
        a.own_target = side ? rhs_target : lhs_target; a.other_target = side ? lhs_target : rhs_target;
        a.kind = op == FG_BIN_MUL ? FG_SEL_TIMES_OTHER : op == FG_BIN_DIV ? (side ? FG_SEL_DENOMINATOR : FG_SEL_OVER_OTHER)
               : (op == FG_BIN_SUB && side) ? FG_SEL_MINUS : FG_SEL_PLUS;
        const bool unique = a.own_target == FG_TARGET_E && !a.own_off, few = n_edges <= kSelFewEdges * n_dst;
        const bool table = !unique && (!few || a.own_off);
        // few features where rows meet; else as many as make whole lines, in tiles of one size
        a.width = !table || few ? (out_len + (out_len + 255) / 256 - 1) / ((out_len + 255) / 256)
                : out_len >= kSelWidth ? kSelWidth : out_len == 1 ? 1 : 2;
        // fewer rows per workgroup where the launch would leave compute units without one
        a.rows = table && !few ? kSelRows : 2 * kSelUnroll * (kSelThreads / a.width);
        int64_t blocks;
        while ((blocks = ((n_dst + a.rows - 1) / a.rows) * ((out_len + a.width - 1) / a.width)) < 192 && a.rows > 512) a.rows /= 2;
        if (blocks > 0x7fffffffLL) return fail(FG_ERR_SHAPE, "grid of %lld workgroups is too large", (long long)blocks);
        const dim3 grid((unsigned)blocks), threads(kSelThreads);
        hipStream_t st = (hipStream_t)stream;
        if (unique) hipLaunchKernelGGL((gspmm_select_backward_kernel<false, true>), grid, threads, 0, st, a);
        else if (table) hipLaunchKernelGGL((gspmm_select_backward_kernel<true, false>), grid, threads, 0, st, a);
        else hipLaunchKernelGGL((gspmm_select_backward_kernel<false, false>), grid, threads, 0, st, a);
    }
    FG_HIP_TRY(hipGetLastError());
    return FG_OK;
}

extern "C" int fg_gsddmm_bcast_f32(const int32_t *row_dev, const int32_t *col_dev, int64_t n_edges, int op,
                                   const float *lhs_dev, int lhs_target, int lhs_len, const int32_t *lhs_off_dev,
                                   const float *rhs_dev, int rhs_target, int rhs_len, const int32_t *rhs_off_dev,
                                   int flags, float *out_dev, int out_len, int reduce_len, void *stream) {
    if (op < FG_BIN_ADD || op > FG_BIN_DOT) return fail(FG_ERR_ARG, "unknown edge operator %d", op);
    if (n_edges < 0) return fail(FG_ERR_ARG, "negative edge count");
    if (out_len < 1) return fail(FG_ERR_SHAPE, "feature length must be positive, got %d", out_len);
    const bool uses_l = op != FG_BIN_COPY_RHS, uses_r = op != FG_BIN_COPY_LHS;
    // with edges every operand has rows to read; without, nothing is read
    if (int rc = check_operand("lhs", uses_l, lhs_dev, n_edges, lhs_len, lhs_target, true)) return rc;
    if (int rc = check_operand("rhs", uses_r, rhs_dev, n_edges, rhs_len, rhs_target, true)) return rc;
    const int R = op == FG_BIN_DOT ? reduce_len : 1;
    if (R < 1) return fail(FG_ERR_SHAPE, "the contracted length must be positive, got %d", reduce_len);
    if (op == FG_BIN_DOT && (lhs_len % R != 0 || rhs_len % R != 0))
        return fail(FG_ERR_SHAPE, "operand lengths %d and %d are not multiples of the contracted length %d", lhs_len, rhs_len, R);
    if ((uses_l && !lhs_off_dev && lhs_len != (int64_t)out_len * R) || (uses_r && !rhs_off_dev && rhs_len != (int64_t)out_len * R))
        return fail(FG_ERR_SHAPE, "an operand without an offset array must have the output's feature length %d (times the contracted length)", out_len);
    if (n_edges == 0) return FG_OK;
    const bool any_u = (uses_l && lhs_target == FG_TARGET_U) || (uses_r && rhs_target == FG_TARGET_U);
    const bool any_v = (uses_l && lhs_target == FG_TARGET_V) || (uses_r && rhs_target == FG_TARGET_V);
    if (!out_dev || (any_u && !col_dev) || (any_v && !row_dev)) return fail(FG_ERR_ARG, "null device pointer");
    const int lmode = vector_mode(uses_l, lhs_len, lhs_off_dev, out_len, flags, FG_BCAST_LHS_VEC4, FG_BCAST_LHS_SPLAT4);
    const int rmode = vector_mode(uses_r, rhs_len, rhs_off_dev, out_len, flags, FG_BCAST_RHS_VEC4, FG_BCAST_RHS_SPLAT4);
    // results over an operand of theirs: no lane may read what another has written, as the two vectors that share features would
    const bool in_place = (uses_l && lhs_target == FG_TARGET_E && lhs_dev == out_dev) || (uses_r && rhs_target == FG_TARGET_E && rhs_dev == out_dev);
    const int vec = vector_variant(op != FG_BIN_DOT && out_len >= 4 && !(in_place && out_len % 4 != 0), lmode, rmode);
    const int V = vec ? 4 : 1;
    // every lane reads its operands' row indices without a branch: an operand on the edges reads (and discards) an
    // index array that exists, or the start of out when the call has none
    const int32_t *some = col_dev ? col_dev : row_dev ? row_dev : reinterpret_cast<const int32_t *>(out_dev);
    EdgeArgs a;
    a.lhs_index = lhs_target == FG_TARGET_U ? col_dev : lhs_target == FG_TARGET_V ? row_dev : some;
    a.rhs_index = rhs_target == FG_TARGET_U ? col_dev : rhs_target == FG_TARGET_V ? row_dev : some;
    a.n_edges = n_edges;
    a.lhs = lhs_dev; a.rhs = rhs_dev; a.lhs_off = lhs_off_dev; a.rhs_off = rhs_off_dev;
    a.lhs_len = lhs_len; a.rhs_len = rhs_len; a.lhs_target = lhs_target; a.rhs_target = rhs_target;
    a.out = out_dev; a.F = out_len; a.L = lanes_for((out_len + V - 1) / V); a.R = R;
    const int64_t waves = (n_edges + 63) / 64;
    const int64_t blocks = (waves + kWavesPerBlock - 1) / kWavesPerBlock;
    if (blocks > 0x7fffffffLL) return fail(FG_ERR_SHAPE, "grid of %lld workgroups is too large", (long long)blocks);
    hipStream_t st = (hipStream_t)stream;
    const dim3 grid((unsigned)blocks);
    switch (op) {
        case FG_BIN_ADD: launch_sddmm<FG_BIN_ADD>(vec, grid, st, a); break;
        case FG_BIN_SUB: launch_sddmm<FG_BIN_SUB>(vec, grid, st, a); break;
        case FG_BIN_MUL: launch_sddmm<FG_BIN_MUL>(vec, grid, st, a); break;
        case FG_BIN_DIV: launch_sddmm<FG_BIN_DIV>(vec, grid, st, a); break;
        case FG_BIN_COPY_LHS: launch_sddmm<FG_BIN_COPY_LHS>(vec, grid, st, a); break;
        case FG_BIN_COPY_RHS: launch_sddmm<FG_BIN_COPY_RHS>(vec, grid, st, a); break;
        default: {
            const bool wide = R % 4 == 0 && lhs_len % 4 == 0 && rhs_len % 4 == 0 && (((uintptr_t)lhs_dev | (uintptr_t)rhs_dev) & 15) == 0;
            if (!wide) hipLaunchKernelGGL((gsddmm_bcast_kernel<FG_BIN_DOT, 1, true, true, false, 4>), grid, dim3(kBlock), 0, st, a);
            else if (R <= 16) hipLaunchKernelGGL(gsddmm_dot_kernel<4>, grid, dim3(kBlock), 0, st, a);
            else if (R <= 32) hipLaunchKernelGGL(gsddmm_dot_kernel<8>, grid, dim3(kBlock), 0, st, a);
            else if (R <= 64) hipLaunchKernelGGL(gsddmm_dot_kernel<16>, grid, dim3(kBlock), 0, st, a);
            else if (R <= 128) hipLaunchKernelGGL(gsddmm_dot_kernel<32>, grid, dim3(kBlock), 0, st, a);
            else hipLaunchKernelGGL(gsddmm_dot_kernel<64>, grid, dim3(kBlock), 0, st, a);
            break;
        }
    }
    FG_HIP_TRY(hipGetLastError());
    return FG_OK;
}
