// The walk over a plan's items that the weighted sum (fg_spmm.hip) and the sum with dots (fg_spmm_dot.hip) share: what a
// wavefront stages, gathers, adds up and stores (fg_spmm.hip says how the work is laid out).  The two are files of their own because
// the sum's kernels are held to 64 registers: with the kernels with dots beside them in one module the compiler spilled 12 to 16 bytes a
// lane in those that add to `out` (58,000 nodes, 12.5 M edges, F=512 in 8 passes: 1439 -> 1451 us).
#pragma once

#include <hip/hip_runtime.h>

#include "fg_common.h"
#include "fg_device.h"

namespace fg_items {

using fg::Item;
using fg::wave_lds_sync;

constexpr int kWavesPerBlock = 4;
constexpr int kBlock = 64 * kWavesPerBlock;
constexpr int kPad = 8;

template <int V> struct Vec;
template <> struct Vec<4> { using type = float4; };
template <> struct Vec<1> { using type = float; };

__device__ __forceinline__ float4 vzero(float4) { return make_float4(0.f, 0.f, 0.f, 0.f); }
__device__ __forceinline__ float vzero(float) { return 0.f; }
__device__ __forceinline__ void vfma(float4 &a, float w, const float4 &x) {
    a.x += w * x.x; a.y += w * x.y; a.z += w * x.z; a.w += w * x.w;
}
__device__ __forceinline__ void vfma(float &a, float w, const float &x) { a += w * x; }
__device__ __forceinline__ void vadd(float4 &a, const float4 &b) { a.x += b.x; a.y += b.y; a.z += b.z; a.w += b.w; }
__device__ __forceinline__ void vadd(float &a, const float &b) { a += b; }
__device__ __forceinline__ float4 vshfl_xor(const float4 &a, int off) {
    return make_float4(__shfl_xor(a.x, off), __shfl_xor(a.y, off), __shfl_xor(a.z, off), __shfl_xor(a.w, off));
}
__device__ __forceinline__ float vshfl_xor(const float &a, int off) { return __shfl_xor(a, off); }
// a where `keep`, else zeros
__device__ __forceinline__ float4 vkeep(bool keep, const float4 &a) {
    return make_float4(keep ? a.x : 0.f, keep ? a.y : 0.f, keep ? a.z : 0.f, keep ? a.w : 0.f);
}
__device__ __forceinline__ float vkeep(bool keep, const float &a) { return keep ? a : 0.f; }

struct SpmmArgs {
    const Item *items;
    int64_t n_items;
    const int32_t *pos;    // this partition's position array (row boundaries), n_dst + 1 entries
    const int32_t *indices;
    const uint16_t *indices16 = nullptr;   // the plan's 16-bit copy of `indices` (null: none), read by the sum kernel
    const float *vals;
    const float *x;        // already offset to the partition's first source row
    // Sum, max and min kernels, 32-bit offsets only.  Bytes between consecutive source rows, and, when the
    // kernel tiles of x are stored one after the other ([tile][row][tile floats]), the bytes from
    // one tile's block to the next; 0: rows of F floats that hold all tiles.
    uint32_t x_row_bytes;
    uint32_t x_tile_bytes;
    float *out;
    float *partial;        // pieces of split rows: columns [partial_f0, partial_f0 + partial_ld) of each
    int partial_ld, partial_f0 = 0;
    int F;                 // row stride of x / out in floats
    int tile_w;            // floats per requested feature tile (F / num_feat_partitions)
    int sub_per_tile;      // kernel tiles (V*L*K floats each) per requested tile
    int n_ftiles;          // kernel tiles handled by this launch (consecutive, starting at tile_base)
    int tile_base;
    int accumulate;        // add to out instead of overwriting it
    int heads;             // weights are [nnz, heads]; a kernel tile lies inside one head
    int head_len;          // floats per head (F / heads)
    int32_t *arg;          // arg kernel: stored position of the element that gave out[v, f]
    int vstride;           // weight of element t, head h: vals[t * vstride + h * head_stride]
    int64_t head_stride;
    // One launch over the items of all source partitions (sum kernel, every pass into a buffer of its own): the
    // plan's item_off on the device (n_parts + 1 entries; null: the launch holds one partition's items and the
    // strides are unused) and the distance from one partition's pos / x / out / partial to the next, in elements.
    const int64_t *item_off = nullptr;
    int n_parts = 1;
    int64_t pos_stride = 0, x_stride = 0, out_stride = 0, partial_stride = 0;
    // Sum with dots: every element's dot product of its gathered row with its output row's row of `own`, per head or, with
    // one head, per kernel tile.  Rows of `own` lie own_ld floats apart and hold heads of own_len <= head_len floats (the
    // kernel's columns beyond own_len meet zeros).  dots[(tile * HPT + head of the tile) * dots_stride + element].
    const float *own = nullptr;
    int64_t own_ld = 0;
    int own_len = 0;
    float *dots = nullptr;
    int64_t dots_stride = 0;
    // Kernels that store rows shorter than the ones they compute (x is a zero-padded copy): rows of `out` lie out_ld floats
    // apart and hold heads of out_len <= head_len floats.
    int out_ld = 0, out_len = 0;
};


// Address of this lane's part of a staged source row.  OFF32: the staged word is the row's byte
// offset from the (wave-uniform) start of X and fits 32 bits, so the load takes a scalar base
// plus a 32-bit lane offset and no 64-bit multiply is left in the loop; otherwise it is the
// column id.
template <bool OFF32>
__device__ __forceinline__ const float *row_ptr(const float *x, uint32_t lane_bytes, int64_t F, int staged) {
    if (OFF32) return reinterpret_cast<const float *>(reinterpret_cast<const char *>(x) + ((uint32_t)staged + lane_bytes));
    return reinterpret_cast<const float *>(reinterpret_cast<const char *>(x + (int64_t)staged * F) + lane_bytes);
}

// Sum over the L (a power of two up to 64) consecutive lanes of a lane group; every lane of the group gets it.
template <int L>
__device__ __forceinline__ float lanes_sum(float v) {
    if constexpr (L == 2) { return v + fg::dpp_move<0xB1>(v); }
    else {
        v = fg::group_sum<(L < 16 ? L : 16)>(v);
        if constexpr (L >= 32) {
            float w = v;
            fg::swap_rows(v, w);
            v += w;
        }
        if constexpr (L >= 64) {
            float w = v;
            fg::swap_halves(v, w);
            v += w;
        }
        return v;
    }
}

// Where the dot products of a sum with dots go: into the staging row, in the place of the element's weight.  RL lanes hold
// a head's part of a row; ON == false: no dots, nothing is done.
template <bool ON, int RL>
struct Dots {
    float4 own;                     // this lane's four floats of the output row's row of `own`
    __device__ __forceinline__ void put(int lane, const float4 &x, bool ok, int32_t *slot) const {
        if constexpr (ON) {
            const float d = lanes_sum<RL>(x.x * own.x + x.y * own.y + x.z * own.z + x.w * own.w);
            if (ok && lane % RL == 0) *slot = __float_as_int(d);
        }
    }
    __device__ __forceinline__ void put(int, float, bool, int32_t *) const {}
};

// The last, partly filled batch of gather_rows: exactly `nu` steps (1 <= nu <= NU, uniform over
// the wavefront), so that no step is spent re-reading the row's last element; inside the last
// step a lane without an element still re-reads it (no load under a branch) and replaces what it
// loaded by zeros -- a select, not a product with weight zero, so that a non-finite source row
// only ever reaches the rows that reference it.
template <int V, int L, int K, bool FULL, int NU, bool OFF32, int HPT, typename DOTS>
__device__ __forceinline__ void gather_tail(int nu, int2 *s_edge, float *wrow, int s0, int e, int g,
                                            const float *x, uint32_t lane_bytes, int64_t F, const bool (&on)[K],
                                            typename Vec<V>::type (&acc)[K], const DOTS &dots) {
    using vec = typename Vec<V>::type;
    constexpr int G = 64 / L;
    if (nu < NU) {
        if constexpr (NU > 1) gather_tail<V, L, K, FULL, NU - 1, OFF32, HPT>(nu, s_edge, wrow, s0, e, g, x, lane_bytes, F, on, acc, dots);
        return;
    }
    int2 cw[NU];
    vec xv[NU][K];
#pragma unroll
    for (int u = 0; u < NU; ++u) {
        const int j = s0 + u * G + g;
        cw[u] = s_edge[j < e ? j : e - 1];
        if (HPT > 1) cw[u].y = __float_as_int(wrow[j < e ? j : e - 1]);
        if (j >= e) cw[u].y = 0;
    }
#pragma unroll
    for (int u = 0; u < NU; ++u)
#pragma unroll
        for (int k = 0; k < K; ++k)
            if (FULL || on[k])
                xv[u][k] = *reinterpret_cast<const vec *>(row_ptr<OFF32>(x, lane_bytes, F, cw[u].x) + k * L * V);
    const bool last_has = s0 + (NU - 1) * G + g < e;      // steps before the last are full
#pragma unroll
    for (int u = 0; u < NU; ++u)
#pragma unroll
        for (int k = 0; k < K; ++k)
            if (FULL || on[k]) {
                if (u == NU - 1) xv[u][k] = vkeep(last_has, xv[u][k]);
                vfma(acc[k], __int_as_float(cw[u].y), xv[u][k]);
                const int j = u < NU - 1 || last_has ? s0 + u * G + g : e - 1;
                dots.put(threadIdx.x & 63, xv[u][k], u < NU - 1 || last_has,
                         HPT > 1 ? reinterpret_cast<int32_t *>(wrow + j) : &s_edge[j].y);
            }
}

// Adds vals * X rows for the staged elements [b, e) of s_edge (x = staged column word, y =
// weight bits) into acc.  The G lane groups take elements b+g, b+g+G, ...; U steps' loads are
// issued back to back before the first use.  No load sits under a branch: in the last, partly
// filled batch a lane without an element re-reads the row's last element and discards it.
// HPT > 1: the kernel tile holds HPT heads and the lane's weight is wrow[slot] (its head's staged
// weights) instead of the word staged next to the column.
// dots: with ON, each element's weight is replaced by its dot product once it has been used.
template <int V, int L, int K, bool FULL, int U, bool OFF32, int HPT, typename DOTS>
__device__ __forceinline__ void gather_rows(int2 *s_edge, float *wrow, int b, int e, int g, const float *x,
                                            uint32_t lane_bytes, int64_t F, const bool (&on)[K],
                                            typename Vec<V>::type (&acc)[K], const DOTS &dots) {
    using vec = typename Vec<V>::type;
    constexpr int G = 64 / L;
    int s0 = b;
    for (; s0 + G * U <= e; s0 += G * U) {
        int2 cw[U];
        vec xv[U][K];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            cw[u] = s_edge[s0 + u * G + g];
            if (HPT > 1) cw[u].y = __float_as_int(wrow[s0 + u * G + g]);
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int k = 0; k < K; ++k)
                if (FULL || on[k])
                    xv[u][k] = *reinterpret_cast<const vec *>(row_ptr<OFF32>(x, lane_bytes, F, cw[u].x) + k * L * V);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int k = 0; k < K; ++k)
                if (FULL || on[k]) {
                    vfma(acc[k], __int_as_float(cw[u].y), xv[u][k]);
                    const int j = s0 + u * G + g;
                    dots.put(threadIdx.x & 63, xv[u][k], true, HPT > 1 ? reinterpret_cast<int32_t *>(wrow + j) : &s_edge[j].y);
                }
    }
    if (s0 < e)                            // uniform: fewer than G*U elements left
        gather_tail<V, L, K, FULL, U, OFF32, HPT>((e - s0 + G - 1) / G, s_edge, wrow, s0, e, g, x, lane_bytes, F, on, acc, dots);
}

// Stores a lane's columns f_lo, f_lo + L * V, .. of a row that holds heads of out_len floats, out_len <= head_len: 16-byte stores
// at 4-byte alignment, the head's last words one by one.
template <int V, int L, int K, bool FULL>
__device__ __forceinline__ void store_short(const SpmmArgs &a, const typename Vec<V>::type (&v)[K], const bool (&on)[K], float *row, int f_lo) {
    if constexpr (V == 4) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            if (!(FULL || on[k])) continue;
            const int f = f_lo + k * L * V, h = a.heads == 1 ? 0 : f / a.head_len, d = f - h * a.head_len, left = a.out_len - d;
            float *p = row + h * a.out_len + d;
            if (left >= 4) {
                *reinterpret_cast<fg::Words4<float> *>(p) = {{v[k].x, v[k].y, v[k].z, v[k].w}};
            } else {
                if (left > 0) p[0] = v[k].x;
                if (left > 1) p[1] = v[k].y;
                if (left > 2) p[2] = v[k].z;
            }
        }
    }
}

// Adds the lane groups' sums (group 0 gets the total).
template <int V, int L, int K>
__device__ __forceinline__ void add_groups(typename Vec<V>::type (&acc)[K]) {
#pragma unroll
    for (int off = L; off < 64; off <<= 1)
#pragma unroll
        for (int k = 0; k < K; ++k) vadd(acc[k], vshfl_xor(acc[k], off));
}

// Adds the lane groups' sums and stores one output row; `old` is what the row held before (only read when ADD).
template <int V, int L, int K, bool FULL, bool ADD>
__device__ __forceinline__ void finish_row(typename Vec<V>::type (&acc)[K], const typename Vec<V>::type (&old)[K],
                                           int g, const bool (&on)[K], float *dst) {
    using vec = typename Vec<V>::type;
    add_groups<V, L, K>(acc);
    if (g == 0) {
#pragma unroll
        for (int k = 0; k < K; ++k)
            if (FULL || on[k]) {
                vec r = acc[k];
                if (ADD) vadd(r, old[k]);
                if constexpr (V == 4 && !ADD) {
                    // written once, read back by another kernel: a non-temporal store leaves the L2 to the gathered rows
                    // (232,965-node graph: 11.24 -> 11.17 ms at F=512, 5.75 -> 5.72 ms at F=256)
                    typedef float f4 __attribute__((ext_vector_type(4)));
                    f4 t; t.x = r.x; t.y = r.y; t.z = r.z; t.w = r.w;
                    __builtin_nontemporal_store(t, reinterpret_cast<f4 *>(dst + k * L * V));
                } else {
                    *reinterpret_cast<vec *>(dst + k * L * V) = r;
                }
            }
    }
}

// Loads elements [base, base + min(n, 256)) of (indices, vals) into registers, lane l holding
// elements 4l .. 4l + 3.  n >= 1.
// `scale` turns a column id into the staged word: the row's byte size (OFF32) or 1.  The weight of
// element t is vals[t * vstride + voff] (one weight per head), or 1 when there are no weights.
// indices16 (uniform; null: none): the same ids as 16-bit words, read instead of `indices`.
__device__ __forceinline__ void stage_load(const int32_t *indices, const uint16_t *indices16, const float *vals, int64_t base, int n,
                                           int lane, uint32_t scale, int vstride, int64_t voff, int2 (&r)[4]) {
    int32_t c[4];
    float w[4] = {1.0f, 1.0f, 1.0f, 1.0f};
    fg::load_four_ids(indices, indices16, base, n, lane, c);
    if (vals) fg::load_four(vals + base * vstride + voff, n, lane, vstride, w);
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = make_int2((int)((uint32_t)c[i] * scale), __float_as_int(w[i]));
}
// Writes the staged words to the wavefront's staging row (16-byte aligned), two elements per store.
__device__ __forceinline__ void stage_store(int2 *edge, int lane, const int2 (&r)[4]) {
    int4 *e4 = reinterpret_cast<int4 *>(edge);
    e4[2 * lane] = make_int4(r[0].x, r[0].y, r[1].x, r[1].y);
    e4[2 * lane + 1] = make_int4(r[2].x, r[2].y, r[3].x, r[3].y);
    if (lane < kPad) edge[fg::kItemEdges + lane] = r[3];      // a valid element: slots past the end stay loadable
}

// The same for the weights of the HPT heads of a kernel tile (head h of the tile: vals[t * vstride + voff + h * hstride]).
template <int HPT>
__device__ __forceinline__ void stage_load_w(const float *vals, int64_t base, int n, int lane, int vstride,
                                             int64_t voff, int64_t hstride, float (&w)[HPT][4]) {
#pragma unroll
    for (int h = 0; h < HPT; ++h) {
        if (vals) {
            fg::load_four(vals + base * vstride + voff + h * hstride, n, lane, vstride, w[h]);
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) w[h][i] = 1.0f;
        }
    }
}
template <int HPT, int ROW>
__device__ __forceinline__ void stage_store_w(float (*rows)[ROW], int lane, const float (&w)[HPT][4]) {
#pragma unroll
    for (int h = 0; h < HPT; ++h) {
        *reinterpret_cast<float4 *>(&rows[h][4 * lane]) = make_float4(w[h][0], w[h][1], w[h][2], w[h][3]);
        if (lane < kPad) rows[h][fg::kItemEdges + lane] = w[h][3];
    }
}

// V: floats per lane per load; L: lanes per source row; K: loads per lane per source row;
// FULL: every lane's columns are inside the tile (no masking needed); ACC: add to out;
// OFF32: X spans less than 4 GiB, rows are addressed by 32-bit byte offsets; HPT: heads (with
// their own weights) per kernel tile, each covered by L / HPT lanes; DOT: each element's dot product with the output
// row's row of `own` as well; SHORT: the rows of out are shorter than the computed ones (SpmmArgs: out_ld, out_len).
template <int V, int L, int K, bool FULL, bool ACC, bool OFF32, int HPT = 1, bool DOT = false, bool SHORT = false>
__device__ __forceinline__ void spmm_items_body(const SpmmArgs &a) {
    using vec = typename Vec<V>::type;
    static_assert(fg::kItemEdges == 256, "stage_load/stage_store move 4 x 64 elements");
    constexpr int FT = V * L * K;          // floats per kernel tile
    constexpr int G = 64 / L;              // lane groups per wavefront
    constexpr int U = (K >= 2) ? 2 : 4;   // steps whose loads are issued back to back
    static_assert(U <= kPad, "reads past a row's end must stay inside the padded staging row");
    // kPad extra slots: the lane-group-per-row walk may read up to U - 1 slots past a row's end
    __shared__ __align__(16) int2 s_edge[kWavesPerBlock][fg::kItemEdges + kPad];
    __shared__ int32_t s_end[kWavesPerBlock][fg::kItemRows];
    __shared__ int32_t s_next[kWavesPerBlock];
    constexpr int kWRow = HPT > 1 ? fg::kItemEdges + kPad : 1;
    __shared__ __align__(16) float s_w[kWavesPerBlock][HPT][kWRow];
    static_assert(HPT == 1 || (L % HPT == 0 && K == 1 && FULL), "heads of a tile split its lanes evenly");
    static_assert(!SHORT || (V == 4 && !ACC), "short rows: 128-bit lanes, one pass");
    static_assert(!DOT || (V == 4 && K == 1 && FULL && !ACC), "dots: whole tiles of 128-bit lanes, every pass in its own buffer");

    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int tile = a.tile_base + (int)(blockIdx.x % (unsigned)a.n_ftiles);
    const int64_t item_id = (int64_t)(blockIdx.x / (unsigned)a.n_ftiles) * kWavesPerBlock + wave;
    if (item_id >= a.n_items) return;      // uniform per wavefront; no workgroup barriers below
    Item it = a.items[item_id];
    if (DOT) {                             // the item's fields as scalars: fewer vector registers, scalar loop bounds
        it.start = __builtin_amdgcn_readfirstlane(it.start); it.len = __builtin_amdgcn_readfirstlane(it.len);
        it.row = __builtin_amdgcn_readfirstlane(it.row); it.info = __builtin_amdgcn_readfirstlane(it.info);
    }
    // the partition this item belongs to (uniform per wavefront): selects its position array, its slice of x,
    // its output buffer and its share of the split rows' scratch
    int part = 0;
    if (a.item_off) {
        const int64_t id = ((int64_t)__builtin_amdgcn_readfirstlane((int)(item_id >> 32)) << 32) |
                           (uint32_t)__builtin_amdgcn_readfirstlane((int)item_id);
        while (part + 1 < a.n_parts && id >= a.item_off[part + 1]) ++part;
    }
    const int32_t *const pos_p = a.pos + part * a.pos_stride;
    const float *const x_p = a.x + part * a.x_stride;
    float *const out_p = a.out + part * a.out_stride;
    float *const partial_p = a.partial + part * a.partial_stride;
    const int g = lane / L, li = lane % L;

    const int rt = tile / a.sub_per_tile, st = tile % a.sub_per_tile;
    const int f_end = (rt + 1) * a.tile_w;
    const int f_lo = rt * a.tile_w + st * FT + li * V;      // first column of this lane, k = 0
    bool on[K];
#pragma unroll
    for (int k = 0; k < K; ++k) on[k] = FULL || (f_lo + k * L * V < f_end);
    const uint32_t lane_bytes = (OFF32 && a.x_tile_bytes) ? (uint32_t)tile * a.x_tile_bytes + (uint32_t)(li * V) * 4u
                                                          : (uint32_t)f_lo * 4u;
    const uint32_t scale = OFF32 ? a.x_row_bytes : 1u;
    const int64_t voff = (int64_t)((rt * a.tile_w + st * FT) / a.head_len) * a.head_stride;     // head of this kernel tile
    const int64_t F = a.F;
    int2 *edge = s_edge[wave];
    float *wrow = s_w[wave][HPT > 1 ? (lane % L) / (L / HPT) : 0];
    const float *col_vals = HPT > 1 ? nullptr : a.vals;     // HPT > 1: weights are staged per head instead
    vec acc[K], old[K];
    int2 regs[4];
    float wregs[HPT][4];
    Dots<DOT, L / HPT> dots;
    // the lane's floats of a row of `own`, in two halves (the load is far from its use); columns that `own` lacks are 0
    const int own_head = DOT ? f_lo / a.head_len : 0, own_d = DOT ? f_lo - own_head * a.head_len : 0;
    auto load_own = [&](int64_t row) {
        if constexpr (DOT) {
            const float *p = a.own + row * a.own_ld + (int64_t)own_head * a.own_len + own_d;
            if (own_d + 4 <= a.own_len) {
                const fg::Words4<float> w = *reinterpret_cast<const fg::Words4<float> *>(p);
                dots.own = make_float4(w.v[0], w.v[1], w.v[2], w.v[3]);
            } else {
                const int left = a.own_len - own_d;
                dots.own = make_float4(left > 0 ? p[0] : 0.f, left > 1 ? p[1] : 0.f, left > 2 ? p[2] : 0.f, 0.f);
            }
        }
    };
    // the staged elements' dot products, [0, n) of the staging row, as runs; `first`: element 0's position in the layout
    auto flush_dots = [&](int64_t first, int n) {
        if constexpr (DOT) {
            wave_lds_sync();
            for (int j = lane; j < n; j += 64) {
#pragma unroll
                for (int h = 0; h < HPT; ++h)
                    __builtin_nontemporal_store(HPT > 1 ? s_w[wave][h][j] : __int_as_float(edge[j].y),
                                                a.dots + ((int64_t)tile * HPT + h) * a.dots_stride + first + j);
            }
        }
    };

    if (it.info < -1) {
        // Several whole rows: stage all their elements once.
        const int nrows = -it.info;
        // ACC: the rows this item adds to are read once here, one word per 128 bytes, while the
        // elements are on their way.  Loads return in order, so a row of `out` fetched from memory
        // at the moment it is needed would hold up every gather issued after it; fetched here, all
        // rows' misses overlap each other and the staging loads, and the later reads hit the cache.
        constexpr int kLines = (FT * 4 + 127) / 128;
        constexpr int kTouch = ACC ? (fg::kItemRows * kLines + 63) / 64 : 1;
        float touched[kTouch];
        if (ACC) {
            const int f_tile = rt * a.tile_w + st * FT;
            const int f_last = min(f_tile + FT, f_end) - 1;
#pragma unroll
            for (int i = 0; i < kTouch; ++i) {
                const int t = lane + 64 * i;
                const int r = min(t / kLines, nrows - 1);
                const int f = min(f_tile + (t % kLines) * 32, f_last);
                touched[i] = out_p[(int64_t)(it.row + r) * F + f];
            }
        }
        // (the rows of `own` likewise)
        constexpr int kOwnTouch = DOT ? (fg::kItemRows * kLines + 63) / 64 : 1;
        float own_touched[kOwnTouch];
        if constexpr (DOT) {
#pragma unroll
            for (int i = 0; i < kOwnTouch; ++i) {
                const int t = lane + 64 * i;
                const int f = rt * a.tile_w + st * FT + (t % kLines) * 32, h = f / a.head_len;
                own_touched[i] = a.own[(int64_t)(it.row + min(t / kLines, nrows - 1)) * a.own_ld + (int64_t)h * a.own_len +
                                       min(f - h * a.head_len, a.own_len - 1)];
            }
        }
        if (it.len > 0) {
            stage_load(a.indices, a.indices16, col_vals, it.start, it.len, lane, scale, a.vstride, voff, regs);
            if (HPT > 1) stage_load_w<HPT>(a.vals, it.start, it.len, lane, a.vstride, voff, a.head_stride, wregs);
            stage_store(edge, lane, regs);
            if (HPT > 1) stage_store_w<HPT>(s_w[wave], lane, wregs);
        }
        s_end[wave][lane] = pos_p[it.row + min(lane, nrows - 1) + 1] - it.start;
        if (lane == 0) s_next[wave] = 0;
        wave_lds_sync();
        if (ACC) {
#pragma unroll
            for (int i = 0; i < kTouch; ++i) asm volatile("" ::"v"(touched[i]));    // keeps the loads
        }
        if constexpr (DOT) {
#pragma unroll
            for (int i = 0; i < kOwnTouch; ++i) asm volatile("" ::"v"(own_touched[i]));
        }
        // Rows in the middle: many at a time, `share` neighbouring groups to a row.  us with every such row on all groups, or from 2 * G rows on one
        // group each / as here: 120,000 rows of 8, F=16 31 / 16, power-law 30 / 19, F=32 22 / 22, 32 / 22; of 16, F=8 34 / 21, F=16 36 / 26; of 60, power-law, F=8 56 /
        // 60, F=128 300 / 293; 20,000 of 8, F=16 11 / 8, of 60, power-law, F=64 29 / 27.
        const int share = fg::groups_per_row<L>(nrows, it.len);
        if (share > 1 && share < G) {
            const int sub = g & (share - 1);
            for (int q0 = 0; q0 < nrows; q0 += G / share) {
                const int q = q0 + g / share;
                const bool mine = q < nrows;
                const int b = mine && q ? s_end[wave][q - 1] : 0, e = mine ? s_end[wave][q] : 0;
#pragma unroll
                for (int k = 0; k < K; ++k) acc[k] = vzero(vec());
                load_own(it.row + min(q, nrows - 1));
                if (ACC && e > b) {
                    const float *src = out_p + (int64_t)(it.row + q) * F + f_lo;
#pragma unroll
                    for (int k = 0; k < K; ++k)
                        if (FULL || on[k]) old[k] = *reinterpret_cast<const vec *>(src + k * L * V);
                }
                for (int j = b + sub; j < e; j += share * U) {
                    int2 cw[U];
                    vec xv[U][K];
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        const int t = j + u * share, at = t < e ? t : j;      // beyond the row: its element once more, replaced by zeros
                        cw[u] = edge[at];
                        if (HPT > 1) cw[u].y = __float_as_int(wrow[at]);
                        if (t >= e) cw[u].y = 0;
                    }
#pragma unroll
                    for (int u = 0; u < U; ++u)
#pragma unroll
                        for (int k = 0; k < K; ++k)
                            if (FULL || on[k])
                                xv[u][k] = *reinterpret_cast<const vec *>(row_ptr<OFF32>(x_p, lane_bytes, F, cw[u].x) + k * L * V);
#pragma unroll
                    for (int u = 0; u < U; ++u)
#pragma unroll
                        for (int k = 0; k < K; ++k)
                            if (FULL || on[k]) {
                                const int t = j + u * share;
                                if (u > 0) xv[u][k] = vkeep(t < e, xv[u][k]);
                                vfma(acc[k], __int_as_float(cw[u].y), xv[u][k]);
                                const int at = t < e ? t : j;
                                dots.put(lane, xv[u][k], t < e, HPT > 1 ? reinterpret_cast<int32_t *>(wrow + at) : &edge[at].y);
                            }
                }
                for (int off = L; off < L * share; off <<= 1)
#pragma unroll
                    for (int k = 0; k < K; ++k) vadd(acc[k], vshfl_xor(acc[k], off));
                if (mine && sub == 0 && (!ACC || e > b)) {
                    if constexpr (SHORT) {
                        store_short<V, L, K, FULL>(a, acc, on, out_p + (int64_t)(it.row + q) * a.out_ld, f_lo);
                    } else {
                        float *dst = out_p + (int64_t)(it.row + q) * F + f_lo;
#pragma unroll
                        for (int k = 0; k < K; ++k)
                            if (FULL || on[k]) {
                                vec r = acc[k];
                                if (ACC) vadd(r, old[k]);
                                *reinterpret_cast<vec *>(dst + k * L * V) = r;
                            }
                    }
                }
            }
            flush_dots(it.start, it.len);
            return;
        }
        if (nrows < 2 * G) {
            // Few, longer rows: all lane groups share each row in turn.
            int b = 0;
            for (int q = 0; q < nrows; ++q) {
                const int e = __builtin_amdgcn_readfirstlane(s_end[wave][q]);
                if (e > b || !ACC) {
                    float *dst = out_p + (int64_t)(it.row + q) * F + f_lo;
                    if (ACC) {
#pragma unroll
                        for (int k = 0; k < K; ++k)
                            if (FULL || on[k]) old[k] = *reinterpret_cast<const vec *>(dst + k * L * V);
                    }
#pragma unroll
                    for (int k = 0; k < K; ++k) acc[k] = vzero(vec());
                    load_own(it.row + q);
                    gather_rows<V, L, K, FULL, U, OFF32, HPT>(edge, wrow, b, e, g, x_p, lane_bytes, F, on, acc, dots);
                    if constexpr (SHORT) {
                        add_groups<V, L, K>(acc);
                        if (g == 0) store_short<V, L, K, FULL>(a, acc, on, out_p + (int64_t)(it.row + q) * a.out_ld, f_lo);
                    } else {
                        finish_row<V, L, K, FULL, ACC>(acc, old, g, on, dst);
                    }
                }
                b = e;
            }
            flush_dots(it.start, it.len);
            return;
        }
        // Many short rows: every lane group takes rows of its own (next free row from a counter
        // in LDS), walks each row's elements U at a time and writes the row itself, so G rows
        // are in flight per wavefront and no sums cross lane groups.
        int q = -1, j = 0, e = 0;
        bool done = false, nonempty = false;
        for (;;) {
            if (!done && j >= e) {
                if (SHORT && q >= 0) {
                    store_short<V, L, K, FULL>(a, acc, on, out_p + (int64_t)(it.row + q) * a.out_ld, f_lo);
                } else if (q >= 0 && (!ACC || nonempty)) {       // the row this group just finished
                    float *dst = out_p + (int64_t)(it.row + q) * F + f_lo;
#pragma unroll
                    for (int k = 0; k < K; ++k)
                        if (FULL || on[k]) {
                            vec r = acc[k];
                            if (ACC) vadd(r, old[k]);
                            *reinterpret_cast<vec *>(dst + k * L * V) = r;
                        }
                }
                int qn = 0;
                if (li == 0) qn = atomicAdd(&s_next[wave], 1);
                q = __shfl(qn, g * L);
                if (q >= nrows) {
                    done = true;
                } else {
                    j = q ? s_end[wave][q - 1] : 0;
                    e = s_end[wave][q];
                    nonempty = e > j;
                    load_own(it.row + q);
#pragma unroll
                    for (int k = 0; k < K; ++k) acc[k] = vzero(vec());
                    if (ACC && nonempty) {
                        const float *src = out_p + (int64_t)(it.row + q) * F + f_lo;
#pragma unroll
                        for (int k = 0; k < K; ++k)
                            if (FULL || on[k]) old[k] = *reinterpret_cast<const vec *>(src + k * L * V);
                    }
                }
            }
            if (__all(done)) break;
            if (!done && j < e) {
                int2 cw[U];
                vec xv[U][K];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    // past the row's end this is a later row's element (or the padding): a loadable
                    // source row whose values are replaced by zeros below
                    cw[u] = edge[j + u];
                    if (HPT > 1) cw[u].y = __float_as_int(wrow[j + u]);
                    if (j + u >= e) cw[u].y = 0;
                }
#pragma unroll
                for (int u = 0; u < U; ++u)
#pragma unroll
                    for (int k = 0; k < K; ++k)
                        if (FULL || on[k])
                            xv[u][k] = *reinterpret_cast<const vec *>(row_ptr<OFF32>(x_p, lane_bytes, F, cw[u].x) + k * L * V);
#pragma unroll
                for (int u = 0; u < U; ++u)
#pragma unroll
                    for (int k = 0; k < K; ++k)
                        if (FULL || on[k]) {
                            // u == 0 is always the row's own element (j < e)
                            if (u > 0) xv[u][k] = vkeep(j + u < e, xv[u][k]);
                            vfma(acc[k], __int_as_float(cw[u].y), xv[u][k]);
                            dots.put(lane, xv[u][k], j + u < e, HPT > 1 ? reinterpret_cast<int32_t *>(wrow + j + u) : &edge[j + u].y);
                        }
                j += U;
            }
        }
        flush_dots(it.start, it.len);
        return;
    }

    // one row, or one piece of a long row: 256 elements at a time, the next 256 on their way
    // while the current ones are used
    float *dst = (it.info < 0 ? out_p + (int64_t)it.row * F : partial_p + (int64_t)it.info * a.partial_ld - a.partial_f0) + f_lo;
    const bool add = ACC && it.info < 0;
    load_own(it.row);
#pragma unroll
    for (int k = 0; k < K; ++k) acc[k] = vzero(vec());
    if (it.len > 0) {
        stage_load(a.indices, a.indices16, col_vals, it.start, it.len, lane, scale, a.vstride, voff, regs);
        if (HPT > 1) stage_load_w<HPT>(a.vals, it.start, it.len, lane, a.vstride, voff, a.head_stride, wregs);
    }
    if (ACC) {
#pragma unroll
        for (int k = 0; k < K; ++k)
            if (FULL || on[k]) old[k] = add ? *reinterpret_cast<const vec *>(dst + k * L * V) : vzero(vec());
    }
    for (int32_t base = 0; base < it.len; base += fg::kItemEdges) {
        const int n = min(fg::kItemEdges, it.len - base);
        wave_lds_sync();                   // earlier reads of the staging row are done
        stage_store(edge, lane, regs);
        if (HPT > 1) stage_store_w<HPT>(s_w[wave], lane, wregs);
        wave_lds_sync();
        if (base + fg::kItemEdges < it.len) {
            stage_load(a.indices, a.indices16, col_vals, (int64_t)it.start + base + fg::kItemEdges,
                       it.len - base - fg::kItemEdges, lane, scale, a.vstride, voff, regs);
            if (HPT > 1)
                stage_load_w<HPT>(a.vals, (int64_t)it.start + base + fg::kItemEdges, it.len - base - fg::kItemEdges,
                                  lane, a.vstride, voff, a.head_stride, wregs);
        }
        gather_rows<V, L, K, FULL, U, OFF32, HPT>(edge, wrow, 0, n, g, x_p, lane_bytes, F, on, acc, dots);
        flush_dots((int64_t)it.start + base, n);
    }
    if constexpr (SHORT) {
        if (it.info < 0) {
            add_groups<V, L, K>(acc);
            if (g == 0) store_short<V, L, K, FULL>(a, acc, on, out_p + (int64_t)it.row * a.out_ld, f_lo);
            return;
        }
    }
    finish_row<V, L, K, FULL, ACC>(acc, old, g, on, dst);
}

// The sum with dots: hpt heads per kernel tile, L lanes per source row (fg_spmm_dot.hip).  a.out_len > 0: short rows of out.
int launch_dot(int L, int hpt, dim3 grid, hipStream_t st, const SpmmArgs &a);
// The sum with short rows of out, one pass: L lanes of K loads of 4 floats per source row (fg_spmm_padded.hip).
int launch_padded(int L, int K, bool full, bool off32, int hpt, dim3 grid, hipStream_t st, const SpmmArgs &a);

}  // namespace fg_items
