// Attention with additive scores (GAT layers) and its gradients, without any [nnz, H] array:
//
//   z[e, h] = el[col e, h] + er[row e, h],  s = leaky_relu(z),  a[e, h] = softmax of s[., h] over the edges of row(e)
//   out[r, h, :] = sum over the edges e of row r of a[e, h] * V[col e, h, :]
//
// With delta[r] = <dout[r], out[r]>, da = <dout[r], V[c]> and gate = z > 0 ? 1 : slope, the gradients are
//
//   columns: dV[c] = sum a * dout[r],   dEl[c] = sum gate * a * (da - delta[r])
//   rows:    dEr[r] = sum gate * a * (da - delta[r]) = (1 - slope) * (<dout[r], plus[r]> - delta[r] * share[r]),
//            plus[r] = sum_{z > 0} a * V[c],  share[r] = sum_{z > 0} a
//
// (the gate takes two values and the sum of a * (da - delta) over a whole row is 0), so a forward pass that is told to
// keep `plus` and `share` leaves nothing of dEr to sweep the graph for: a step with gradients is two sweeps.  Against
// float64, that dEr is closer than the edge-by-edge sum (3.4e-7 against 5.5e-7 relative, 58,000 nodes, 3 M edges); by column
// the same form is not (cancellation that the edge-by-edge difference has not), so dEl is summed edge by edge.
// Not in the reference (no attention operator exists there); the result is defined by the composition of
// gather-add, leaky ReLU, edge softmax and per-head weighted SpMM: a row with a NaN score, or one of +inf, is NaN and so is
// every gradient it takes part in.  (A row whose scores are all -inf counts as one without edges, though: 0.)
//
// Layout of the work: one head (16, 32 or 64 floats) per kernel tile, the tile index fastest in the workgroup id so
// that every XCD gathers one head's slices; items, staging and tile-by-tile copies are those of the SpMM kernels.
// What bounds it: the latency of a row's steps one after the other (ids, scalars, weights, gathers, totals), with the
// vector units about half busy; 8 wavefronts per SIMD (64 registers) are worth 3 % over 6 or 7.  The weights of a staged row
// are formed by all 64 lanes, an edge each, and written back to the staging row, instead of by every lane of a group.
// Step with gradients, 58,000 nodes, 12.5 M edges, 4 x 32: 1494 -> 1021 us (three sweeps of 502 + 553 + 500 before, two of
// 490 + 540 now, the first of which also writes `plus`); 200,000 nodes of degree 20: 1224 -> 859 us.
#include <hip/hip_runtime.h>

#include <cmath>
#include <type_traits>

#include "fg_common.h"
#include "fg_device.h"

using fg::fail;
using fg::Item;
using fg::group_sum;
using fg::wave_lds_sync;
using std::integral_constant;

namespace {

constexpr int kWavesPerBlock = 4;
constexpr int kBlock = 64 * kWavesPerBlock;
constexpr int kPad = 8;
constexpr int kU = 4;                  // elements per lane group whose gathers are issued back to back
constexpr int kOwnLen = 8;             // rows up to this long on average: a lane group each

enum Sweep { kForward, kByRow, kByColumn };
// forward: the only pass over a row (divided by the sum of exponentials at once), a pass into a buffer of its own, or
// a later pass that merges into what the earlier ones left.  Gradients: write, or add to what the earlier passes left.
enum Pass { kOnly, kWrite, kMerge };

struct AdditiveArgs {
    const Item *items;
    int64_t n_items;
    const int32_t *pos;       // this partition's row boundaries
    const int32_t *indices;   // partition-local ids of the far side
    const uint16_t *indices16 = nullptr;   // the plan's 16-bit copy of them, read instead (null: none)
    const float *x;           // gathered rows: V, or dout by column; offset to the partition's first far row
    uint32_t x_row_bytes;     // bytes between consecutive rows of x
    uint32_t x_tile_bytes;    // x stored head by head: bytes from one head's block to the next; 0: rows of F floats
    // What is staged per element: el of the source, or (by column) the destination's coef (m + log l, delta, er, 0);
    // head by head, offset to the partition's first far row.
    const float *far;
    int64_t far_head_floats;
    const float *own;         // the own side's scalar, er or (by column) el: own[row * own_row + head * own_head]
    int64_t own_row, own_head;
    const float *coef;        // by row: [H, n_own, 4] (m + log l, delta, er, 0)
    int64_t coef_head_floats;
    const float *own_x;       // gradients: the own side's rows of dout, or (by column) V
    float *out;               // [n_own, F]: weighted sums; by column: dV
    float *plus;              // forward: [n_own, F] weighted sums over the edges with z > 0
    float *state;             // forward: [n_own, H, 2] maximum and sum of exponentials
    float *share;             // forward: [n_own, H] sum of exponentials over the edges with z > 0
    float *res;               // gradients: dEr or dEl, res[row * own_row + head * own_head]
    int F, H;
    int n_heads, head_base;   // heads of this launch
    float slope;
    // One launch over the items of all source partitions (forward, every pass into buffers of its own): the plan's
    // item_off on the device (n_parts + 1 entries; null: one partition's items, strides unused) and the distance from
    // one partition's arrays to the next, in elements.
    const int64_t *item_off = nullptr;
    int n_parts = 1;
    int64_t pos_stride = 0, far_stride = 0, x_stride = 0, out_stride = 0, state_stride = 0, share_stride = 0;
};

__device__ __forceinline__ float4 zero4() { return make_float4(0.f, 0.f, 0.f, 0.f); }
__device__ __forceinline__ float dot4(const float4 &a, const float4 &b) { return a.x * b.x + a.y * b.y + a.z * b.z + a.w * b.w; }
__device__ __forceinline__ void fma4(float4 &acc, float w, const float4 &x) {
    acc.x += w * x.x; acc.y += w * x.y; acc.z += w * x.z; acc.w += w * x.w;
}
__device__ __forceinline__ void scale4(float4 &a, float f) { a.x *= f; a.y *= f; a.z *= f; a.w *= f; }
__device__ __forceinline__ void add4(float4 &a, const float4 &b) { a.x += b.x; a.y += b.y; a.z += b.z; a.w += b.w; }
__device__ __forceinline__ float4 shfl_xor4(const float4 &a, int off) {
    return make_float4(__shfl_xor(a.x, off), __shfl_xor(a.y, off), __shfl_xor(a.z, off), __shfl_xor(a.w, off));
}
__device__ __forceinline__ float wave_sum(float v) { return fg::rows_sum(group_sum<16>(v)); }
// the largest value of the wavefront, as a scalar
__device__ __forceinline__ float wave_max(float v) {
    v = fmaxf(v, fg::dpp_move<0xB1>(v));
    v = fmaxf(v, fg::dpp_move<0x4E>(v));
    v = fmaxf(v, fg::dpp_move<0x141>(v));
    v = fmaxf(v, fg::dpp_move<0x140>(v));
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(fg::rows_max(v))));
}

// Running sums of one row: over all its elements and over those with z > 0.  fmaxf passes a NaN score by, so the sum of
// exponentials alone carries it: a score makes it NaN where any is above -inf, and where none is, as the score itself (nan_term).  acc / plus: weighted rows, this lane's four
// floats (in the totals of a row that the wavefront shared: one of them, fg::word_of_row); a / p: weights (by column a is the sum of gate * a * (da - delta)).  m: the maximum that the forward weights are
// relative to.
template <typename T>
struct SumsOf {
    T acc, plus;
    float a, p, m;
};
using Sums = SumsOf<float4>;
// s, a score that is -inf or NaN, as a term of a sum of exponentials
__device__ __forceinline__ float nan_term(float s) { return s == -INFINITY ? 0.f : s; }
__device__ __forceinline__ Sums sums_empty() { return {zero4(), zero4(), 0.f, 0.f, -INFINITY}; }

__device__ __forceinline__ void scale4(float &a, float f) { a *= f; }
__device__ __forceinline__ void fma4(float &acc, float w, float x) { acc += w * x; }
__device__ __forceinline__ void add4(float &a, float b) { a += b; }
__device__ __forceinline__ void set_zero(float4 &a) { a = zero4(); }
__device__ __forceinline__ void set_zero(float &a) { a = 0.f; }
// written once and read back by another kernel: non-temporal stores leave the L2 to the gathered rows
__device__ __forceinline__ void store_nt(const float4 &v, float *p) {
    typedef float f4 __attribute__((ext_vector_type(4)));
    f4 t; t.x = v.x; t.y = v.y; t.z = v.z; t.w = v.w;
    __builtin_nontemporal_store(t, reinterpret_cast<f4 *>(p));
}
__device__ __forceinline__ void store_nt(float v, float *p) { __builtin_nontemporal_store(v, p); }

template <bool PLUS, typename T>
__device__ __forceinline__ void rescale(SumsOf<T> &r, float f) {
    scale4(r.acc, f);
    r.a *= f;
    if (PLUS) { scale4(r.plus, f); r.p *= f; }
}
// r <- r and s merged (both relative to their own maxima)
template <bool PLUS, typename T>
__device__ __forceinline__ void merge(SumsOf<T> &r, const SumsOf<T> &s) {
    const float m = fmaxf(r.m, s.m);
    if (m == -INFINITY) { r.a += s.a; return; }      // both empty, or NaN scores alone in one of them
    const float fs = __expf(s.m - m);         // exp(-inf) = 0 for the empty side
    rescale<PLUS>(r, __expf(r.m - m));
    fma4(r.acc, fs, s.acc);
    r.a += fs * s.a;
    if (PLUS) { fma4(r.plus, fs, s.plus); r.p += fs * s.p; }
    r.m = m;
}

// The own side's scalars: er (forward, by row) or el (by column); by row also m + log l and delta.
struct Own { float s, c1, delta; };

template <int L, int SWEEP, int PASS, bool PLUS>
__global__ __launch_bounds__(kBlock, PASS == kMerge ? 5 : 8) void additive_sweep_kernel(const AdditiveArgs a) {
    constexpr int G = 64 / L, D = 4 * L;
    constexpr bool FWD = SWEEP == kForward, BY_COLUMN = SWEEP == kByColumn;
    constexpr bool ACC = SWEEP != kByRow;              // dEr needs the sum over z > 0 alone
    static_assert(PLUS == (SWEEP == kByRow) || FWD, "by row the sums over z > 0, by column those over all edges");
    static_assert(FWD || PASS != kOnly, "gradients write or add");
    // {byte offset of the far row, its scalar} -> {offset, weight, negative where z <= 0}; by column
    // {offset, delta, er, m + log l} -> {offset, delta, weight, gate * weight}
    using W = typename std::conditional<BY_COLUMN, int4, int2>::type;
    __shared__ __align__(16) W s_far[kWavesPerBlock][fg::kItemEdges + kPad];
    __shared__ int32_t s_end[kWavesPerBlock][fg::kItemRows];
    __shared__ int32_t s_next[kWavesPerBlock];

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int head = a.head_base + (int)(blockIdx.x % (unsigned)a.n_heads);
    const int64_t item_id = (int64_t)(blockIdx.x / (unsigned)a.n_heads) * kWavesPerBlock + wave;
    if (item_id >= a.n_items) return;      // uniform per wavefront; no workgroup barriers below
    Item it = a.items[item_id];
    it.start = __builtin_amdgcn_readfirstlane(it.start); it.len = __builtin_amdgcn_readfirstlane(it.len);
    it.row = __builtin_amdgcn_readfirstlane(it.row); it.info = __builtin_amdgcn_readfirstlane(it.info);
    int part = 0;                          // the partition this item belongs to (uniform per wavefront)
    if (a.item_off) {
        const int64_t id = ((int64_t)__builtin_amdgcn_readfirstlane((int)(item_id >> 32)) << 32) |
                           (uint32_t)__builtin_amdgcn_readfirstlane((int)item_id);
        while (part + 1 < a.n_parts && id >= a.item_off[part + 1]) ++part;
    }
    const int32_t *const pos_p = a.pos + part * a.pos_stride;
    const float *const x_p = a.x + part * a.x_stride;
    const float *const far_p = a.far + part * a.far_stride + (int64_t)head * a.far_head_floats;
    const int g = lane / L, li = lane % L;
    const int f_lo = head * D + li * 4;
    const uint32_t lane_bytes = a.x_tile_bytes ? (uint32_t)head * a.x_tile_bytes + (uint32_t)li * 16u : (uint32_t)f_lo * 4u;
    const int64_t F = a.F;
    W *far = s_far[wave];
    auto out_row = [&](int64_t row) { return a.out + part * a.out_stride + row * F; };
    auto plus_row = [&](int64_t row) { return a.plus + part * a.out_stride + row * F; };
    auto state_row = [&](int64_t row) { return a.state + part * a.state_stride + (row * a.H + head) * 2; };
    auto share_row = [&](int64_t row) { return a.share + part * a.share_stride + row * a.H + head; };
    auto scalar_at = [&](int64_t row) { return row * a.own_row + (int64_t)head * a.own_head; };

    auto stage = [&](int64_t base, int n) {
        int32_t c[4];
        fg::load_four_ids(a.indices, a.indices16, base, n, lane, c);
        W w[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int off = (int)((uint32_t)c[i] * a.x_row_bytes);
            if constexpr (BY_COLUMN) {
                const float4 cf = *reinterpret_cast<const float4 *>(far_p + (int64_t)c[i] * 4);
                w[i] = make_int4(off, __float_as_int(cf.y), __float_as_int(cf.z), __float_as_int(cf.x));
            } else {
                w[i] = make_int2(off, __float_as_int(far_p[c[i]]));
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) far[4 * lane + i] = w[i];
        if (lane < kPad) far[fg::kItemEdges + lane] = w[3];
    };
    auto own_at = [&](int64_t row) {
        Own o = {0.f, 0.f, 0.f};
        if constexpr (SWEEP == kByRow) {
            const float4 cf = *reinterpret_cast<const float4 *>(a.coef + (int64_t)head * a.coef_head_floats + row * 4);
            o.c1 = cf.x; o.delta = cf.y; o.s = cf.z;
        } else {
            o.s = a.own[scalar_at(row)];
        }
        return o;
    };
    auto score = [&](const W &w, const Own &o, bool &pos) {
        float z;
        if constexpr (BY_COLUMN) z = __int_as_float(w.z) + o.s;
        else z = __int_as_float(w.y) + o.s;
        pos = z > 0.f;
        return pos ? z : z * a.slope;
    };
    // gradients: the softmax value of a staged element with score s
    auto softmax_of = [&](const W &w, const Own &o, float s) {
        if constexpr (BY_COLUMN) return __expf(s - __int_as_float(w.w));
        else return __expf(s - o.c1);
    };

    // The weights of the staged elements [b, e) of one row (1 .. 256 of them), an element per lane and step; false: no
    // score above -inf so far, nothing to add (forward only).
    auto weigh = [&](int b, int e, const Own &o, Sums &r) {
        const int n = e - b;
        float s[4];
        bool pos[4];
        if constexpr (FWD) {
            float mx = -INFINITY;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                s[i] = -INFINITY; pos[i] = false;
                if (64 * i < n) {
                    const int j = b + lane + 64 * i;
                    const float t = score(far[min(j, e - 1)], o, pos[i]);
                    s[i] = j < e ? t : -INFINITY;
                    mx = fmaxf(mx, s[i]);
                }
            }
            const float m = fmaxf(r.m, wave_max(mx));
            if (m == -INFINITY) {
#pragma unroll
                for (int i = 0; i < 4; ++i) r.a += nan_term(s[i]);
                return false;
            }
            if (r.m != -INFINITY) rescale<PLUS>(r, __expf(r.m - m));      // a later batch of a long row
            r.m = m;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (64 * i < n) {
                const int j = b + lane + 64 * i;
                float p;
                if constexpr (FWD) {
                    p = __expf(s[i] - r.m);
                } else {
                    const W w = far[min(j, e - 1)];
                    p = softmax_of(w, o, score(w, o, pos[i]));
                }
                if (j < e) {
                    if constexpr (BY_COLUMN) {
                        *reinterpret_cast<int2 *>(&far[j].z) = make_int2(__float_as_int(p), __float_as_int(pos[i] ? p : p * a.slope));
                    } else {
                        far[j].y = __float_as_int(pos[i] ? p : -p);
                        r.a += p;
                        if (PLUS) r.p += pos[i] ? p : 0.f;
                    }
                }
            }
        }
        return true;
    };
    // Adds one gathered row with signed weight w (by column: weight w, gated weight gw); keep == false: a slot without an
    // element, whose row is dropped by a select (a product with zero would turn a non-finite row into NaN in rows that do
    // not reference it).
    auto apply = [&](float w, float gw, float delta, bool keep, float4 x, const float4 &ox, Sums &r) {
        if constexpr (BY_COLUMN) {
            const float ds = gw * (group_sum<L>(dot4(x, ox)) - delta);
            r.a += keep ? ds : 0.f;
        }
        if (!keep) { w = 0.f; x = zero4(); }
        if (ACC) fma4(r.acc, BY_COLUMN ? w : fabsf(w), x);
        if (PLUS) fma4(r.plus, fmaxf(w, 0.f), x);
    };
    auto gathered = [&](const W &w) {
        return *reinterpret_cast<const float4 *>(reinterpret_cast<const char *>(x_p) + ((uint32_t)w.x + lane_bytes));
    };
    // NU steps of one row (weighed elements s0 + g, s0 + g + G, ...), all gathers issued before the first is used; only
    // the last step may have groups without an element, which re-read element e - 1.
    auto batch = [&](auto nu_tag, auto all_tag, int s0, int e, const float4 &ox, Sums &r) {
        constexpr int NU = decltype(nu_tag)::value;
        constexpr bool ALL = decltype(all_tag)::value;
        const bool last = ALL || s0 + (NU - 1) * G + g < e;
        W w[NU];
        float4 x[NU];
#pragma unroll
        for (int u = 0; u < NU; ++u) {
            w[u] = far[(u < NU - 1 || last) ? s0 + u * G + g : e - 1];
            x[u] = gathered(w[u]);
        }
#pragma unroll
        for (int u = 0; u < NU; ++u) {
            const bool keep = u < NU - 1 || last;
            if constexpr (BY_COLUMN)
                apply(__int_as_float(w[u].z), __int_as_float(w[u].w), __int_as_float(w[u].y), keep, x[u], ox, r);
            else
                apply(__int_as_float(w[u].y), 0.f, 0.f, keep, x[u], ox, r);
        }
    };
    auto walk = [&](int b, int e, const float4 &ox, Sums &r) {
        int s0 = b;
        for (; s0 + G * kU <= e; s0 += G * kU) batch(integral_constant<int, kU>(), integral_constant<bool, true>(), s0, e, ox, r);
        if (s0 >= e) return;
        const int nu = (e - s0 + G - 1) / G;    // uniform: 1 .. kU
        static_assert(kU == 4, "the tail below lists the step counts");
        if (nu == 1) batch(integral_constant<int, 1>(), integral_constant<bool, false>(), s0, e, ox, r);
        else if (nu == 2) batch(integral_constant<int, 2>(), integral_constant<bool, false>(), s0, e, ox, r);
        else if (nu == 3) batch(integral_constant<int, 3>(), integral_constant<bool, false>(), s0, e, ox, r);
        else batch(integral_constant<int, 4>(), integral_constant<bool, false>(), s0, e, ox, r);
    };
    // kU staged elements j .. of a row that a lane group walks alone, forming their weights as it goes (slots behind e hold
    // later rows' elements or the padding: loadable, given no weight).
    auto own_batch = [&](int j, int e, const Own &o, const float4 &ox, Sums &r) {
        W w[kU];
        float4 x[kU];
        float s[kU], m = r.m;
        bool pos[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u) { w[u] = far[j + u]; x[u] = gathered(w[u]); }
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            s[u] = score(w[u], o, pos[u]);
            if (FWD) m = fmaxf(m, j + u < e ? s[u] : -INFINITY);
        }
        if constexpr (FWD) {
            if (m == -INFINITY) {               // uniform inside a lane group
#pragma unroll
                for (int u = 0; u < kU; ++u) r.a += j + u < e ? nan_term(s[u]) : 0.f;
                return;
            }
            rescale<PLUS>(r, __expf(r.m - m));
            r.m = m;
        }
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const bool keep = j + u < e;
            if constexpr (BY_COLUMN) {
                const float p = softmax_of(w[u], o, s[u]);
                apply(p, pos[u] ? p : p * a.slope, __int_as_float(w[u].y), keep, x[u], ox, r);
            } else {
                float p;
                if constexpr (FWD) p = __expf(s[u] - m);
                else p = softmax_of(w[u], o, s[u]);
                r.a += keep ? p : 0.f;
                if (PLUS) r.p += (keep && pos[u]) ? p : 0.f;
                apply(pos[u] ? p : -p, 0.f, 0.f, keep, x[u], ox, r);
            }
        }
    };
    // What a row holds from earlier passes (read before its gathers are issued) and, for the gradients, its row of dout / V.
    auto load_old = [&](int64_t row, int f, auto &old, float4 &ox) {
        using T = decltype(old.acc);
        set_zero(old.acc); set_zero(old.plus);
        old.a = old.p = 0.f; old.m = -INFINITY;
        if constexpr (!FWD) ox = *reinterpret_cast<const float4 *>(a.own_x + row * F + f_lo);
        if constexpr (PASS == kMerge) {
            if constexpr (ACC) old.acc = *reinterpret_cast<const T *>(out_row(row) + f);
            if constexpr (FWD) {
                old.m = state_row(row)[0]; old.a = state_row(row)[1];
                if (PLUS) { old.plus = *reinterpret_cast<const T *>(plus_row(row) + f); old.p = *share_row(row); }
            } else {
                old.a = a.res[scalar_at(row)];
            }
        }
    };
    // Stores a row from its totals: column f on (one or four floats) in this lane, the scalars in each lane, stored where `first`.
    auto store = [&](int64_t row, int f, bool first, const Own &o, auto r, const auto &old, const float4 &ox) {
        if constexpr (FWD) {
            if (PASS == kMerge) merge<PLUS>(r, old);
            float l = r.a, share = r.p;
            if (PASS == kOnly) {
                const float inv = l == 0.f ? 0.f : 1.0f / l;
                rescale<PLUS>(r, inv);
                if (l == 0.f) { set_zero(r.acc); set_zero(r.plus); r.p = 0.f; }
                share = r.p;
            }
            store_nt(r.acc, out_row(row) + f);
            if (PLUS) store_nt(r.plus, plus_row(row) + f);
            if (first) {
                float *st = state_row(row);
                st[0] = r.m; st[1] = l;
                if (PLUS) *share_row(row) = share;
            }
        } else if constexpr (BY_COLUMN) {
            if (first) a.res[scalar_at(row)] = PASS == kMerge ? r.a + old.a : r.a;
            if (PASS == kMerge) add4(r.acc, old.acc);
            *reinterpret_cast<decltype(r.acc) *>(out_row(row) + f) = r.acc;
        } else {
            const float d = (1.f - a.slope) * (group_sum<L>(dot4(ox, r.plus)) - o.delta * r.p);
            if (first) a.res[scalar_at(row)] = PASS == kMerge ? d + old.a : d;
        }
    };
    // Rows that the wavefront shares: the lane groups' and lanes' parts are added up first.  By row the four words of a lane
    // stay together (the dot product with dout needs them), otherwise each 16-lane row of the wavefront keeps one of them.
    using Total = SumsOf<typename std::conditional<SWEEP == kByRow, float4, float>::type>;
    const int f_total = SWEEP == kByRow ? f_lo : f_lo + fg::word_of_row(lane);
    auto finish = [&](int64_t row, const Own &o, const Sums &r, const Total &old, const float4 &ox) {
        Total t;
        t.m = r.m;
        if constexpr (SWEEP == kByRow) {
            t.acc = r.acc; t.plus = r.plus;
#pragma unroll
            for (int off = L; off < 64; off <<= 1) add4(t.plus, shfl_xor4(t.plus, off));
            t.a = 0.f; t.p = wave_sum(r.p);
            if (g == 0) store(row, f_total, li == 0, o, t, old, ox);
        } else {
            t.acc = fg::groups_sum<L>(r.acc);
            t.plus = PLUS ? fg::groups_sum<L>(r.plus) : 0.f;
            t.p = PLUS ? wave_sum(r.p) : 0.f;
            if (FWD) {
                t.a = wave_sum(r.a);
            } else {                                 // the lanes of a group hold the same sum
                t.a = fg::rows_sum(r.a);
                if (L <= 8) t.a += fg::dpp_move<0x128>(t.a);
                if (L <= 4) t.a += fg::dpp_move<0x124>(t.a);
            }
            if (lane % 16 < L) store(row, f_total, lane == 0, o, t, old, ox);
        }
    };

    Total old_total;
    float4 ox = zero4();
    if (it.info < -1) {
        // several whole rows, at most 256 elements: staged once
        const int nrows = -it.info;
        // The rows that are read whole besides the gathers are touched once here, one word per row and 128 bytes, while the
        // ids are on their way: loads return in order, so a row fetched when it is needed would hold up every gather behind it.
        float touched = 0.f;
        constexpr int kLines = (D * 4 + 127) / 128;
        static_assert(fg::kItemRows * kLines <= 128, "two touches per lane cover an item's rows");
        if constexpr (!FWD || PASS == kMerge) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int t = lane + 64 * i;
                const int64_t at = (int64_t)(it.row + min(t / kLines, nrows - 1)) * F + head * D + min((t % kLines) * 32, D - 1);
                if constexpr (!FWD) touched += a.own_x[at];
                if constexpr (PASS == kMerge && ACC) touched += a.out[at];
            }
        }
        if (it.len > 0) stage(it.start, it.len);
        s_end[wave][lane] = pos_p[it.row + min(lane, nrows - 1) + 1] - it.start;
        if (lane == 0) s_next[wave] = 0;
        wave_lds_sync();
        asm volatile("" ::"v"(touched));      // keeps the loads
        if (nrows >= 2 * G && it.len <= nrows * kOwnLen) {
            // Many rows of a few elements: every lane group takes rows of its own (the next free one from a counter in LDS),
            // forms its elements' weights itself and stores the row: G rows in flight per wavefront, nothing crosses lane
            // groups.  (Against every row shared by the wavefront, gradients at 200,000 nodes of degree 7.5, 4 x 32: 790 -> 710 us.)
            int r = 0, j = 0, e = 0;
            bool live = false;
            Sums sum = sums_empty(), old;
            Own o = {0.f, 0.f, 0.f};
            for (;;) {
                if (j >= e) {
                    if (live) store(it.row + r, f_lo, li == 0, o, sum, old, ox);       // the row this group just finished
                    int rn = 0;
                    if (li == 0) rn = atomicAdd(&s_next[wave], 1);
                    r = __shfl(rn, g * L);
                    if (r >= nrows) break;
                    j = r ? s_end[wave][r - 1] : 0;
                    e = s_end[wave][r];
                    live = PASS != kMerge || e > j;
                    if (live) { o = own_at(it.row + r); load_old(it.row + r, f_lo, old, ox); }
                    sum = sums_empty();
                }
                if (j < e) { own_batch(j, e, o, ox, sum); j += kU; }
            }
            return;
        }
        int b = 0;
        for (int r = 0; r < nrows; ++r) {
            const int e = __builtin_amdgcn_readfirstlane(s_end[wave][r]);
            if (e > b || PASS != kMerge) {
                const Own o = own_at(it.row + r);
                load_old(it.row + r, f_total, old_total, ox);
                Sums sum = sums_empty();
                if (e > b && weigh(b, e, o, sum)) {
                    wave_lds_sync();
                    walk(b, e, ox, sum);
                }
                finish(it.row + r, o, sum, old_total, ox);
            }
            b = e;
        }
        return;
    }
    // one row of any length: 256 elements at a time
    const Own o = own_at(it.row);
    load_old(it.row, f_total, old_total, ox);
    Sums sum = sums_empty();
    for (int32_t base = 0; base < it.len; base += fg::kItemEdges) {
        const int n = min(fg::kItemEdges, it.len - base);
        wave_lds_sync();
        stage((int64_t)it.start + base, n);
        wave_lds_sync();
        if (weigh(0, n, o, sum)) {
            wave_lds_sync();
            walk(0, n, ox, sum);
        }
    }
    if (it.len > 0 || PASS != kMerge) finish(it.row, o, sum, old_total, ox);
}

// The passes' sums merged and divided by the sum of exponentials: from buffers [P][n_dst][...] of every pass, or (P == 1,
// buf_* == the results themselves) only divided.  plus / share may be null.
__global__ __launch_bounds__(256) void additive_merge_kernel(float4 *out, float4 *plus, float *state, float *share,
                                                             const float4 *buf_out, const float4 *buf_plus,
                                                             const float *buf_state, const float *buf_share,
                                                             uint32_t n_words, uint32_t row_words, uint32_t head_words,
                                                             int H, int P) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= n_words) return;
    const uint32_t r = i / row_words, w = i - r * row_words, h = w / head_words;
    const uint64_t pair = (uint64_t)r * H + h, pairs = (uint64_t)(n_words / row_words) * H;
    // the row's maximum over the passes first, so that every buffer enters with one factor and the loads of the running
    // sums do not wait for each other
    float m = -INFINITY;
    for (int p = 0; p < P; ++p) m = fmaxf(m, buf_state[(p * pairs + pair) * 2]);
    Sums run = sums_empty();
    run.m = m;
    if (m != -INFINITY) {
#pragma unroll 4
        for (int p = 0; p < P; ++p) {
            const float f = __expf(buf_state[(p * pairs + pair) * 2] - m);      // exp(-inf) = 0 for a pass without elements
            typedef float f4 __attribute__((ext_vector_type(4)));
            const f4 b = __builtin_nontemporal_load(reinterpret_cast<const f4 *>(buf_out) + (uint64_t)p * n_words + i);   // read once
            fma4(run.acc, f, make_float4(b.x, b.y, b.z, b.w));
            run.a += buf_state[(p * pairs + pair) * 2 + 1] * f;
            if (plus) {
                const f4 c = __builtin_nontemporal_load(reinterpret_cast<const f4 *>(buf_plus) + (uint64_t)p * n_words + i);
                fma4(run.plus, f, make_float4(c.x, c.y, c.z, c.w));
                run.p += buf_share[p * pairs + pair] * f;
            }
        }
    } else {
        for (int p = 0; p < P; ++p) run.a += buf_state[(p * pairs + pair) * 2 + 1];      // 0, or NaN
    }
    const float l = run.a;
    const float inv = l == 0.f ? 0.f : 1.0f / l;
    scale4(run.acc, inv);
    out[i] = l == 0.f ? zero4() : run.acc;
    if (plus) {
        scale4(run.plus, inv);
        plus[i] = l == 0.f ? zero4() : run.plus;
    }
    // (P == 1: the state and share in place are read by the row's other words in this launch, so they are not rewritten here)
    if (P > 1 && w == h * head_words) {
        state[pair * 2] = m; state[pair * 2 + 1] = l;
        if (plus) share[pair] = l == 0.f ? 0.f : run.p * inv;
    }
}
// share /= sum of exponentials, after the passes that merged in place
__global__ __launch_bounds__(256) void additive_share_kernel(float *share, const float *state, int64_t n_pairs) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n_pairs) return;
    const float l = state[i * 2 + 1];
    share[i] = l == 0.f ? 0.f : share[i] / l;
}

// coef[h, r] = (m + log l, <dout[r, h, :], out[r, h, :]>, er[r, h], 0), head by head so that the gathers of one head stay
// inside 16 * n_dst bytes; rows without edges (l == 0): (+inf, 0), so that every softmax value formed from them is 0.
// With plus / share also der = (1 - slope) * (<dout, plus> - delta * share).  One lane group per (row, head).
template <int L>
__global__ __launch_bounds__(256) void additive_coef_kernel(const float *out, const float *dout, const float *state,
                                                            const float *er, int64_t er_row, int64_t er_head, float *coef,
                                                            const float *plus, const float *share, float *der, float slope,
                                                            int64_t n_pairs, int64_t n_rows, int H) {
    const int64_t pair = ((int64_t)blockIdx.x * 256 + threadIdx.x) / L;
    const int li = threadIdx.x % L;
    const bool on = pair < n_pairs;
    const int64_t at = (on ? pair : 0) * (4 * L) + li * 4;
    const float4 d = *reinterpret_cast<const float4 *>(dout + at);
    const float delta = group_sum<L>(dot4(*reinterpret_cast<const float4 *>(out + at), d));
    float up = 0.f;
    if (plus) up = group_sum<L>(dot4(*reinterpret_cast<const float4 *>(plus + at), d));
    if (on && li == 0) {
        const float m = state[pair * 2], l = state[pair * 2 + 1];
        const int64_t r = pair / H, h = pair - r * H;
        const float c1 = l == 0.f ? INFINITY : m + __logf(l), dl = l == 0.f ? 0.f : delta;
        *reinterpret_cast<float4 *>(coef + (h * n_rows + r) * 4) = make_float4(c1, dl, er[r * er_row + h * er_head], 0.f);
        if (plus) der[r * er_row + h * er_head] = (1.f - slope) * (up - dl * share[pair]);
    }
}

template <int SWEEP, int PASS, bool PLUS>
int launch(int head_len, const AdditiveArgs &base, hipStream_t st) {
    AdditiveArgs a = base;
    const int per_launch = (a.H > 8 && a.H % 8 == 0) ? 8 : a.H;
    for (int hb = 0; hb < a.H; hb += per_launch) {
        a.n_heads = per_launch; a.head_base = hb;
        const int64_t blocks = ((a.n_items + kWavesPerBlock - 1) / kWavesPerBlock) * per_launch;
        if (blocks > 0x7fffffffLL) return fail(FG_ERR_SHAPE, "grid of %lld workgroups is too large", (long long)blocks);
        const dim3 grid((unsigned)blocks);
        if (head_len == 64) hipLaunchKernelGGL((additive_sweep_kernel<16, SWEEP, PASS, PLUS>), grid, dim3(kBlock), 0, st, a);
        else if (head_len == 32) hipLaunchKernelGGL((additive_sweep_kernel<8, SWEEP, PASS, PLUS>), grid, dim3(kBlock), 0, st, a);
        else hipLaunchKernelGGL((additive_sweep_kernel<4, SWEEP, PASS, PLUS>), grid, dim3(kBlock), 0, st, a);
    }
    return FG_OK;
}

int check_plan(const fg_spmm_plan *pl, int heads, int head_len) {
    if (!pl) return fail(FG_ERR_ARG, "plan is null");
    if (int drc = fg::check_device(pl)) return drc;
    if (heads < 1 || !(head_len == 16 || head_len == 32 || head_len == 64))
        return fail(FG_ERR_SHAPE, "attention takes heads of 16, 32 or 64 floats, got %d heads of %d", heads, head_len);
    if (pl->n_fixups > 0)
        return fail(FG_ERR_ARG, "attention needs a plan without split rows (fg_plan_opts.split_threshold = INT32_MAX)");
    const uint64_t F = (uint64_t)heads * head_len;
    if ((uint64_t)pl->n_src * F * 4u >= (1ull << 32) || (uint64_t)pl->n_dst * F >= (1ull << 32))
        return fail(FG_ERR_SHAPE, "attention operands of 4 GiB and more are not supported");
    return FG_OK;
}

// Floats that one pass's buffers take: running sums, maxima and sums of exponentials, and the same over z > 0.
uint64_t pass_floats(const fg_spmm_plan *pl, int heads, int head_len, bool plus) {
    return (uint64_t)pl->n_dst * heads * (head_len + 2 + (plus ? head_len + 1 : 0));
}
// Every pass into buffers of its own: several partitions, unless the plan's pass_buffers option says never or the buffers
// would take more than 8 GiB.
bool pass_buffers(const fg_spmm_plan *pl, int heads, int head_len, bool plus) {
    const int P = pl->num_col_partitions;
    return P >= 2 && pl->pass_buffers != 2 && pass_floats(pl, heads, head_len, plus) * 4u * (uint64_t)P <= (8ull << 30);
}

// x gathered head by head when that pays (the plan's scratch then holds the copy); sets the args' gathered side.
int gathered_side(const fg_spmm_plan *pl, const fg::ScratchNeed &need, const float *x_dev, int heads, int head_len, void *stream,
                  AdditiveArgs &a, int *row_floats) {
    const int F = heads * head_len;
    const bool tiled = need.tiled > 0;
    a.x = x_dev;
    if (tiled) {
        if (int rc = fg::make_tile_major(pl, x_dev, pl->n_src, F, head_len, stream)) return rc;
        a.x = pl->tiled_dev;
    }
    *row_floats = tiled ? head_len : F;
    a.x_row_bytes = (uint32_t)*row_floats * 4u;
    a.x_tile_bytes = tiled ? (uint32_t)((uint64_t)pl->n_src * head_len * 4u) : 0u;
    return FG_OK;
}

// PLUS: also plus_dev [n_dst, F] and share_dev [n_dst, H].
template <bool PLUS>
int run_forward(fg_spmm_plan *pl, const int32_t *pos_dev, const int32_t *idx_dev, const float *er_dev, int64_t er_row,
                int64_t er_head, const float *el_dev, const float *v_dev, float *out_dev, float *row_state_dev,
                float *plus_dev, float *share_dev, int heads, int head_len, float slope, void *stream) {
    if (int rc = check_plan(pl, heads, head_len)) return rc;
    if (pl->n_dst == 0) return FG_OK;
    if (!pos_dev || !er_dev || !out_dev || (pl->nnz > 0 && (!idx_dev || !el_dev || !v_dev)) ||
        (PLUS && (!row_state_dev || !plus_dev || !share_dev)))
        return fail(FG_ERR_ARG, "null device pointer");
    if ((((uintptr_t)v_dev | (uintptr_t)out_dev | (uintptr_t)plus_dev) & 15) != 0)
        return fail(FG_ERR_ARG, "attention needs 16-byte aligned arrays");
    const int F = heads * head_len;
    fg::ScratchNeed need;
    int rc = fg::additive_scratch_need(pl, heads, head_len, !row_state_dev, PLUS, &need);
    if (rc == FG_OK) rc = fg::ensure_scratch(pl, need, stream);
    if (rc != FG_OK) return rc;
    if (!row_state_dev) row_state_dev = pl->partial_dev;
    hipStream_t st = (hipStream_t)stream;
    const int P = pl->num_col_partitions;
    const int64_t width = (pl->n_src + P - 1) / P;
    AdditiveArgs a;
    int row_floats = 0;
    if ((rc = gathered_side(pl, need, v_dev, heads, head_len, stream, a, &row_floats)) != FG_OK) return rc;
    a.indices = idx_dev; a.indices16 = fg::narrow_indices(pl, idx_dev);
    a.far = el_dev; a.far_head_floats = pl->n_src;
    a.own = er_dev; a.own_row = er_row; a.own_head = er_head;
    a.coef = nullptr; a.coef_head_floats = 0; a.own_x = nullptr; a.res = nullptr;
    a.pos = pos_dev; a.items = pl->items_dev; a.n_items = pl->n_items;
    a.out = out_dev; a.plus = plus_dev; a.state = row_state_dev; a.share = share_dev;
    a.F = F; a.H = heads; a.slope = slope;
    const uint32_t n_words = (uint32_t)((uint64_t)pl->n_dst * F / 4);
    const dim3 word_grid((n_words + 255u) / 256u);
    float4 *out4 = reinterpret_cast<float4 *>(out_dev), *plus4 = reinterpret_cast<float4 *>(plus_dev);
    if (P == 1) {
        // every row is finished by the wavefront that walks it
        if (pl->n_items > 0 && (rc = launch<kForward, kOnly, PLUS>(head_len, a, st)) != FG_OK) return rc;
    } else if (pass_buffers(pl, heads, head_len, PLUS) && pl->n_items > 0) {
        // Every partition into buffers of its own (no reads of the rows' earlier state inside the gather kernel, no order
        // between the passes): one launch walks all partitions' items, one kernel merges the buffers.
        const size_t own_state = row_state_dev == pl->partial_dev ? (size_t)pl->n_dst * heads * 2 : 0;
        const size_t rows = (size_t)pl->n_dst * F, pairs = (size_t)pl->n_dst * heads;
        float *buf_out = pl->partial_dev + ((own_state + 3) & ~(size_t)3);
        float *buf_plus = PLUS ? buf_out + (size_t)P * rows : nullptr;
        float *buf_state = buf_out + (size_t)P * rows * (PLUS ? 2 : 1);
        float *buf_share = buf_state + (size_t)P * pairs * 2;
        a.item_off = pl->item_off_dev; a.n_parts = P;
        a.pos_stride = pl->n_dst + 1; a.far_stride = width; a.x_stride = width * row_floats;
        a.out = buf_out; a.plus = buf_plus; a.out_stride = (int64_t)rows;
        a.state = buf_state; a.state_stride = (int64_t)pairs * 2;
        a.share = buf_share; a.share_stride = (int64_t)pairs;
        if ((rc = launch<kForward, kWrite, PLUS>(head_len, a, st)) != FG_OK) return rc;
        hipLaunchKernelGGL(additive_merge_kernel, word_grid, dim3(256), 0, st, out4, plus4, row_state_dev, share_dev,
                           reinterpret_cast<const float4 *>(buf_out), reinterpret_cast<const float4 *>(buf_plus), buf_state,
                           buf_share, n_words, (uint32_t)(F / 4), (uint32_t)(head_len / 4), heads, P);
    } else {
        for (int p = 0; p < P; ++p) {
            const int64_t i0 = pl->item_off[p], i1 = pl->item_off[p + 1];
            if (i1 == i0) continue;
            AdditiveArgs b = a;
            b.items = a.items + i0; b.n_items = i1 - i0;
            b.pos = a.pos + (int64_t)p * (pl->n_dst + 1);
            b.far = a.far + (int64_t)p * width;
            b.x = a.x + (int64_t)p * width * row_floats;
            rc = p == 0 ? launch<kForward, kWrite, PLUS>(head_len, b, st) : launch<kForward, kMerge, PLUS>(head_len, b, st);
            if (rc != FG_OK) return rc;
        }
        hipLaunchKernelGGL(additive_merge_kernel, word_grid, dim3(256), 0, st, out4, plus4, row_state_dev, share_dev, out4, plus4,
                           row_state_dev, share_dev, n_words, (uint32_t)(F / 4), (uint32_t)(head_len / 4), heads, 1);
        if (PLUS) {
            const int64_t pairs = pl->n_dst * heads;
            hipLaunchKernelGGL(additive_share_kernel, dim3((unsigned)((pairs + 255) / 256)), dim3(256), 0, st, share_dev, row_state_dev, pairs);
        }
    }
    FG_HIP_TRY(hipGetLastError());
    return FG_OK;
}

// The gradients' passes over the far side's partitions; res is addressed by (own_row, own_head) as own is.
template <int SWEEP>
int run_backward(fg_spmm_plan *pl, const int32_t *pos_dev, const int32_t *idx_dev, const float *x_dev, const float *far_dev,
                 int far_floats, const float *own_dev, int64_t own_row, int64_t own_head, const float *coef_dev,
                 const float *own_x_dev, float *dv_dev, float *res_dev, int heads, int head_len, float slope, void *stream) {
    hipStream_t st = (hipStream_t)stream;
    const int P = pl->num_col_partitions;
    const int64_t width = (pl->n_src + P - 1) / P;
    fg::ScratchNeed need;
    int rc = fg::additive_scratch_need(pl, heads, head_len, false, false, &need, false);
    if (rc == FG_OK) rc = fg::ensure_scratch(pl, need, stream);
    if (rc != FG_OK) return rc;
    AdditiveArgs a;
    int row_floats = 0;
    if ((rc = gathered_side(pl, need, x_dev, heads, head_len, stream, a, &row_floats)) != FG_OK) return rc;
    a.indices = idx_dev; a.indices16 = fg::narrow_indices(pl, idx_dev);
    a.far = far_dev; a.far_head_floats = (int64_t)far_floats * pl->n_src;
    a.own = own_dev; a.own_row = own_row; a.own_head = own_head;
    a.coef = coef_dev; a.coef_head_floats = 4 * pl->n_dst;
    a.own_x = own_x_dev; a.out = dv_dev; a.res = res_dev;
    a.plus = a.state = a.share = nullptr;
    a.F = heads * head_len; a.H = heads; a.slope = slope;
    for (int p = 0; p < P; ++p) {
        const int64_t i0 = pl->item_off[p], i1 = pl->item_off[p + 1];
        if (i1 == i0) continue;
        AdditiveArgs b = a;
        b.items = pl->items_dev + i0; b.n_items = i1 - i0;
        b.pos = pos_dev + (int64_t)p * (pl->n_dst + 1);
        b.far = a.far + (int64_t)p * width * far_floats;
        b.x = a.x + (int64_t)p * width * row_floats;
        constexpr bool PLUS = SWEEP == kByRow;
        rc = p == 0 ? launch<SWEEP, kWrite, PLUS>(head_len, b, st) : launch<SWEEP, kMerge, PLUS>(head_len, b, st);
        if (rc != FG_OK) return rc;
    }
    FG_HIP_TRY(hipGetLastError());
    return FG_OK;
}

int run_coef(const float *out_dev, const float *dout_dev, const float *row_state_dev, const float *er_dev, int64_t er_row,
             int64_t er_head, float *coef_dev, const float *plus_dev, const float *share_dev, float *der_dev, float slope,
             int64_t n_dst, int heads, int head_len, void *stream) {
    if (n_dst < 0 || heads < 1 || !(head_len == 16 || head_len == 32 || head_len == 64))
        return fail(FG_ERR_SHAPE, "attention takes heads of 16, 32 or 64 floats, got %d heads of %d", heads, head_len);
    if (n_dst == 0) return FG_OK;
    if (!out_dev || !dout_dev || !row_state_dev || !coef_dev) return fail(FG_ERR_ARG, "null device pointer");
    if ((((uintptr_t)out_dev | (uintptr_t)dout_dev | (uintptr_t)coef_dev | (uintptr_t)plus_dev) & 15) != 0)
        return fail(FG_ERR_ARG, "attention needs 16-byte aligned arrays");
    const int64_t n_pairs = n_dst * heads;
    const int L = head_len / 4;
    const dim3 grid((unsigned)((n_pairs * L + 255) / 256));
    hipStream_t st = (hipStream_t)stream;
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(256), 0, st, out_dev, dout_dev, row_state_dev, er_dev, er_row, er_head, coef_dev,
                           plus_dev, share_dev, der_dev, slope, n_pairs, n_dst, heads);
    };
    if (L == 16) go(additive_coef_kernel<16>);
    else if (L == 8) go(additive_coef_kernel<8>);
    else go(additive_coef_kernel<4>);
    FG_HIP_TRY(hipGetLastError());
    return FG_OK;
}

int run_elv(fg_spmm_plan *pl, const int32_t *pos_t_dev, const int32_t *idx_t_dev, const float *dout_dev, const float *el_dev,
            int64_t el_row, int64_t el_head, const float *v_dev, const float *row_coef_dev, float *del_dev, float *dv_dev,
            int heads, int head_len, float slope, void *stream) {
    if (int rc = check_plan(pl, heads, head_len)) return rc;
    if ((uint64_t)pl->n_src * 16u >= (1ull << 32)) return fail(FG_ERR_SHAPE, "attention operands of 4 GiB and more are not supported");
    if (pl->n_dst == 0) return FG_OK;
    if (!pos_t_dev || !el_dev || !v_dev || !del_dev || !dv_dev || (pl->nnz > 0 && (!idx_t_dev || !dout_dev || !row_coef_dev)))
        return fail(FG_ERR_ARG, "null device pointer");
    if ((((uintptr_t)v_dev | (uintptr_t)dout_dev | (uintptr_t)dv_dev | (uintptr_t)row_coef_dev) & 15) != 0)
        return fail(FG_ERR_ARG, "attention needs 16-byte aligned arrays");
    return run_backward<kByColumn>(pl, pos_t_dev, idx_t_dev, dout_dev, row_coef_dev, 4, el_dev, el_row, el_head, nullptr, v_dev,
                                   dv_dev, del_dev, heads, head_len, slope, stream);
}

}  // namespace

namespace fg {
// The rows' (max, sum) state when the caller passes none, the passes' buffers (forward), and the head-by-head copy of the
// gathered operand.
int additive_scratch_need(const fg_spmm_plan *pl, int heads, int head_len, bool own_row_state, bool plus, ScratchNeed *need,
                          bool forward) {
    if (int rc = attention_scratch_need(pl, heads, head_len, 1, own_row_state, need, false)) return rc;
    if (forward && pass_buffers(pl, heads, head_len, plus))
        need->partial = ((need->partial + 3) & ~(size_t)3) + (size_t)pl->num_col_partitions * pass_floats(pl, heads, head_len, plus);
    return FG_OK;
}
}  // namespace fg

extern "C" int fg_graph_attention_additive_f32(fg_spmm_plan *pl, const int32_t *pos_dev, const int32_t *idx_dev,
                                               const float *er_dev, const float *el_dev, const float *v_dev,
                                               float *out_dev, float *row_state_dev, int heads, int head_len,
                                               float negative_slope, void *stream) {
    return run_forward<false>(pl, pos_dev, idx_dev, er_dev, 1, pl ? pl->n_dst : 0, el_dev, v_dev, out_dev, row_state_dev, nullptr,
                              nullptr, heads, head_len, negative_slope, stream);
}

extern "C" int fg_graph_attention_additive_train_f32(fg_spmm_plan *pl, const int32_t *pos_dev, const int32_t *idx_dev,
                                                     const float *er_dev, const float *el_dev, const float *v_dev,
                                                     float *out_dev, float *row_state_dev, float *plus_dev,
                                                     float *share_dev, int heads, int head_len, float negative_slope,
                                                     void *stream) {
    return run_forward<true>(pl, pos_dev, idx_dev, er_dev, heads, 1, el_dev, v_dev, out_dev, row_state_dev, plus_dev, share_dev,
                             heads, head_len, negative_slope, stream);
}

extern "C" int fg_graph_attention_additive_coef_f32(const float *out_dev, const float *dout_dev, const float *row_state_dev,
                                                    const float *er_dev, float *row_coef_dev, int64_t n_dst, int heads,
                                                    int head_len, void *stream) {
    if (!er_dev) return fail(FG_ERR_ARG, "null device pointer");
    return run_coef(out_dev, dout_dev, row_state_dev, er_dev, 1, n_dst, row_coef_dev, nullptr, nullptr, nullptr, 0.f, n_dst, heads,
                    head_len, stream);
}

extern "C" int fg_graph_attention_additive_train_coef_f32(const float *out_dev, const float *dout_dev,
                                                          const float *row_state_dev, const float *er_dev,
                                                          const float *plus_dev, const float *share_dev,
                                                          float *row_coef_dev, float *der_dev, int64_t n_dst, int heads,
                                                          int head_len, float negative_slope, void *stream) {
    if (n_dst > 0 && (!er_dev || !plus_dev || !share_dev || !der_dev)) return fail(FG_ERR_ARG, "null device pointer");
    return run_coef(out_dev, dout_dev, row_state_dev, er_dev, heads, 1, row_coef_dev, plus_dev, share_dev, der_dev, negative_slope,
                    n_dst, heads, head_len, stream);
}

extern "C" int fg_graph_attention_additive_backward_er_f32(fg_spmm_plan *pl, const int32_t *pos_dev,
                                                           const int32_t *idx_dev, const float *el_dev, const float *v_dev,
                                                           const float *dout_dev, const float *row_coef_dev,
                                                           float *der_dev, int heads, int head_len,
                                                           float negative_slope, void *stream) {
    if (int rc = check_plan(pl, heads, head_len)) return rc;
    if (pl->n_dst == 0) return FG_OK;
    if (!pos_dev || !dout_dev || !row_coef_dev || !der_dev || (pl->nnz > 0 && (!idx_dev || !el_dev || !v_dev)))
        return fail(FG_ERR_ARG, "null device pointer");
    if ((((uintptr_t)v_dev | (uintptr_t)dout_dev | (uintptr_t)row_coef_dev) & 15) != 0)
        return fail(FG_ERR_ARG, "attention needs 16-byte aligned arrays");
    return run_backward<kByRow>(pl, pos_dev, idx_dev, v_dev, el_dev, 1, nullptr, 1, pl->n_dst, row_coef_dev, dout_dev, nullptr,
                                der_dev, heads, head_len, negative_slope, stream);
}

extern "C" int fg_graph_attention_additive_backward_elv_f32(fg_spmm_plan *pl, const int32_t *pos_t_dev,
                                                            const int32_t *idx_t_dev, const float *dout_dev,
                                                            const float *el_dev, const float *v_dev,
                                                            const float *row_coef_dev, float *del_dev, float *dv_dev,
                                                            int heads, int head_len, float negative_slope, void *stream) {
    return run_elv(pl, pos_t_dev, idx_t_dev, dout_dev, el_dev, 1, pl ? pl->n_dst : 0, v_dev, row_coef_dev, del_dev, dv_dev, heads,
                   head_len, negative_slope, stream);
}

extern "C" int fg_graph_attention_additive_train_elv_f32(fg_spmm_plan *pl, const int32_t *pos_t_dev,
                                                         const int32_t *idx_t_dev, const float *dout_dev,
                                                         const float *el_dev, const float *v_dev,
                                                         const float *row_coef_dev, float *del_dev, float *dv_dev,
                                                         int heads, int head_len, float negative_slope, void *stream) {
    return run_elv(pl, pos_t_dev, idx_t_dev, dout_dev, el_dev, heads, 1, v_dev, row_coef_dev, del_dev, dv_dev, heads, head_len,
                   negative_slope, stream);
}
