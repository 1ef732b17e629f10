// Softmax over the stored elements of every CSR row, per head, and its gradient (gfx950).
//
//   forward : y[e, h] = exp(x[e, h] - m[v, h]) / sum_{e' in row v} exp(x[e', h] - m[v, h]),  m = row maximum
//   backward: dx[e, h] = a[e, h] * (g[e, h] - sum_{e' in row v} a[e', h] * g[e', h])
//
// x, y are [nnz, H] row-major, so a row's values are one contiguous run of len * H floats.  Both operators move
// 2 * nnz * H * 4 bytes at best (read + write; the gradient reads two arrays): they are bound by HBM bandwidth, so what
// counts is that every value is read once and that enough 128-bit loads are in flight.  The work is cut by the plan's
// items (one wavefront per run of short rows, per row, or per piece of a long row) and by its list of split rows:
//   a run of short rows   staged in LDS, several lanes per (row, head);
//   a row that fits the registers of one wavefront (Chunks::capacity; 4 heads: 8 KB of scores, 4 KB each of a and g)   finished there;
//   a row that fits those of a workgroup (four times that)   finished by four wavefronts, split or not; up to group_floats() in two
//                         sweeps by them;
//   a longer row          by its pieces: (max, sum) per head, a small kernel that merges them, a second sweep.
// That is for the head counts that are measured to gain by it, 1, 2, 3, 4, 6, 8, 16, 32 and 64 (edge_softmax_rows_kernel); any other number goes through 32-bit loads, with
// every split row in two sweeps (edge_softmax_kernel).
// Forward + backward on 232,965 nodes / 114.8 M edges against that general form: 4 heads 2529 -> 2067 us (9.2 GB that
// have to move, 4.45 TB/s; a copy of arrays this large reaches 4.8, a sum of two 5.9), 1 head 788 -> 611 us, 8 heads
// 5025 -> 4330 us; 30,000 edges, 4 heads 45 -> 19 us (one launch each way instead of three).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "fg_common.h"
#include "fg_device.h"

using fg::fail;
using fg::Fixup;
using fg::Item;
using fg::wave_lds_sync;

namespace {

constexpr int kWavesPerBlock = 4;
constexpr int kBlock = 64 * kWavesPerBlock;
constexpr int kStage = 1024;          // floats of a multi-row item staged in LDS per wavefront
// Longest row that one workgroup takes: 2^15 floats, about 13 us of it, up to 2^17 where all rows together hold 128 times as much
// (there are 256 compute units); longer ones are spread by their pieces.  us forward + backward with 2^15 / 2^16 / 2^17: one row of
// 64,000 floats among short ones 24 / 45 / 46, of 128,000 26 / 26 / 84; 500 rows of 40,000 111 / 95 / 95, 128 of 48,000 52 / 44 / 44.
constexpr int64_t kGroupFloats = 1 << 15, kGroupFloatsMost = 1 << 17;
// (A caller's own longer pieces are not worth spreading a row for: 2^17.)
int group_floats(const fg_spmm_plan *pl, int H) {
    return (int)(pl->split_threshold > 1024 ? kGroupFloatsMost : std::min(std::max(kGroupFloats, pl->nnz * H / 128), kGroupFloatsMost));
}

struct SoftmaxArgs {
    const Item *items;
    int64_t n_items;
    const Fixup *fixups;  // the split rows
    int64_t n_fixups;
    const int32_t *indptr;
    const float *x;       // forward: scores; backward: the softmax output a
    const float *g;       // backward: dL/da
    float *y;
    float2 *stats;        // per (piece, head): forward (max, sum of exp); backward (sum of a * g, 0)
    int group_floats;     // rows of more floats are left to their pieces
    int H;
    int W;                // lanes of a wavefront in use when lanes are tied to heads: the largest multiple of H <= 64
};

// Combines `v` over the lanes that hold the same head (lane % H, H a power of two <= 64), or over
// the whole wavefront when H == 1.
template <bool IS_MAX>
__device__ __forceinline__ float head_reduce(float v, int H) {
    for (int off = 32; off >= H; off >>= 1) {
        const float o = __shfl_xor(v, off);
        v = IS_MAX ? fmaxf(v, o) : v + o;
    }
    return v;
}

// The same for any H <= 64: the lanes below W (the largest multiple of H that a wavefront holds) carry head
// lane % H, the others carry nothing.  Windows of doubling length are folded towards the lanes below H, which
// then hand every lane the result of its head.
template <bool IS_MAX>
__device__ __forceinline__ float head_reduce_any(float v, int H, int W, int lane) {
    for (int off = H; off < W; off <<= 1) {
        const float o = __shfl_down(v, off);
        if (lane + off < W) v = IS_MAX ? fmaxf(v, o) : v + o;
    }
    return __shfl(v, lane % H);
}

// MODE 1: H a power of two, all 64 lanes in use; MODE 2: any H <= 64, W lanes in use.
template <bool IS_MAX, int MODE>
__device__ __forceinline__ float lanes_reduce(float v, int H, int W, int lane) {
    return MODE == 2 ? head_reduce_any<IS_MAX>(v, H, W, lane) : head_reduce<IS_MAX>(v, H);
}


// A whole row of n <= 64 * R floats (H a power of two <= 64, so lane i always meets head i % H):
// every lane's R loads are issued back to back, the row is read from memory once and the result
// is formed in registers.  No load sits under a branch: lanes past the end re-read the last float.
// l0: the lane's first index (its lane number; past every run for a lane that is not in use), W: lanes in use.
template <bool BWD, int R, int MODE>
__device__ __forceinline__ void row_in_registers(const float *x, const float *g, float *y, int n, int lane, int l0, int W, int H) {
    float v[R], w[BWD ? R : 1];
#pragma unroll
    for (int k = 0; k < R; ++k) {
        const int i = min(l0 + W * k, n - 1);
        v[k] = x[i];
        if (BWD) w[k] = g[i];
    }
    if (!BWD) {
        float m = -INFINITY;
#pragma unroll
        for (int k = 0; k < R; ++k) m = (l0 + W * k < n) ? fmaxf(m, v[k]) : m;
        m = lanes_reduce<true, MODE>(m, H, W, lane);
        float s = 0.f;
#pragma unroll
        for (int k = 0; k < R; ++k) {
            v[k] = (l0 + W * k < n) ? __expf(v[k] - m) : 0.f;
            s += v[k];
        }
        s = lanes_reduce<false, MODE>(s, H, W, lane);
        const float inv = 1.0f / s;
#pragma unroll
        for (int k = 0; k < R; ++k)
            if (l0 + W * k < n) y[l0 + W * k] = v[k] * inv;
    } else {
        float d = 0.f;
#pragma unroll
        for (int k = 0; k < R; ++k) d += (l0 + W * k < n) ? v[k] * w[k] : 0.f;
        d = lanes_reduce<false, MODE>(d, H, W, lane);
#pragma unroll
        for (int k = 0; k < R; ++k)
            if (l0 + W * k < n) y[l0 + W * k] = v[k] * (w[k] - d);
    }
}

// One run of `len` elements starting at element e0, all lanes together.
//   LANEHEAD 1: H divides 64, lane i always meets head i % H, values are read as one coalesced run.
//   LANEHEAD 2: any H <= 64: the same with the first W lanes (the largest multiple of H), the rest idle.
//   LANEHEAD 0: one head at a time, lanes stride over the elements.
// STATS_ONLY: write (max, sum) / (dot, 0) to stats[slot * H + h] instead of the result.
// NORMALISE : the row statistics come from stats[slot * H + h] (merged over the row's pieces).
template <bool BWD, int LANEHEAD, bool STATS_ONLY, bool NORMALISE>
__device__ __forceinline__ void run_together(const SoftmaxArgs &a, int64_t e0, int len, int lane, int slot) {
    const int H = a.H;
    const int64_t base = e0 * H;
    const float *x = a.x + base;
    const float *g = BWD ? a.g + base : nullptr;
    float *y = a.y + base;
    if (LANEHEAD) {
        const int n = len * H;
        const int W = LANEHEAD == 2 ? a.W : 64;
        const int l0 = (LANEHEAD == 2 && lane >= W) ? (1 << 29) : lane;
        if (!STATS_ONLY && !NORMALISE) {
            if (n <= W * 2) { row_in_registers<BWD, 2, LANEHEAD>(x, g, y, n, lane, l0, W, H); return; }
            if (n <= W * 4) { row_in_registers<BWD, 4, LANEHEAD>(x, g, y, n, lane, l0, W, H); return; }
            if (n <= W * 8) { row_in_registers<BWD, 8, LANEHEAD>(x, g, y, n, lane, l0, W, H); return; }
        }
        // longer runs: sweeps of 8 loads per lane issued back to back (lanes past the end re-read
        // the last float, so no load sits under a branch)
        constexpr int U = 8;
        const int h = LANEHEAD == 2 ? lane % H : lane & (H - 1);
        float m = 0.f, s = 0.f;
        if (NORMALISE) {
            const float2 st = a.stats[(int64_t)slot * H + h];
            m = st.x; s = st.y;
        } else if (!BWD) {
            // one sweep: running maximum, the sum rescaled whenever the maximum grows
            m = -INFINITY;
            for (int i0 = l0, b0 = 0; b0 < n; i0 += W * U, b0 += W * U) {
                float v[U];
#pragma unroll
                for (int k = 0; k < U; ++k) v[k] = x[min(i0 + W * k, n - 1)];
#pragma unroll
                for (int k = 0; k < U; ++k) {
                    const float vk = (i0 + W * k < n) ? v[k] : -INFINITY;
                    const float mn = fmaxf(m, vk);
                    s = (m == mn ? s : s * __expf(m - mn)) + (vk == -INFINITY ? 0.f : __expf(vk - mn));
                    m = mn;
                }
            }
            const float mw = lanes_reduce<true, LANEHEAD>(m, H, W, lane);
            // a lane that met no number has s = 0 (nothing, or -inf only) or NaN (a NaN among them): either stays
            s = (m == -INFINITY) ? s : s * __expf(m - mw);
            m = mw;
            s = lanes_reduce<false, LANEHEAD>(s, H, W, lane);
        } else {
            for (int i0 = l0, b0 = 0; b0 < n; i0 += W * U, b0 += W * U) {
                float v[U], w[U];
#pragma unroll
                for (int k = 0; k < U; ++k) { const int i = min(i0 + W * k, n - 1); v[k] = x[i]; w[k] = g[i]; }
#pragma unroll
                for (int k = 0; k < U; ++k) m += (i0 + W * k < n) ? v[k] * w[k] : 0.f;
            }
            m = lanes_reduce<false, LANEHEAD>(m, H, W, lane);
        }
        if (STATS_ONLY) {
            if (lane < H) a.stats[(int64_t)slot * H + lane] = make_float2(m, s);
            return;
        }
        if (!BWD) {
            const float inv = 1.0f / s;
            for (int i0 = l0, b0 = 0; b0 < n; i0 += W * U, b0 += W * U) {
                float v[U];
#pragma unroll
                for (int k = 0; k < U; ++k) v[k] = x[min(i0 + W * k, n - 1)];
#pragma unroll
                for (int k = 0; k < U; ++k)
                    if (i0 + W * k < n) y[i0 + W * k] = __expf(v[k] - m) * inv;
            }
        } else {
            for (int i0 = l0, b0 = 0; b0 < n; i0 += W * U, b0 += W * U) {
                float v[U], w[U];
#pragma unroll
                for (int k = 0; k < U; ++k) { const int i = min(i0 + W * k, n - 1); v[k] = x[i]; w[k] = g[i]; }
#pragma unroll
                for (int k = 0; k < U; ++k)
                    if (i0 + W * k < n) y[i0 + W * k] = v[k] * (w[k] - m);
            }
        }
        return;
    }
    for (int h = 0; h < H; ++h) {
        float m = 0.f, s = 0.f;
        if (NORMALISE) {
            const float2 st = a.stats[(int64_t)slot * H + h];
            m = st.x; s = st.y;
        } else if (!BWD) {
            m = -INFINITY;
            for (int j = lane; j < len; j += 64) m = fmaxf(m, x[(int64_t)j * H + h]);
            m = head_reduce<true>(m, 1);
            // -inf adds nothing, also where the run (a piece of a row) holds nothing else and m is -inf
            for (int j = lane; j < len; j += 64) { const float v = x[(int64_t)j * H + h]; s += v == -INFINITY ? 0.f : __expf(v - m); }
            s = head_reduce<false>(s, 1);
        } else {
            for (int j = lane; j < len; j += 64) m += x[(int64_t)j * H + h] * g[(int64_t)j * H + h];
            m = head_reduce<false>(m, 1);
        }
        if (STATS_ONLY) {
            if (lane == 0) a.stats[(int64_t)slot * H + h] = make_float2(m, s);
            continue;
        }
        if (!BWD) {
            const float inv = 1.0f / s;
            for (int j = lane; j < len; j += 64) y[(int64_t)j * H + h] = __expf(x[(int64_t)j * H + h] - m) * inv;
        } else {
            for (int j = lane; j < len; j += 64) y[(int64_t)j * H + h] = x[(int64_t)j * H + h] * (g[(int64_t)j * H + h] - m);
        }
    }
}

// ---- 128-bit lanes: a lane holds chunks of CH = 4 * Q consecutive floats of a run -------------------------------
//
// A chunk starts at a multiple of CH, CH a multiple of H or H one of CH, so a float's place in its chunk says its head:
//   Q = 1, A = 1, 2, 4 : H = A;        Q = 3, A = 3, 6 : H = A;
//   Q = 1, A = 4, PER  : H = 4 * G, lane i holds heads 4 * (i % G) .. + 3 (G a power of two <= 16).
// A: heads a lane sees.  The last chunk of a run is moved back to end with the run (by a multiple of H, so heads keep
// their places) and the floats that the chunk before it holds too are masked: no load is conditional or out of range.
constexpr int stage_floats(bool bwd) { return bwd ? 512 : 1024; }

template <int Q, int A, bool PER>
struct Chunks {
    static constexpr int CH = 4 * Q;
    static constexpr bool EXACT = A % CH == 0;                // a run is a whole number of chunks
    // Chunks per lane, and the wavefronts per SIMD that the registers are held to.  Measured forward + backward on
    // 114.8 M edges: 4 heads (8 and 4 chunks, 6 and 5 wavefronts) 2102 us, (16, 8; 4, 4) 2112, (4, 4; 8, 6) 2139;
    // 1 head 693, 843, 635.
    static constexpr int max_chunks(bool bwd) { return Q == 3 ? 2 : (A < 4 || bwd) ? 4 : 8; }
    static constexpr int waves(bool bwd) { return A == 4 || Q == 3 ? (bwd ? 5 : 6) : (bwd ? 6 : 8); }
    static constexpr int capacity(bool bwd, int threads) { return threads * CH * max_chunks(bwd); }
};

template <bool IS_MAX>
__device__ __forceinline__ float combine(float a, float b) { return IS_MAX ? fmaxf(a, b) : a + b; }

// Over the lanes of a wavefront that hold the same heads.
template <bool IS_MAX, int A, bool PER>
__device__ __forceinline__ void fold_lanes(float (&v)[A], int G) {
#pragma unroll
    for (int c = 0; c < A; ++c) {
        if (!PER) {
            v[c] = combine<IS_MAX>(v[c], fg::dpp_move<0xB1>(v[c]));     // quad_perm [1,0,3,2]
            v[c] = combine<IS_MAX>(v[c], fg::dpp_move<0x4E>(v[c]));     // quad_perm [2,3,0,1]
            v[c] = combine<IS_MAX>(v[c], fg::dpp_move<0x141>(v[c]));    // row_half_mirror
            v[c] = combine<IS_MAX>(v[c], fg::dpp_move<0x140>(v[c]));    // row_mirror
            v[c] = combine<IS_MAX>(v[c], __shfl_xor(v[c], 16));
            v[c] = combine<IS_MAX>(v[c], __shfl_xor(v[c], 32));
        } else {
            for (int off = 32; off >= G; off >>= 1) v[c] = combine<IS_MAX>(v[c], __shfl_xor(v[c], off));
        }
    }
}

// ... and over the workgroup's wavefronts when THREADS is a workgroup: red[wavefront][head place], one array per use.
template <bool IS_MAX, int A, bool PER, int THREADS>
__device__ __forceinline__ void fold(float (&v)[A], int G, float (*red)[64]) {
    fold_lanes<IS_MAX, A, PER>(v, G);
    if (THREADS == 64) return;
    const int lane = threadIdx.x & 63, at = PER ? (lane & (G - 1)) * A : 0;
    if (lane < (PER ? G : 1)) {
#pragma unroll
        for (int c = 0; c < A; ++c) red[threadIdx.x >> 6][at + c] = v[c];
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < A; ++c) {
        v[c] = red[0][at + c];
#pragma unroll
        for (int w = 1; w < THREADS / 64; ++w) v[c] = combine<IS_MAX>(v[c], red[w][at + c]);
    }
}

// R chunks per lane from float b0 of a run of n (n >= CH), chunk k of lane l at b0 + (l + THREADS * k) * CH.
template <int Q, int R>
__device__ __forceinline__ void load_chunks(const float *x, int n, int i0, int step, float (&v)[R][4 * Q]) {
#pragma unroll
    for (int k = 0; k < R; ++k) {
        const int s = min(i0 + step * k, n - 4 * Q);
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const fg::Words4<float> c = *reinterpret_cast<const fg::Words4<float> *>(x + s + 4 * q);
#pragma unroll
            for (int j = 0; j < 4; ++j) v[k][4 * q + j] = c.v[j];
        }
    }
}

// Whether float j of the chunk loaded for place i belongs to that place.
template <int CH, bool EXACT>
__device__ __forceinline__ bool chunk_holds(int i, int n, int j) { return EXACT ? i < n : (i < n && j >= i - (n - CH)); }

template <int Q, bool EXACT>
__device__ __forceinline__ void store_chunk(float *y, int n, int i, const float (&v)[4 * Q]) {
    if (i >= n) return;
    if (EXACT || i <= n - 4 * Q) {
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            typedef float words4 __attribute__((ext_vector_type(4), aligned(4)));
            const words4 c = {v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
            // a wavefront's stores cover whole lines when Q = 1: past the caches, 4 heads 2102 -> 2021 us; with Q = 3
            // each covers a third of its lines: 1674 -> 1842 us
            if (Q == 1) __builtin_nontemporal_store(c, reinterpret_cast<words4 *>(y + i + 4 * q));
            else *reinterpret_cast<words4 *>(y + i + 4 * q) = c;
        }
    } else {
#pragma unroll
        for (int j = 0; j < 4 * Q; ++j)
            if (j >= i - (n - 4 * Q)) y[n - 4 * Q + j] = v[j];
    }
}

// A whole row of CH <= n <= THREADS * CH * R floats: read once, finished in registers, written.
template <bool BWD, int Q, int A, bool PER, int THREADS, int R>
__device__ __forceinline__ void chunk_row(const float *x, const float *g, float *y, int n, int G, float (*red)[kWavesPerBlock][64]) {
    constexpr int CH = 4 * Q;
    constexpr bool EXACT = Chunks<Q, A, PER>::EXACT;
    const int i0 = (THREADS == 64 ? (int)(threadIdx.x & 63) : (int)threadIdx.x) * CH;
    float v[R][CH], w[BWD ? R : 1][CH];
    load_chunks<Q, R>(x, n, i0, THREADS * CH, v);
    if constexpr (BWD) load_chunks<Q, R>(g, n, i0, THREADS * CH, w);
    if constexpr (!BWD) {
        float m[A], s[A];
#pragma unroll
        for (int c = 0; c < A; ++c) { m[c] = -INFINITY; s[c] = 0.f; }
#pragma unroll
        for (int k = 0; k < R; ++k)
#pragma unroll
            for (int j = 0; j < CH; ++j) {
                if (!chunk_holds<CH, EXACT>(i0 + THREADS * CH * k, n, j)) v[k][j] = -INFINITY;
                m[j % A] = fmaxf(m[j % A], v[k][j]);
            }
        fold<true, A, PER, THREADS>(m, G, red[0]);
#pragma unroll
        for (int k = 0; k < R; ++k)
#pragma unroll
            for (int j = 0; j < CH; ++j) {
                v[k][j] = __expf(v[k][j] - m[j % A]);
                s[j % A] += v[k][j];
            }
        fold<false, A, PER, THREADS>(s, G, red[1]);
#pragma unroll
        for (int c = 0; c < A; ++c) s[c] = 1.0f / s[c];
#pragma unroll
        for (int k = 0; k < R; ++k) {
#pragma unroll
            for (int j = 0; j < CH; ++j) v[k][j] *= s[j % A];
            store_chunk<Q, EXACT>(y, n, i0 + THREADS * CH * k, v[k]);
        }
    } else {
        float d[A];
#pragma unroll
        for (int c = 0; c < A; ++c) d[c] = 0.f;
#pragma unroll
        for (int k = 0; k < R; ++k)
#pragma unroll
            for (int j = 0; j < CH; ++j)
                d[j % A] += chunk_holds<CH, EXACT>(i0 + THREADS * CH * k, n, j) ? v[k][j] * w[k][j] : 0.f;
        fold<false, A, PER, THREADS>(d, G, red[0]);
#pragma unroll
        for (int k = 0; k < R; ++k) {
#pragma unroll
            for (int j = 0; j < CH; ++j) v[k][j] *= w[k][j] - d[j % A];
            store_chunk<Q, EXACT>(y, n, i0 + THREADS * CH * k, v[k]);
        }
    }
}

// A run of n >= CH floats of any length, R chunks per thread at a time: its statistics per head, (max, sum of exp) or (sum of a * g, 0).
template <bool BWD, int Q, int A, bool PER, int THREADS>
__device__ __forceinline__ void sweep_stats(const float *x, const float *g, int n, int G, float (*red)[kWavesPerBlock][64], float (&m)[A], float (&s)[A]) {
    constexpr int CH = 4 * Q, R = Chunks<Q, A, PER>::max_chunks(BWD) > 4 ? 4 : 2;
    constexpr bool EXACT = Chunks<Q, A, PER>::EXACT;
    const int l0 = (THREADS == 64 ? (int)(threadIdx.x & 63) : (int)threadIdx.x) * CH;
#pragma unroll
    for (int c = 0; c < A; ++c) { m[c] = BWD ? 0.f : -INFINITY; s[c] = 0.f; }
    for (int i0 = l0, b0 = 0; b0 < n; i0 += THREADS * CH * R, b0 += THREADS * CH * R) {
        float v[R][CH], w[BWD ? R : 1][CH];
        load_chunks<Q, R>(x, n, i0, THREADS * CH, v);
        if constexpr (BWD) {
            load_chunks<Q, R>(g, n, i0, THREADS * CH, w);
#pragma unroll
            for (int k = 0; k < R; ++k)
#pragma unroll
                for (int j = 0; j < CH; ++j)
                    m[j % A] += chunk_holds<CH, EXACT>(i0 + THREADS * CH * k, n, j) ? v[k][j] * w[k][j] : 0.f;
        } else {
            float mn[A];
#pragma unroll
            for (int c = 0; c < A; ++c) mn[c] = m[c];
#pragma unroll
            for (int k = 0; k < R; ++k)
#pragma unroll
                for (int j = 0; j < CH; ++j) {
                    if (!chunk_holds<CH, EXACT>(i0 + THREADS * CH * k, n, j)) v[k][j] = -INFINITY;
                    mn[j % A] = fmaxf(mn[j % A], v[k][j]);
                }
            // the sum so far is rescaled once per R chunks, and only where the maximum grew
#pragma unroll
            for (int c = 0; c < A; ++c) { s[c] = m[c] == mn[c] ? s[c] : s[c] * __expf(m[c] - mn[c]); m[c] = mn[c]; }
#pragma unroll
            for (int k = 0; k < R; ++k)
#pragma unroll
                for (int j = 0; j < CH; ++j) s[j % A] += v[k][j] == -INFINITY ? 0.f : __expf(v[k][j] - m[j % A]);
        }
    }
    if constexpr (BWD) {
        fold<false, A, PER, THREADS>(m, G, THREADS == 64 ? nullptr : red[0]);
    } else {
        float own[A];
#pragma unroll
        for (int c = 0; c < A; ++c) own[c] = m[c];
        fold<true, A, PER, THREADS>(m, G, THREADS == 64 ? nullptr : red[0]);
#pragma unroll
        for (int c = 0; c < A; ++c) s[c] = own[c] == -INFINITY ? s[c] : s[c] * __expf(own[c] - m[c]);     // 0, or NaN where one was met
        fold<false, A, PER, THREADS>(s, G, THREADS == 64 ? nullptr : red[1]);
    }
}

// ... and its result from those statistics.
template <bool BWD, int Q, int A, bool PER, int THREADS>
__device__ __forceinline__ void sweep_result(const float *x, const float *g, float *y, int n, const float (&m)[A], const float (&s)[A]) {
    constexpr int CH = 4 * Q, R = Chunks<Q, A, PER>::max_chunks(BWD) > 4 ? 4 : 2;
    constexpr bool EXACT = Chunks<Q, A, PER>::EXACT;
    const int l0 = (THREADS == 64 ? (int)(threadIdx.x & 63) : (int)threadIdx.x) * CH;
    float inv[A];
#pragma unroll
    for (int c = 0; c < A; ++c) inv[c] = BWD ? 0.f : 1.0f / s[c];
    for (int i0 = l0, b0 = 0; b0 < n; i0 += THREADS * CH * R, b0 += THREADS * CH * R) {
        float v[R][CH], w[BWD ? R : 1][CH];
        load_chunks<Q, R>(x, n, i0, THREADS * CH, v);
        if constexpr (BWD) load_chunks<Q, R>(g, n, i0, THREADS * CH, w);
#pragma unroll
        for (int k = 0; k < R; ++k) {
#pragma unroll
            for (int j = 0; j < CH; ++j) {
                if constexpr (BWD) v[k][j] *= w[k][j] - m[j % A];
                else v[k][j] = __expf(v[k][j] - m[j % A]) * inv[j % A];
            }
            store_chunk<Q, EXACT>(y, n, i0 + THREADS * CH * k, v[k]);
        }
    }
}

// A whole row by one wavefront: from registers, or in two sweeps (a long row of a multi-row item at many heads).
template <bool BWD, int Q, int A, bool PER>
__device__ __forceinline__ void wave_row(const SoftmaxArgs &a, int64_t e0, int len, int lane, int G) {
    constexpr int CH = 4 * Q, RM = Chunks<Q, A, PER>::max_chunks(BWD);
    const int64_t base = e0 * a.H;
    const int n = len * a.H;
    const float *x = a.x + base, *g = BWD ? a.g + base : nullptr;
    float *y = a.y + base;
    if (n < CH) { row_in_registers<BWD, 1, Q == 1 ? 1 : 2>(x, g, y, n, lane, (Q == 3 && lane >= a.W) ? (1 << 29) : lane, a.W, a.H); return; }
    if (n <= 64 * CH) { chunk_row<BWD, Q, A, PER, 64, 1>(x, g, y, n, G, nullptr); return; }
    if constexpr (RM > 2) { if (n <= 64 * CH * 2) { chunk_row<BWD, Q, A, PER, 64, 2>(x, g, y, n, G, nullptr); return; } }
    if constexpr (RM > 4) { if (n <= 64 * CH * 4) { chunk_row<BWD, Q, A, PER, 64, 4>(x, g, y, n, G, nullptr); return; } }
    if (n <= 64 * CH * RM) { chunk_row<BWD, Q, A, PER, 64, RM>(x, g, y, n, G, nullptr); return; }
    float m[A], s[A];
    sweep_stats<BWD, Q, A, PER, 64>(x, g, n, G, nullptr, m, s);
    sweep_result<BWD, Q, A, PER, 64>(x, g, y, n, m, s);
}

// A whole row of n >= CH floats by the workgroup (every thread of it calls this): from registers, or in two sweeps.
template <bool BWD, int Q, int A, bool PER>
__device__ __forceinline__ void group_row(const SoftmaxArgs &a, int64_t e0, int len, int G, float (*red)[kWavesPerBlock][64]) {
    constexpr int CH = 4 * Q, RM = Chunks<Q, A, PER>::max_chunks(BWD), RH = (RM + 1) / 2;
    const int64_t base = e0 * a.H;
    const int n = len * a.H;
    const float *x = a.x + base, *g = BWD ? a.g + base : nullptr;
    float *y = a.y + base;
    if (n <= kBlock * CH * RH) { chunk_row<BWD, Q, A, PER, kBlock, RH>(x, g, y, n, G, red); return; }
    if (n <= kBlock * CH * RM) { chunk_row<BWD, Q, A, PER, kBlock, RM>(x, g, y, n, G, red); return; }
    float m[A], s[A];
    sweep_stats<BWD, Q, A, PER, kBlock>(x, g, n, G, red, m, s);
    sweep_result<BWD, Q, A, PER, kBlock>(x, g, y, n, m, s);
}

// Rows [row, row + nrows) of a multi-row item, as many at a time as LDS holds: their values are one contiguous run, which
// is copied to LDS with all loads in flight at once, worked on there by T lanes per (row, head), T the largest power
// of two that a wavefront has for each, and copied out.  A row that LDS does not hold goes to wave_row.
template <bool BWD, int Q, int A, bool PER>
__device__ __forceinline__ void short_rows(const SoftmaxArgs &a, const Item &it, int lane, int G, float *sx, float *sg) {
    constexpr int STAGE = stage_floats(BWD);
    const int nrows = -it.info, H = a.H;
    const int ends = a.indptr[it.row + min(lane, nrows - 1) + 1];
    int b = it.start;
    for (int q0 = 0; q0 < nrows;) {
        const int fit = __popcll(__ballot(lane >= q0 && lane < nrows && (int64_t)(ends - b) * H <= STAGE));   // ends ascend
        if (fit == 0) {
            const int e = __shfl(ends, q0);
            wave_row<BWD, Q, A, PER>(a, b, e - b, lane, G);
            b = e; ++q0;
            continue;
        }
        const int64_t base = (int64_t)b * H;
        const int nf = (__shfl(ends, q0 + fit - 1) - b) * H;
        const float *x = a.x + base, *g = BWD ? a.g + base : nullptr;
        float *y = a.y + base;
        if (nf >= 4) {
            float v[STAGE / 256][4], w[BWD ? STAGE / 256 : 1][4];
            load_chunks<1, STAGE / 256>(x, nf, lane * 4, 256, v);
            if constexpr (BWD) load_chunks<1, STAGE / 256>(g, nf, lane * 4, 256, w);
#pragma unroll
            for (int k = 0; k < STAGE / 256; ++k) {
                const int i = lane * 4 + 256 * k;
                if (i <= nf - 4) {
                    *reinterpret_cast<float4 *>(sx + i) = make_float4(v[k][0], v[k][1], v[k][2], v[k][3]);
                    if constexpr (BWD) *reinterpret_cast<float4 *>(sg + i) = make_float4(w[k][0], w[k][1], w[k][2], w[k][3]);
                } else if (i < nf) {
#pragma unroll
                    for (int j = 1; j < 4; ++j)
                        if (j >= i - (nf - 4)) { sx[nf - 4 + j] = v[k][j]; if constexpr (BWD) sg[nf - 4 + j] = w[k][j]; }
                }
            }
        } else if (lane < nf) {
            sx[lane] = x[lane];
            if (BWD) sg[lane] = g[lane];
        }
        wave_lds_sync();
        const int tasks = fit * H;
        const int T = tasks >= 64 ? 1 : 1 << (31 - __clz(64 / tasks)), slots = 64 / T;
        for (int t0 = 0; t0 < tasks; t0 += slots) {
            const int tt = t0 + lane / T, t = min(tt, tasks - 1), j0 = lane & (T - 1);
            const int q = t / H, h = t - q * H;
            const int e = __shfl(ends, q0 + q) - b, prev = __shfl(ends, max(q0 + q - 1, 0)) - b;
            const int rb = q ? prev : 0, len = tt < tasks ? e - rb : 0;
            float *r = sx + rb * H + h;
            if (!BWD) {
                float m = -INFINITY, sum = 0.f;
                for (int j = j0; j < len; j += T) m = fmaxf(m, r[j * H]);
                for (int off = 1; off < T; off <<= 1) m = fmaxf(m, __shfl_xor(m, off));
                for (int j = j0; j < len; j += T) { const float ex = __expf(r[j * H] - m); r[j * H] = ex; sum += ex; }
                for (int off = 1; off < T; off <<= 1) sum += __shfl_xor(sum, off);
                const float inv = 1.0f / sum;
                for (int j = j0; j < len; j += T) r[j * H] *= inv;
            } else {
                const float *gr = sg + rb * H + h;
                float d = 0.f;
                for (int j = j0; j < len; j += T) d += r[j * H] * gr[j * H];
                for (int off = 1; off < T; off <<= 1) d += __shfl_xor(d, off);
                for (int j = j0; j < len; j += T) r[j * H] *= gr[j * H] - d;
            }
        }
        wave_lds_sync();
#pragma unroll
        for (int k = 0; k < STAGE / 256; ++k) {
            const int i = lane * 4 + 256 * k;
            if (i <= nf - 4) {
                const float4 o = *reinterpret_cast<const float4 *>(sx + i);
                fg::Words4<float> c;
                c.v[0] = o.x; c.v[1] = o.y; c.v[2] = o.z; c.v[3] = o.w;
                *reinterpret_cast<fg::Words4<float> *>(y + i) = c;
            } else {
                for (int j = i; j < nf; ++j) y[j] = sx[j];
            }
        }
        wave_lds_sync();
        b += nf / H;
        q0 += fit;
    }
}

// A piece of a row that no workgroup takes: its statistics go to its slot, or come from there for its result.
template <bool BWD, int Q, int A, bool PER, bool STATS>
__device__ __forceinline__ void piece(const SoftmaxArgs &a, const Item &it, int lane, int G) {
    const int64_t base = (int64_t)it.start * a.H;
    const int n = it.len * a.H;
    const float *x = a.x + base, *g = BWD ? a.g + base : nullptr;
    const int at = PER ? (lane & (G - 1)) * A : 0;
    float2 *st = a.stats + (int64_t)it.info * a.H + at;
    if (n < 4 * Q) {                              // the last elements of a row, fewer floats than a chunk: one lane per head
        if (lane >= a.H) return;
        st = a.stats + (int64_t)it.info * a.H + lane;
        if (STATS) {
            float m = BWD ? 0.f : -INFINITY, s = 0.f;
            for (int i = lane; i < n; i += a.H) m = BWD ? m + x[i] * g[i] : fmaxf(m, x[i]);
            for (int i = lane; !BWD && i < n; i += a.H) s += x[i] == -INFINITY ? 0.f : __expf(x[i] - m);
            *st = make_float2(m, s);
        } else {
            const float2 t = *st;
            for (int i = lane; i < n; i += a.H) a.y[base + i] = BWD ? x[i] * (g[i] - t.x) : __expf(x[i] - t.x) * (1.0f / t.y);
        }
        return;
    }
    float m[A], s[A];
    if (STATS) {
        sweep_stats<BWD, Q, A, PER, 64>(x, g, n, G, nullptr, m, s);
        if (lane < (PER ? G : 1)) {
#pragma unroll
            for (int c = 0; c < A; ++c) st[c] = make_float2(m[c], s[c]);
        }
    } else {
#pragma unroll
        for (int c = 0; c < A; ++c) { const float2 t = st[c]; m[c] = t.x; s[c] = t.y; }
        sweep_result<BWD, Q, A, PER, 64>(x, g, a.y + base, n, m, s);
    }
}

// One workgroup per split row first (a row longer than a workgroup holds is left to its pieces), then four items each.
template <bool BWD, int Q, int A, bool PER>
__device__ __forceinline__ void rows_body(const SoftmaxArgs &a) {
    __shared__ __align__(16) float s_x[kWavesPerBlock][stage_floats(BWD)];
    __shared__ __align__(16) float s_g[BWD ? kWavesPerBlock : 1][BWD ? stage_floats(BWD) : 4];
    __shared__ float red[2][kWavesPerBlock][64];
    constexpr int wave_cap = Chunks<Q, A, PER>::capacity(BWD, 64);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int H = a.H, G = PER ? H / 4 : 1;
    if ((int64_t)blockIdx.x < a.n_fixups) {
        const int row = a.fixups[blockIdx.x].row;
        const int b = a.indptr[row], len = a.indptr[row + 1] - b;
        const int64_t n = (int64_t)len * H;
        if (n > a.group_floats) return;
        if (n <= wave_cap) { if (wave == 0) wave_row<BWD, Q, A, PER>(a, b, len, lane, G); }
        else group_row<BWD, Q, A, PER>(a, b, len, G, red);
        return;
    }
    const int64_t first = ((int64_t)blockIdx.x - a.n_fixups) * kWavesPerBlock;
    // a whole row of one item that only the workgroup holds is everybody's work, after each wavefront's own
    auto shared_row = [&](const Item &it) { return it.info == -1 && (int64_t)it.len * H > wave_cap; };
    if (first + wave < a.n_items) {
        const Item it = a.items[first + wave];
        if (it.len == 0 || shared_row(it)) {
        } else if (it.info >= 0) {
            const int len = a.indptr[it.row + 1] - a.indptr[it.row];
            if ((int64_t)len * H > a.group_floats) piece<BWD, Q, A, PER, true>(a, it, lane, G);
        } else if (it.info == -1) {
            wave_row<BWD, Q, A, PER>(a, it.start, it.len, lane, G);
        } else {
            short_rows<BWD, Q, A, PER>(a, it, lane, G, s_x[wave], s_g[BWD ? wave : 0]);
        }
    }
    for (int q = 0; q < kWavesPerBlock && first + q < a.n_items; ++q) {     // uniform over the workgroup
        const Item it = a.items[first + q];
        if (!shared_row(it)) continue;
        group_row<BWD, Q, A, PER>(a, it.start, it.len, G, red);
        __syncthreads();                                                    // red is free again
    }
}

template <int Q, int A, bool PER>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(Chunks<Q, A, PER>::waves(false), 8))) void edge_softmax_rows_kernel(const SoftmaxArgs a) { rows_body<false, Q, A, PER>(a); }
template <int Q, int A, bool PER>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(Chunks<Q, A, PER>::waves(true), 8))) void edge_softmax_rows_backward_kernel(const SoftmaxArgs a) { rows_body<true, Q, A, PER>(a); }

// The pieces of the rows that no workgroup holds, with their rows' merged statistics.
template <bool BWD, int Q, int A, bool PER>
__global__ __launch_bounds__(kBlock) void edge_softmax_pieces_kernel(const SoftmaxArgs a) {
    const int lane = threadIdx.x & 63;
    const int64_t item_id = (int64_t)blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6);
    if (item_id >= a.n_items) return;         // uniform per wavefront; no workgroup barriers below
    const Item it = a.items[item_id];
    if (it.info < 0) return;
    if ((int64_t)(a.indptr[it.row + 1] - a.indptr[it.row]) * a.H > a.group_floats) piece<BWD, Q, A, PER, false>(a, it, lane, PER ? a.H / 4 : 1);
}

// PIECES == false: rows held whole by an item are finished, pieces write their statistics.
// PIECES == true : pieces only, normalised with the merged statistics of their row.
template <bool BWD, int LANEHEAD, bool PIECES>
__device__ __forceinline__ void edge_softmax_body(const SoftmaxArgs &a) {
    __shared__ float s_x[kWavesPerBlock][kStage];
    __shared__ float s_g[BWD ? kWavesPerBlock : 1][BWD ? kStage : 1];
    const int lane = threadIdx.x & 63;
    const int64_t item_id = (int64_t)blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6);
    if (item_id >= a.n_items) return;         // uniform per wavefront; no workgroup barriers below
    const Item it = a.items[item_id];
    if (it.len == 0) return;
    if (it.info >= 0) {
        if (PIECES) run_together<BWD, LANEHEAD, false, true>(a, it.start, it.len, lane, it.info);
        else run_together<BWD, LANEHEAD, true, false>(a, it.start, it.len, lane, it.info);
        return;
    }
    if (PIECES) return;
    if (it.info == -1) {
        run_together<BWD, LANEHEAD, false, false>(a, it.start, it.len, lane, 0);
        return;
    }
    // several whole rows: lane q keeps the end of row q
    const int nrows = -it.info;
    const int H = a.H;
    const int ends = a.indptr[it.row + min(lane, nrows - 1) + 1];
    const int nf = it.len * H;
    if (nf <= kStage) {
        // The item's values are one contiguous run: copy it to LDS with coalesced loads, let one
        // lane per (row, head) work on its row there, and copy the result out the same way.
        float *sx = s_x[threadIdx.x >> 6];
        float *sg = s_g[BWD ? (threadIdx.x >> 6) : 0];
        const int64_t base = (int64_t)it.start * H;
        for (int i0 = 0; i0 < nf; i0 += 256) {
            float v[4], w[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int i = min(i0 + lane + 64 * k, nf - 1);
                v[k] = a.x[base + i];
                if (BWD) w[k] = a.g[base + i];
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int i = i0 + lane + 64 * k;
                if (i < nf) { sx[i] = v[k]; if (BWD) sg[i] = w[k]; }
            }
        }
        wave_lds_sync();
        const int tasks = nrows * H;
        for (int t0 = 0; t0 < tasks; t0 += 64) {
            const int t = min(t0 + lane, tasks - 1);
            const int q = t / H, h = t - q * H;
            const int prev = __shfl(ends, max(q - 1, 0));
            const int e = __shfl(ends, q) - it.start;
            const int b = q ? prev - it.start : 0;
            if (t0 + lane < tasks && e > b) {
                float *r = sx + b * H + h;
                const int len = e - b;
                if (!BWD) {
                    float m = r[0];
                    for (int j = 1; j < len; ++j) m = fmaxf(m, r[j * H]);
                    float sum = 0.f;
                    for (int j = 0; j < len; ++j) { const float ex = __expf(r[j * H] - m); r[j * H] = ex; sum += ex; }
                    const float inv = 1.0f / sum;
                    for (int j = 0; j < len; ++j) r[j * H] *= inv;
                } else {
                    const float *gr = sg + b * H + h;
                    float d = 0.f;
                    for (int j = 0; j < len; ++j) d += r[j * H] * gr[j * H];
                    for (int j = 0; j < len; ++j) r[j * H] *= gr[j * H] - d;
                }
            }
        }
        wave_lds_sync();
        for (int i = lane; i < nf; i += 64) a.y[base + i] = sx[i];
        return;
    }
    if ((int64_t)it.len * H >= 32 * (int64_t)nrows) {
        // long enough rows: the wavefront takes them one after the other
        int b = it.start;
        for (int q = 0; q < nrows; ++q) {
            const int e = __shfl(ends, q);
            if (e > b) run_together<BWD, LANEHEAD, false, false>(a, b, e - b, lane, 0);
            b = e;
        }
        return;
    }
    // short rows: one lane per (row, head), walking that row's values for its head
    const int tasks = nrows * H;
    for (int t0 = 0; t0 < tasks; t0 += 64) {
        const int t = min(t0 + lane, tasks - 1);
        const int q = t / H, h = t - q * H;
        const int prev = __shfl(ends, max(q - 1, 0));
        const int e = __shfl(ends, q);
        const int b = q ? prev : it.start;
        if (t0 + lane < tasks && e > b) {
            const float *x = a.x + (int64_t)b * H + h;
            float *y = a.y + (int64_t)b * H + h;
            const int len = e - b;
            if (!BWD) {
                float m = x[0];
                for (int j = 1; j < len; ++j) m = fmaxf(m, x[(int64_t)j * H]);
                float s = 0.f;
                for (int j = 0; j < len; ++j) s += __expf(x[(int64_t)j * H] - m);
                const float inv = 1.0f / s;
                for (int j = 0; j < len; ++j) y[(int64_t)j * H] = __expf(x[(int64_t)j * H] - m) * inv;
            } else {
                const float *g = a.g + (int64_t)b * H + h;
                float d = 0.f;
                for (int j = 0; j < len; ++j) d += x[(int64_t)j * H] * g[(int64_t)j * H];
                for (int j = 0; j < len; ++j) y[(int64_t)j * H] = x[(int64_t)j * H] * (g[(int64_t)j * H] - d);
            }
        }
    }
}

// The forward kernel is held to 64 registers (8 wavefronts per SIMD); the gradient kernel is bound
// by its two LDS staging rows per wavefront instead.
template <int LANEHEAD, bool PIECES>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(8, 8))) void edge_softmax_kernel(const SoftmaxArgs a) {
    edge_softmax_body<false, LANEHEAD, PIECES>(a);
}
template <int LANEHEAD, bool PIECES>
__global__ __launch_bounds__(kBlock) void edge_softmax_backward_kernel(const SoftmaxArgs a) {
    edge_softmax_body<true, LANEHEAD, PIECES>(a);
}

// Merges the pieces' statistics of every split row of more than `above` floats and writes the row's statistics back to each of
// its pieces.  kMergeLanes lanes per (split row, head): a row of 24,000 elements is 190 pieces on a small graph, which one lane
// takes longer over than the two sweeps around this launch (4 heads, whole call: 32 us, 20 with pieces of 1024).
constexpr int kMergeLanes = 16;
template <bool IS_MAX>
__device__ __forceinline__ float merge_lanes(float v) {
    for (int off = 1; off < kMergeLanes; off <<= 1) { const float o = __shfl_xor(v, off); v = IS_MAX ? fmaxf(v, o) : v + o; }
    return v;
}
template <bool BWD>
__device__ __forceinline__ float2 merged_stats(const float2 *s, int n, int H, int lane) {
    auto load = [&](int q) { return s[(int64_t)(lane + q * kMergeLanes) * H]; };
    const int mine = lane < n ? (n - lane + kMergeLanes - 1) / kMergeLanes : 0;
    float m = BWD ? 0.f : -INFINITY, sum = 0.f;
    fg::each_piece(0, mine, load, [&](int, const float2 &c) { m = BWD ? m + c.x : fmaxf(m, c.x); });
    m = merge_lanes<!BWD>(m);
    if (!BWD) {
        fg::each_piece(0, mine, load, [&](int, const float2 &c) { sum += c.y * __expf(c.x - m); });
        sum = merge_lanes<false>(sum);
    }
    return make_float2(m, sum);
}
template <bool BWD>
__global__ __launch_bounds__(256) void edge_softmax_merge_kernel(const Fixup *fixups, int64_t n_fixups, const int32_t *indptr,
                                                                 int above, float2 *stats, int H) {
    const int64_t t = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kMergeLanes;
    if (t >= n_fixups * H) return;
    const Fixup fx = fixups[t / H];
    if ((int64_t)(indptr[fx.row + 1] - indptr[fx.row]) * H <= above) return;
    const int lane = threadIdx.x % kMergeLanes;
    float2 *s = stats + (int64_t)fx.slot0 * H + (int)(t % H);
    const float2 row = merged_stats<BWD>(s, fx.n_pieces, H, lane);
    for (int p = lane; p < fx.n_pieces; p += kMergeLanes) s[(int64_t)p * H] = row;
}

// ---- statistics only, and the fused normalise-and-relayout step ------------------------------------
//
// For attention without a stored softmax: row_stats[v, h] = (max, sum of exp(x - max)) over row v, then
// edge_softmax_head_major_kernel writes exp(x - max) / sum straight into the head-major, traversal-ordered
// weight array that the per-head SpMM streams -- the [nnz, H] softmax array is never written or re-read.

template <int LANEHEAD>
__global__ __launch_bounds__(kBlock) void edge_softmax_stats_kernel(const SoftmaxArgs a, float2 *row_stats) {
    const int lane = threadIdx.x & 63;
    const int64_t item_id = (int64_t)blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6);
    if (item_id >= a.n_items) return;         // uniform per wavefront; no workgroup barriers below
    const Item it = a.items[item_id];
    if (it.len == 0) return;
    if (it.info >= 0) {                       // a piece: its statistics go to the plan's scratch, merged later
        run_together<false, LANEHEAD, true, false>(a, it.start, it.len, lane, it.info);
        return;
    }
    SoftmaxArgs rows = a;
    rows.stats = row_stats;                   // whole rows write their own entry, slot = row
    const int nrows = -it.info;
    const int ends = a.indptr[it.row + min(lane, nrows - 1) + 1];
    int b = it.start;
    for (int q = 0; q < nrows; ++q) {
        const int e = __shfl(ends, q);
        if (e > b) run_together<false, LANEHEAD, true, false>(rows, b, e - b, lane, it.row + q);
        b = e;
    }
}

// Merges the pieces of every split row and writes the row's entry of row_stats.
__global__ __launch_bounds__(256) void edge_softmax_stats_merge_kernel(const Fixup *fixups, int64_t n_fixups,
                                                                       const float2 *stats, float2 *row_stats, int H) {
    const int64_t t = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kMergeLanes;
    if (t >= n_fixups * H) return;
    const Fixup fx = fixups[t / H];
    const int h = (int)(t % H), lane = threadIdx.x % kMergeLanes;
    const float2 row = merged_stats<false>(stats + (int64_t)fx.slot0 * H + h, fx.n_pieces, H, lane);
    if (lane == 0) row_stats[(int64_t)fx.row * H + h] = row;
}

// dst[h, e'] = exp(x[pos[e'], h] - max) / sum with the statistics of the row of stored element pos[e'].
__global__ __launch_bounds__(256) void edge_softmax_head_major_kernel(const float *x, const float2 *row_stats,
                                                                      const int32_t *edge_row, const int32_t *pos,
                                                                      int64_t n, int H, float *dst) {
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n) return;
    const int64_t at = pos ? (int64_t)pos[e] : e;
    const float *xs = x + at * H;
    const float2 *st = row_stats + (int64_t)edge_row[at] * H;
    for (int h = 0; h < H; ++h) dst[(int64_t)h * n + e] = __expf(xs[h] - st[h].x) / st[h].y;
}

// The same for H = 4 * Q heads and 16-byte aligned arrays: an element's scores by Q 128-bit loads and its row's
// statistics by 2 Q, two elements per lane (a block apart: every store of a wavefront covers 64 consecutive elements
// of one head); exp and division as in the kernel above, so both give the same bits.
template <int Q>
__global__ __launch_bounds__(256) void edge_softmax_head_major_vec_kernel(const float *x, const float2 *row_stats,
                                                                          const int32_t *edge_row, const int32_t *pos,
                                                                          int64_t n, float *dst) {
    constexpr int H = 4 * Q;
    const int64_t e0 = (int64_t)blockIdx.x * 512 + threadIdx.x;
    float4 xs[2][Q], st[2][2 * Q];
    bool ok[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int64_t e = e0 + 256 * j;
        ok[j] = e < n;
        const int64_t ec = ok[j] ? e : n - 1;                   // clamped: no branch around the loads
        const int64_t at = pos ? (int64_t)pos[ec] : ec;
        const float4 *xp = reinterpret_cast<const float4 *>(x + at * H);
        const float4 *sp = reinterpret_cast<const float4 *>(row_stats + (int64_t)edge_row[at] * H);
#pragma unroll
        for (int q = 0; q < Q; ++q) xs[j][q] = xp[q];
#pragma unroll
        for (int q = 0; q < 2 * Q; ++q) st[j][q] = sp[q];       // (max, sum) of heads 2q and 2q + 1
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        if (!ok[j]) continue;
        float *d = dst + e0 + 256 * j;
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            d[(int64_t)(4 * q + 0) * n] = __expf(xs[j][q].x - st[j][2 * q].x) / st[j][2 * q].y;
            d[(int64_t)(4 * q + 1) * n] = __expf(xs[j][q].y - st[j][2 * q].z) / st[j][2 * q].w;
            d[(int64_t)(4 * q + 2) * n] = __expf(xs[j][q].z - st[j][2 * q + 1].x) / st[j][2 * q + 1].y;
            d[(int64_t)(4 * q + 3) * n] = __expf(xs[j][q].w - st[j][2 * q + 1].z) / st[j][2 * q + 1].w;
        }
    }
}

template <bool BWD>
void launch_merge(const fg_spmm_plan *pl, const SoftmaxArgs &a, int above, hipStream_t st) {
    const int64_t threads = pl->n_fixups * a.H * kMergeLanes;
    hipLaunchKernelGGL(edge_softmax_merge_kernel<BWD>, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, st,
                       pl->fixups_dev, pl->n_fixups, a.indptr, above, a.stats, a.H);
}

template <bool BWD, int LANEHEAD>
void launch_both(const fg_spmm_plan *pl, const SoftmaxArgs &a, hipStream_t st) {
    const dim3 grid((unsigned)((pl->n_items + kWavesPerBlock - 1) / kWavesPerBlock));
    if (BWD) hipLaunchKernelGGL((edge_softmax_backward_kernel<LANEHEAD, false>), grid, dim3(kBlock), 0, st, a);
    else hipLaunchKernelGGL((edge_softmax_kernel<LANEHEAD, false>), grid, dim3(kBlock), 0, st, a);
    if (pl->n_fixups > 0) {
        launch_merge<BWD>(pl, a, 0, st);
        if (BWD) hipLaunchKernelGGL((edge_softmax_backward_kernel<LANEHEAD, true>), grid, dim3(kBlock), 0, st, a);
        else hipLaunchKernelGGL((edge_softmax_kernel<LANEHEAD, true>), grid, dim3(kBlock), 0, st, a);
    }
}

template <bool BWD, int Q, int A, bool PER>
void launch_rows(const fg_spmm_plan *pl, const SoftmaxArgs &a, hipStream_t st) {
    const int64_t item_blocks = (pl->n_items + kWavesPerBlock - 1) / kWavesPerBlock;
    const dim3 grid((unsigned)(item_blocks + pl->n_fixups));
    if (BWD) hipLaunchKernelGGL((edge_softmax_rows_backward_kernel<Q, A, PER>), grid, dim3(kBlock), 0, st, a);
    else hipLaunchKernelGGL((edge_softmax_rows_kernel<Q, A, PER>), grid, dim3(kBlock), 0, st, a);
    if (pl->n_fixups == 0 || pl->max_len * a.H <= a.group_floats) return;
    launch_merge<BWD>(pl, a, a.group_floats, st);
    hipLaunchKernelGGL((edge_softmax_pieces_kernel<BWD, Q, A, PER>), dim3((unsigned)item_blocks), dim3(kBlock), 0, st, a);
}

// How a wavefront's lanes meet the heads: 1: H divides 64; 2: any other H <= 64 (the lanes past the largest multiple of
// H stay idle); 0: more heads than lanes, one head at a time.
int lane_mode(int H) { return H > 64 ? 0 : (H & (H - 1)) == 0 ? 1 : 2; }

template <bool BWD>
void launch_heads(const fg_spmm_plan *pl, const SoftmaxArgs &a, int mode, hipStream_t st) {
    switch (a.H) {
        case 1: return launch_rows<BWD, 1, 1, false>(pl, a, st);
        case 2: return launch_rows<BWD, 1, 2, false>(pl, a, st);
        case 3: return launch_rows<BWD, 3, 3, false>(pl, a, st);
        case 4: return launch_rows<BWD, 1, 4, false>(pl, a, st);
        case 6: return launch_rows<BWD, 3, 6, false>(pl, a, st);
        case 8: case 16: case 32: case 64: return launch_rows<BWD, 1, 4, true>(pl, a, st);
        default: break;
    }
    if (mode == 2) launch_both<BWD, 2>(pl, a, st);
    else launch_both<BWD, 0>(pl, a, st);
}

int softmax_run(fg_spmm_plan *pl, const int32_t *indptr, const float *x, const float *g, float *y,
                int H, void *stream, bool bwd) {
    if (!pl) return fail(FG_ERR_ARG, "plan is null");
    if (int drc = fg::check_device(pl)) return drc;
    if (pl->num_col_partitions != 1) return fail(FG_ERR_ARG, "edge softmax needs a plan with one column partition");
    if (H < 1) return fail(FG_ERR_SHAPE, "number of heads must be positive, got %d", H);
    if (pl->nnz == 0 || pl->n_items == 0) return FG_OK;
    if (!indptr || !x || !y || (bwd && !g)) return fail(FG_ERR_ARG, "null device pointer");
    if ((pl->n_items + kWavesPerBlock - 1) / kWavesPerBlock + pl->n_fixups > 0x7fffffffLL)
        return fail(FG_ERR_SHAPE, "too many work items for one grid");
    fg::ScratchNeed need;
    int rc = fg::softmax_scratch_need(pl, H, &need);
    if (rc == FG_OK) rc = fg::ensure_scratch(pl, need, stream);
    if (rc != FG_OK) return rc;
    SoftmaxArgs a;
    a.items = pl->items_dev; a.n_items = pl->n_items; a.indptr = indptr;
    a.fixups = pl->fixups_dev; a.n_fixups = pl->n_fixups;
    a.x = x; a.g = g; a.y = y; a.stats = reinterpret_cast<float2 *>(pl->partial_dev); a.H = H;
    a.group_floats = group_floats(pl, H);
    hipStream_t st = (hipStream_t)stream;
    const int mode = lane_mode(H);
    a.W = H <= 64 ? 64 / H * H : 64;
    if (bwd) launch_heads<true>(pl, a, mode, st);
    else launch_heads<false>(pl, a, mode, st);
    FG_HIP_TRY(hipGetLastError());
    return FG_OK;
}

}  // namespace

namespace fg {
// (max, sum) per head for every piece of a split row
int softmax_scratch_need(const fg_spmm_plan *pl, int heads, ScratchNeed *need) {
    if (heads < 1) return fail(FG_ERR_SHAPE, "number of heads must be positive, got %d", heads);
    need->partial = (size_t)pl->max_slots_in_partition * 2 * (size_t)heads;
    need->tiled = 0;
    return FG_OK;
}
}  // namespace fg

extern "C" int fg_edge_softmax_f32(fg_spmm_plan *plan, const int32_t *indptr_dev, const float *scores_dev,
                                   float *out_dev, int heads, void *stream) {
    return softmax_run(plan, indptr_dev, scores_dev, nullptr, out_dev, heads, stream, false);
}

extern "C" int fg_edge_softmax_stats_f32(fg_spmm_plan *pl, const int32_t *indptr_dev, const float *scores_dev,
                                         float *row_stats_dev, int heads, void *stream) {
    if (!pl) return fail(FG_ERR_ARG, "plan is null");
    if (int drc = fg::check_device(pl)) return drc;
    if (pl->num_col_partitions != 1) return fail(FG_ERR_ARG, "edge softmax needs a plan with one column partition");
    if (heads < 1) return fail(FG_ERR_SHAPE, "number of heads must be positive, got %d", heads);
    if (pl->nnz == 0 || pl->n_items == 0) return FG_OK;
    if (!indptr_dev || !scores_dev || !row_stats_dev) return fail(FG_ERR_ARG, "null device pointer");
    if (((uintptr_t)row_stats_dev & 7) != 0) return fail(FG_ERR_ARG, "row_stats must be 8-byte aligned");
    fg::ScratchNeed need;
    int rc = fg::softmax_scratch_need(pl, heads, &need);
    if (rc == FG_OK) rc = fg::ensure_scratch(pl, need, stream);
    if (rc != FG_OK) return rc;
    SoftmaxArgs a;
    a.items = pl->items_dev; a.n_items = pl->n_items; a.indptr = indptr_dev;
    a.fixups = pl->fixups_dev; a.n_fixups = pl->n_fixups;
    a.x = scores_dev; a.g = nullptr; a.y = nullptr; a.stats = reinterpret_cast<float2 *>(pl->partial_dev); a.H = heads;
    hipStream_t st = (hipStream_t)stream;
    float2 *row_stats = reinterpret_cast<float2 *>(row_stats_dev);
    const dim3 grid((unsigned)((pl->n_items + kWavesPerBlock - 1) / kWavesPerBlock));
    a.W = heads <= 64 ? 64 / heads * heads : 64;
    const int mode = lane_mode(heads);
    if (mode == 1) hipLaunchKernelGGL(edge_softmax_stats_kernel<1>, grid, dim3(kBlock), 0, st, a, row_stats);
    else if (mode == 2) hipLaunchKernelGGL(edge_softmax_stats_kernel<2>, grid, dim3(kBlock), 0, st, a, row_stats);
    else hipLaunchKernelGGL(edge_softmax_stats_kernel<0>, grid, dim3(kBlock), 0, st, a, row_stats);
    if (pl->n_fixups > 0) {
        const int64_t threads = pl->n_fixups * heads * kMergeLanes;
        hipLaunchKernelGGL(edge_softmax_stats_merge_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, st,
                           pl->fixups_dev, pl->n_fixups, a.stats, row_stats, heads);
    }
    FG_HIP_TRY(hipGetLastError());
    return FG_OK;
}

extern "C" int fg_edge_softmax_head_major_f32(const float *scores_dev, const float *row_stats_dev,
                                              const int32_t *edge_row_dev, const int32_t *edge_pos_dev, int64_t n_edges,
                                              int heads, float *dst_dev, void *stream) {
    if (n_edges < 0 || heads < 1) return fail(FG_ERR_ARG, "fg_edge_softmax_head_major_f32: bad size");
    if (n_edges == 0) return FG_OK;
    if (!scores_dev || !row_stats_dev || !edge_row_dev || !dst_dev) return fail(FG_ERR_ARG, "null device pointer");
    const int64_t blocks = (n_edges + 255) / 256;
    if (blocks > 0x7fffffffLL) return fail(FG_ERR_SHAPE, "too many edges for one grid");
    hipStream_t st = (hipStream_t)stream;
    const float2 *stats = reinterpret_cast<const float2 *>(row_stats_dev);
    const dim3 wide((unsigned)((n_edges + 511) / 512));
    const bool aligned = (((uintptr_t)scores_dev | (uintptr_t)row_stats_dev) & 15) == 0;
    if (aligned && heads == 4)
        hipLaunchKernelGGL(edge_softmax_head_major_vec_kernel<1>, wide, dim3(256), 0, st, scores_dev, stats, edge_row_dev,
                           edge_pos_dev, n_edges, dst_dev);
    else if (aligned && heads == 8)
        hipLaunchKernelGGL(edge_softmax_head_major_vec_kernel<2>, wide, dim3(256), 0, st, scores_dev, stats, edge_row_dev,
                           edge_pos_dev, n_edges, dst_dev);
    else
        hipLaunchKernelGGL(edge_softmax_head_major_kernel, dim3((unsigned)blocks), dim3(256), 0, st,
                           scores_dev, stats, edge_row_dev, edge_pos_dev, n_edges, heads, dst_dev);
    FG_HIP_TRY(hipGetLastError());
    return FG_OK;
}

extern "C" int fg_edge_softmax_backward_f32(fg_spmm_plan *plan, const int32_t *indptr_dev,
                                            const float *softmax_dev, const float *grad_softmax_dev,
                                            float *grad_scores_dev, int heads, void *stream) {
    return softmax_run(plan, indptr_dev, softmax_dev, grad_softmax_dev, grad_scores_dev, heads, stream, true);
}
