// Device-side helpers shared by the kernels (included by .hip files only).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace fg {

// Four consecutive elements that are only known to be aligned like one of them (4 bytes for 32-bit words, 2 for
// 16-bit ones): read with one 128-bit or 64-bit load.
template <typename T> struct __attribute__((packed, aligned(sizeof(T) < 4 ? sizeof(T) : 4))) Words4 { T v[4]; };

// o[i] = p[min(4 * lane + i, n - 1) * stride], n >= 1: the lane's four consecutive elements of a
// stream of n, lanes past the end repeating the last element so that no load is conditional.
// With unit stride and n >= 4 (both uniform) that is one 128-bit load per lane from a window that
// is shifted back to end at the last element.
template <typename T>
__device__ __forceinline__ void load_four(const T *p, int n, int lane, int stride, T (&o)[4]) {
    if (stride == 1 && n >= 4) {
        const int s = min(4 * lane, n - 4), d = 4 * lane - s;
        const Words4<T> c = *reinterpret_cast<const Words4<T> *>(p + s);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int k = min(d + i, 3);
            o[i] = k == 0 ? c.v[0] : k == 1 ? c.v[1] : k == 2 ? c.v[2] : c.v[3];
        }
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = p[(int64_t)min(4 * lane + i, n - 1) * stride];
    }
}

// The lane's four column ids of a stream of n (as load_four): from the 16-bit copy `ids16` when there is one
// (uniform over the wavefront), else from `ids`.
__device__ __forceinline__ void load_four_ids(const int32_t *ids, const uint16_t *ids16, int64_t base, int n, int lane,
                                              int32_t (&c)[4]) {
    if (ids16) {
        uint16_t c16[4];
        load_four(ids16 + base, n, lane, 1, c16);
#pragma unroll
        for (int i = 0; i < 4; ++i) c[i] = c16[i];
    } else {
        load_four(ids + base, n, lane, 1, c);
    }
}

// Orders this wavefront's LDS writes before its later LDS reads (and the reverse); for staging buffers
// that are private to one wavefront, so no workgroup barrier is involved.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// v from another lane of the same 16-lane row, chosen by a DPP control word (no LDS traffic).
template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}

// Sum over the L (4, 8 or 16) consecutive lanes of a lane group; every lane of the group gets it.
template <int L>
__device__ __forceinline__ float group_sum(float v) {
    static_assert(L == 4 || L == 8 || L == 16, "lane groups inside one 16-lane row");
    v += dpp_move<0xB1>(v);                  // quad_perm [1,0,3,2]
    v += dpp_move<0x4E>(v);                  // quad_perm [2,3,0,1]
    if (L >= 8) v += dpp_move<0x141>(v);     // row_half_mirror
    if (L >= 16) v += dpp_move<0x140>(v);    // row_mirror
    return v;
}

// The workgroup's place in a one-dimensional grid when every XCD (workgroups are dealt to the 8 of them in turn) is to work
// on one contiguous share: of n blocks the XCD of block b takes [x * n / 8, (x + 1) * n / 8), x = b mod 8.  For kernels
// that read or write through a permutation with locality (edges in column order, results in row order): what one XCD
// touches around the same time shares lines, which its own L2 then fills or reads whole.  58,000 nodes, 12.5 M edges, 64-float
// rows: step of a weighted sum with both gradients 738 -> 722 us, and 605 once all its results are placed this way.
__device__ __forceinline__ unsigned xcd_contiguous_block() {
    const unsigned n = gridDim.x, x = blockIdx.x & 7u, i = blockIdx.x >> 3;
    const unsigned q = n >> 3, r = n & 7u;             // the first r XCDs hold q + 1 blocks
    return x * q + (x < r ? x : r) + i;
}

// Lanes l and l + 32 (l < 32) trade: afterwards a holds {a of the lower half, b of the lower half} and b the two upper
// halves.  a + b is then a's sum over l and l + 32 in the lower half and b's in the upper one: two values reduced by one
// vector instruction and one add, where ds_bpermute takes a trip through LDS for each.
__device__ __forceinline__ void swap_halves(float &a, float &b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(r[0]); b = __uint_as_float(r[1]);
}
// The same between the odd 16-lane rows of a and the even rows of b.
__device__ __forceinline__ void swap_rows(float &a, float &b) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(r[0]); b = __uint_as_float(r[1]);
}
// Sum (maximum) over lanes l, l ^ 16, l ^ 32, l ^ 48; every lane gets it.
__device__ __forceinline__ float rows_sum(float v) {
    float w = v;
    swap_halves(v, w);
    v += w; w = v;
    swap_rows(v, w);
    return v + w;
}
__device__ __forceinline__ float rows_max(float v) {
    float w = v;
    swap_halves(v, w);
    v = fmaxf(v, w); w = v;
    swap_rows(v, w);
    return fmaxf(v, w);
}
// Sum of v over the 64 / L lane groups of the wavefront (lanes l, l + L, ...): component word_of_row() of it in every
// lane, i.e. a lane's four words end up in the wavefront's four 16-lane rows.
template <int L>
__device__ __forceinline__ float groups_sum(float4 v) {
    swap_halves(v.x, v.y);
    swap_halves(v.z, v.w);
    float a = v.x + v.y, b = v.z + v.w;      // lower half x / z, upper half y / w
    swap_rows(a, b);
    a += b;                                  // rows 0 .. 3: x, z, y, w
    if (L <= 8) a += dpp_move<0x128>(a);     // row_ror:8
    if (L <= 4) a += dpp_move<0x124>(a);     // row_ror:4
    return a;
}
__device__ __forceinline__ int word_of_row(int lane) { return ((lane >> 5) & 1) | ((lane >> 3) & 2); }

// use(p, load(p)) for p in [first, n), in order, eight loads in flight: a row's pieces added up one load at a time take
// about 0.3 us each.  3 M elements with rows of up to 60,000 (240 pieces), whole calls: F=16 weighted sum 84 -> 51 us,
// maximum 176 -> 121; 100 rows of 5,000, F=16 maximum 32 -> 18; the results are the same bits.
template <typename Load, typename Use>
__device__ __forceinline__ void each_piece(int first, int n, Load load, Use use) {
    constexpr int U = 8;
    for (int p0 = first; p0 < n; p0 += U) {
        decltype(load(0)) v[U];
#pragma unroll
        for (int k = 0; k < U; ++k) v[k] = load(min(p0 + k, n - 1));
#pragma unroll
        for (int k = 0; k < U; ++k)
            if (p0 + k < n) use(p0 + k, v[k]);
    }
}

// How many neighbouring lane groups (of L lanes) share a row of an item of `nrows` rows and `len` elements that are walked many at a
// time: the fewest, a power of two, that are spread / nrows of all 64 / L groups.  Wide apart (a small spread) rows take fewer steps,
// together uneven rows leave fewer groups idle.
template <int L>
__device__ __forceinline__ int groups_per_row(int nrows, int len) {
    constexpr int G = 64 / L;
    const int spread = L <= 4 && len <= 48 * nrows ? 2 : 4;
    int share = 1;
    while (share < G && share * nrows < spread * G) share *= 2;
    return share;
}
}  // namespace fg
