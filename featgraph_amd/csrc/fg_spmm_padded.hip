// The weighted sum over rows of a length that suits no tile: the kernels gather from a zero-padded copy of x, which one kernel lays
// out the way they read it, and store the caller's shorter rows themselves.
#include <hip/hip_runtime.h>

#include "fg_spmm_items.h"

using fg::fail;
using namespace fg_items;

namespace {

// Bound as the plain sum is, by the gathers (58,000 nodes, 12.5 M edges, rows of 602 floats as 640 in 2 passes: see fg_spmm.hip).  Files of their
// own, as fg_spmm_dot.hip, keep the plain kernels' registers what they are.
template <int L, int K, bool FULL, bool OFF32, int HPT>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(8, 8))) void spmm_padded_kernel(const SpmmArgs a) {
    spmm_items_body<4, L, K, FULL, false, OFF32, HPT, false, true>(a);
}
// (wider rows per lane and tiles of several heads keep the compiler's own register budget)
template <int L, int K, bool FULL, bool OFF32, int HPT>
__global__ __launch_bounds__(kBlock) void spmm_padded_wide_kernel(const SpmmArgs a) {
    spmm_items_body<4, L, K, FULL, false, OFF32, HPT, false, true>(a);
}

template <int L, int K, bool FULL, int HPT>
int launch(bool off32, dim3 grid, hipStream_t st, const SpmmArgs &a) {
    if constexpr (K == 1 && HPT == 1) {
        if (off32) hipLaunchKernelGGL((spmm_padded_kernel<L, K, FULL, true, HPT>), grid, dim3(kBlock), 0, st, a);
        else hipLaunchKernelGGL((spmm_padded_kernel<L, K, FULL, false, HPT>), grid, dim3(kBlock), 0, st, a);
    } else {
        if (off32) hipLaunchKernelGGL((spmm_padded_wide_kernel<L, K, FULL, true, HPT>), grid, dim3(kBlock), 0, st, a);
        else hipLaunchKernelGGL((spmm_padded_wide_kernel<L, K, FULL, false, HPT>), grid, dim3(kBlock), 0, st, a);
    }
    return FG_OK;
}

template <int L, int K>
int launch_full(bool full, bool off32, dim3 grid, hipStream_t st, const SpmmArgs &a) {
    return full ? launch<L, K, true, 1>(off32, grid, st, a) : launch<L, K, false, 1>(off32, grid, st, a);
}

}  // namespace

namespace fg_items {
int launch_padded(int L, int K, bool full, bool off32, int hpt, dim3 grid, hipStream_t st, const SpmmArgs &a) {
    if (hpt > 1 && K == 1 && full) {
        if (L == 16 && hpt == 2) return launch<16, 1, true, 2>(off32, grid, st, a);
        if (L == 16 && hpt == 4) return launch<16, 1, true, 4>(off32, grid, st, a);
        if (L == 8 && hpt == 4) return launch<8, 1, true, 4>(off32, grid, st, a);
        if (L == 4 && hpt == 4) return launch<4, 1, true, 4>(off32, grid, st, a);
    } else if (hpt == 1 && K == 1) {
        switch (L) {
            case 4: return launch_full<4, 1>(full, off32, grid, st, a);
            case 8: return launch_full<8, 1>(full, off32, grid, st, a);
            case 16: return launch_full<16, 1>(full, off32, grid, st, a);
            case 32: return launch_full<32, 1>(full, off32, grid, st, a);
            case 64: return launch_full<64, 1>(full, off32, grid, st, a);
        }
    } else if (hpt == 1 && K == 2 && L == 64) {
        return launch_full<64, 2>(full, off32, grid, st, a);
    }
    return fail(FG_ERR_SHAPE, "no SpMM kernel for padded rows with L=%d K=%d and %d heads per tile", L, K, hpt);
}
}  // namespace fg_items
