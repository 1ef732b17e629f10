// The weighted sum that also leaves every element's dot product (fg_spmm_dot_f32; host side and closing kernels: fg_spmm.hip).
#include <hip/hip_runtime.h>

#include "fg_spmm_items.h"

using fg::fail;
using namespace fg_items;

namespace {

// The sum with dots: one gather of a source row serves the row's weighted sum and its dot product with the output row's
// own vector, which is what the two gradients of a weighted sum need from the transposed graph (dx = A^T dy and
// dw[e] = <dy[row e], x[col e]>).  Bound as the plain sum is, by the gathers' L2 misses.  58,000 nodes, 12.5 M elements, rows
// of 602 floats: 1.80 ms and 0.17 ms to add the tiles' parts up, in the place of a sum of 1.47 ms and an SDDMM of 1.72 (whole
// step 5194 -> 3850 us); 7 wavefronts per SIMD without spills beat 8 with them (step 4172 against 3990 before the last kernel's
// own gain).
template <int L, int HPT, bool SHORT>
__global__ __launch_bounds__(kBlock, HPT == 1 ? 7 : 4) void spmm_dot_kernel(const SpmmArgs a) {
    spmm_items_body<4, L, 1, true, false, true, HPT, true, SHORT>(a);
}

template <int L, int HPT>
int launch(dim3 grid, hipStream_t st, const SpmmArgs &a) {
    if (a.out_len > 0) hipLaunchKernelGGL((spmm_dot_kernel<L, HPT, true>), grid, dim3(kBlock), 0, st, a);
    else hipLaunchKernelGGL((spmm_dot_kernel<L, HPT, false>), grid, dim3(kBlock), 0, st, a);
    return FG_OK;
}

}  // namespace

namespace fg_items {
int launch_dot(int L, int hpt, dim3 grid, hipStream_t st, const SpmmArgs &a) {
    if (hpt == 1) {
        switch (L) {
            case 4: return launch<4, 1>(grid, st, a);
            case 8: return launch<8, 1>(grid, st, a);
            case 16: return launch<16, 1>(grid, st, a);
            case 32: return launch<32, 1>(grid, st, a);
            case 64: return launch<64, 1>(grid, st, a);
        }
    } else if (L == 16 && hpt == 2) { return launch<16, 2>(grid, st, a); }
    else if (L == 16 && hpt == 4) { return launch<16, 4>(grid, st, a); }
    else if (L == 8 && hpt == 4) { return launch<8, 4>(grid, st, a); }
    return fail(FG_ERR_SHAPE, "no SpMM kernel with dots for %d heads per tile with L=%d", hpt, L);
}
}  // namespace fg_items
