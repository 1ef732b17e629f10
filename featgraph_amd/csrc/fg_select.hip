// Gradients of a max / min aggregation by a sweep over the edges.  Every result out[v, f] is the message at stored position
// arg[v, f], so that edge's operands get dout[v, f]; fg_gspmm_select_backward_f32 (fg_general.hip) takes the results one by one and adds
// each to its operand with a float atomic.  Here every edge looks at its row's positions instead and keeps what is its own:
//   sources : grad[u, f] = sum over the edges e out of u with arg[row e, f] == e of dout[row e, f] (op other[e, f]), over the
//             transposed graph, 8 gathered bytes per edge and feature, no atomics, every element of grad written once;
//   edges   : grad[e, f] = dout[row e, f] (op other[col e, f]) where arg[row e, f] == e, else 0, over the graph; with one value per edge
//             the sum of these over f.
// The sums are in a fixed order.  Atomics on scattered addresses run at 24 G a second whatever the degree, the sweeps' reads grow with
// it: the caller takes the sweeps on graphs of few edges per row.  A lane group holds 16 bytes per lane of one row and has 4 elements'
// loads in flight; rows shorter than an item go one to a lane group, so that short rows need no reduction between lanes.
// 120,000 rows of 8 elements, F = 64: sources 344 us by atomics -> 76 us here (6.9 TB/s of gathered rows, mostly from the
// memory-side cache), edges 136 -> 96 us (2.6 TB/s written), one value per edge 264 -> 34 us.
#include <hip/hip_runtime.h>

#include "fg_common.h"
#include "fg_device.h"

using fg::fail;
using fg::Fixup;
using fg::Item;
using fg::wave_lds_sync;

namespace {

constexpr int kWavesPerBlock = 4;
constexpr int kBlock = 64 * kWavesPerBlock;
constexpr int kSteps = 4;                      // elements per lane group whose loads are issued back to back

enum { kNoOther = 0, kOneOther = 1, kRowOther = 2 };      // the other operand: none, one value per row of it, F values

struct SweepArgs {
    const Item *items;
    int64_t n_items;
    const int32_t *pos;       // row boundaries of the layout
    const int32_t *idx;       // per element: its row of arg / dout (sources), its row of `other` (edges)
    const int32_t *edge_pos;  // sources: per element, its position (what arg holds)
    const int32_t *arg;
    const float *dout, *other;
    float *grad, *partial;
    int F, tiles;             // tiles of 4 * L features
    int divide;               // dout / other instead of dout * other
    float sign;
};

using F4 = fg::Words4<float>;
using I4 = fg::Words4<int32_t>;

// The lane's four features: words `from` .. `from` + 3 of a row, of which the first `skip` are another lane's (4: all of them).
struct Span {
    int from, skip;
    __device__ Span(int tile, int L, int li, int F) {
        const int c0 = (tile * L + li) * 4;
        from = min(c0, F - 4);
        skip = min(c0 - from, 4);
    }
    __device__ void store(float *row, const float (&v)[4]) const {
        if (skip == 0) {
            F4 w;
#pragma unroll
            for (int i = 0; i < 4; ++i) w.v[i] = v[i];
            *reinterpret_cast<F4 *>(row + from) = w;
        } else {
#pragma unroll
            for (int i = 1; i < 4; ++i)
                if (i >= skip) row[from + i] = v[i];
        }
    }
};

__device__ __forceinline__ float message(float d, float x, int divide) { return divide ? d / x : d * x; }

template <int L, int OTHER>
__global__ __launch_bounds__(kBlock) void select_sources_kernel(const SweepArgs a) {
    constexpr int G = 64 / L, U = kSteps;
    __shared__ int2 s_el[kWavesPerBlock][fg::kItemEdges];        // x = row, y = position
    __shared__ int32_t s_end[kWavesPerBlock][fg::kItemRows];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int g = lane / L, li = lane % L;
    const int64_t item_id = (int64_t)(blockIdx.x / (unsigned)a.tiles) * kWavesPerBlock + wave;
    if (item_id >= a.n_items) return;      // uniform per wavefront; no workgroup barriers below
    const Item it = a.items[item_id];
    const Span span((int)(blockIdx.x % (unsigned)a.tiles), L, li, a.F);
    int2 *el = s_el[wave];
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    auto stage = [&](int64_t base, int n) {
        wave_lds_sync();                   // earlier reads of the staging row are done
        for (int t = lane; t < n; t += 64) el[t] = make_int2(a.idx[base + t], a.edge_pos[base + t]);
        wave_lds_sync();
    };
    auto walk = [&](int first, int step, int end) {
        for (int j = first; j < end; j += step * U) {
            int2 e[U];
            I4 at[U];
            F4 d[U], x[U];
#pragma unroll
            for (int u = 0; u < U; ++u) e[u] = el[min(j + u * step, end - 1)];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int64_t row = (int64_t)e[u].x * a.F + span.from;
                at[u] = *reinterpret_cast<const I4 *>(a.arg + row);
                d[u] = *reinterpret_cast<const F4 *>(a.dout + row);
                if (OTHER == kOneOther) x[u].v[0] = a.other[e[u].y];
                if (OTHER == kRowOther) x[u] = *reinterpret_cast<const F4 *>(a.other + (int64_t)e[u].y * a.F + span.from);
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int mine = j + u * step < end ? e[u].y : -2;      // -2: no element (arg holds -1 where a row has none)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float m = OTHER == kNoOther ? d[u].v[i] : message(d[u].v[i], x[u].v[OTHER == kOneOther ? 0 : i], a.divide);
                    acc[i] += at[u].v[i] == mine ? m : 0.f;
                }
            }
        }
    };
    auto put = [&](float *row) {
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = a.sign * acc[i];
        span.store(row, v);
    };
    if (it.info < -1) {
        // several whole rows: every lane group takes rows of its own
        const int nrows = -it.info;
        if (lane < nrows) s_end[wave][lane] = a.pos[it.row + lane + 1] - it.start;
        stage(it.start, it.len);
        for (int q = g; q < nrows; q += G) {
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i] = 0.f;
            walk(q ? s_end[wave][q - 1] : 0, 1, s_end[wave][q]);
            put(a.grad + (int64_t)(it.row + q) * a.F);
        }
        return;
    }
    // one row, or one piece of a long row: all lane groups share it
    for (int32_t base = 0; base < it.len; base += fg::kItemEdges) {
        const int n = min(fg::kItemEdges, it.len - base);
        stage((int64_t)it.start + base, n);
        walk(g, G, n);
    }
#pragma unroll
    for (int off = L; off < 64; off <<= 1)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] += __shfl_xor(acc[i], off);
    if (g == 0) put(it.info < 0 ? a.grad + (int64_t)it.row * a.F : a.partial + (int64_t)it.info * a.F);
}

// Rows that were cut into pieces: the pieces added up in order.
__global__ __launch_bounds__(256) void select_fixup_kernel(const Fixup *fixups, const float *partial, float *grad, int F) {
    const Fixup fx = fixups[blockIdx.x];
    for (int f = threadIdx.x; f < F; f += 256) {
        float s = 0.f;
        fg::each_piece(0, fx.n_pieces, [&](int p) { return partial[(int64_t)(fx.slot0 + p) * F + f]; }, [&](int, float v) { s += v; });
        grad[(int64_t)fx.row * F + f] = s;
    }
}

// ONE: one value per edge, the sum over the features (a.tiles == 1).
template <int L, int OTHER, bool ONE>
__global__ __launch_bounds__(kBlock) void select_edges_kernel(const SweepArgs a) {
    constexpr int G = 64 / L, U = kSteps;
    __shared__ int32_t s_idx[kWavesPerBlock][fg::kItemEdges];
    __shared__ int32_t s_end[kWavesPerBlock][fg::kItemRows];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int g = lane / L, li = lane % L;
    const int64_t item_id = (int64_t)(blockIdx.x / (unsigned)a.tiles) * kWavesPerBlock + wave;
    if (item_id >= a.n_items) return;
    const Item it = a.items[item_id];
    if (it.len == 0) return;
    const Span span((int)(blockIdx.x % (unsigned)a.tiles), L, li, a.F);
    int32_t *idx = s_idx[wave];
    I4 at;
    F4 d;
    auto load_row = [&](int64_t row) {
        at = *reinterpret_cast<const I4 *>(a.arg + row * a.F + span.from);
        d = *reinterpret_cast<const F4 *>(a.dout + row * a.F + span.from);
    };
    auto stage = [&](int64_t base, int n) {
        wave_lds_sync();
        if (OTHER != kNoOther)
            for (int t = lane; t < n; t += 64) idx[t] = a.idx[base + t];
        wave_lds_sync();
    };
    // elements first, first + step, .. of the staged ones whose first has position `base`
    auto walk = [&](int64_t base, int first, int step, int end) {
        for (int j = first; j < end; j += step * U) {
            F4 x[U];
            if (OTHER != kNoOther) {
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int64_t row = idx[min(j + u * step, end - 1)];
                    if (OTHER == kOneOther) x[u].v[0] = a.other[row];
                    else x[u] = *reinterpret_cast<const F4 *>(a.other + row * a.F + span.from);
                }
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int64_t p = base + j + u * step;
                float v[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float m = OTHER == kNoOther ? d.v[i] : message(d.v[i], x[u].v[OTHER == kOneOther ? 0 : i], a.divide);
                    v[i] = at.v[i] == (int32_t)p ? a.sign * m : 0.f;
                }
                const bool ok = j + u * step < end;
                if constexpr (ONE) {
                    float s = 0.f;
#pragma unroll
                    for (int i = 0; i < 4; ++i) s += i >= span.skip ? v[i] : 0.f;
#pragma unroll
                    for (int off = 1; off < L; off <<= 1) s += __shfl_xor(s, off);
                    if (ok && li == 0) a.grad[p] = s;
                } else if (ok) {
                    span.store(a.grad + p * a.F, v);
                }
            }
        }
    };
    if (it.info < -1) {
        const int nrows = -it.info;
        if (lane < nrows) s_end[wave][lane] = a.pos[it.row + lane + 1] - it.start;
        stage(it.start, it.len);
        for (int q = g; q < nrows; q += G) {
            const int b = q ? s_end[wave][q - 1] : 0, e = s_end[wave][q];
            load_row(it.row + q);
            walk(it.start, b, 1, e);
        }
        return;
    }
    load_row(it.row);
    for (int32_t base = 0; base < it.len; base += fg::kItemEdges) {
        const int n = min(fg::kItemEdges, it.len - base);
        stage((int64_t)it.start + base, n);
        walk((int64_t)it.start + base, g, G, n);
    }
}

int lanes_for(int F, int most) {
    int L = 4;
    while (L < most && L * 4 < F) L *= 2;
    return L;
}

template <int OTHER>
void launch_sources(int L, dim3 grid, hipStream_t st, const SweepArgs &a) {
    switch (L) {
        case 4: hipLaunchKernelGGL((select_sources_kernel<4, OTHER>), grid, dim3(kBlock), 0, st, a); break;
        case 8: hipLaunchKernelGGL((select_sources_kernel<8, OTHER>), grid, dim3(kBlock), 0, st, a); break;
        case 16: hipLaunchKernelGGL((select_sources_kernel<16, OTHER>), grid, dim3(kBlock), 0, st, a); break;
        default: hipLaunchKernelGGL((select_sources_kernel<32, OTHER>), grid, dim3(kBlock), 0, st, a); break;
    }
}

template <int OTHER, bool ONE>
void launch_edges(int L, dim3 grid, hipStream_t st, const SweepArgs &a) {
    switch (L) {
        case 4: hipLaunchKernelGGL((select_edges_kernel<4, OTHER, ONE>), grid, dim3(kBlock), 0, st, a); break;
        case 8: hipLaunchKernelGGL((select_edges_kernel<8, OTHER, ONE>), grid, dim3(kBlock), 0, st, a); break;
        case 16: hipLaunchKernelGGL((select_edges_kernel<16, OTHER, ONE>), grid, dim3(kBlock), 0, st, a); break;
        case 32: hipLaunchKernelGGL((select_edges_kernel<32, OTHER, ONE>), grid, dim3(kBlock), 0, st, a); break;
        default: hipLaunchKernelGGL((select_edges_kernel<64, OTHER, ONE>), grid, dim3(kBlock), 0, st, a); break;
    }
}

// What the two calls share; other_len 0: no other operand.
int prepare(const fg_spmm_plan *pl, const int32_t *pos, const int32_t *idx, int op, const int32_t *arg, const float *dout, const float *other,
            int other_len, float *grad, int F, int L, dim3 *grid, SweepArgs *a) {
    if (F < 4) return fail(FG_ERR_SHAPE, "the sweeps take rows of 4 features or more, got %d", F);
    if (other_len != 0 && other_len != 1 && other_len != F) return fail(FG_ERR_SHAPE, "the other operand has 1 or %d features, got %d", F, other_len);
    if ((op == FG_BIN_MUL || op == FG_BIN_DIV) != (other_len != 0)) return fail(FG_ERR_ARG, "operator %d with%s another operand", op, other_len ? "" : "out");
    if (!pos || !idx || !arg || !dout || (other_len && !other) || !grad) return fail(FG_ERR_ARG, "null device pointer");
    a->items = pl->items_dev; a->n_items = pl->n_items; a->pos = pos; a->idx = idx; a->edge_pos = nullptr;
    a->arg = arg; a->dout = dout; a->other = other; a->grad = grad; a->partial = pl->partial_dev; a->F = F;
    a->tiles = (F + 4 * L - 1) / (4 * L);
    a->divide = op == FG_BIN_DIV; a->sign = op == FG_BIN_SUB ? -1.f : 1.f;
    const int64_t blocks = (pl->n_items + kWavesPerBlock - 1) / kWavesPerBlock * a->tiles;
    if (blocks > 0x7fffffffLL) return fail(FG_ERR_SHAPE, "grid too large");
    *grid = dim3((unsigned)blocks);
    return FG_OK;
}

}  // namespace

extern "C" int fg_select_sources_f32(fg_spmm_plan *plan, const int32_t *pos_dev, const int32_t *idx_dev, const int32_t *edge_pos_dev, int op,
                                     const int32_t *arg_dev, const float *dout_dev, const float *other_dev, int other_len,
                                     float *grad_dev, int F, void *stream) {
    if (!plan) return fail(FG_ERR_ARG, "plan is null");
    if (int rc = fg::check_device(plan)) return rc;
    if (plan->num_col_partitions != 1) return fail(FG_ERR_ARG, "fg_select_sources_f32 needs a plan with one column partition");
    if (op != FG_BIN_ADD && op != FG_BIN_SUB && op != FG_BIN_MUL && op != FG_BIN_DIV) return fail(FG_ERR_ARG, "operator %d has no sweep", op);
    if (plan->n_dst == 0) return FG_OK;
    if (plan->nnz > 0 && !edge_pos_dev) return fail(FG_ERR_ARG, "null device pointer");
    const int L = lanes_for(F, 32);
    SweepArgs a;
    dim3 grid;
    if (int rc = prepare(plan, pos_dev, idx_dev, op, arg_dev, dout_dev, other_dev, other_len, grad_dev, F, L, &grid, &a)) return rc;
    fg::ScratchNeed need;
    need.partial = (size_t)plan->max_slots_in_partition * (size_t)F;
    if (int rc = fg::ensure_scratch(plan, need, stream)) return rc;
    a.edge_pos = edge_pos_dev; a.partial = plan->partial_dev;
    hipStream_t st = (hipStream_t)stream;
    if (grid.x > 0) {
        if (other_len == 0) launch_sources<kNoOther>(L, grid, st, a);
        else if (other_len == 1) launch_sources<kOneOther>(L, grid, st, a);
        else launch_sources<kRowOther>(L, grid, st, a);
    }
    if (plan->n_fixups > 0)
        hipLaunchKernelGGL(select_fixup_kernel, dim3((unsigned)plan->n_fixups), dim3(256), 0, st, plan->fixups_dev, plan->partial_dev, grad_dev, F);
    FG_HIP_TRY(hipGetLastError());
    return FG_OK;
}

extern "C" int fg_select_edges_f32(const fg_spmm_plan *plan, const int32_t *pos_dev, const int32_t *idx_dev, int op, const int32_t *arg_dev,
                                   const float *dout_dev, const float *other_dev, int other_len, float *grad_dev, int grad_len, int F,
                                   void *stream) {
    if (!plan) return fail(FG_ERR_ARG, "plan is null");
    if (int rc = fg::check_device(plan)) return rc;
    if (plan->num_col_partitions != 1) return fail(FG_ERR_ARG, "fg_select_edges_f32 needs a plan with one column partition");
    if (op != FG_BIN_ADD && op != FG_BIN_SUB && op != FG_BIN_MUL && op != FG_BIN_DIV) return fail(FG_ERR_ARG, "operator %d has no sweep", op);
    if (grad_len != F && (grad_len != 1 || F > 256)) return fail(FG_ERR_SHAPE, "gradients of %d features, or 1 for rows of up to 256, got %d", F, grad_len);
    if (plan->nnz == 0) return FG_OK;
    const bool one = grad_len == 1;
    const int L = lanes_for(F, one ? 64 : 32);
    SweepArgs a;
    dim3 grid;
    if (int rc = prepare(plan, pos_dev, idx_dev, op, arg_dev, dout_dev, other_dev, other_len, grad_dev, F, L, &grid, &a)) return rc;
    hipStream_t st = (hipStream_t)stream;
    if (other_len == 0) one ? launch_edges<kNoOther, true>(L, grid, st, a) : launch_edges<kNoOther, false>(L, grid, st, a);
    else if (other_len == 1) one ? launch_edges<kOneOther, true>(L, grid, st, a) : launch_edges<kOneOther, false>(L, grid, st, a);
    else one ? launch_edges<kRowOther, true>(L, grid, st, a) : launch_edges<kRowOther, false>(L, grid, st, a);
    FG_HIP_TRY(hipGetLastError());
    return FG_OK;
}
