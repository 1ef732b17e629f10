/*
 * featgraph_hip.h -- C ABI of libfeatgraph_hip.so, the gfx950 (MI355X) build of
 * FeatGraph's SpMM / SDDMM hot path.
 *
 * Every pointer named *_dev is device memory owned by the caller (any allocator:
 * hipMalloc, a PyTorch-ROCm tensor's data_ptr(), ...).  Pointers named *_host are
 * host memory.  `stream` is a hipStream_t passed as void* (NULL = default stream);
 * kernels are enqueued on it and the call returns without synchronising.
 * All index arrays are int32, all values fp32, all feature matrices row-major and
 * contiguous.  Functions return FG_OK (0) or a negative fg_status;
 * fg_last_error() gives the thread's last message.
 *
 * The reference has no C interface: its kernels are generated by TVM at run time
 * and called as PackedFuncs from python/featgraph/module/{spmm,sddmm}.py.  Each
 * entry point below cites the reference call it stands in for.
 */
#ifndef FEATGRAPH_HIP_H
#define FEATGRAPH_HIP_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

typedef enum {
    FG_OK = 0,
    FG_ERR_ARG = -1,      /* null pointer, negative size, bad option            */
    FG_ERR_SHAPE = -2,    /* feature length / partition count does not fit      */
    FG_ERR_GRAPH = -3,    /* non-monotone positions, index out of range, dups   */
    FG_ERR_HIP = -4,      /* a HIP runtime call failed (text in fg_last_error)  */
    FG_ERR_NOMEM = -5
} fg_status;

int fg_version(void);
const char *fg_last_error(void);

/* ---- host-side graph preprocessing --------------------------------------------------- */

/*
 * CSR -> DDS, 1-D source-column partitioning.
 * Replaces util_convert_csr_to_dds (python/featgraph/util/adj_partitioning.py:7-57),
 * called from SpMMbase.__init__ (python/featgraph/module/spmm.py:40-45).
 * data32/vals32 are arrays of 32-bit words (fp32 weights or int32 ids), moved unchanged.
 * Outputs: s1_pos [P*(n_rows+1)], s1_idx [nnz] partition-local column ids, vals32 [nnz].
 */
int fg_csr_to_dds(int64_t n_rows, int64_t n_cols, const int32_t *indptr_host,
                  const int32_t *indices_host, const void *data32_host,
                  int num_col_partitions, int32_t *s1_pos_host, int32_t *s1_idx_host,
                  void *vals32_host);

/*
 * 2-D COO partitioning.
 * Replaces util_partition_adj_coo_2d (python/featgraph/util/adj_partitioning.py:60-128),
 * called from SDDMMbase.__init__ (python/featgraph/module/sddmm.py:45-49).
 * Outputs (each [nnz]): 1-based edge ids in traversal order, and the global row / col of
 * each traversed edge.  The input arrays are not modified.  Duplicate (row, col) pairs
 * are rejected with FG_ERR_GRAPH.
 */
int fg_partition_coo_2d(int64_t n_rows, int64_t n_cols, int64_t nnz,
                        const int32_t *row_host, const int32_t *col_host,
                        int num_row_partitions, int num_col_partitions,
                        int32_t *edge_id_host, int32_t *out_row_host, int32_t *out_col_host);

/*
 * Structural check of a CSR / DDS position array and its column ids, on the host:
 * positions start at 0, never decrease, end at nnz; ids lie in [0, n_cols).
 * (The reference performs no such check; TVM would read out of bounds.)
 */
int fg_check_csr_host(int64_t n_rows, int64_t n_cols, const int32_t *indptr_host,
                      const int32_t *indices_host);

/* ---- SpMM ---------------------------------------------------------------------------- */

typedef struct fg_spmm_plan fg_spmm_plan;

typedef struct {
    int32_t split_threshold; /* rows longer than this are split over wavefronts; 0 = default: 128 elements on graphs
                                of fewer than 2^20 elements, 256 below 2^23, 512 below 2^25, doubled up to 1024 while a
                                partition's split rows would make more than 8192 pieces; 1024 on larger graphs and
                                where no row is longer than 256 (512, if the graph has 1,700 times as many elements) */
    int32_t item_edges;      /* short rows are packed into items of at most this many elements
                                (and at most 64 rows); 0 = default: 256, or 16 .. 128 on graphs that would have fewer
                                than about 1,700 such items; 1 = one row per item */
    int32_t wide_offsets;    /* non-zero: address feature rows with 64-bit offsets even when the matrix
                                is smaller than 4 GiB (the path larger matrices take; for testing it) */
    int32_t tile_major;      /* SpMM / tiled SDDMM gather from a copy of the source features stored tile by
                                tile ([T][n_src][tile floats], made at the start of every call) instead of
                                from the caller's row-major matrix: 0 = when it pays (4 or more feature
                                tiles and a matrix of 64 MB or more), 1 = whenever the kernel allows it,
                                2 = never                                                              */
    int32_t pass_buffers;    /* SpMM over several source partitions: every pass writes a buffer of its own
                                ([P][n_dst][F] floats of plan scratch) and a last kernel adds them up, instead of
                                later passes reading and rewriting out (same sums, same order); the passes then run
                                as one launch: 0 = whenever the buffers take 8 GiB or less, 1 = always, 2 = never */
    int32_t reserved[3];
} fg_plan_opts;

/*
 * Builds the load-balance plan of one adjacency: a list of per-wavefront work items
 * (runs of whole short rows, pieces of long rows) resident on the current device.
 * pos_host is indptr [n_dst+1] when num_col_partitions == 1, or the DDS s1_pos
 * [P*(n_dst+1)] otherwise.  Stands where SpMMbase.__init__ uploads the adjacency and
 * fixes the partitioning (python/featgraph/module/spmm.py:40-69).
 *
 * A plan owns device scratch that the calls taking a non-const plan fill and read (partial sums
 * of split rows, per-tile partial scores, softmax statistics, attention row state, the tile-by-tile
 * copy of the gathered operand).  Calls that share a plan must therefore be ordered on one stream;
 * calls on different plans are independent.  The scratch is sized by fg_spmm_plan_reserve; a call that
 * finds it too small grows it on the spot (hipFree + hipMalloc: a device synchronisation inside an
 * otherwise asynchronous call), or, when its stream is being captured into a graph, changes nothing
 * and returns FG_ERR_ARG.
 */
int fg_spmm_plan_create(const int32_t *pos_host, int64_t n_dst, int64_t n_src,
                        int num_col_partitions, const fg_plan_opts *opts,
                        fg_spmm_plan **plan_out);
void fg_spmm_plan_destroy(fg_spmm_plan *plan);

/*
 * Sizes the plan's scratch for later calls of one operator, so that those calls allocate nothing:
 * op names the operator, (heads, head_len) its feature shape (heads = 1 and head_len = F for the
 * single-head operators) and num_feat_partitions the value the calls will pass.  The scratch only ever
 * grows; reserving for several operators or shapes keeps the largest.  No counterpart in the reference
 * (TVM allocates its workspaces inside the generated function).
 */
typedef enum {
    FG_OP_SPMM_SUM = 0,           /* fg_spmm_csr_f32, fg_spmm_dds_f32, fg_gspmm_f32 with FG_REDUCE_SUM */
    FG_OP_SPMM_EXTREME = 1,       /* fg_gspmm_f32 / fg_gspmm_arg_f32 with FG_REDUCE_MAX / FG_REDUCE_MIN */
    FG_OP_SDDMM_DDS = 2,          /* fg_sddmm_dds_f32 */
    FG_OP_EDGE_SOFTMAX = 3,       /* fg_edge_softmax_f32, _backward_f32, _stats_f32 (head_len ignored) */
    FG_OP_ATTENTION = 4,          /* fg_graph_attention_f32 and its two gradient calls */
    FG_OP_ATTENTION_ADDITIVE = 5, /* fg_graph_attention_additive_f32 and its two gradient calls */
    FG_OP_GSPMM_BCAST = 6,        /* fg_gspmm_bcast_f32 / _dds_f32 without arg_dev (heads * head_len = out_len) */
    FG_OP_GSPMM_BCAST_ARG = 7,    /* fg_gspmm_bcast_f32 / _dds_f32 with arg_dev */
    FG_OP_ATTENTION_ADDITIVE_TRAIN = 8, /* fg_graph_attention_additive_train_f32 and _train_elv_f32 */
    FG_OP_SPMM_SUM_DOTS = 9,      /* fg_spmm_dot_f32 (FG_ERR_SHAPE where fg_spmm_dot_takes says no) */
    FG_OP_SPMM_SUM_PADDED = 10,   /* fg_gspmm_padded_f32 (head_len: F / heads) */
    FG_OP_SPMM_SUM_DOTS_PADDED = 11 /* fg_spmm_dot_padded_f32 (likewise) */
} fg_op;
int fg_spmm_plan_reserve(fg_spmm_plan *plan, int op, int heads, int head_len, int num_feat_partitions);

/*
 * Makes, on the device, a 16-bit copy of the layout's column ids (idx_dev: indices [nnz] of a CSR plan, or the
 * partition-local s1_idx [nnz] of a DDS plan) that the plan owns from then on.  The gather kernels of
 * fg_spmm_csr_f32 / fg_spmm_dds_f32 / fg_gspmm_f32 (sums), fg_sddmm_dds_f32, the fg_graph_attention_* calls and fg_gspmm_bcast_f32 / _dds_f32 then stream 2 bytes per stored
 * element instead of 4 on every call that hands them this same idx_dev (compared by address; any other array is read
 * as int32, as before).  Results are bit-identical either way.  The binding is by ADDRESS: the caller must neither
 * change the contents of idx_dev afterwards nor free it and pass another array that an allocator placed at the same
 * address (a caching allocator does that readily) without calling this again (or with NULL) first -- the kernels would
 * gather through the stale copy.  fg_debug_checks(1) makes every operator call compare a fingerprint of the array (its
 * length and its first and last 1,024 ids) with the one taken here, at the price of a device round trip per call, and
 * read the int32 array when they differ.  The ids are checked while they are copied: FG_ERR_GRAPH when one lies outside
 * [0, partition width).  Allocates nnz * 2 bytes; FG_ERR_SHAPE when a partition is more than 65,536 columns wide.
 * idx_dev == NULL releases the copy.  The call returns after the copy has been made (it waits for `stream`).  No counterpart in the reference, whose index arrays are
 * whatever scipy holds (python/featgraph/module/spmm.py:47-49,62-64).  The copy is made by a kernel on `stream`: operator
 * calls on other streams must be ordered after it.  To be called next to fg_spmm_plan_create,
 * like fg_spmm_plan_reserve, not between operator calls that are in flight on the plan.
 */
int fg_spmm_plan_narrow_indices(fg_spmm_plan *plan, const int32_t *idx_dev, void *stream);

/* Switches the library's debug checks on (non-zero) or off for the whole process and returns the previous setting.
 * Off by default.  On: see fg_spmm_plan_narrow_indices.  No counterpart in the reference. */
int fg_debug_checks(int on);

/* Device memory the plan holds at the moment, in bytes: work items and fix-up list, the scratch buffers as far as
 * fg_spmm_plan_reserve or the operator calls have grown them, the tile-by-tile copy buffer, the 16-bit column ids.
 * (The reference's counterpart is whatever TVM allocates for its temporaries, python/featgraph/op/vanilla_spmm.py:43-60.) */
int64_t fg_spmm_plan_bytes(const fg_spmm_plan *plan);

/* Human-readable description of the plan and of the launch it would use for feature
 * length F (the counterpart of lower_to_ir, python/featgraph/module/spmm.py:113-140).
 * Returns the number of bytes written (excluding the NUL) or a negative status. */
int fg_spmm_plan_describe(const fg_spmm_plan *plan, int F, int num_feat_partitions,
                          char *buf, size_t buf_len);

/*
 * out[v, :] = sum_{e in row v} vals[e] * X[indices[e], :]   (every element of out written).
 * Replaces the function built from vanilla_spmm_csr_cuda + schedule_vanilla_spmm_csr_cuda
 * (python/featgraph/op/vanilla_spmm.py:83-146) that SpMMbase.run launches
 * (python/featgraph/module/spmm.py:156-160).
 * num_feat_partitions: 0 = choose; T >= 1 = split the feature axis into T tiles handled by
 * different workgroups (the knob of vanilla_spmm_csr_x86, vanilla_spmm.py:41-56); F % T == 0.
 */
int fg_spmm_csr_f32(fg_spmm_plan *plan, const int32_t *indptr_dev,
                    const int32_t *indices_dev, const float *vals_dev, const float *x_dev,
                    float *out_dev, int F, int num_feat_partitions, void *stream);

/*
 * fg_spmm_csr_f32 for callers that cannot allocate device memory or have it allocated under them:
 * code that records a HIP graph, tight serving loops, harnesses that forbid hipMalloc.  It has no
 * counterpart in the reference.  Same arguments and result as fg_spmm_csr_f32 (bit-identical), but
 * the partial sums of split rows go to a 16 MiB array that is part of the library's device image
 * instead of plan-owned memory, X is always gathered from the caller's row-major matrix, and the call
 * itself performs no hipMalloc / hipFree; the plan is not modified.
 * Limit: (pieces of 1024 elements that the plan's longer rows make) * F <= 4,194,304 floats, else FG_ERR_SHAPE
 * (the 232,965-node benchmark graph needs 2.7 M floats at F = 512); a plan whose rows are cut finer than that
 * fills the array a range of columns at a time.
 * Each GPU holds one such array for the life of the process and every call on that GPU uses it: calls
 * that overlap on one GPU (two streams, two threads) race on it and must be ordered by the caller.
 * Nothing in it needs clearing between calls (every piece's row is written before it is read).
 */
int fg_spmm_csr_noalloc_f32(const fg_spmm_plan *plan, const int32_t *indptr_dev,
                            const int32_t *indices_dev, const float *vals_dev, const float *x_dev,
                            float *out_dev, int F, int num_feat_partitions, void *stream);

/*
 * Same product over the DDS format: partition p's elements contribute
 * vals[e] * X[s1_idx[e] + p*ceil(n_src/P), :], partitions are processed in ascending p,
 * each adding its partial row sums to out.
 * Replaces vanilla_spmm_dds_x86 + schedule_vanilla_spmm_dds_x86
 * (python/featgraph/op/vanilla_spmm.py:149-246).
 */
int fg_spmm_dds_f32(fg_spmm_plan *plan, const int32_t *s1_pos_dev,
                    const int32_t *s1_idx_dev, const float *vals_dev, const float *x_dev,
                    float *out_dev, int F, int num_feat_partitions, void *stream);

/*
 * Generalised SpMM (aggregation other than the weighted sum; the generalisation the reference's
 * README.md:9-11 points to but does not contain):
 *   out[v, h, :] = reduce over the row's elements of vals[e, h] * X[indices[e], h, :]
 * reduce: FG_REDUCE_SUM, or FG_REDUCE_MAX / FG_REDUCE_MIN (rows without elements give 0; plan with
 * one column partition; a NaN message beats every number, so that it reaches the result as it does through a
 * sum -- the behaviour of numpy's maximum / minimum reductions; the same holds for fg_gspmm_bcast_f32 / _dds_f32).  heads = H >= 1: vals is [nnz, H], or [H, nnz] when vals_head_major is
 * non-zero (each head's weights contiguous, which is what the kernels stream best), and F = H * D
 * with D a multiple of 64 or a power of two >= 4 (sum; heads shorter than 16 floats need H % 4 == 0)
 * or >= 16 (max / min).  vals_dev == NULL: every weight is 1 (copy_u).
 * pos/idx are indptr/indices for a one-partition plan, s1_pos/s1_idx (and vals in DDS order) otherwise.
 */
typedef enum { FG_REDUCE_SUM = 0, FG_REDUCE_MAX = 1, FG_REDUCE_MIN = 2 } fg_reduce;
int fg_gspmm_f32(fg_spmm_plan *plan, const int32_t *pos_dev, const int32_t *idx_dev,
                 const float *vals_dev, const float *x_dev, float *out_dev, int F, int heads,
                 int vals_head_major, int reduce, int num_feat_partitions, void *stream);

/*
 * The two gradients of a weighted sum y[r] = sum over e of w[e] * x[col e] in one sweep over the TRANSPOSED adjacency (its
 * rows are y's sources; no counterpart in the reference): out as fg_gspmm_f32 (sum) with x_dev = dL/dy, and
 *   dots[edge_pos[t], h] = <own[row of element t, h, :], x[idx[t], h, :]>
 * for every element t of the layout, own_dev [n_dst, heads, own_len] (own_len <= F / heads; columns of x beyond it count
 * as zeros of own).  Without elements this is fg_gspmm_f32: own_dev, edge_pos_dev and dots_dev are not read and may be
 * NULL.  fg_spmm_dot_takes says whether this plan and shape do (arrays 16-byte aligned): whole tiles of 16 to 256
 * floats, X below 4 GiB (whether one sweep is also the faster way depends on the graph: tuning.sum_gradients_in_one_sweep), with several partitions every pass in a buffer of its own, and at most 8 GiB of scratch for the
 * dots (nnz floats per head, or per tile with one head).  FG_ERR_NOMEM leaves a plan that a plain sum can still use.
 */
int fg_spmm_dot_takes(const fg_spmm_plan *plan, int F, int heads, int num_feat_partitions);
int fg_spmm_dot_f32(fg_spmm_plan *plan, const int32_t *pos_dev, const int32_t *idx_dev, const float *vals_dev,
                    const float *x_dev, const float *own_dev, int own_len, float *out_dev, const int32_t *edge_pos_dev,
                    float *dots_dev, int F, int heads, int vals_head_major, int num_feat_partitions, void *stream);

/*
 * fg_gspmm_f32 (sum) and fg_spmm_dot_f32 over rows whose length suits no tile: x, out and own hold heads of given_len floats, at any
 * 4-byte alignment, and the kernels run at heads of F / heads >= given_len floats (a length that fg_gspmm_f32 takes, tiles of a
 * multiple of 4), on a zero-padded copy of x in the plan's scratch (n_src * F floats).  Zero columns change no sum.
 */
int fg_gspmm_padded_f32(fg_spmm_plan *plan, const int32_t *pos_dev, const int32_t *idx_dev, const float *vals_dev,
                        const float *x_dev, int given_len, float *out_dev, int F, int heads, int vals_head_major,
                        int num_feat_partitions, void *stream);
int fg_spmm_dot_padded_f32(fg_spmm_plan *plan, const int32_t *pos_dev, const int32_t *idx_dev, const float *vals_dev,
                           const float *x_dev, const float *own_dev, int given_len, float *out_dev, const int32_t *edge_pos_dev,
                           float *dots_dev, int F, int heads, int vals_head_major, int num_feat_partitions, void *stream);

/*
 * fg_gspmm_f32 with FG_REDUCE_MAX / FG_REDUCE_MIN that also reports which element was selected (no
 * counterpart in the reference; what the gradient of a max / min aggregation needs):
 * arg_dev[v, f] = position in the CSR element order of the first element of row v whose message
 * equals out[v, f] (for a NaN result: the row's first NaN message, as numpy's argmax / argmin report it), or -1 for
 * a row without elements.  arg_dev is int32 [n_dst, F].
 */
int fg_gspmm_arg_f32(fg_spmm_plan *plan, const int32_t *indptr_dev, const int32_t *indices_dev,
                     const float *vals_dev, const float *x_dev, float *out_dev, int32_t *arg_dev, int F,
                     int heads, int vals_head_major, int reduce, int num_feat_partitions, void *stream);

/*
 * Brings per-edge, per-head values into the order and layout fg_gspmm_f32 streams best (no
 * counterpart in the reference): dst[h, e] = src[edge_pos[e], h] for e < n_edges, src is
 * [n_edges, heads], dst is [heads, n_edges]; edge_pos_dev == NULL means the identity.  With the
 * positions that fg_csr_to_dds produces for 0-based edge numbers as data, this turns values given in
 * CSR edge order into head-major values in DDS order.
 */
int fg_edge_values_head_major_f32(const float *src_dev, const int32_t *edge_pos_dev, int64_t n_edges,
                                  int heads, float *dst_dev, void *stream);
/*
 * The same for values that are head-major already, result[h, e] = src[h, edge_pos[e]], both arrays [heads, n_edges]; src is
 * overwritten as well, and *result tells which of the two (src_dev or dst_dev) holds the result once the stream is there.
 * edge_pos 16-byte aligned.
 */
int fg_edge_values_permute_f32(float *src_dev, const int32_t *edge_pos_dev, int64_t n_edges, int heads, float *dst_dev,
                               float **result, void *stream);

/* ---- SDDMM --------------------------------------------------------------------------- */

/*
 * out[e, h] = sum_{d<D} src[col[e], h, d] * dst[row[e], h, d],  e in stored COO order.
 * H == 1 is the reference's vanilla_sddmm (python/featgraph/op/vanilla_sddmm.py:6-63,
 * CUDA schedules :77-100) launched by SDDMMbase.run (python/featgraph/module/sddmm.py:128):
 * src is gathered by the COLUMN index and dst by the ROW index (:47).
 * H > 1 is the multi-head form (src/dst contiguous [n, H, D], out row-major [E, H]); it
 * has no counterpart in the reference.
 */
int fg_sddmm_coo_f32(const int32_t *row_dev, const int32_t *col_dev, int64_t n_edges,
                     const float *src_dev, const float *dst_dev, float *out_dev, int H,
                     int D, void *stream);

/*
 * The same for edges listed in an order of the caller's choice, best by row (a destination row is then read once for many
 * edges): the results of edge e go to out[edge_pos[e] * H ..] (edge_pos null: to out[e * H ..]).  n_src / n_dst: rows of src and
 * dst, which let the kernel address them with 32 bits; 0: not known.
 */
int fg_sddmm_edges_f32(const int32_t *row_dev, const int32_t *col_dev, const int32_t *edge_pos_dev, int64_t n_edges,
                       int64_t n_src, int64_t n_dst, const float *src_dev, const float *dst_dev, float *out_dev, int H, int D,
                       void *stream);

/*
 * Same result for edges in CSR order (edge e of row v at position indptr[v] + k), using the
 * SpMM plan's row items, so that no row-id array is read; dst[v] is read once per batch of edges (8 .. 128 of them) that
 * share it, and once per edge in a batch of several rows.  The plan must have num_col_partitions == 1.
 */
int fg_sddmm_csr_f32(const fg_spmm_plan *plan, const int32_t *indptr_dev,
                     const int32_t *indices_dev, const float *src_dev, const float *dst_dev,
                     float *out_dev, int H, int D, void *stream);

/*
 * Same result for large graphs, over a source-column-partitioned (DDS) copy of the adjacency
 * (fg_csr_to_dds with the 0-based CSR positions of the edges as data, giving edge_pos) and
 * with the feature axis cut into num_feat_partitions tiles handled by different workgroups
 * (the tiling the reference applies on x86 only, python/featgraph/op/vanilla_sddmm.py:48-60,
 * and rules out on CUDA, :79-80).  out is written in the caller's CSR edge order:
 * out[edge_pos[e'] * H + h].  The tile width H*D / num_feat_partitions must be a power of two
 * between 16 and 256 floats and hold whole heads, or (H == 1) divide the head.  `plan` is
 * built from s1_pos with the same num_col_partitions; it also owns the per-tile partial sums.
 */
int fg_sddmm_dds_f32(fg_spmm_plan *plan, const int32_t *s1_pos_dev, const int32_t *s1_idx_dev,
                     const int32_t *edge_pos_dev, const float *src_dev, const float *dst_dev,
                     float *out_dev, int H, int D, int num_feat_partitions, void *stream);

/*
 * Element-wise edge operators of a generalised SDDMM (no counterpart in the reference, which has
 * the dot product only): out[e, f] = src[col[e], f] op dst[row[e], f], out is [n_edges, F] in
 * stored edge order.
 */
typedef enum { FG_EDGE_ADD = 0, FG_EDGE_SUB = 1, FG_EDGE_MUL = 2 } fg_edge_op;
int fg_gsddmm_elementwise_f32(const int32_t *row_dev, const int32_t *col_dev, int64_t n_edges,
                              const float *src_dev, const float *dst_dev, float *out_dev, int F,
                              int op, void *stream);

/*
 * Generalised SpMM / SDDMM whose two operands may live on the source nodes (FG_TARGET_U: the row of the
 * operand is the element's column), on the stored elements (FG_TARGET_E: its position) or, for the SDDMM,
 * on the destination nodes (FG_TARGET_V: its row), with feature shapes that broadcast against each other.
 * No counterpart in the reference (its README.md:9-11 only names "generalized SpMM and SDDMM"); the
 * vocabulary is that of DGL's gspmm / gsddmm.  An operand is [rows, len] row-major; output feature f
 * reads operand feature off[f] (off == NULL: the identity, and then len must equal out_len).
 *
 *   fg_gspmm_bcast_f32 : out[v, f] = reduce over the elements e of row v of  lhs[.., lhs_off[f]] op rhs[.., rhs_off[f]]
 *     op: FG_BIN_ADD .. FG_BIN_COPY_RHS; reduce: FG_REDUCE_SUM / MAX / MIN; rows without elements give 0.
 *     row_scale_dev (optional, [n_dst]) multiplies each finished row (1 / degree gives the mean).
 *     arg_dev (optional, max / min only, int32 [n_dst, out_len]): the stored position of the first element
 *     whose message equals the result, -1 for rows without elements.  `plan` is a plan of this CSR with one
 *     column partition.  Messages and sums are rounded separately (no fused multiply-add).  With an operand on
 *     the source nodes, 128-bit accesses and 128 features or more in a multiple of 64, the feature axis is cut
 *     into 64-float tiles that different workgroups take (the tiling the reference applies to the weighted sum,
 *     python/featgraph/op/vanilla_spmm.py:43-60).  Otherwise, with 256 output features or more (64 without
 *     128-bit accesses), a row's sum is formed in stored element order (rows longer than the split threshold:
 *     piece by piece); with fewer, several lane groups may take every so many elements of a row each and their sums are
 *     added, in a fixed order.
 *   fg_gspmm_bcast_dds_f32 : the same result over a source-column-partitioned (DDS) copy of the adjacency, so that
 *     an operand gathered from the source nodes is read partition by partition and its rows stay in the L2s
 *     (the reference's 1-D graph partitioning, python/featgraph/op/vanilla_spmm.py:198-222, applied to these
 *     messages).  `plan` is built from s1_pos with the same num_col_partitions; s1_pos / s1_idx come from
 *     fg_csr_to_dds, and edge_pos (the data of fg_csr_to_dds called with the 0-based CSR positions of the
 *     elements) gives every DDS element's stored position: operands on the elements, and arg_dev, stay in the
 *     caller's CSR order.  Every partition's rows go to a buffer of plan scratch ([P][n_dst][out_len] floats, as
 *     much again with arg_dev; more than 8 GiB is refused) and a closing kernel combines them in partition
 *     order: sums add the partitions' sums, max / min and the selected positions are the same as without partitions.
 *     In general edge_pos[i] is the row of element i in the operands on the elements, and the position reported
 *     for it: a caller whose edge operands lie in another order than the plan's adjacency (the transposed graph's
 *     calls over arrays kept in the original edge order, say) composes that order into edge_pos; with a plan of
 *     one partition (s1_pos / s1_idx = indptr / indices) edge_pos may be NULL for the identity.
 *   fg_gsddmm_bcast_f32 : out[e, f] = lhs[.., lhs_off[f]] op rhs[.., rhs_off[f]], or, with FG_BIN_DOT,
 *     out[e, f] = sum_{i < reduce_len} lhs[.., lhs_off[f] * reduce_len + i] * rhs[.., rhs_off[f] * reduce_len + i];
 *     row_dev / col_dev give each stored edge's row and column (needed for the targets that are used).  out may be an operand on
 *     the elements of out_len features without an offset array.
 */
typedef enum {
    FG_BIN_ADD = 0, FG_BIN_SUB = 1, FG_BIN_MUL = 2, FG_BIN_DIV = 3, FG_BIN_COPY_LHS = 4, FG_BIN_COPY_RHS = 5,
    FG_BIN_DOT = 6   /* SDDMM only */
} fg_binary_op;
typedef enum { FG_TARGET_U = 0, FG_TARGET_E = 1, FG_TARGET_V = 2 } fg_target;
/* flags: what the caller knows about an offset array, which lets the kernels use 128-bit accesses when out_len
 * is a multiple of 4 (0 is always valid).  An operand without an offset array, or of one feature, needs no flag: where all operands are
 * such, 128-bit accesses are used from 4 output features on, at any length and 4-byte alignment (but in short odd rows with an operand
 * streamed from the elements, and at odd lengths where out_dev is an operand).  _VEC4: every aligned group of 4 output features reads 4 consecutive operand features that
 * start at a multiple of 4.  _SPLAT4: every such group reads one operand feature 4 times.
 * FG_BCAST_EDGES_ASCEND: edge_pos ascends along every row segment of the layout (it does for the positions that
 * fg_csr_to_dds gives), which lets max / min with positions skip comparing positions on ties. */
enum { FG_BCAST_LHS_VEC4 = 1, FG_BCAST_LHS_SPLAT4 = 2, FG_BCAST_RHS_VEC4 = 4, FG_BCAST_RHS_SPLAT4 = 8, FG_BCAST_EDGES_ASCEND = 16 };
int fg_gspmm_bcast_f32(fg_spmm_plan *plan, const int32_t *indptr_dev, const int32_t *indices_dev, int op,
                       int reduce, const float *lhs_dev, int lhs_target, int lhs_len,
                       const int32_t *lhs_off_dev, const float *rhs_dev, int rhs_target, int rhs_len,
                       const int32_t *rhs_off_dev, int flags, const float *row_scale_dev, float *out_dev,
                       int32_t *arg_dev, int out_len, void *stream);
int fg_gspmm_bcast_dds_f32(fg_spmm_plan *plan, const int32_t *s1_pos_dev, const int32_t *s1_idx_dev,
                           const int32_t *edge_pos_dev, int op, int reduce, const float *lhs_dev, int lhs_target,
                           int lhs_len, const int32_t *lhs_off_dev, const float *rhs_dev, int rhs_target, int rhs_len,
                           const int32_t *rhs_off_dev, int flags, const float *row_scale_dev, float *out_dev,
                           int32_t *arg_dev, int out_len, void *stream);
/*
 * Gradient of a max / min aggregation: dlhs / drhs (either may be NULL; both are added to, so clear them first) receive
 * d(out[v, f]) / d(operand) * dout[v, f] at the operands of the element arg[v, f] that fg_gspmm_bcast_f32 reported
 * (-1: nothing).  op: FG_BIN_ADD .. FG_BIN_COPY_LHS; operands on FG_TARGET_U or FG_TARGET_E with the offset arrays of
 * the forward call; lhs_dev / rhs_dev are read for FG_BIN_MUL / FG_BIN_DIV only; col_dev [n_edges] holds every stored
 * element's column.  Additions are atomic, in no fixed order.
 */
int fg_gspmm_select_backward_f32(const int32_t *arg_dev, const int32_t *col_dev, int64_t n_dst, int64_t n_edges, int op,
                                 const float *lhs_dev, int lhs_target, int lhs_len, const int32_t *lhs_off_dev,
                                 const float *rhs_dev, int rhs_target, int rhs_len, const int32_t *rhs_off_dev,
                                 const float *dout_dev, int out_len, float *dlhs_dev, float *drhs_dev, void *stream);
/*
 * The same gradient of one operand by a sweep over the edges, in a fixed order and without atomics, for graphs of few edges per
 * row.  op: FG_BIN_ADD (also for copies), FG_BIN_SUB (the operand that is subtracted), FG_BIN_MUL, FG_BIN_DIV (the numerator); other_dev: the other
 * operand of FG_BIN_MUL / _DIV, other_len = out_len or 1 features (other_len 0: none).  Every element of grad is written.
 *   _sources : the operand on FG_TARGET_U, out_len features.  `plan`, pos, idx and edge_pos are the TRANSPOSED adjacency's (one column
 *              partition): its elements' rows of arg / dout and their positions in the order that arg refers to.
 *   _edges   : the operand on FG_TARGET_E, grad_len = out_len features, or 1 (the sum over up to 256).  `plan`, pos, idx: the adjacency's, whose
 *              element order is the one that arg refers to.
 * Rows of 4 features or more.  _sources keeps rows' pieces in the plan's scratch, as FG_OP_GSPMM_BCAST with out_len sizes it.
 */
int fg_select_sources_f32(fg_spmm_plan *plan, const int32_t *pos_dev, const int32_t *idx_dev, const int32_t *edge_pos_dev, int op,
                          const int32_t *arg_dev, const float *dout_dev, const float *other_dev, int other_len, float *grad_dev,
                          int out_len, void *stream);
int fg_select_edges_f32(const fg_spmm_plan *plan, const int32_t *pos_dev, const int32_t *idx_dev, int op, const int32_t *arg_dev,
                        const float *dout_dev, const float *other_dev, int other_len, float *grad_dev, int grad_len, int out_len,
                        void *stream);

int fg_gsddmm_bcast_f32(const int32_t *row_dev, const int32_t *col_dev, int64_t n_edges, int op,
                        const float *lhs_dev, int lhs_target, int lhs_len, const int32_t *lhs_off_dev,
                        const float *rhs_dev, int rhs_target, int rhs_len, const int32_t *rhs_off_dev,
                        int flags, float *out_dev, int out_len, int reduce_len, void *stream);

/*
 * Softmax over the stored elements of every row, separately per head (no counterpart in the
 * reference, which stops at SpMM and SDDMM; this is the step between them in an attention layer):
 *   out[e, h] = exp(scores[e, h] - m) / sum over the row's e' of exp(scores[e', h] - m), m = row maximum.
 * scores / out are [nnz, heads] in CSR element order; rows without elements write nothing; out may
 * alias scores.  `plan` is a plan of this CSR with one column partition (it also owns the scratch).
 */
int fg_edge_softmax_f32(fg_spmm_plan *plan, const int32_t *indptr_dev, const float *scores_dev,
                        float *out_dev, int heads, void *stream);

/*
 * Gradient of fg_edge_softmax_f32 with respect to scores, given its output and dL/d(output):
 *   grad_scores[e, h] = softmax[e, h] * (grad_softmax[e, h] - sum over the row's e' of softmax * grad_softmax).
 */
int fg_edge_softmax_backward_f32(fg_spmm_plan *plan, const int32_t *indptr_dev,
                                 const float *softmax_dev, const float *grad_softmax_dev,
                                 float *grad_scores_dev, int heads, void *stream);

/*
 * The two halves of a softmax that is consumed at once by the per-head weighted SpMM (attention without a
 * stored softmax; no counterpart in the reference):
 *   fg_edge_softmax_stats_f32     : row_stats[v, h] = (max, sum of exp(scores - max)) over row v, as float pairs
 *                                   [n_dst, heads, 2]; rows without elements are left untouched.
 *   fg_edge_softmax_head_major_f32: dst[h, e] = exp(scores[edge_pos[e], h] - max) / sum, with the statistics of
 *                                   row edge_row[edge_pos[e]]; dst is [heads, n_edges], i.e. what
 *                                   fg_gspmm_f32(..., vals_head_major = 1, ...) reads; edge_pos_dev == NULL means
 *                                   the identity; edge_row_dev [n_edges] holds the row of every stored element.
 */
int fg_edge_softmax_stats_f32(fg_spmm_plan *plan, const int32_t *indptr_dev, const float *scores_dev,
                              float *row_stats_dev, int heads, void *stream);
int fg_edge_softmax_head_major_f32(const float *scores_dev, const float *row_stats_dev,
                                   const int32_t *edge_row_dev, const int32_t *edge_pos_dev, int64_t n_edges,
                                   int heads, float *dst_dev, void *stream);

/* ---- attention ------------------------------------------------------------------------ */

/*
 * out[v, h, :] = sum over the edges e of row v of softmax_e(scale * <K[col e, h, :], Q[v, h, :]>) * V[col e, h, :]
 * (rows without edges: 0): multi-head SDDMM, edge softmax and per-head weighted SpMM in one sweep per
 * source-column partition, without storing the [nnz, heads] scores.  q is [n_dst, heads, head_len], k and v
 * are [n_src, heads, head_len], out is [n_dst, heads, head_len]; head_len is 16, 32 or 64; pos / idx are the
 * plan's CSR (one partition) or DDS arrays.  The plan must hold no split rows (create it with
 * fg_plan_opts.split_threshold = INT32_MAX).  row_state_dev, when not NULL, is [n_dst, heads, 2] and receives
 * every row's maximum score and sum of exponentials (what the gradient kernels below start from).
 * No counterpart in the reference: the result is defined by the composition of the three operators above.
 */
int fg_graph_attention_f32(fg_spmm_plan *plan, const int32_t *pos_dev, const int32_t *idx_dev,
                           const float *q_dev, const float *k_dev, const float *v_dev, float *out_dev,
                           float *row_state_dev, int heads, int head_len, float scale, void *stream);

/*
 * The same with additive scores (the attention of GAT layers): s[e, h] = leaky_relu(el[col e, h] + er[row e, h])
 * with the given negative slope.  er_dev is [heads, n_dst] and el_dev [heads, n_src] (one scalar per vertex and
 * head, head by head); v, out, row_state, plan and head lengths as above.
 */
int fg_graph_attention_additive_f32(fg_spmm_plan *plan, const int32_t *pos_dev, const int32_t *idx_dev,
                                    const float *er_dev, const float *el_dev, const float *v_dev, float *out_dev,
                                    float *row_state_dev, int heads, int head_len, float negative_slope,
                                    void *stream);

/*
 * Gradients of fg_graph_attention_f32: the scores are formed anew from Q and K, the softmax from row_state.
 *   fg_graph_attention_coef_f32: row_coef[h, v] = (max + log(sum), <dout[v, h, :], out[v, h, :]>), an
 *     [heads, n_dst, 2] array, from the forward pass's row_state and output (one small pass over the rows);
 *   fg_graph_attention_backward_q_f32: dq, on the plan and arrays of the forward pass (gathers K and V);
 *   fg_graph_attention_backward_kv_f32: dk and dv, on a plan and arrays of the TRANSPOSED adjacency (rows =
 *     sources; gathers Q, dout and row_coef of the destinations);
 *   fg_graph_attention_backward_kv_ds_f32: the same, and ds[h, t] = scale * the gradient of element t's score, a
 *     [heads, nnz] array in the layout's element order.  dq[v, h, :] is the sum of ds * k over v's elements: brought into
 *     the order of a layout of the adjacency (fg_edge_values_permute_f32) they are fg_gspmm_f32's head-major weights, and
 *     _backward_q_f32, which gathers V as well, is not needed.
 * Same restrictions as the forward pass.
 */
int fg_graph_attention_coef_f32(const float *out_dev, const float *dout_dev, const float *row_state_dev,
                                float *row_coef_dev, int64_t n_dst, int heads, int head_len, void *stream);
int fg_graph_attention_backward_q_f32(fg_spmm_plan *plan, const int32_t *pos_dev, const int32_t *idx_dev,
                                      const float *q_dev, const float *k_dev, const float *v_dev,
                                      const float *dout_dev, const float *row_coef_dev, float *dq_dev,
                                      int heads, int head_len, float scale, void *stream);
int fg_graph_attention_backward_kv_f32(fg_spmm_plan *plan_t, const int32_t *pos_t_dev, const int32_t *idx_t_dev,
                                       const float *q_dev, const float *dout_dev, const float *k_dev,
                                       const float *v_dev, const float *row_coef_dev, float *dk_dev, float *dv_dev,
                                       int heads, int head_len, float scale, void *stream);
int fg_graph_attention_backward_kv_ds_f32(fg_spmm_plan *plan_t, const int32_t *pos_t_dev, const int32_t *idx_t_dev,
                                          const float *q_dev, const float *dout_dev, const float *k_dev,
                                          const float *v_dev, const float *row_coef_dev, float *dk_dev, float *dv_dev,
                                          float *ds_dev, int heads, int head_len, float scale, void *stream);

/*
 * Gradients of fg_graph_attention_additive_f32.  row_coef is [heads, n_dst, 4] here: (max + log(sum),
 * <dout, out>, er, 0) per row and head, made by fg_graph_attention_additive_coef_f32 from the forward pass's
 * row_state and output.  _er: d_er [heads, n_dst], on the forward pass's plan and arrays (gathers el and V);
 * _elv: d_el [heads, n_src] and dv [n_src, heads, head_len], on a plan and arrays of the transposed adjacency
 * (gathers dout and row_coef of the destinations).
 */
int fg_graph_attention_additive_coef_f32(const float *out_dev, const float *dout_dev, const float *row_state_dev,
                                         const float *er_dev, float *row_coef_dev, int64_t n_dst, int heads,
                                         int head_len, void *stream);
int fg_graph_attention_additive_backward_er_f32(fg_spmm_plan *plan, const int32_t *pos_dev,
                                                const int32_t *idx_dev, const float *el_dev, const float *v_dev,
                                                const float *dout_dev, const float *row_coef_dev, float *der_dev,
                                                int heads, int head_len, float negative_slope, void *stream);
int fg_graph_attention_additive_backward_elv_f32(fg_spmm_plan *plan_t, const int32_t *pos_t_dev,
                                                 const int32_t *idx_t_dev, const float *dout_dev,
                                                 const float *el_dev, const float *v_dev, const float *row_coef_dev,
                                                 float *del_dev, float *dv_dev, int heads, int head_len,
                                                 float negative_slope, void *stream);

/*
 * The same operator and gradients for a training step, with one sweep each way.  er and el's gradient-side uses are
 * vertex by vertex here: er_dev [n_dst, heads], der_dev [n_dst, heads], and in _train_elv el_dev / del_dev [n_src, heads]
 * (the forward call still takes el_dev [heads, n_src], which it gathers).
 *   _train: also plus[v, h, :] and share[v, h], the sums of a * V and of a over the edges with el + er > 0
 *     ([n_dst, heads, head_len] and [n_dst, heads]); row_state_dev must be given.
 *   _train_coef: row_coef as above, and der = (1 - slope) * (<dout, plus> - <dout, out> * share).
 *   _train_elv: as _backward_elv.
 */
int fg_graph_attention_additive_train_f32(fg_spmm_plan *plan, const int32_t *pos_dev, const int32_t *idx_dev,
                                          const float *er_dev, const float *el_dev, const float *v_dev, float *out_dev,
                                          float *row_state_dev, float *plus_dev, float *share_dev, int heads,
                                          int head_len, float negative_slope, void *stream);
int fg_graph_attention_additive_train_coef_f32(const float *out_dev, const float *dout_dev, const float *row_state_dev,
                                               const float *er_dev, const float *plus_dev, const float *share_dev,
                                               float *row_coef_dev, float *der_dev, int64_t n_dst, int heads,
                                               int head_len, float negative_slope, void *stream);
int fg_graph_attention_additive_train_elv_f32(fg_spmm_plan *plan_t, const int32_t *pos_t_dev, const int32_t *idx_t_dev,
                                              const float *dout_dev, const float *el_dev, const float *v_dev,
                                              const float *row_coef_dev, float *del_dev, float *dv_dev, int heads,
                                              int head_len, float negative_slope, void *stream);

/* ---- synthetic graphs ---------------------------------------------------------------- */

/*
 * Seeded power-law (Chung-Lu style) directed graph in CSR form, rows = destinations:
 * row v draws in_degree[v] sources from the distribution cdf (length n, non-decreasing,
 * last element 1) over RANKS, rank -> vertex id through perm (length n); duplicates are
 * merged, a self-loop is added, columns are sorted.  Bit-identical for a given seed on
 * any host and any thread count.  Call once with indices_host == NULL to get indptr
 * (and nnz = indptr[n]); call again with the buffer to fill the column ids.
 * Stands in for benchmark/download_reddit_dataset.py, which needs a network.
 */
int fg_synth_powerlaw_csr(int64_t n, const int32_t *in_degree_host, const double *cdf_host,
                          const int32_t *perm_host, uint64_t seed, int num_threads,
                          int32_t *indptr_host, int32_t *indices_host);

/*
 * The same with planted communities, for a graph whose rows have locality (the Reddit adjacency that
 * benchmark/bench_vanilla_spmm.py:78-79 loads is made of subreddit communities; no network here): every draw of row v
 * comes, with probability p_in, from v's own community c = comm_of_vertex[v] -- the members
 * comm_member[comm_off[c] .. comm_off[c + 1]) under their own distribution comm_cdf (same layout, each
 * community's part non-decreasing with last element 1) -- and from the whole graph's distribution otherwise
 * (a row with in_degree above half its community's size s uses p_in * (s / 2) / in_degree instead, so that
 * hubs reach beyond their community instead of drawing the same members over and over).
 * Same two-call protocol and the same guarantees as fg_synth_powerlaw_csr.
 */
int fg_synth_community_csr(int64_t n, const int32_t *in_degree_host, const double *cdf_host, const int32_t *perm_host,
                           int n_comm, const int32_t *comm_of_vertex_host, const int64_t *comm_off_host,
                           const int32_t *comm_member_host, const double *comm_cdf_host, double p_in, uint64_t seed,
                           int num_threads, int32_t *indptr_host, int32_t *indices_host);

#ifdef __cplusplus
}
#endif
#endif /* FEATGRAPH_HIP_H */
