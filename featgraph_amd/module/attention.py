"""Dot-product attention over a graph's edges in one operator: multi-head SDDMM, edge softmax and per-head
weighted SpMM without the [nnz, H] scores being stored (the gradients of larger calls keep the scores' gradients for a
while: tuning.attention_keeps_score_gradients).  The reference has no such operator; the
class follows the build()/run() conventions of its modules (python/featgraph/module/spmm.py:81-161)."""
import ctypes

import numpy as np
import scipy.sparse
import torch

from .. import _lib
from .. import tuning
from ..util import util_convert_csr_to_dds
from . import common
from .gspmm import GSpMMhip

_INT32_MAX = 2 ** 31 - 1


class GraphAttentionhip(object):
    """out[v, h, :] = sum over the edges e into v of softmax_v(scale * <K[col e, h, :], Q[v, h, :]>) * V[col e, h, :]

    Q is (num_rows, H, D), K and V are (num_cols, H, D), D in {16, 32, 64}; rows without edges give 0.
    compute_args: 'scale' (default 1 / sqrt(D)); 'scores': 'dot' (default) | 'additive' -- the attention of GAT
    layers, scores leaky_relu(El[col e, h] + Er[v, h]) with 'negative_slope' (default 0.2); the inputs are then
    [Er (num_rows, H), El (num_cols, H), V (num_cols, H, D)].  schedule_args: 'num_src_partitions': 'auto' (default: chosen
    for the L2 size, as for SpMM) | int | None (plain CSR); 'num_dst_partitions': the same for the transposed
    adjacency that backward() sweeps.
    Equal, within rounding, to MultiHeadSDDMMhip -> EdgeSoftmaxhip -> GSpMMhip with per-head weights.
    """

    def __init__(self, adj_scipy):
        csr = adj_scipy.tocsr() if adj_scipy.format != 'csr' else adj_scipy
        self._num_rows, self._num_cols = csr.shape
        self._target = 'rocm'
        self._ctx = common.device()
        self._indptr = np.ascontiguousarray(csr.indptr, dtype=np.int32)
        self._indices = np.ascontiguousarray(csr.indices, dtype=np.int32)
        _lib.check(_lib.lib().fg_check_csr_host(self._num_rows, self._num_cols, _lib.host_ptr(self._indptr),
                                                _lib.host_ptr(self._indices)))
        self._csr = csr
        self._layouts = {}
        self._sum = None
        self._new_sum = None        # a Graph gives a function here that builds backward()'s weighted sum on layouts it has
        self._placeholders = None
        self.out_tvm = None

    def _layout(self, P):
        """Device arrays and a plan without split rows for P source-column partitions (built once per P)."""
        if P in self._layouts:
            return self._layouts[P]
        if P > 1:
            pos, idx, _ = util_convert_csr_to_dds(self._csr, P)
        else:
            pos, idx = self._indptr, self._indices
        lay = {'P': P, 'pos': common.to_device_i32(pos, self._ctx), 'idx': common.to_device_i32(idx, self._ctx),
               'plan': ctypes.c_void_p()}
        base = _lib.plan_opts
        opts = _lib.FgPlanOpts(split_threshold=_INT32_MAX, item_edges=base.item_edges if base is not None else 0,
                               wide_offsets=0, tile_major=base.tile_major if base is not None else 0,
                               pass_buffers=base.pass_buffers if base is not None else 0)
        with torch.cuda.device(self._ctx):
            _lib.check(_lib.lib().fg_spmm_plan_create(_lib.host_ptr(np.ascontiguousarray(pos, dtype=np.int32)),
                                                      self._num_rows, self._num_cols, P, ctypes.byref(opts),
                                                      ctypes.byref(lay['plan'])))
        common.narrow_indices(lay['plan'], lay['idx'], self._num_cols, P, self._ctx)
        self._layouts[P] = lay
        return lay

    def __del__(self):
        for lay in getattr(self, "_layouts", {}).values():
            plan = lay.get('plan')
            if plan is not None and plan.value:
                try:
                    _lib.lib().fg_spmm_plan_destroy(plan)
                except Exception:
                    pass
                lay['plan'] = None

    def build(self, input_placeholders, compute_args=None, schedule_args=None):
        """input_placeholders: [Q (num_rows, H, D), K (num_cols, H, D), V (num_cols, H, D)]."""
        compute_args = common.take_args(compute_args or {}, ('scale', 'scores', 'negative_slope'), "compute_func")
        self._additive = compute_args.get('scores', 'dot') == 'additive'
        if compute_args.get('scores', 'dot') not in ('dot', 'additive'):
            raise ValueError("scores must be 'dot' or 'additive'")
        if self._additive:
            return self._build_additive(input_placeholders, compute_args, schedule_args)
        schedule_args = common.take_args(schedule_args or {}, ('num_src_partitions', 'num_dst_partitions'), "schedule_func")
        if len(input_placeholders) != 3:
            raise ValueError("attention takes three inputs (Q, K, V), got %d" % len(input_placeholders))
        q_ph, k_ph, v_ph = input_placeholders
        if len(q_ph.shape) != 3 or q_ph.shape[0] != self._num_rows:
            raise ValueError("Q must be (num_rows=%d, H, D), got %s" % (self._num_rows, q_ph.shape))
        heads, head_len = int(q_ph.shape[1]), int(q_ph.shape[2])
        for name, ph in (("K", k_ph), ("V", v_ph)):
            if tuple(ph.shape) != (self._num_cols, heads, head_len):
                raise ValueError("%s must be (num_cols=%d, %d, %d), got %s" % (name, self._num_cols, heads, head_len, ph.shape))
        if head_len not in (16, 32, 64):
            raise ValueError("heads of 16, 32 or 64 floats, got %d" % head_len)
        P = self._partitions(schedule_args, 2 * 4 * head_len)
        self._heads, self._head_len = heads, head_len
        t_parts = schedule_args.get('num_dst_partitions')       # backward(): partitions of the transposed adjacency
        self._t_parts = None if t_parts in (None, 'auto') else int(t_parts)
        self._scale = float(compute_args.get('scale', 1.0 / np.sqrt(head_len)))
        self._active = self._layout(P)
        common.reserve(self._active['plan'], common.OP_ATTENTION, heads, head_len, 0, self._ctx)
        self._placeholders = [q_ph, k_ph, v_ph]
        self.out_tvm = torch.zeros((self._num_rows, heads, head_len), dtype=torch.float32, device=self._ctx)
        # every row's maximum score and sum of exponentials, per head: what backward() starts from
        self.state_tvm = torch.zeros((self._num_rows, heads, 2), dtype=torch.float32, device=self._ctx)
        self._coef = None
        self._sum = None
        self._scores_kept = True            # until an allocation fails
        for lay in self._layouts.values():
            lay.pop('sum_position', None)

    def _partitions(self, schedule_args, slice_row_bytes):
        """Source partitions: one head per XCD, whose L2 holds the head's slices of the gathered operands."""
        src_parts = schedule_args.get('num_src_partitions', 'auto')
        if src_parts is None:
            return 1
        if src_parts == 'auto':
            return tuning._partitions(self._num_cols, slice_row_bytes, self._indices.shape[0], self._num_rows,
                                      tuning.SPMM_SLICE_BYTES, min_segment=24)
        if int(src_parts) < 1:
            raise ValueError("num_src_partitions must be >= 1")
        return int(src_parts)

    def _build_additive(self, input_placeholders, compute_args, schedule_args):
        schedule_args = common.take_args(schedule_args or {}, ('num_src_partitions', 'num_dst_partitions'), "schedule_func")
        if len(input_placeholders) != 3:
            raise ValueError("additive attention takes three inputs (Er, El, V), got %d" % len(input_placeholders))
        er_ph, el_ph, v_ph = input_placeholders
        if len(v_ph.shape) != 3 or v_ph.shape[0] != self._num_cols:
            raise ValueError("V must be (num_cols=%d, H, D), got %s" % (self._num_cols, v_ph.shape))
        heads, head_len = int(v_ph.shape[1]), int(v_ph.shape[2])
        if tuple(er_ph.shape) != (self._num_rows, heads) or tuple(el_ph.shape) != (self._num_cols, heads):
            raise ValueError("Er must be (num_rows=%d, %d) and El (num_cols=%d, %d), got %s and %s"
                             % (self._num_rows, heads, self._num_cols, heads, er_ph.shape, el_ph.shape))
        if head_len not in (16, 32, 64):
            raise ValueError("heads of 16, 32 or 64 floats, got %d" % head_len)
        self._heads, self._head_len = heads, head_len
        self._slope = float(compute_args.get('negative_slope', 0.2))
        self._scale = 1.0
        t_parts = schedule_args.get('num_dst_partitions')
        self._t_parts = None if t_parts in (None, 'auto') else int(t_parts)
        self._active = self._layout(self._partitions(schedule_args, 4 * head_len))
        common.reserve(self._active['plan'], common.OP_ATTENTION_ADDITIVE, heads, head_len, 0, self._ctx)
        self._placeholders = [er_ph, el_ph, v_ph]
        self.out_tvm = torch.zeros((self._num_rows, heads, head_len), dtype=torch.float32, device=self._ctx)
        self.state_tvm = torch.zeros((self._num_rows, heads, 2), dtype=torch.float32, device=self._ctx)
        self._coef = None

    def _launch_additive(self, er, el, v):
        lay = self._active
        self._er_t, self._el_t = er.t().contiguous(), el.t().contiguous()      # head by head
        _lib.check(_lib.lib().fg_graph_attention_additive_f32(
            lay['plan'], _lib.dev_ptr(lay['pos']), _lib.dev_ptr(lay['idx']), _lib.dev_ptr(self._er_t),
            _lib.dev_ptr(self._el_t), _lib.dev_ptr(v), _lib.dev_ptr(self.out_tvm), _lib.dev_ptr(self.state_tvm),
            self._heads, self._head_len, ctypes.c_float(self._slope), common.stream_ptr()))

    def _launch(self, q, k, v):
        if self._additive:
            return self._launch_additive(q, k, v)
        lay = self._active
        _lib.check(_lib.lib().fg_graph_attention_f32(lay['plan'], _lib.dev_ptr(lay['pos']), _lib.dev_ptr(lay['idx']),
                                                     _lib.dev_ptr(q), _lib.dev_ptr(k), _lib.dev_ptr(v),
                                                     _lib.dev_ptr(self.out_tvm), _lib.dev_ptr(self.state_tvm),
                                                     self._heads, self._head_len,
                                                     ctypes.c_float(self._scale), common.stream_ptr()))

    def run(self, input_tvm_ndarrays):
        """[Q, K, V] -> self.out_tvm (the same tensor on every call); nothing is synchronised."""
        if self._placeholders is None:
            raise RuntimeError("call build() before run()")
        common.ensure_output(self)
        common.check_inputs(input_tvm_ndarrays, self._placeholders, self._ctx)
        self._launch(*input_tvm_ndarrays)
        return self.out_tvm

    def _transposed(self, P):
        """Position array, column ids and, for every element, its position in the adjacency's CSR order."""
        nnz = self._indices.shape[0]
        tr = scipy.sparse.csr_matrix((np.arange(nnz, dtype=np.int32), self._indices, self._indptr), shape=self._csr.shape).T.tocsr()
        tr.sort_indices()
        return util_convert_csr_to_dds(tr, P) if P > 1 else (tr.indptr, tr.indices, tr.data)

    def _layout_t(self, P):
        """The transposed adjacency (rows = sources) with P partitions over the destinations."""
        key = ('t', P)
        if key in self._layouts:
            return self._layouts[key]
        pos, idx, csr_pos = self._transposed(P)
        pos = np.ascontiguousarray(pos, dtype=np.int32)
        lay = {'P': P, 'pos': common.to_device_i32(pos, self._ctx),
               'idx': common.to_device_i32(np.ascontiguousarray(idx, dtype=np.int32), self._ctx), 'plan': ctypes.c_void_p()}
        base = _lib.plan_opts
        opts = _lib.FgPlanOpts(split_threshold=_INT32_MAX, item_edges=base.item_edges if base is not None else 0,
                               wide_offsets=0, tile_major=base.tile_major if base is not None else 0,
                               pass_buffers=base.pass_buffers if base is not None else 0)
        with torch.cuda.device(self._ctx):
            _lib.check(_lib.lib().fg_spmm_plan_create(_lib.host_ptr(pos), self._num_cols, self._num_rows, P,
                                                      ctypes.byref(opts), ctypes.byref(lay['plan'])))
        common.narrow_indices(lay['plan'], lay['idx'], self._num_rows, P, self._ctx)      # the transposed graph gathers from the rows
        if not self._additive and self._keeps_scores():
            lay['csr_pos_host'] = csr_pos                   # until _query_sum has made its positions of it
        self._layouts[key] = lay
        return lay

    def backward(self, q, k, v, out, state, grad_out):
        """(dQ, dK, dV) for dL/d(out) = grad_out, given the inputs, the output and the row state
        (out_tvm / state_tvm as they were after run() on these inputs).  The scores are formed again from Q
        and K; dK and dV come from a sweep like the forward pass over the transposed adjacency, dQ from a weighted sum
        with the scores' gradients that this sweep leaves (two arrays of nnz * H floats while the call lasts), or, where
        that does not pay or does not fit, from a sweep of its own over the adjacency.  Returns new tensors."""
        if self._placeholders is None:
            raise RuntimeError("call build() before backward()")
        common.check_inputs([q, k, v], self._placeholders, self._ctx)
        if self._additive:
            return self._backward_additive(q, k, v, out, state, grad_out)
        common.check_inputs([out, grad_out], [self._placeholders[0]] * 2, self._ctx)
        L, s = _lib.lib(), common.stream_ptr()
        coef = torch.empty_like(state)
        _lib.check(L.fg_graph_attention_coef_f32(_lib.dev_ptr(out), _lib.dev_ptr(grad_out), _lib.dev_ptr(state),
                                                 _lib.dev_ptr(coef), self._num_rows, self._heads, self._head_len, s))
        dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
        # partitions over the destinations, sized like the forward pass's over the sources
        lt = self._layout_t(self._dst_partitions(2 * 4 * self._head_len))
        kv = (lt['plan'], _lib.dev_ptr(lt['pos']), _lib.dev_ptr(lt['idx']), _lib.dev_ptr(q), _lib.dev_ptr(grad_out),
              _lib.dev_ptr(k), _lib.dev_ptr(v), _lib.dev_ptr(coef), _lib.dev_ptr(dk), _lib.dev_ptr(dv))
        tail = (self._heads, self._head_len, ctypes.c_float(self._scale), s)
        if not self._backward_with_kept_scores(lt, kv, tail, k, dq):
            lay = self._active
            _lib.check(L.fg_graph_attention_backward_q_f32(lay['plan'], _lib.dev_ptr(lay['pos']), _lib.dev_ptr(lay['idx']),
                                                           _lib.dev_ptr(q), _lib.dev_ptr(k), _lib.dev_ptr(v),
                                                           _lib.dev_ptr(grad_out), _lib.dev_ptr(coef), _lib.dev_ptr(dq), *tail))
            _lib.check(L.fg_graph_attention_backward_kv_f32(*kv, *tail))
        self._coef = coef
        return dq, dk, dv

    def _backward_with_kept_scores(self, lt, kv, tail, k, dq):
        """dK and dV, and dQ from the scores' gradients that their sweep leaves; False, and nothing of them to use, where that
        does not pay or memory for it was not to be had (not tried again before the next build(): an attempt that fails
        costs device synchronisations)."""
        if not self._keeps_scores():
            return False
        try:
            self._kept_scores_sweeps(lt, kv, tail, k, dq)
        except (MemoryError, torch.cuda.OutOfMemoryError):
            self._scores_kept = False
        if not self._scores_kept:
            # what was taken goes back to the device, where the other way's plans look for memory
            self._sum = None
            lt.pop('sum_position', None)
            if not torch.cuda.is_current_stream_capturing():
                torch.cuda.empty_cache()
        return self._scores_kept

    def _keeps_scores(self):
        return self._scores_kept and tuning.attention_keeps_score_gradients(self._indices.shape[0], self._num_rows, self._heads, self._head_len)

    def _kept_scores_sweeps(self, lt, kv, tail, k, dq):
        L, H, nnz = _lib.lib(), self._heads, self._indices.shape[0]
        # the sum's plan and positions before the arrays: the library allocates beside torch, not from what torch holds
        total, position = self._query_sum(lt)
        ds, other = torch.empty((2, H, nnz), dtype=torch.float32, device=self._ctx)
        _lib.check(L.fg_graph_attention_backward_kv_ds_f32(*kv, _lib.dev_ptr(ds), *tail))
        result = ctypes.c_void_p()
        _lib.check(L.fg_edge_values_permute_f32(_lib.dev_ptr(ds), _lib.dev_ptr(position), nnz, H, _lib.dev_ptr(other),
                                                ctypes.byref(result), tail[-1]))
        flat = total._placeholders[0].shape
        total.run_laid_out(k.view(flat), ds if result.value == ds.data_ptr() else other, dq.view((self._num_rows,) + flat[1:]))

    def _own_sum(self, inputs):
        csr = self._csr
        total = GSpMMhip(scipy.sparse.csr_matrix((np.ones(csr.nnz, np.float32), csr.indices, csr.indptr), shape=csr.shape))
        total.build(inputs, {}, {})
        return total

    def _query_sum(self, lt):
        """(weighted sum over the adjacency with H heads, position in lt's element order of each element of its layout)."""
        if self._sum is None:
            H, D, nnz = self._heads, self._head_len, self._indices.shape[0]
            total = (self._new_sum or self._own_sum)([common.placeholder((self._num_cols,) + ((D,) if H == 1 else (H, D))),
                                                      common.placeholder((nnz,) if H == 1 else (nnz, H))])
            total.out_tvm = None                    # its results go to tensors of backward()'s own
            self._sum = total
        if 'sum_position' not in lt:
            csr_pos = lt.pop('csr_pos_host', None)
            if csr_pos is None:                             # positions of another build were made of it
                csr_pos = self._transposed(lt['P'])[2]
            csr_pos = common.to_device_i32(csr_pos, self._ctx).long()
            of_csr = torch.empty(csr_pos.shape, dtype=torch.int32, device=self._ctx)
            of_csr[csr_pos] = torch.arange(csr_pos.shape[0], dtype=torch.int32, device=self._ctx)
            pos = self._sum.layout_positions()
            lt['sum_position'] = of_csr if pos is None else of_csr[pos.long()]
        return self._sum, lt['sum_position']

    def _dst_partitions(self, slice_row_bytes):
        if self._t_parts is not None:
            return self._t_parts
        if self._active['P'] == 1:
            return 1
        return max(1, tuning._partitions(self._num_rows, slice_row_bytes, self._indices.shape[0], self._num_cols,
                                         tuning.SPMM_SLICE_BYTES, min_segment=24))

    def _backward_additive(self, er, el, v, out, state, grad_out):
        """(dEr, dEl, dV) of the additive-score operator."""
        out_ph = common.placeholder((self._num_rows, self._heads, self._head_len))
        common.check_inputs([out, grad_out], [out_ph] * 2, self._ctx)
        L, s = _lib.lib(), common.stream_ptr()
        H, D = self._heads, self._head_len
        er_t, el_t = er.t().contiguous(), el.t().contiguous()
        coef = torch.empty((H, self._num_rows, 4), dtype=torch.float32, device=self._ctx)
        _lib.check(L.fg_graph_attention_additive_coef_f32(_lib.dev_ptr(out), _lib.dev_ptr(grad_out), _lib.dev_ptr(state),
                                                          _lib.dev_ptr(er_t), _lib.dev_ptr(coef), self._num_rows, H, D, s))
        der_t = torch.empty_like(er_t)
        del_t = torch.empty_like(el_t)
        dv = torch.empty_like(v)
        lay = self._active
        _lib.check(L.fg_graph_attention_additive_backward_er_f32(
            lay['plan'], _lib.dev_ptr(lay['pos']), _lib.dev_ptr(lay['idx']), _lib.dev_ptr(el_t), _lib.dev_ptr(v),
            _lib.dev_ptr(grad_out), _lib.dev_ptr(coef), _lib.dev_ptr(der_t), H, D, ctypes.c_float(self._slope), s))
        lt = self._layout_t(self._dst_partitions(4 * D))
        _lib.check(L.fg_graph_attention_additive_backward_elv_f32(
            lt['plan'], _lib.dev_ptr(lt['pos']), _lib.dev_ptr(lt['idx']), _lib.dev_ptr(grad_out), _lib.dev_ptr(el_t),
            _lib.dev_ptr(v), _lib.dev_ptr(coef), _lib.dev_ptr(del_t), _lib.dev_ptr(dv), H, D,
            ctypes.c_float(self._slope), s))
        self._coef = coef
        return der_t.t().contiguous(), del_t.t().contiguous(), dv

    def reserve_train(self):
        """Sizes the plan's scratch for train_forward() of the built shape (build() sizes it for run(), which needs less): to be
        called after build() by a program whose first train_forward() is one that it captures."""
        if self._placeholders is None or not self._additive:
            raise RuntimeError("build() with additive scores before reserve_train()")
        common.reserve(self._active['plan'], common.OP_ATTENTION_ADDITIVE_TRAIN, self._heads, self._head_len, 0, self._ctx)

    def train_forward(self, er, el, v):
        """Additive scores: (out, saved) as new tensors, `saved` being what train_backward() starts from -- the row state and
        the sums over the edges with a positive score (as large as `out`), with which dEr takes no sweep of its own.  The first call
        on a plan may grow its scratch: reserve_train()."""
        if self._placeholders is None or not self._additive:
            raise RuntimeError("build() with additive scores before train_forward()")
        common.check_inputs([er, el, v], self._placeholders, self._ctx)
        H, D, lay = self._heads, self._head_len, self._active
        new = lambda *shape: torch.empty(shape, dtype=torch.float32, device=self._ctx)
        n = self._num_rows
        out, plus, state, share = new(n, H, D), new(n, H, D), new(n, H, 2), new(n, H)
        el_t = el.t().contiguous()                      # head by head: one head's scalars are what an XCD gathers
        _lib.check(_lib.lib().fg_graph_attention_additive_train_f32(
            lay['plan'], _lib.dev_ptr(lay['pos']), _lib.dev_ptr(lay['idx']), _lib.dev_ptr(er), _lib.dev_ptr(el_t),
            _lib.dev_ptr(v), _lib.dev_ptr(out), _lib.dev_ptr(state), _lib.dev_ptr(plus), _lib.dev_ptr(share), H, D,
            ctypes.c_float(self._slope), common.stream_ptr()))
        return out, (state, plus, share)

    def train_backward(self, er, el, v, out, saved, grad_out):
        """(dEr, dEl, dV) from what train_forward() returned on these inputs."""
        out_ph = common.placeholder((self._num_rows, self._heads, self._head_len))
        common.check_inputs([er, el, v], self._placeholders, self._ctx)
        common.check_inputs([out, grad_out], [out_ph] * 2, self._ctx)
        L, s = _lib.lib(), common.stream_ptr()
        H, D = self._heads, self._head_len
        state, plus, share = saved
        coef = torch.empty((H, self._num_rows, 4), dtype=torch.float32, device=self._ctx)
        der, del_, dv = torch.empty_like(er), torch.empty_like(el), torch.empty_like(v)
        _lib.check(L.fg_graph_attention_additive_train_coef_f32(
            _lib.dev_ptr(out), _lib.dev_ptr(grad_out), _lib.dev_ptr(state), _lib.dev_ptr(er), _lib.dev_ptr(plus),
            _lib.dev_ptr(share), _lib.dev_ptr(coef), _lib.dev_ptr(der), self._num_rows, H, D, ctypes.c_float(self._slope), s))
        lt = self._layout_t(self._dst_partitions(4 * D))
        _lib.check(L.fg_graph_attention_additive_train_elv_f32(
            lt['plan'], _lib.dev_ptr(lt['pos']), _lib.dev_ptr(lt['idx']), _lib.dev_ptr(grad_out), _lib.dev_ptr(el),
            _lib.dev_ptr(v), _lib.dev_ptr(coef), _lib.dev_ptr(del_), _lib.dev_ptr(dv), H, D, ctypes.c_float(self._slope), s))
        return der, del_, dv

    def measure_average_time(self, input_tvm_ndarrays, num_runs):
        if self._placeholders is None:
            raise RuntimeError("call build() before measure_average_time()")
        common.ensure_output(self)
        common.check_inputs(input_tvm_ndarrays, self._placeholders, self._ctx)
        q, k, v = input_tvm_ndarrays
        return common.timed_mean_seconds(lambda: self._launch(q, k, v), num_runs)

    @property
    def ctx(self):
        return self._ctx

    @property
    def target(self):
        return self._target
