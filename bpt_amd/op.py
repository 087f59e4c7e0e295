"""Autograd operators with the surface of the reference's modules/op.py:10-70 (same Function
names, argument orders, saved tensors and `None` gradient slots), running on the HIP kernels,
plus `bpt_attention`, the fused layer core.
"""
import math

import torch
from torch.autograd import Function

from . import graphop as _g
from ._native import native as _native
from .graphop import (maskedmm_csr_backward, maskedmm_csr_forward, node_mul_edge_backward, node_mul_edge_forward,
                      sparse_softmax_backward, sparse_softmax_forward, vector_spmm_backward, vector_spmm_forward)

__all__ = ["SparseSoftmax", "MaskedMMCSR", "NodeMulEdge", "VectorSPMM", "BPTAttention", "EdgeTypeEmbedding",
           "sparse_softmax", "masked_mm", "node_mul_edge", "vec_spmm", "bpt_attention", "edge_type_embedding"]


class SparseSoftmax(Function):
    # modules/op.py:10-20
    @staticmethod
    def forward(ctx, row, indptr, eid, x):
        y = sparse_softmax_forward(row, indptr, eid, x)
        ctx.save_for_backward(row, indptr, eid, y)
        return y

    @staticmethod
    def backward(ctx, dy):
        row, indptr, eid, y = ctx.saved_tensors
        return None, None, None, sparse_softmax_backward(row, indptr, eid, y, dy.contiguous())


class MaskedMMCSR(Function):
    # modules/op.py:23-33
    @staticmethod
    def forward(ctx, row, indptr_r, eid_r, indices_r, col, indptr_c, eid_c, indices_c, A, B):
        ctx.save_for_backward(row, indptr_r, eid_r, indices_r, col, indptr_c, eid_c, indices_c, A, B)
        return maskedmm_csr_forward(row, indptr_r, eid_r, indices_r, A, B)

    @staticmethod
    def backward(ctx, grad):
        row, indptr_r, eid_r, indices_r, col, indptr_c, eid_c, indices_c, A, B = ctx.saved_tensors
        dA, dB = maskedmm_csr_backward(row, indptr_r, eid_r, indices_r, col, indptr_c, eid_c, indices_c, A, B, grad)
        return None, None, None, None, None, None, None, None, dA, dB


class NodeMulEdge(Function):
    # modules/op.py:35-45
    @staticmethod
    def forward(ctx, row, indptr, eid, A, B):
        ctx.save_for_backward(row, indptr, eid, A, B)
        return node_mul_edge_forward(row, indptr, eid, A, B)

    @staticmethod
    def backward(ctx, grad):
        row, indptr, eid, A, B = ctx.saved_tensors
        dA, dB = node_mul_edge_backward(row, indptr, eid, A, B, grad)
        return None, None, None, dA, dB


class VectorSPMM(Function):
    # modules/op.py:47-58
    @staticmethod
    def forward(ctx, row, indptr, eid, indices, col, ptr_t, eid_t, indices_t, edata, x, n_rows=None):
        # n_rows (not in the reference): rows of y when the operator is rectangular (y = zeros_like(x) there, :527)
        y = vector_spmm_forward(row, indptr, eid, indices, edata, x, n_rows=n_rows)
        ctx.save_for_backward(row, indptr, eid, indices, col, ptr_t, eid_t, indices_t, edata, x)
        return y

    @staticmethod
    def backward(ctx, dy):
        row, indptr, eid, indices, col, ptr_t, eid_t, indices_t, edata, x = ctx.saved_tensors
        dedata, dx = vector_spmm_backward(row, indptr, eid, indices, col, ptr_t, eid_t, indices_t, edata, dy, x)
        return None, None, None, None, None, None, None, None, dedata, dx, None


class BPTAttention(Function):
    """Fused masked_mm -> scale -> sparse_softmax -> dropout -> vec_spmm (modules/attention.py:66-77 with
    rel_pos off).  Saves q, k, v, o and the per-(node, head) log-sum-exp instead of the (E, h) score and
    probability tensors; the dropout mask is regenerated in backward from (dropout_p, seed)."""

    @staticmethod
    def forward(ctx, row, indptr_r, eid_r, indices_r, col, indptr_c, eid_c, indices_c, q, k, v, scale, dropout_p=0.0, seed=0):
        o, lse = _g.attention_forward(col, indptr_c, eid_c, indices_c, q, k, v, scale, dropout_p, seed)
        ctx.save_for_backward(row, indptr_r, eid_r, indices_r, col, indptr_c, eid_c, indices_c, q, k, v, o, lse)
        ctx.scale, ctx.dropout_p, ctx.seed = scale, dropout_p, seed
        return o

    @staticmethod
    def backward(ctx, do):
        row, indptr_r, eid_r, indices_r, col, indptr_c, eid_c, indices_c, q, k, v, o, lse = ctx.saved_tensors
        dq, dk, dv = _g.attention_backward(row, indptr_r, eid_r, indices_r, col, indptr_c, eid_c, indices_c,
                                           q, k, v, o, lse, do, ctx.scale, ctx.dropout_p, ctx.seed)
        return None, None, None, None, None, None, None, None, dq, dk, dv, None, None, None


class BPTRelAttention(Function):
    """BPTAttention with the rel_pos score term of modules/attention.py:69-71, s = (q.k + q.table[etype]) * scale,
    without the (E, d) rows of the embedding lookup: a small kernel writes the (E, h) term q[dst].table[etype], the
    fused kernels add it to the scores, and the backward kernel returns ds = dL/d(q.k + term) per edge and head,
    from which the term's gradients follow: dq += sum_e ds[e] table[etype[e]] over the in-CSR and
    dtable[t] = sum_h sum_{e of type t} ds[e, h] q[dst(e), h].  One kernel forms both where the shape has it
    (graphop.rel_bias_backward); otherwise two SpMMs do, the first over the in-CSR with the edge types as column indices,
    the second over a CSR whose rows are the edge types.  All sums are row-owned (no atomics)."""

    @staticmethod
    def forward(ctx, row, indptr_r, eid_r, indices_r, col, indptr_c, eid_c, indices_c, q, k, v, scale, dropout_p, seed,
                table, etype, on_tiles=None, train=False):
        """on_tiles: None or, outside of stream capture, a list, which receives the term's index tensors (_rel_aux, and those in the order of the
        tiles) and, for a call that is going to have a backward (train), both passes' plans, where the term is formed over the tiles."""
        aux = _rel_aux(etype, col, indptr_c, eid_c, table.size(0))
        table = table.contiguous()
        # (the gradient kernel's configuration is asked for here: the SpMM form is then chosen for both passes up front)
        ctx.on_chip = (_g.rel_rows_supported(q) and aux["n_used"] <= _g.REL_MAX_USED_TYPES and not _g.force_generic_enabled()
                       and _g.rel_bias_backward_supported(q, aux["n_used"]))
        # where forward and backward both run on the tile kernels, the term and its gradient are stored head-major in the
        # order in which the tiles meet the edges (rows_slot: the place of every in-CSR slot) instead of by edge id
        graph = (row, indptr_r, eid_r, indices_r, col, indptr_c, eid_c, indices_c, q, k)
        order = _g.attention_pair_order(*graph, dropout_p) if ctx.on_chip else None
        ctx.rows_slot = None
        if order is not None:
            pair = order[1]["pair_of_eid"]
            held, plans = aux.get("rows_slot"), None
            new = held is None or held[0] is not pair
            if new:
                rows_slot = pair.index_select(0, eid_c).contiguous()
                # per pair number: the number of its edge's type and which row of its tile its destination is
                types = torch.empty_like(aux["number_slot"]).index_copy_(0, rows_slot, aux["number_slot"]).to(torch.int32)
                held = (pair, rows_slot, (types | (order[1]["member_of_pair"] << 8)).contiguous())
            ctx.rows_slot = held[1]
            if on_tiles is not None and train:
                plans = _g.prepare_rel_backward(*graph, order, held[1], aux["number_slot"], aux["n_used"])
            if new and not _g.capturing(q):                       # (what a captured graph fills is there after its replays only)
                _written(q.device)                                # (a new plan, where one was just built, has been waited for with these)
                aux["rows_slot"] = held
            try:
                bias = _g.rel_bias_forward_tiles(*graph, table, aux["used_types"], held[2], dropout_p)
                if on_tiles is not None:
                    on_tiles.extend((aux, held, order, plans))
            except _g.BptStatusError as err:
                # (many types in use need more than 64 KB of LDS there, which a runtime may refuse: the kernel over the
                # in-CSR writes the same layout from within 64 KB)
                if err.status != _g.BPT_ERR_UNSUPPORTED:
                    raise
                bias = _g.rel_bias_forward(col, indptr_c, ctx.rows_slot, aux["number_slot"], q, table, used_types=aux["used_types"],
                                           by_pair=True)
        elif ctx.on_chip:
            bias = _g.rel_bias_forward(col, indptr_c, eid_c, aux["number_slot"], q, table, used_types=aux["used_types"])
        else:
            bias = _g.rel_bias_forward(col, indptr_c, eid_c, aux["etype_slot"], q, table)
        o, lse = _g.attention_forward(col, indptr_c, eid_c, indices_c, q, k, v, scale, dropout_p, seed, bias=bias,
                                      bias_by_pair=ctx.rows_slot is not None)
        ctx.save_for_backward(row, indptr_r, eid_r, indices_r, col, indptr_c, eid_c, indices_c, q, k, v, o, lse, bias, table)
        ctx.scale, ctx.dropout_p, ctx.seed, ctx.aux, ctx.etype = scale, dropout_p, seed, aux, etype
        return o

    @staticmethod
    def backward(ctx, do):
        row, indptr_r, eid_r, indices_r, col, indptr_c, eid_c, indices_c, q, k, v, o, lse, bias, table = ctx.saved_tensors
        aux = ctx.aux
        if ctx.rows_slot is not None:
            dq, dk, dv, dtable = _rel_backward(*ctx.saved_tensors, do, ctx.scale, ctx.dropout_p, ctx.seed, ctx.rows_slot, aux["number_slot"],
                                               aux["used"], aux["used_types"])
            return None, None, None, None, None, None, None, None, dq, dk, dv, None, None, None, dtable, None, None, None
        dq, dk, dv, ds = _g.attention_backward(row, indptr_r, eid_r, indices_r, col, indptr_c, eid_c, indices_c,
                                               q, k, v, o, lse, do, ctx.scale, ctx.dropout_p, ctx.seed, bias=bias)
        if ctx.on_chip:
            dtable = _g.rel_bias_backward(col, indptr_c, eid_c, aux["number_slot"], aux["used"], aux["used_types"], ds, q, table, dq)
        else:
            t_row, t_indptr, t_order, t_dst = _rel_type_rows(aux, ctx.etype, col, indptr_c, eid_c, table.size(0))
            h = q.size(1)
            ds = ds.to(q.dtype)
            table_h = table.unsqueeze(1).expand(-1, h, -1).contiguous()
            dq = vector_spmm_forward(col, indptr_c, eid_c, aux["etype_slot"], ds, table_h, n_rows=q.size(0), out=dq)
            dtable = vector_spmm_forward(t_row, t_indptr, t_order, t_dst, ds, q, n_rows=table.size(0))
            dtable = dtable.float().sum(1).to(table.dtype)
        return None, None, None, None, None, None, None, None, dq, dk, dv, None, None, None, dtable, None, None, None


def _rel_backward(row, indptr_r, eid_r, indices_r, col, indptr_c, eid_c, indices_c, q, k, v, o, lse, bias, table, do, scale, dropout_p, seed, rows_slot,
                  number_slot, used, used_types):
    """(dq, dk, dv, dtable) where the term and its gradient are stored in the order of the tiles' pairs; also what the native host path's
    node comes to with a call that its table does not serve."""
    dq, dk, dv, ds = _g.attention_backward(row, indptr_r, eid_r, indices_r, col, indptr_c, eid_c, indices_c, q, k, v, o, lse, do, scale, dropout_p,
                                           seed, bias=bias, bias_by_pair=True)
    return dq, dk, dv, _g.rel_bias_backward(col, indptr_c, rows_slot, number_slot, used, used_types, ds, q, table, dq, by_pair=True)


_REL_FORM = _g.rel_bias_forward_tiles        # what the native host path stands for: where a caller has put another function in its place, it does not


def _rel_attention(*args):
    """BPTRelAttention, by the native host path where it knows the call (the second one of a graph, shape and type on).  What the first one leaves
    with that path is made before its kernels are queued and waits for none of them, so that the backward can be queued behind the forward; a
    call under stream capture leaves nothing."""
    graph, (q, k, v, scale, dropout_p, seed, table, etype) = args[:8], args[8:]
    if not (_served_natively(graph) and _native_takes(etype) and _g.rel_bias_forward_tiles is _REL_FORM):
        return BPTRelAttention.apply(*args)
    o = _native.rel_attention(*graph, q, k, v, scale, dropout_p, seed & (2 ** 64 - 1), table, etype)
    if o is not None:
        return o
    if not q.is_cuda or _g.capturing(q):
        return BPTRelAttention.apply(*args)
    generation, on_tiles = _native.generation(), []
    train = torch.is_grad_enabled() and any(x.requires_grad for x in (q, k, v, table))
    if train and _rel_aux_key(etype, *graph[4:7], table.size(0)) not in _rel_aux_cache:      # (a new graph)
        _g.prepare_rel_training(*graph, q, k, dropout_p)
    o = BPTRelAttention.apply(*args, on_tiles, train)
    if on_tiles:
        _g.remember_rel(generation, *graph, q, k, dropout_p, table, etype, *on_tiles, train)
    return o


_rel_aux_cache = {}


def _rel_aux_key(etype, col, indptr_c, eid_c, n_types):
    return tuple((t.data_ptr(), t.numel(), t._version) for t in (etype, col, indptr_c, eid_c)) + (str(etype.device), n_types)


def _written(device):
    """Waits until the current stream has written the index tensors just made: whichever stream serves the next call reads them."""
    if device.type == "cuda":
        torch.cuda.current_stream(device).synchronize()


def _rel_aux(etype, col, indptr_c, eid_c, n_types):
    """Index tensors of the rel_pos term, cached per (etype, in-CSR): etype_slot, the edge type of every in-CSR slot;
    used_types (n_used,) int32, the types that occur in a slot, ascending; used (n_types,) int32, the number of every
    type in that list (-1 for the others); number_slot, the number of every slot's type.  Built where etype lives;
    two scalars are read back (the range check and n_used)."""
    key = _rel_aux_key(etype, col, indptr_c, eid_c, n_types)
    hit = _rel_aux_cache.get(key)
    if hit is None:
        et = etype.detach()
        if et.dim() != 1 or et.dtype != torch.int64:
            raise ValueError("etype must be a 1-D int64 tensor")
        if et.numel() and (int(et.min()) < 0 or int(et.max()) >= n_types):
            raise ValueError("edge type out of range")
        etype_slot = et.index_select(0, eid_c).contiguous()
        present = torch.zeros(n_types, dtype=torch.bool, device=et.device).index_fill_(0, etype_slot, True)
        number = torch.cumsum(present, 0) - 1
        used = torch.where(present, number, -1).to(torch.int32)
        # every type in use at its number, the others behind all of them
        types = torch.empty(n_types + 1, dtype=torch.int32, device=et.device).scatter_(
            0, torch.where(present, number, n_types), torch.arange(n_types, dtype=torch.int32, device=et.device))
        number_slot = number.index_select(0, etype_slot)
        # the read-back of n_used comes last: all of them are there for whichever stream serves the next call
        n_used = int(number[-1]) + 1 if n_types else 0
        hit = {"etype_slot": etype_slot, "used": used, "used_types": types[:n_used], "n_used": n_used, "number_slot": number_slot,
               "keep": (etype, col, indptr_c, eid_c)}
        if len(_rel_aux_cache) > 16:
            _rel_aux_cache.clear()
        _rel_aux_cache[key] = hit           # "keep" holds the tensors so that their data_ptrs are not reused while cached
    return hit


def _rel_type_rows(aux, etype, col, indptr_c, eid_c, n_types):
    """For the SpMM form of the table's gradient: the CSR whose row t lists the edges of type t (_type_csr) and the
    destination node of each of its slots; kept with the other index tensors of the graph."""
    if "type_rows" not in aux:
        t_row, t_indptr, t_order = _type_csr(etype, n_types)
        slot_dst = torch.repeat_interleave(col, indptr_c[1:] - indptr_c[:-1], output_size=eid_c.numel())   # destination of every in-CSR slot
        dst_of_eid = torch.empty_like(slot_dst)
        dst_of_eid[eid_c] = slot_dst
        aux["type_rows"] = (t_row, t_indptr, t_order, dst_of_eid.index_select(0, t_order).contiguous())
    return aux["type_rows"]


def _native_takes(*tensors):
    """Whether bptop.so's function may take a call of one of the separate operators: a trace and the transforms of torch.func work on the
    Python functions, and None (a side that only a backward would read) is no tensor to it."""
    return not torch.jit.is_tracing() and not torch._C._are_functorch_transforms_active() and all(t is not None for t in tensors)


def sparse_softmax(row, indptr, eid, x):
    if _native_takes(row, indptr, eid, x):
        return _native.sparse_softmax(row, indptr, eid, x)
    return SparseSoftmax.apply(row, indptr, eid, x)


def masked_mm(row, indptr_r, eid_r, indices_r, col, indptr_c, eid_c, indices_c, A, B):
    if _native_takes(row, indptr_r, eid_r, indices_r, col, indptr_c, eid_c, indices_c, A, B):
        return _native.masked_mm(row, indptr_r, eid_r, indices_r, col, indptr_c, eid_c, indices_c, A, B)
    return MaskedMMCSR.apply(row, indptr_r, eid_r, indices_r, col, indptr_c, eid_c, indices_c, A, B)


def node_mul_edge(row, indptr, eid, A, B):
    return NodeMulEdge.apply(row, indptr, eid, A, B)


def vec_spmm(row, indptr, eid, indices, col, ptr_t, eid_t, indices_t, edata, x, n_rows=None):
    if n_rows is None and _native_takes(row, indptr, eid, indices, col, ptr_t, eid_t, indices_t, edata, x):
        return _native.vec_spmm(row, indptr, eid, indices, col, ptr_t, eid_t, indices_t, edata, x)
    return VectorSPMM.apply(row, indptr, eid, indices, col, ptr_t, eid_t, indices_t, edata, x, n_rows)


class EdgeTypeEmbedding(Function):
    """table[etype] -> (E, d): what `self.embed_ak(g.edata['etype'])` computes (modules/attention.py:57), with a
    deterministic backward: the (E, d) gradient rows are summed per edge type by the SpMM kernels over a CSR whose
    rows are the edge types (torch's embedding backward scatters with atomics, about 1 ms at E = 430 k)."""

    @staticmethod
    def forward(ctx, table, etype, type_csr):
        ctx.type_csr = type_csr
        ctx.n_types = table.size(0)
        return table.index_select(0, etype)

    @staticmethod
    def backward(ctx, grad):
        row, indptr, order = ctx.type_csr
        grad = grad.contiguous()
        ones = torch.ones(grad.size(0), dtype=grad.dtype, device=grad.device)
        return vector_spmm_forward(row, indptr, order, order, ones, grad, n_rows=ctx.n_types), None, None


_type_csr_cache = {}


def _type_csr(etype, n_types, chunk_size=32):
    """(row, indptr, order) of the CSR whose row t lists the edges of type t (ascending edge id), chunked like the
    reference's other CSRs (builder.pyx:305-321); cached per etype tensor.  Built where etype lives: on the GPU a stable
    sort, a histogram and prefix sums, with two scalars read back (the range check and the number of units), so the
    edge types never travel to the host."""
    key = (etype.data_ptr(), etype.numel(), etype._version, str(etype.device), n_types)
    hit = _type_csr_cache.get(key)
    if hit is None:
        et = etype.detach()
        if et.dim() != 1 or et.dtype != torch.int64:
            raise ValueError("etype must be a 1-D int64 tensor")
        if et.numel() and (int(et.min()) < 0 or int(et.max()) >= n_types):
            raise ValueError("edge type out of range")
        order = torch.argsort(et, stable=True)
        counts = torch.bincount(et, minlength=n_types)
        indptr = torch.zeros(n_types + 1, dtype=torch.int64, device=et.device)
        torch.cumsum(counts, 0, out=indptr[1:])
        # partition_csr on the device: row t gives ceil(count_t / chunk) units; unit u of row t starts at indptr[t] + u * chunk
        units = (counts + (chunk_size - 1)) // chunk_size
        first = torch.cumsum(units, 0) - units                           # number of the first unit of every row
        n_units = int(units.sum())
        row = torch.repeat_interleave(torch.arange(n_types, device=et.device), units, output_size=n_units)
        rank = torch.arange(n_units, device=et.device) - first.index_select(0, row)
        indptr_units = torch.empty(n_units + 1, dtype=torch.int64, device=et.device)
        indptr_units[:n_units] = indptr.index_select(0, row) + rank * chunk_size
        indptr_units[n_units] = et.numel()
        hit = (row, indptr_units, order, etype)
        if len(_type_csr_cache) > 16:
            _type_csr_cache.clear()
        _type_csr_cache[key] = hit          # holds etype so that its data_ptr is not reused while cached
    return hit[:3]


def edge_type_embedding(table, etype):
    """Rows of `table` for every edge, differentiable w.r.t. `table` (deterministic segment-sum backward)."""
    return EdgeTypeEmbedding.apply(table, etype, _type_csr(etype, table.size(0)))


def _served_natively(graph):
    """Whether bptop.so's function may take the call: a trace records the Python function, not what the native one launches, and a
    caller that only wants a forward may leave the out-CSR side out (None), which is no tensor to it."""
    return graph[0] is not None and graph[1] is not None and graph[2] is not None and graph[3] is not None and not torch.jit.is_tracing()


def bpt_attention(row, indptr_r, eid_r, indices_r, col, indptr_c, eid_c, indices_c, q, k, v, scale=None, fused=None,
                  dropout_p=0.0, seed=None, rel_table=None, etype=None):
    """Attention over the graph: (ROW, INDPTR_R, out_eid, out_idx) is the out-CSR side (rows =
    sources), (COL, INDPTR_C, in_eid, in_idx) the in-CSR side (rows = destinations), exactly the
    eight graph arguments modules/attention.py:66-67 passes to masked_mm.

    fused=None picks the fused kernels when they cover (h, d, dtype) and otherwise composes the
    unfused HIP ops in the reference's order; both run on the GPU.

    dropout_p > 0 applies dropout to the attention probabilities (attention.py:73).  The fused path hashes
    (seed, edge, head); seed=None draws one from torch's CPU generator (reproducible under torch.manual_seed).  The
    unfused path uses torch's dropout, so the two paths drop different elements.

    rel_table (n_types, d) and etype (E,) int64 add the rel_pos term q[dst] . rel_table[etype[e]] to the score of
    edge e (attention.py:69-71); the gradient of rel_table is returned like any other."""
    scale = 1.0 / math.sqrt(q.size(-1)) if scale is None else float(scale)
    if (rel_table is None) != (etype is None):
        raise ValueError("rel_table and etype go together")
    padded = None
    if fused is None:
        fused = _g.attention_supported(q)
        if not fused and not _g.force_generic_enabled():
            padded = _g.attention_padded_shape(q)
            fused = padded is not None
        if (dropout_p > 0 or rel_table is not None) and not _g.row_groups_enabled():
            fused = False                       # only the row-group kernels implement dropout and the rel_pos term
    elif fused and not _g.attention_supported(q):
        padded = _g.attention_padded_shape(q)
    if fused and padded is not None:
        # heads of fewer than 64 columns (6 x 50, 8 x 40 in the reference's configs), computed as (h', 64) with the scale of the real d:
        # by kernels that read the rows as they are (attention_reads_narrow), else and with the rel_pos term on zero-padded copies (the
        # pads and the slice are ordinary differentiable torch ops)
        h, d = q.size(1), q.size(2)
        hp, dp = padded
        if dropout_p > 0 and seed is None:
            seed = int(torch.randint(0, 2 ** 62, (1,)).item())
        graph = (row, indptr_r, eid_r, indices_r, col, indptr_c, eid_c, indices_c)
        grow = lambda x: torch.nn.functional.pad(x, (0, dp - d, 0, hp - h))
        if rel_table is None:
            if _served_natively(graph) and _g.attention_reads_narrow(col, eid_c, q, k, hp, dropout_p):
                return _native.attention_narrow(*graph, q, k, v, hp, scale, float(dropout_p), int(seed or 0) & (2 ** 64 - 1))
            o = BPTAttention.apply(*graph, grow(q), grow(k), grow(v), scale, float(dropout_p), int(seed or 0))
            return o[:, :h, :d].contiguous()
        o = _rel_attention(*graph, grow(q), grow(k), grow(v), scale, float(dropout_p), int(seed or 0),
                           torch.nn.functional.pad(rel_table, (0, dp - d)), etype)
        return o[:, :h, :d].contiguous()
    if fused:
        if dropout_p > 0 and seed is None:
            seed = int(torch.randint(0, 2 ** 62, (1,)).item())
        if rel_table is not None:
            return _rel_attention(row, indptr_r, eid_r, indices_r, col, indptr_c, eid_c, indices_c, q, k, v, scale, float(dropout_p), int(seed or 0),
                                  rel_table, etype)
        if not _served_natively((row, indptr_r, eid_r, indices_r)):
            return BPTAttention.apply(row, indptr_r, eid_r, indices_r, col, indptr_c, eid_c, indices_c, q, k, v, scale,
                                      float(dropout_p), int(seed or 0))
        return _native.attention(row, indptr_r, eid_r, indices_r, col, indptr_c, eid_c, indices_c, q, k, v, scale, float(dropout_p),
                                 int(seed or 0) & (2 ** 64 - 1))
    e = masked_mm(row, indptr_r, eid_r, indices_r, col, indptr_c, eid_c, indices_c, k, q)
    if rel_table is not None:
        e = e + node_mul_edge(col, indptr_c, eid_c, q, edge_type_embedding(rel_table, etype))
    a = torch.nn.functional.dropout(sparse_softmax(col, indptr_c, eid_c, e * scale), p=float(dropout_p), training=dropout_p > 0)
    return vec_spmm(col, indptr_c, eid_c, indices_c, row, indptr_r, eid_r, indices_r, a, v,
                    n_rows=None if q.size(0) == v.size(0) else q.size(0))
