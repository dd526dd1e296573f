"""Fused edge-probability operators used by layer-wise samplers
(reference: python/gs/ops/fused_op.py:51-243).

  fused_u_mul_v : two u*v SDDMMs in one sweep over the edges
  e_square_sum  : out[t] = sum of e^2 over the edges of column (axis 0) / row (axis 1) t
  e_div_u_sum   : out[t] = sum of e / u[other endpoint]
"""
import torch

from .. import _library
from ..format import _COO, _CSC, _CSR
from ._common import infer_broadcast_shape
from .sddmm import _after_sddmm, _before_sddmm
from .spmm import _after_spmm, _before_spmm

torch.fx.wrap("_before_e_div_u_sum")

__all__ = ["fused_u_mul_v", "e_square_sum", "e_div_u_sum"]


def _before_e_div_u_sum(num_rows, num_cols, e, u, u_target):
    """Operands of _CAPI_FusedEDivUSum for the compiled rewrite of
    `div` followed by `sum`: both with the broadcast feature shape the two
    separate operators would have produced, and the zero-filled accumulator."""
    if u.device != e.device:
        raise ValueError(f"operand devices differ: {u.device} and {e.device}")
    if u.dtype != e.dtype:
        raise ValueError(f"operand dtypes differ: {u.dtype} and {e.dtype}")
    squeeze = e.dim() == 1 and u.dim() == 1
    e2 = e.unsqueeze(-1) if e.dim() == 1 else e
    u2 = u.unsqueeze(-1) if u.dim() == 1 else u
    feat = infer_broadcast_shape("div", tuple(e2.shape[1:]), tuple(u2.shape[1:]))
    e2 = e2.expand((e2.shape[0],) + feat).contiguous()
    u2 = u2.expand((u2.shape[0],) + feat).contiguous()
    n_out = num_cols if u_target == 0 else num_rows
    v = torch.zeros((n_out,) + feat, dtype=e.dtype, device=e.device)
    return u2, e2, v, squeeze


# kinds of terms, as gs_edge_score numbers them
VALUE, QUOTIENT, PRODUCTS = 0, 1, 2


def _edge_score(g, kinds, lhs, rhs, targets, weights, positive_part, shift, on_format):
    """What a compiled sampler's scores are computed by: a weighted sum of terms per edge
    (no weights: the one term), its positive part, plus a constant -- in one kernel, or by
    the operators that the sampler was written with where that does not take the call."""
    out = _library.native.edge_score(g, kinds, lhs, rhs, targets, weights, positive_part,
                                     shift or 0.0, on_format)
    if out is not None:
        return out
    terms = []
    for k, kind in enumerate(kinds):
        if kind == VALUE:
            terms.append(lhs[k])
            continue
        left, right, out, squeeze = _before_sddmm(
            g._CAPI_GetNumEdges(), "mul" if kind == PRODUCTS else "div", lhs[k], rhs[k])
        g._CAPI_SDDMM("mul" if kind == PRODUCTS else "div", left, right, out, targets[2 * k],
                      targets[2 * k + 1], on_format)
        out = _after_sddmm(out, squeeze)
        terms.append(torch.sum(out, dim=1) if kind == PRODUCTS else out)
    out = terms[0] if weights is None else torch.matmul(torch.stack(terms, dim=1), weights)
    if positive_part:
        out = torch.relu(out)
    return out if shift is None else out + shift * torch.ones_like(out)


def _normalised(g, values, select, divisor, formats):
    """values[select] / divisor[row] (either may be None), divided by its sums over columns: the
    end of a LADIES layer, by two passes over the edges where the operators take four or five."""
    from ..matrix_api.matrix import data_index
    if all(t is None or type(t) is torch.Tensor for t in (values, select, divisor)):
        out = g._CAPI_NormaliseColumns(values, select, divisor)
        if out is not None:
            return out

    def divided(e, by, target, on_format):
        left, right, out, squeeze = _before_sddmm(g._CAPI_GetNumEdges(), "div", e, by)
        g._CAPI_SDDMM("div", left, right, out, 1, target, on_format)
        return _after_sddmm(out, squeeze)

    e = values if select is None else data_index(values, select)
    if divisor is not None:
        e = divided(e, divisor, 0, formats[0])
    sums, arg_u, arg_e, squeeze = _before_spmm(g._CAPI_GetNumRows(), g._CAPI_GetNumCols(), "copy_rhs",
                                               "sum", None, e, 0)
    g._CAPI_SpMM("copy_rhs", "sum", None, e, sums, arg_u, arg_e, 0, formats[1])
    return divided(e, _after_spmm(sums, squeeze), 2, formats[2])


def _relabelled_rows(g, cols, rows, formats, values=None, divisor=None, value_formats=None):
    """What a compiled sampler hands on of the row slice g[rows, cols]: its relabelled edges
    (_CAPI_GraphRelabel) and, if `values` of g's edges are given, these as _normalised leaves
    them on the slice, which is not written where that can be."""
    if all(t is None or type(t) is torch.Tensor for t in (values, divisor)):
        out = g._CAPI_RelabelledRows(cols, rows, values, divisor)
        if out is not None:
            return out[:3] + (None,), out[3]
    sub, index = g._CAPI_ColRowSlicing(cols, rows, *formats)
    e = None if values is None else _normalised(sub, values, index, divisor, value_formats)
    return sub._CAPI_GraphRelabel(cols, rows), e


def _encoded_blocks(part, row_ids, rows_ptr, rows, seeds, values=None, divisor=None,
                    value_formats=None):
    """The same of a super-batched sampler: the blocks of _encoded_row_slice(part, ...)."""
    if (len(part) == 4 and part[1] is seeds and part[3] is rows
            and all(t is None or type(t) is torch.Tensor for t in (values, divisor))):
        out = part[0]._CAPI_EncodedBlocks(*part[1:], row_ids, rows_ptr, values, divisor)
        if out is not None:
            return out
    sub, index, names = _encoded_row_slice(part, row_ids, rows_ptr, rows)
    e = None if values is None else _normalised(sub, values, index, divisor, value_formats)
    return sub._CAPI_BatchBlocks(seeds, names), e


def _subgraph_blocks(g, nodes, nodes_ptr):
    """The blocks of the subgraphs that lists of nodes induce."""
    out = g._CAPI_SubgraphBlocks(nodes, nodes_ptr)
    if out is not None:
        return out
    sub, _ = g._CAPI_BatchColRowSlcing(nodes, nodes_ptr, nodes, nodes_ptr)
    return sub._CAPI_BatchBlocks(nodes, nodes)


def _sliced_square_sums(g, cols, values):
    """Sums of the squared values over the edges of the column slice g[:, cols] onto its rows."""
    if type(values) is torch.Tensor and not values.requires_grad:
        out = g._CAPI_SlicedSquareSums(cols, values)
        if out is not None:
            return out
    out, _, _, squeeze = _before_spmm(g._CAPI_GetNumRows(), cols.numel(), "copy_rhs", "sum", None, values, 2)
    g._CAPI_SlicedESquareSum(cols, values, out)
    return _after_spmm(out, squeeze)


def _encoded_square_sums(g, seeds, seeds_ptr, values, on_format):
    """What a compiled super-batched sampler asks an encoded column slice for: (the slice for
    _encoded_row_slice, its rows, where every batch's begin, sums of the squared values on
    them) -- without writing the slice where that can be."""
    from ..matrix_api.matrix import data_index
    if type(values) is torch.Tensor and not values.requires_grad:
        found = g._CAPI_EncodedSquareSums(seeds, seeds_ptr, values)
        if found is not None:
            rows, rows_ptr, sums = found
            return (g, seeds, seeds_ptr, rows), rows, rows_ptr, sums
    sub, index = g._CAPI_BatchColSlicing(seeds, seeds_ptr, True)
    rows, rows_ptr = sub._CAPI_BatchGetRows()
    values = data_index(values, index)
    out, arg_u, arg_e, squeeze = _before_spmm(sub._CAPI_GetNumRows(), sub._CAPI_GetNumCols(), "copy_rhs",
                                              "sum", None, values, 2)
    sub._CAPI_FusedESquareSum("copy_rhs", "sum", None, values, out, arg_u, arg_e, 2, on_format)
    return (sub, index), rows, rows_ptr, _after_spmm(out, squeeze)


def _encoded_row_slice(part, row_ids, rows_ptr, rows=None):
    """The rows picked of such a slice: (matrix, index into the sliced matrix's edges), and
    rows[row_ids] where its rows are given."""
    from ..matrix_api.matrix import data_index
    if len(part) == 4:
        sub, index, names = part[0]._CAPI_EncodedPickedRows(*part[1:], row_ids, rows_ptr)
        return (sub, index) if rows is None else (sub, index, names)
    sub, index = part[0]._CAPI_BatchRowSlicing(row_ids, rows_ptr)
    index = data_index(part[1], index)
    return (sub, index) if rows is None else (sub, index, rows[row_ids])


def _picks_and_weights(probs, num_picks, replace, ranges=None):
    """(picks of a list by weight, their offsets in a list cut by `ranges`, probs[picks])."""
    out = _library.native.list_sampling(probs, num_picks, replace, ranges)
    if out is not None:
        return out
    if ranges is None:
        picks, offsets = torch.ops.gs_ops._CAPI_ListSamplingWithProbs(probs, num_picks, replace), None
    else:
        picks, offsets = torch.ops.gs_ops._CAPI_BatchListSamplingWithProbs(probs, num_picks, replace, ranges)
    return picks, offsets, probs[picks]


def _leading_rows(x, n):
    """x[torch.arange(n)], to be read only: a view where that is the same."""
    if (type(x) is torch.Tensor and x.is_cuda and x.dim() >= 1 and x.is_contiguous()
            and n <= x.shape[0] and x.device.index == torch.cuda.current_device()):
        return x.narrow(0, 0, n)
    return x[torch.arange(n, dtype=torch.int64, device="cuda")]


def fused_u_mul_v(m, lhs1, rhs1, lhs2, rhs2, on_format=_COO):
    g = m._graph
    if lhs1.device != rhs1.device:
        raise ValueError(f"operand devices differ: {lhs1.device} and {rhs1.device}")
    if lhs1.dtype != rhs1.dtype:
        raise ValueError(f"operand dtypes differ: {lhs1.dtype} and {rhs1.dtype}")
    exp_l = exp_r = False
    if lhs1.dim() == 1:
        lhs1, lhs2, exp_l = lhs1.unsqueeze(-1), lhs2.unsqueeze(-1), True
    if rhs1.dim() == 1:
        rhs1, rhs2, exp_r = rhs1.unsqueeze(-1), rhs2.unsqueeze(-1), True
    num_edges = g._CAPI_GetNumEdges()
    shape = (num_edges,) + infer_broadcast_shape("mul", tuple(lhs1.shape[1:]),
                                                 tuple(rhs1.shape[1:]))
    out1 = torch.zeros(shape, dtype=lhs1.dtype, device=lhs1.device)
    out2 = torch.zeros(shape, dtype=lhs1.dtype, device=lhs1.device)
    if num_edges > 0:
        g._CAPI_FusedUOPV("mul", lhs1, rhs1, out1, lhs2, rhs2, out2, on_format)
    if exp_l and exp_r:
        out1, out2 = out1.squeeze(-1), out2.squeeze(-1)
    return out1, out2


def _reduce_target(g, axis):
    if axis == 0:
        return g._CAPI_GetNumCols(), 0
    if axis == 1:
        return g._CAPI_GetNumRows(), 2
    raise ValueError("axis should be 0 or 1")


def e_square_sum(m, key, axis, on_format=_CSR) -> torch.Tensor:
    g = m._graph
    e = m.edata[key]
    n_out, u_target = _reduce_target(g, axis)
    if e.dim() == 1:
        e = e.unsqueeze(-1)
    v = torch.zeros((n_out,), dtype=e.dtype, device=e.device)
    if g._CAPI_GetNumEdges() > 0:
        fmt = _CSC if axis == 0 else on_format
        g._CAPI_FusedESquareSum("copy_rhs", "sum", None, e, v, None, None, u_target, fmt)
    return v


def e_div_u_sum(m, key, u, axis, on_format=_CSC) -> torch.Tensor:
    g = m._graph
    e = m.edata[key]
    if u.device != e.device:
        raise ValueError(f"operand devices differ: {u.device} and {e.device}")
    if u.dtype != e.dtype:
        raise ValueError(f"operand dtypes differ: {u.dtype} and {e.dtype}")
    n_out, u_target = _reduce_target(g, axis)
    if u.dim() == 1:
        u = u.unsqueeze(-1)
    if e.dim() == 1:
        e = e.unsqueeze(-1)
    v = torch.zeros((n_out,), dtype=e.dtype, device=e.device)
    if g._CAPI_GetNumEdges() > 0:
        g._CAPI_FusedEDivUSum("div", "sum", u, e, v, None, None, u_target, on_format)
    return v
