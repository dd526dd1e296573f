"""Rewrite passes over the traced operator graph.

Structural clean-up: common-subexpression elimination, dead-code elimination,
hoisting of tensor constants.  Operator rewrites (observable in
`compiled.gm.graph`, same set as the reference's python/gs/jit/optimize.py):

  merge_relabel_and_all_nodes   _CAPI_GetValidNodes + _CAPI_GraphRelabel on one
                                matrix            -> one _CAPI_GraphRelabel;
                                _CAPI_BatchGetValidNodes + _CAPI_BatchBlocks
                                                  -> the block batch's frontier
  fuse_slicing_and_sampling     _CAPI_Slicing -> _CAPI_Sampling on one axis
                                                  -> _CAPI_SlicingSampling
  batch_fuse_slicing_and_sampling  _CAPI_BatchColSlicing(encoding=False) ->
                                _CAPI_BatchRowSampling
                                                  -> _CAPI_BatchFusedSlicingSampling
  fuse_square_and_sum           (e ** 2) summed by a copy_rhs / sum SpMM
                                                  -> _CAPI_FusedESquareSum
  fuse_div_and_sum              e / u[endpoint] summed onto the other endpoint,
                                quotient not used otherwise
                                                  -> _CAPI_FusedEDivUSum
  merge_u_mul_v                 two u-op-v SDDMMs on one matrix
                                                  -> _CAPI_FusedUOPV
  read_column_slice_in_place    a column slice that is only summed (squares
                                onto rows) and row-sliced is never written:
                                                  -> _CAPI_SlicedESquareSum,
                                                     _CAPI_ColRowSlicing on the
                                                     parent matrix
  chain_layers                  layers of slice + sample -> relabel
                                                  -> _CAPI_SampleLayers,
                                                     _CAPI_BatchSampleLayers
  select_formats                deterministic on_format / output_format choice

and, in the copy of the graph that calls run (like chain_layers):

  compute_edge_scores           products of features summed over the feature, stacked
                                and multiplied by a vector  -> one kernel
  sum_encoded_slices_in_place   an encoded column slice of a super-batch that is summed
                                (squares onto rows) and sliced by rows picked of it is
                                never written
  normalise_columns             edge values divided by row and by their columns' sums
  share_leading_rows            features of all rows of a column slice: the parent's, once
  sum_slices_into_new_arrays    sums over a column slice that is not written
  weights_of_picks              picks of a list by weight and their weights  -> one operator
  relabel_row_slices            row slices that are only relabelled (and whose normalised
                                values are wanted) are not written
  count_slices_ahead            the size of a row slice is on its way before its rows are
                                picked

A pass rewrites `gm.graph` and checks it; the module's code is generated once, by
whoever runs the passes (gm.recompile()): generating it after each of them was
three quarters of a compilation.
"""
import operator
from typing import Dict, Iterable, List, Optional

import torch
import torch.fx as fx

from .. import _library
from ..format import _COO, _CSC, _CSR

# Operators that write into a caller-allocated tensor: they have no users in the
# graph but must survive dead-code elimination.
IN_PLACE_OPS = ("_CAPI_SDDMM", "_CAPI_SpMM", "_CAPI_FusedUOPV", "_CAPI_FusedESquareSum",
                "_CAPI_FusedEDivUSum", "_CAPI_SlicedESquareSum")


def _input_nodes(node: fx.Node) -> Iterable[fx.Node]:
    return node.all_input_nodes


def _finish(gm: fx.GraphModule) -> fx.GraphModule:
    gm.graph.lint()
    return gm


def _drop_dead_nodes(graph: fx.Graph, replaced=()) -> None:
    """`replaced`: operators that write in place and have been replaced."""
    live = set()
    for node in reversed(graph.nodes):
        if node.op in ("output", "placeholder") or node.target in IN_PLACE_OPS and node not in replaced:
            live.add(node)
        if node in live:
            live.update(_input_nodes(node))
    for node in reversed(graph.nodes):
        if node not in live:
            graph.erase_node(node)


def dce(gm: fx.GraphModule) -> fx.GraphModule:
    _drop_dead_nodes(gm.graph)
    return _finish(gm)


def _draws_random_numbers(node: fx.Node) -> bool:
    """Sampling and walk operators, whether methods of the graph class
    (call_method, target is the name) or free operators of gs_ops
    (call_function, target is the operator object)."""
    name = node.target if isinstance(node.target, str) else str(node.target)
    return any(word in name for word in ("Sampling", "RandomWalk", "Node2Vec"))


def cse(gm: fx.GraphModule) -> fx.GraphModule:
    """Merges nodes with identical target and arguments.  Sampling operators are
    left alone: two textually identical sampling calls draw different samples."""
    seen: Dict[str, fx.Node] = {}
    for node in list(gm.graph.nodes):
        if node.op in ("placeholder", "output"):
            continue
        if _draws_random_numbers(node):
            continue
        if node.target in IN_PLACE_OPS:
            continue
        key = f"{node.op}|{node.target}|{node.args}|{node.kwargs}"
        if key in seen:
            node.replace_all_uses_with(seen[key])
            gm.graph.erase_node(node)
        else:
            seen[key] = node
    return _finish(gm)


def move_constant_to_top(gm: fx.GraphModule) -> fx.GraphModule:
    first = next(iter(gm.graph.nodes))
    constants = [n for n in gm.graph.nodes if n.op == "get_attr" and "constant" in n.name]
    with gm.graph.inserting_before(first):
        for node in constants:
            if node is first:
                continue
            node.replace_all_uses_with(gm.graph.node_copy(node))
            gm.graph.erase_node(node)
    return _finish(gm)


def _is_method(node: fx.Node, name: str) -> bool:
    return node.op == "call_method" and node.target == name


def _getitem_users(node: fx.Node, index: int) -> List[fx.Node]:
    return [u for u in node.users
            if u.op == "call_function" and u.target is operator.getitem and u.args[1] == index]


def merge_relabel_and_all_nodes(gm: fx.GraphModule) -> fx.GraphModule:
    """all_nodes() and to_dgl_block() of one matrix share a single relabel."""
    gm = cse(gm)
    by_graph: Dict[fx.Node, List[fx.Node]] = {}
    for node in gm.graph.nodes:
        if _is_method(node, "_CAPI_GetValidNodes") or _is_method(node, "_CAPI_GraphRelabel"):
            by_graph.setdefault(node.args[0], []).append(node)
    for group in by_graph.values():
        relabels = [n for n in group if n.target == "_CAPI_GraphRelabel"]
        valid = [n for n in group if n.target == "_CAPI_GetValidNodes"]
        if not relabels or not valid:
            continue
        keep = relabels[0]
        first = min(group, key=lambda n: list(gm.graph.nodes).index(n))
        if first is not keep:
            first.prepend(keep)  # the relabel must precede every former user
        with gm.graph.inserting_after(keep):
            frontier = gm.graph.call_function(operator.getitem, args=(keep, 0))
        for v in valid:
            if v.args[1:] == keep.args[1:]:
                v.replace_all_uses_with(frontier)
    return dce(_merge_batch_blocks_and_all_nodes(gm))


def _merge_batch_blocks_and_all_nodes(gm: fx.GraphModule) -> fx.GraphModule:
    """The super-batched twin: all_nodes() reads the frontier and its batch
    pointer off the layer's block batch, which is built first.  The relabel is
    then queued before the host waits for the size of the frontier, so the
    device has work while that number travels."""
    by_graph: Dict[fx.Node, List[fx.Node]] = {}
    for node in gm.graph.nodes:
        if _is_method(node, "_CAPI_BatchGetValidNodes") or _is_method(node, "_CAPI_BatchBlocks"):
            by_graph.setdefault(node.args[0], []).append(node)
    for group in by_graph.values():
        # (numbered anew for every group: the rewrite of an earlier layer added nodes)
        order = {n: i for i, n in enumerate(gm.graph.nodes)}
        builders = [n for n in group if n.target == "_CAPI_BatchBlocks"]
        valid = [n for n in group if n.target == "_CAPI_BatchGetValidNodes"]
        if not builders or not valid:
            continue
        keep = builders[0]
        # only all_nodes() calls with the builder's own id tensors read its frontier
        matching = [v for v in valid if v.args[1:] == keep.args[1:]]
        if not matching:
            continue
        first = min(matching + [keep], key=lambda n: order[n])
        if first is not keep:
            # the builder moves in front of its first reader, but never in front of
            # one of its own arguments
            if any(order[a] > order[first] for a in keep.all_input_nodes):
                continue
            first.prepend(keep)
        with gm.graph.inserting_after(keep):
            ptr = gm.graph.call_method("frontier_ptr", args=(keep,))
            frontier = gm.graph.call_method("frontier", args=(keep,))
        for v in matching:
            for user in list(v.users):
                if (user.op == "call_function" and user.target is operator.getitem
                        and user.args[1] in (0, 1)):
                    user.replace_all_uses_with(frontier if user.args[1] == 0 else ptr)
    gm.graph.lint()
    return gm


def fuse_slicing_and_sampling(gm: fx.GraphModule) -> fx.GraphModule:
    """Slicing(seeds, axis, on, out) -> [0] -> Sampling(axis, K, replace, on, out)
       => SlicingSampling(axis, seeds, K, replace, on, out).

    Edge data gathered through the slice index and then through the sampling
    index is re-gathered from the parent with the fused index, which addresses
    the parent's edges directly."""
    for sampling in list(gm.graph.nodes):
        if not _is_method(sampling, "_CAPI_Sampling"):
            continue
        sliced_graph = sampling.args[0]
        if not (sliced_graph.op == "call_function" and sliced_graph.target is operator.getitem
                and sliced_graph.args[1] == 0):
            continue
        slicing = sliced_graph.args[0]
        if not _is_method(slicing, "_CAPI_Slicing"):
            continue
        if sampling.args[1] != slicing.args[2]:      # same axis
            continue
        if len(sliced_graph.users) > 1:              # the slice itself is used
            continue
        slice_index = _getitem_users(slicing, 1)
        sample_index = _getitem_users(sampling, 1)
        # every tensor gathered with the slice index may only feed a gather with
        # the sampling index
        rewires = []
        ok = True
        for idx_node in slice_index:
            for gathered in idx_node.users:
                users = list(gathered.users)
                if len(users) != 1 or not sample_index or sample_index[0] not in users[0].args:
                    ok = False
                rewires.append((gathered, users[0] if users else None))
        if not ok:
            continue
        with gm.graph.inserting_before(slicing):
            fused = gm.graph.call_method(
                "_CAPI_SlicingSampling",
                args=(slicing.args[0], slicing.args[2], slicing.args[1], sampling.args[2],
                      sampling.args[3], sampling.args[4], sampling.args[5]))
            fused_graph = gm.graph.call_function(operator.getitem, args=(fused, 0))
            fused_index = gm.graph.call_function(operator.getitem, args=(fused, 1))
        for g in _getitem_users(sampling, 0):
            g.replace_all_uses_with(fused_graph)
        for gathered, second in rewires:
            with gm.graph.inserting_before(second):
                direct = gm.graph.call_function(operator.getitem,
                                                args=(gathered.args[0], fused_index))
            second.replace_all_uses_with(direct)
    return dce(gm)


def _fuse_weighted(gm: fx.GraphModule, slice_name: str, sample_name: str,
                   probs_arg: int, compatible, make_fused) -> fx.GraphModule:
    """Shared by the two passes below.  The weights of the sampling call must be
    a gather of some edge tensor through the slice index; the fused operator
    takes that edge tensor itself (the parent's weights), and every edge tensor
    that went through the slice index and then through the sampling index is
    re-gathered from the parent with the fused index."""
    for sampling in list(gm.graph.nodes):
        if not _is_method(sampling, sample_name):
            continue
        sliced_graph = sampling.args[0]
        if not (sliced_graph.op == "call_function" and sliced_graph.target is operator.getitem
                and sliced_graph.args[1] == 0 and len(sliced_graph.users) == 1):
            continue
        slicing = sliced_graph.args[0]
        if not _is_method(slicing, slice_name) or not compatible(slicing, sampling):
            continue
        slice_index = _getitem_users(slicing, 1)
        sample_index = _getitem_users(sampling, 1)
        probs = sampling.args[probs_arg]
        if not (isinstance(probs, fx.Node) and probs.op == "call_function"
                and len(probs.args) == 2 and probs.args[1] in slice_index):
            continue
        rewires, ok = [], True
        for idx_node in slice_index:
            for gathered in idx_node.users:
                for user in list(gathered.users):
                    if user is sampling:
                        continue
                    if not (sample_index and sample_index[0] in user.args):
                        ok = False
                    rewires.append((gathered, user))
        if not ok:
            continue
        with gm.graph.inserting_before(slicing):
            fused = make_fused(gm.graph, slicing, sampling, probs.args[0])
            fused_graph = gm.graph.call_function(operator.getitem, args=(fused, 0))
            fused_index = gm.graph.call_function(operator.getitem, args=(fused, 1))
        for g in _getitem_users(sampling, 0):
            g.replace_all_uses_with(fused_graph)
        for gathered, second in rewires:
            with gm.graph.inserting_before(second):
                direct = gm.graph.call_function(operator.getitem,
                                                args=(gathered.args[0], fused_index))
            second.replace_all_uses_with(direct)
    return dce(gm)


def fuse_slicing_and_weighted_sampling(gm: fx.GraphModule) -> fx.GraphModule:
    """Slicing(seeds, axis, on, out) -> [0] -> SamplingProbs(axis, w[slice index], K, ...)
       => SlicingSamplingProbs(axis, seeds, w, K, replace, on, out): the slice is
    never materialised and the draws go through the parent's weight CDF."""
    def compatible(slicing, sampling):          # same axis, same format
        return sampling.args[1] == slicing.args[2] and sampling.args[5] == slicing.args[3]

    def make(graph, slicing, sampling, weights):
        return graph.call_method(
            "_CAPI_SlicingSamplingProbs",
            args=(slicing.args[0], slicing.args[2], slicing.args[1], weights, sampling.args[3],
                  sampling.args[4], sampling.args[5], sampling.args[6]))

    return _fuse_weighted(gm, "_CAPI_Slicing", "_CAPI_SamplingProbs", 2, compatible, make)


def batch_fuse_slicing_and_weighted_sampling(gm: fx.GraphModule) -> fx.GraphModule:
    """BatchColSlicing(seeds, ptr, encoding=False) -> [0] -> BatchRowSamplingProbs(K, replace,
    w[slice index]) => BatchFusedSlicingSamplingProbs(seeds, ptr, w, K, replace)."""
    def compatible(slicing, sampling):          # encoded rows cannot be fused
        return slicing.args[3] is False

    def make(graph, slicing, sampling, weights):
        return graph.call_method(
            "_CAPI_BatchFusedSlicingSamplingProbs",
            args=(slicing.args[0], slicing.args[1], slicing.args[2], weights, sampling.args[1],
                  sampling.args[2]))

    return _fuse_weighted(gm, "_CAPI_BatchColSlicing", "_CAPI_BatchRowSamplingProbs", 3,
                          compatible, make)


def batch_fuse_slicing_and_sampling(gm: fx.GraphModule) -> fx.GraphModule:
    """BatchColSlicing(seeds, ptr, encoding=False) -> [0] -> BatchRowSampling(K, replace)
       => BatchFusedSlicingSampling(seeds, ptr, K, replace)."""
    for sampling in list(gm.graph.nodes):
        if not _is_method(sampling, "_CAPI_BatchRowSampling"):
            continue
        sliced_graph = sampling.args[0]
        if not (sliced_graph.op == "call_function" and sliced_graph.target is operator.getitem):
            continue
        slicing = sliced_graph.args[0]
        if not _is_method(slicing, "_CAPI_BatchColSlicing"):
            continue
        if slicing.args[3] is not False or len(sliced_graph.users) > 1:
            continue
        # edge data gathered through the slice index cannot be re-routed here
        if any(list(i.users) for i in _getitem_users(slicing, 1)):
            continue
        with gm.graph.inserting_before(slicing):
            fused = gm.graph.call_method(
                "_CAPI_BatchFusedSlicingSampling",
                args=(slicing.args[0], slicing.args[1], slicing.args[2], sampling.args[1],
                      sampling.args[2]))
        sampling.replace_all_uses_with(fused)
    return dce(gm)


def _is_wrapped(node, name: str) -> bool:
    return (isinstance(node, fx.Node) and node.op == "call_function"
            and getattr(node.target, "__name__", "") == name)


def fuse_square_and_sum(gm: fx.GraphModule) -> fx.GraphModule:
    """SpMM("copy_rhs", "sum", _, e ** 2, ...) => FusedESquareSum(..., e, ...)."""
    for spmm in list(gm.graph.nodes):
        if not _is_method(spmm, "_CAPI_SpMM"):
            continue
        if spmm.args[1] != "copy_rhs" or spmm.args[2] != "sum":
            continue
        efeat = spmm.args[4]
        if not (isinstance(efeat, fx.Node) and efeat.op == "call_function"
                and efeat.target is operator.pow and efeat.args[1] == 2):
            continue
        new_args = list(spmm.args)
        new_args[4] = efeat.args[0]
        with gm.graph.inserting_before(spmm):
            gm.graph.call_method("_CAPI_FusedESquareSum", args=tuple(new_args))
        gm.graph.erase_node(spmm)
        # the step that shapes the accumulator only looks at shape and dtype:
        # give it the plain weights, so that the square is dead and goes away
        for user in list(efeat.users):
            if _is_wrapped(user, "_before_spmm"):
                user.replace_input_with(efeat, efeat.args[0])
    return dce(gm)


def fuse_div_and_sum(gm: fx.GraphModule) -> fx.GraphModule:
    """q = e / u[t] (an SDDMM with targets (e, t) and operator "div", or "mul"
    with 1.0 / u as its operand), then SpMM("copy_rhs", "sum", _, q)
    onto the other endpoint, q read by nothing else
        => FusedEDivUSum("div", "sum", u, e, ...): the quotient is never stored.
    The reference names this pass and leaves it empty
    (python/gs/jit/optimize.py:372-374)."""
    from ..ops.fused_op import _before_e_div_u_sum
    for spmm in list(gm.graph.nodes):
        if not _is_method(spmm, "_CAPI_SpMM"):
            continue
        if spmm.args[1] != "copy_rhs" or spmm.args[2] != "sum":
            continue
        quotient, u_target = spmm.args[4], spmm.args[8]
        v_item = spmm.args[5]
        if not (_is_wrapped(quotient, "_after_sddmm") and isinstance(v_item, fx.Node)
                and v_item.target is operator.getitem
                and _is_wrapped(v_item.args[0], "_before_spmm")):
            continue
        before_spmm = v_item.args[0]
        if set(quotient.users) != {spmm, before_spmm}:
            continue                      # the quotient itself is wanted as well
        out_item = quotient.args[0]
        if not (isinstance(out_item, fx.Node) and out_item.target is operator.getitem
                and _is_wrapped(out_item.args[0], "_before_sddmm")):
            continue
        before_sddmm = out_item.args[0]
        writers = [n for n in out_item.users if _is_method(n, "_CAPI_SDDMM")]
        if len(writers) != 1 or set(out_item.users) != {writers[0], quotient}:
            continue
        sddmm = writers[0]
        if not (sddmm.args[0] is spmm.args[0] and sddmm.args[4] is out_item
                and sddmm.args[5] == 1 and sddmm.args[6] == u_target and u_target in (0, 2)):
            continue
        op, e, rhs = before_sddmm.args[1], before_sddmm.args[2], before_sddmm.args[3]
        if op == "div":
            u = rhs
        elif (op == "mul" and isinstance(rhs, fx.Node) and rhs.op == "call_function"
              and rhs.target is operator.truediv and rhs.args[0] == 1.0):
            u = rhs.args[1]
        else:
            continue
        # the accumulator's users: the SpMM and the step that squeezes the result
        finish = [n for n in v_item.users if _is_wrapped(n, "_after_spmm")]
        if len(finish) != 1 or set(v_item.users) != {spmm, finish[0]}:
            continue
        with gm.graph.inserting_before(spmm):
            parts = gm.graph.call_function(
                _before_e_div_u_sum,
                args=(before_spmm.args[0], before_spmm.args[1], e, u, u_target))
            u2, e2, v, squeeze = (gm.graph.call_function(operator.getitem, args=(parts, i))
                                  for i in range(4))
            gm.graph.call_method("_CAPI_FusedEDivUSum",
                                 args=(spmm.args[0], "div", "sum", u2, e2, v, None, None,
                                       u_target, spmm.args[9]))
        finish[0].args = (v, squeeze)
        gm.graph.erase_node(spmm)
        gm.graph.erase_node(sddmm)
    return dce(gm)


def merge_u_mul_v(gm: fx.GraphModule) -> fx.GraphModule:
    """Two SDDMMs with targets (u, v), the same operator, graph and format
       => one FusedUOPV that sweeps the edges once."""
    groups: Dict[str, List[fx.Node]] = {}
    for node in gm.graph.nodes:
        if _is_method(node, "_CAPI_SDDMM") and node.args[5] == 0 and node.args[6] == 2:
            groups.setdefault(f"{node.args[0]}|{node.args[1]}|{node.args[7]}", []).append(node)
    order = {n: i for i, n in enumerate(gm.graph.nodes)}
    for pair in groups.values():
        if len(pair) != 2:
            continue
        first, second = sorted(pair, key=order.get)
        # The fused operator runs where the second product ran.  Readers of the
        # first output that sit in between (its squeeze step) move behind it;
        # that is only sound when their own users come later still.
        early = [u for u in first.args[4].users
                 if u is not first and order[u] < order[second]]
        if any(order[uu] < order[second] for u in early for uu in u.users):
            continue
        for u in sorted(early, key=order.get, reverse=True):
            second.append(u)
        with gm.graph.inserting_before(second):
            gm.graph.call_method(
                "_CAPI_FusedUOPV",
                args=(first.args[0], first.args[1], first.args[2], first.args[3], first.args[4],
                      second.args[2], second.args[3], second.args[4], second.args[7]))
        gm.graph.erase_node(first)
        gm.graph.erase_node(second)
    return dce(gm)


def read_column_slice_in_place(gm: fx.GraphModule) -> fx.GraphModule:
    """s = A._CAPI_Slicing(cols, axis=1, ...) whose matrix s[0] is only asked for its
    shape, summed by _CAPI_FusedESquareSum(copy_rhs, sum, e = w[s[1]]) onto rows, and
    row-sliced (s[0]._CAPI_Slicing(rows, axis=0, ...)), and whose edge index s[1] only
    gathers edge data that feeds those operators
        => A._CAPI_SlicedESquareSum(cols, w, out)
           A._CAPI_ColRowSlicing(cols, rows, on, out)   (edge index into A's edges)
    The slice -- row id, edge position and column of every edge, and every edge
    tensor gathered through it -- is then dead and is not computed: a layer-wise
    sampler slices a few hundred long columns, sums them onto rows, keeps a quarter
    of the edges and never looks at the rest again (examples/ladies/ladies.py:7-21 of
    the reference, which fuses neither step for a single matrix)."""
    for slicing in list(gm.graph.nodes):
        if not _is_method(slicing, "_CAPI_Slicing") or slicing.args[2] != 1:
            continue
        parent, cols = slicing.args[0], slicing.args[1]
        sliced = _getitem_users(slicing, 0)
        index = _getitem_users(slicing, 1)
        if len(sliced) != 1 or len(index) > 1 or len(slicing.users) != len(sliced) + len(index):
            continue
        g = sliced[0]
        gathered = list(index[0].users) if index else []
        if not all(_is_wrapped(n, "data_index") and n.args[1] is index[0] for n in gathered):
            continue
        sums, row_slices, shapes, ok = [], [], [], True
        for user in g.users:
            if (_is_method(user, "_CAPI_FusedESquareSum") and user.args[0] is g
                    and user.args[1] == "copy_rhs" and user.args[2] == "sum"
                    and user.args[8] == 2 and user.args[4] in gathered):
                sums.append(user)
            elif (_is_method(user, "_CAPI_Slicing") and user.args[0] is g
                  and user.args[2] == 0):
                row_slices.append(user)
            elif (_is_method(user, "_CAPI_GetNumRows") or _is_method(user, "_CAPI_GetNumCols")):
                shapes.append(user)
            else:
                ok = False
        if not ok or not row_slices:
            continue
        # what was gathered through the slice may only be summed, looked at for its
        # shape, or gathered again through the index of one of the row slices
        regather = []
        row_indices = [i for rs in row_slices for i in _getitem_users(rs, 1)]
        for w in gathered:
            for user in w.users:
                if user in sums and user.args[4] is w and list(user.all_input_nodes).count(w) == 1:
                    continue
                if _is_wrapped(user, "_before_spmm"):
                    continue
                if (_is_wrapped(user, "data_index") and user.args[0] is w
                        and user.args[1] in row_indices):
                    regather.append(user)
                    continue
                ok = False
        if not ok:
            continue
        for node in shapes:
            with gm.graph.inserting_before(node):
                if node.target == "_CAPI_GetNumRows":      # a column slice keeps the rows
                    fresh = gm.graph.call_method("_CAPI_GetNumRows", args=(parent,))
                else:
                    fresh = gm.graph.call_method("numel", args=(cols,))
            node.replace_all_uses_with(fresh)
        for node in sums:
            w = node.args[4]
            with gm.graph.inserting_before(node):
                gm.graph.call_method("_CAPI_SlicedESquareSum",
                                     args=(parent, cols, w.args[0], node.args[5]))
            gm.graph.erase_node(node)
        for w in gathered:
            for user in list(w.users):
                if _is_wrapped(user, "_before_spmm"):      # reads shape and dtype only
                    user.replace_input_with(w, w.args[0])
        for rs in row_slices:
            with gm.graph.inserting_before(rs):
                fused = gm.graph.call_method(
                    "_CAPI_ColRowSlicing", args=(parent, cols, rs.args[1], _CSC, rs.args[4]))
            rs.replace_all_uses_with(fused)
        for node in regather:                              # the new index addresses the parent
            node.replace_input_with(node.args[0], node.args[0].args[0])
    return dce(gm)


def sink_block_construction(gm: fx.GraphModule) -> fx.GraphModule:
    """Splitting results per batch and building blocks is host work (and, for the
    splits, a blocking read of the offsets).  Done where the sampler wrote it,
    it holds back the launches of the next layer; nothing on the device depends
    on it, so it moves to the end of the graph, in its original order."""
    host_functions = {"batch_gen_block", "batch_block_list", "create_block_from_coo", "create_block_from_csc",
                      "assign_block", "_CAPI_BatchSplitByOffset",
                      "_CAPI_BatchIndptrSplitByOffset"}

    def is_host_work(n: fx.Node) -> bool:
        if n.op == "call_method":
            return n.target == "_CAPI_BatchGetColCounts"
        if n.op != "call_function":
            return False
        name = getattr(n.target, "__name__", None) or str(n.target)
        return name.split(".")[-1] in host_functions

    output = next(n for n in gm.graph.nodes if n.op == "output")
    moving = set()
    for n in gm.graph.nodes:            # topological order: users come later
        if n.op == "output":
            continue
        if is_host_work(n) or any(a in moving for a in n.all_input_nodes):
            moving.add(n)
    for n in [n for n in gm.graph.nodes if n in moving]:
        output.prepend(n)
    return _finish(gm)


def _is_empty_constant(gm: fx.GraphModule, node) -> bool:
    """The null tensor that stands for "no id mapping"."""
    return (isinstance(node, fx.Node) and node.op == "get_attr"
            and getattr(getattr(gm, node.target, None), "numel", lambda: -1)() == 0)


def chain_layers(gm: fx.GraphModule, copy: fx.Graph) -> None:
    """In a copy of gm's graph: layer after layer of  slice + sample -> relabel,  each
    layer's frontier the next one's seeds and the sampled matrix and its edge index
    used for nothing else, becomes one operator call:
        _CAPI_SlicingSampling[Probs] -> _CAPI_GraphRelabel          (one mini-batch)
            => _CAPI_SampleLayers(seeds, fanouts, replace, weights)
        _CAPI_BatchFusedSlicingSampling[Probs] -> _CAPI_BatchBlocks  (a super-batch)
            => _CAPI_BatchSampleLayers(seeds, ptr, fanouts, replace, weights)
        _CAPI_BatchFusedSlicingSampling[Probs] -> _CAPI_BatchGetValidNodes
            => the nodes of such layers, without their blocks
    (called through the native binding, which makes the block objects).
    The operator draws the same samples.  The operator graph that a compiled sampler
    shows keeps its layers."""
    single = {"_CAPI_SlicingSampling": (2, None, 3, 4, 5), "_CAPI_SlicingSamplingProbs": (2, 3, 4, 5, 6)}
    batch = {"_CAPI_BatchFusedSlicingSampling": (1, None, 3, 4), "_CAPI_BatchFusedSlicingSamplingProbs": (1, 3, 4, 5)}
    order = {n: i for i, n in enumerate(copy.nodes)}
    draws = [n for n in copy.nodes if _draws_random_numbers(n)]

    def layer_of(node):
        """(matrix, seeds, ptr, weights, fanout, replace, relabel) of one layer, or None."""
        if node.op != "call_method" or (node.target not in single and node.target not in batch):
            return None
        is_batch = node.target in batch
        at = (batch if is_batch else single)[node.target]
        args = node.args
        if not is_batch and (args[1] != 1 or args[at[4]] != _CSC):
            return None
        sampled = _getitem_users(node, 0)
        if len(sampled) != 1 or len(node.users) != 1 or len(sampled[0].users) != 1:
            return None
        relabel = next(iter(sampled[0].users))
        nodes_only = is_batch and _is_method(relabel, "_CAPI_BatchGetValidNodes")
        if nodes_only:
            if any(not _call(u, operator.getitem) or u.args[1] not in (0, 1) for u in relabel.users):
                return None
        elif not _is_method(relabel, "_CAPI_BatchBlocks" if is_batch else "_CAPI_GraphRelabel"):
            return None
        seeds, fanout, replace = args[at[0]], args[at[2]], args[at[3]]
        if (relabel.args[0] is not sampled[0] or relabel.args[1] is not seeds
                or not _is_empty_constant(gm, relabel.args[2])
                or type(fanout) is not int or type(replace) is not bool):
            return None
        return (args[0], seeds, args[2] if is_batch else None,
                args[at[1]] if at[1] is not None else None, fanout, replace, relabel)

    chains, current = [], []
    for node in draws:
        layer = layer_of(node)
        if layer is None:
            current = []
            continue
        if current:
            (graph, _, _, weights, _, replace, prev) = current[-1][1]
            follows = (layer[0] is graph and layer[3] is weights and layer[5] == replace
                       and (layer[2] is None) == (current[-1][1][2] is None))
            if follows and layer[2] is None:
                follows = layer[1] in _getitem_users(prev, 0)
            elif follows and layer[6].target != prev.target:
                follows = False
            elif follows and _is_method(prev, "_CAPI_BatchGetValidNodes"):
                follows = layer[1] in _getitem_users(prev, 0) and layer[2] in _getitem_users(prev, 1)
            elif follows:
                follows = (_is_method(layer[1], "frontier") and layer[1].args[0] is prev
                           and _is_method(layer[2], "frontier_ptr") and layer[2].args[0] is prev)
            if follows:
                current.append((node, layer))
                continue
        current = [(node, layer)]
        chains.append(current)
    for chain in chains:
        first, (graph, seeds, ptr, weights, _, replace, end) = chain[0]
        nodes_only = _is_method(end, "_CAPI_BatchGetValidNodes")
        if any(a is not None and order[a] > order[first] for a in (graph, seeds, ptr, weights)):
            continue
        fanouts = [layer[4] for _, layer in chain]
        with copy.inserting_before(first):
            if ptr is None:
                out = copy.call_function(_library.native.sample_layers,
                                         args=(graph, seeds, fanouts, replace, weights))
            else:
                out = copy.call_function(_library.native.batch_sample_nodes if nodes_only
                                         else _library.native.batch_sample_layers,
                                         args=(graph, seeds, ptr, fanouts, replace, weights))
            for i, (_, layer) in enumerate(chain):
                relabel = layer[6]
                if ptr is not None and not nodes_only:
                    blocks = copy.call_function(operator.getitem, args=(out, i))
                    relabel.replace_all_uses_with(blocks)
                    continue
                outputs = 2 if nodes_only else 4
                for j in range(outputs):
                    users = _getitem_users(relabel, j)
                    if users:
                        item = copy.call_function(operator.getitem, args=(out, outputs * i + j))
                        for u in users:
                            u.replace_all_uses_with(item)
    if chains:
        _drop_dead_nodes(copy)


IN_PLACE_FUNCTIONS = {getattr(operator, name) for name in (
    "iadd", "iand", "iconcat", "ifloordiv", "ilshift", "imatmul", "imod", "imul", "ior", "ipow",
    "irshift", "isub", "itruediv", "ixor", "setitem", "delitem")}


def _writes_in_place(node: fx.Node) -> bool:
    """Whether a node of the sampler's own may change a tensor that others read.  Of the
    functions only those of torch, Python's operators and this package are known; any other
    (one given to torch.fx.wrap) may write."""
    if node.op not in ("call_method", "call_function"):
        return node.op == "call_module"
    if "out" in node.kwargs or node.kwargs.get("inplace") is True:
        return True
    if node.op == "call_method":
        return node.target.endswith("_") and not node.target.endswith("__")
    if node.target in IN_PLACE_FUNCTIONS:
        return True
    if isinstance(node.target, torch._ops.OpOverload):
        return node.target._schema.is_mutable
    if isinstance(node.target, torch._ops.OpOverloadPacket):
        schemas = [getattr(node.target, name)._schema for name in node.target.overloads()]
        return node.target.__name__.endswith("_") or all(s.is_mutable for s in schemas)
    name, module = getattr(node.target, "__name__", ""), getattr(node.target, "__module__", None) or ""
    known = (module.partition(".")[0] in ("torch", "_operator", "builtins", "math", __name__.partition(".")[0])
             or node.target in (_library.native.sample_layers, _library.native.batch_sample_layers,
                                _library.native.batch_sample_nodes)
             or getattr(torch, name, None) is node.target)
    return not known or name.endswith("_") and not name.endswith("__")


def _written_between(order: Dict[fx.Node, int], nodes) -> bool:
    """Whether a node of the sampler's own may write from the first of `nodes` to the last:
    what they read must then be read where they stand."""
    first, last = min(order[n] for n in nodes), max(order[n] for n in nodes)
    return any(first < at < last and _writes_in_place(n) for n, at in order.items())


def _call(node, *targets) -> bool:
    return isinstance(node, fx.Node) and node.op == "call_function" and node.target in targets


def _only_user(node: fx.Node, user: fx.Node) -> bool:
    return set(node.users) == {user}


def _dim_one(node: fx.Node, position: int) -> bool:
    """Whether a call's one option is dim = 1."""
    given = list(node.args[position:]) + list(node.kwargs.values())
    return given == [1] and set(node.kwargs) <= {"dim"} and type(given[0]) is int


def _sddmm_of(out):
    """(graph, op, lhs data, rhs data, targets, format, node) of the SDDMM that wrote `out`,
    an _after_sddmm node, into an array that nothing else sees; else None."""
    if not _is_wrapped(out, "_after_sddmm") or len(out.args) != 2:
        return None
    item = out.args[0]
    if not (_call(item, operator.getitem) and item.args[1] == 2
            and _is_wrapped(item.args[0], "_before_sddmm")):
        return None
    before = item.args[0]
    writers = [n for n in item.users if _is_method(n, "_CAPI_SDDMM")]
    if len(writers) != 1 or set(item.users) != {writers[0], out}:
        return None
    w = writers[0]
    for i, arg in ((0, w.args[2]), (1, w.args[3])):
        if not (_call(arg, operator.getitem) and arg.args == (before, i)):
            return None
    if w.args[1] != before.args[1] or w.args[4] is not item:
        return None
    return w.args[0], w.args[1], before.args[2], before.args[3], [w.args[5], w.args[6]], w.args[7], w


def compute_edge_scores(copy: fx.Graph) -> None:
    """In a copy of a graph: (u * v).sum(1) of an SDDMM's products, alone or as a term of
    stack([...], dim=1) @ weights, whose other terms are quotients e / u and values an edge
    has; then relu and the addition of a constant times ones_like, where they follow
    => one _edge_score, which falls back to those operators where it has to (values that
    carry gradients, other types and shapes)."""
    from ..ops.fused_op import PRODUCTS, QUOTIENT, VALUE, _edge_score
    if any(_writes_in_place(n) for n in copy.nodes):
        return

    def products_of(node):
        """The SDDMM behind a sum over the feature of its products, or None."""
        if not ((_call(node, torch.sum) or (isinstance(node, fx.Node) and _is_method(node, "sum")))
                and len(node.args) >= 1 and _dim_one(node, 1)):
            return None
        found = _sddmm_of(node.args[0])
        if found is None or found[1] != "mul" or not _only_user(node.args[0], node):
            return None
        return found

    written = []

    def replace(node, terms, weights, positive_part, shift):
        """terms: (kind, the SDDMM as _sddmm_of gives it, or the value)"""
        kinds, lhs, rhs, targets = [], [], [], []
        for kind, of in terms:
            kinds.append(kind)
            lhs.append(of if kind == VALUE else of[2])
            rhs.append(None if kind == VALUE else of[3])
            targets += [1, 1] if kind == VALUE else of[4]
            if kind != VALUE:
                written.append(of[6])
                g, on_format = of[0], of[5]
        with copy.inserting_before(node):
            new = copy.call_function(_edge_score, args=(g, kinds, lhs, rhs, targets, weights,
                                                        positive_part, shift, on_format))
        node.replace_all_uses_with(new)

    for product in list(copy.nodes):
        if not (_call(product, torch.matmul, operator.matmul) and len(product.args) == 2
                and not product.kwargs):
            continue
        stack, weights = product.args
        if not (_call(stack, torch.stack) and len(stack.args) >= 1 and _dim_one(stack, 1)
                and isinstance(stack.args[0], (list, tuple)) and _only_user(stack, product)
                and all(isinstance(v, fx.Node) for v in (weights, *stack.args[0]))):
            continue
        terms = []
        for value in stack.args[0]:
            found = products_of(value) if _only_user(value, stack) else None
            if found is not None:
                terms.append((PRODUCTS, found))
                continue
            found = _sddmm_of(value) if _only_user(value, stack) else None
            quotient = found is not None and found[1] == "div"
            terms.append((QUOTIENT, found) if quotient else (VALUE, value))
        if (not any(kind == PRODUCTS for kind, _ in terms)
                or len({(of[0], of[5]) for kind, of in terms if kind != VALUE}) != 1):
            continue
        last, positive_part, shift = product, False, None
        after = list(last.users)
        if (len(after) == 1 and len(after[0].args) == 1 and after[0].args[0] is last
                and (_call(after[0], torch.relu) and not after[0].kwargs
                     or _call(after[0], torch.nn.functional.relu)
                     and after[0].kwargs.get("inplace", False) is False)):
            last, positive_part = after[0], True
        ones = [n for n in last.users if _call(n, torch.ones_like) and n.args == (last,) and not n.kwargs]
        if len(ones) == 1 and len(last.users) == 2:
            add = next(n for n in last.users if n is not ones[0])
            scaled = list(ones[0].users)
            if (_call(add, operator.add, torch.add) and not add.kwargs and len(add.args) == 2
                    and len(scaled) == 1 and _call(scaled[0], operator.mul, torch.mul)
                    and len(scaled[0].args) == 2 and not scaled[0].kwargs
                    and _only_user(scaled[0], add) and set(add.args) == {last, scaled[0]}):
                constant = [a for a in scaled[0].args if a is not ones[0]]
                if len(constant) == 1 and type(constant[0]) is float:
                    last, shift = add, constant[0]
        replace(last, terms, weights, positive_part, shift)
    for node in list(copy.nodes):
        found = products_of(node)
        if found is not None and node.users and not any(_call(u, torch.stack) for u in node.users):
            replace(node, [(PRODUCTS, found)], None, False, None)
    if written:
        _drop_dead_nodes(copy, written)


def normalise_columns(copy: fx.Graph) -> None:
    """In a copy of a graph: q / s[column] with s = sum of q over columns, where q = e /
    r[row], or an edge value itself, is used for nothing else; and the gather that e comes
    from, if only this reads it  => one _normalised, in the last one's place."""
    from ..ops.fused_op import _normalised
    order = {n: i for i, n in enumerate(copy.nodes)}
    written = []
    for out in list(copy.nodes):
        last = _sddmm_of(out) if out.users else None
        if last is None or last[1] != "div" or last[4] != [1, 2]:
            continue
        g, q, s = last[0], last[2], last[3]
        if not (isinstance(q, fx.Node) and _is_wrapped(s, "_after_spmm") and len(s.users) == 1
                and _call(s.args[0], operator.getitem) and s.args[0].args[1] == 0
                and _is_wrapped(s.args[0].args[0], "_before_spmm")):
            continue
        total, before_total = s.args[0], s.args[0].args[0]
        sums = [n for n in total.users if _is_method(n, "_CAPI_SpMM")]
        before_last = next(iter(s.users))
        if len(sums) != 1 or set(total.users) != {sums[0], s} or not _is_wrapped(before_last, "_before_sddmm"):
            continue
        spmm = sums[0]
        if not (spmm.args[0] is g and spmm.args[1] == "copy_rhs" and spmm.args[2] == "sum"
                and spmm.args[4] is q and spmm.args[8] == 0 and before_total.args[5] is q):
            continue
        readers = {spmm, before_total, before_last}
        first = _sddmm_of(q)
        values, divisor, formats = q, None, (last[5], spmm.args[9], last[5])
        replaced = [before_total, spmm, before_last, last[6], out]
        if (first is not None and first[1] == "div" and first[4] == [1, 0] and first[0] is g
                and set(q.users) == readers and isinstance(first[2], fx.Node)):
            values, divisor, formats = first[2], first[3], (first[5], spmm.args[9], last[5])
            readers = {n.args[0] for n in first[6].all_input_nodes if _call(n, operator.getitem)
                       and _is_wrapped(n.args[0], "_before_sddmm")}
            replaced += [first[6], *readers]
        select = None
        if _is_wrapped(values, "data_index") and set(values.users) == readers:
            replaced.append(values)
            values, select = values.args
        if _written_between(order, replaced):
            continue
        if divisor is not None:
            written.append(first[6])
        with copy.inserting_before(out):
            new = copy.call_function(_normalised, args=(g, values, select, divisor, formats))
        out.replace_all_uses_with(new)
        written += [spmm, last[6]]
    if written:
        _drop_dead_nodes(copy, written)


def sum_encoded_slices_in_place(copy: fx.Graph) -> None:
    """In a copy of a graph: s = A._CAPI_BatchColSlicing(seeds, ptr, True) whose matrix s[0]
    is only asked for its rows and shape, summed once by _CAPI_FusedESquareSum(copy_rhs, sum,
    e = w[s[1]]) onto rows, and row-sliced by what _CAPI_BatchListSampling[WithProbs] picked of
    those rows, whose edge index s[1] only gathers edge data that feeds those operators, and
    nothing written to from there to the row slice
        => _encoded_square_sums(A, seeds, ptr, w) and _encoded_row_slice, whose index
           addresses A's edges and which has the ids of the picked rows at hand."""
    from ..ops.fused_op import _encoded_row_slice, _encoded_square_sums
    order = {n: i for i, n in enumerate(copy.nodes)}

    def free_operator(node, *names):
        return (node.op == "call_function"
                and str(getattr(node.target, "__name__", node.target)).split(".")[0] in names)

    for slicing in list(copy.nodes):
        if not _is_method(slicing, "_CAPI_BatchColSlicing") or slicing.args[3] is not True:
            continue
        parent, seeds, ptr = slicing.args[:3]
        sliced, index = _getitem_users(slicing, 0), _getitem_users(slicing, 1)
        if len(sliced) != 1 or len(index) != 1 or len(slicing.users) != 2:
            continue
        g, idx = sliced[0], index[0]
        gathered = list(idx.users)
        if not all(_is_wrapped(n, "data_index") and n.args[1] is idx and n.args[0] is not idx
                   and isinstance(n.args[0], fx.Node) and n.args[0] in order
                   and order[n.args[0]] < order[slicing] for n in gathered):
            continue
        sums, row_slices, rows, shapes, ok = [], [], [], [], True
        for user in g.users:
            if (_is_method(user, "_CAPI_FusedESquareSum") and user.args[0] is g
                    and user.args[1] == "copy_rhs" and user.args[2] == "sum" and user.args[8] == 2
                    and user.args[4] in gathered and list(user.all_input_nodes).count(g) == 1):
                sums.append(user)
            elif _is_method(user, "_CAPI_BatchRowSlicing") and user.args[0] is g:
                row_slices.append(user)
            elif _is_method(user, "_CAPI_BatchGetRows"):
                rows.append(user)
            elif _is_method(user, "_CAPI_GetNumRows") or _is_method(user, "_CAPI_GetNumCols"):
                shapes.append(user)
            else:
                ok = False
        if not ok or len(sums) != 1 or not row_slices:
            continue
        total = sums[0]
        accumulator, before = total.args[5], total.args[5].args[0]
        if not (_call(accumulator, operator.getitem) and accumulator.args[1] == 0
                and _is_wrapped(before, "_before_spmm")):
            continue
        after = [n for n in accumulator.users if _is_wrapped(n, "_after_spmm")]
        if (len(after) != 1 or set(accumulator.users) != {total, after[0]}
                or any(not _only_user(n, before) for n in shapes)
                or any(not _call(n, operator.getitem) or n.args[1] not in (0, 1)
                       for r in rows for n in r.users)):
            continue
        row_ptrs = [n for r in rows for n in _getitem_users(r, 1)]
        regather = []
        row_indices = [i for rs in row_slices for i in _getitem_users(rs, 1)]
        for w in gathered:
            for user in w.users:
                if user is total or user is before:
                    continue
                if _is_wrapped(user, "data_index") and user.args[0] is w and user.args[1] in row_indices:
                    regather.append(user)
                else:
                    ok = False
        for rs in row_slices:
            picked, picked_ptr = rs.args[1], rs.args[2]
            if not (_call(picked, operator.getitem) and picked.args[1] == 0
                    and _call(picked_ptr, operator.getitem) and picked_ptr.args[1] == 1
                    and picked.args[0] is picked_ptr.args[0]
                    and free_operator(picked.args[0], "_CAPI_BatchListSampling",
                                      "_CAPI_BatchListSamplingWithProbs")
                    and picked.args[0].args and picked.args[0].args[-1] in row_ptrs):
                ok = False            # rows that may not be the slice's
        names = [n for r in rows for ids in _getitem_users(r, 0) for n in ids.users
                 if _call(n, operator.getitem) and n.args[0] is ids
                 and any(n.args[1] is rs.args[1] and order[rs] < order[n] for rs in row_slices)]
        if not ok or _written_between(order, [slicing, *gathered, total, *row_slices, *regather, *names]):
            continue
        with copy.inserting_before(slicing):
            found = copy.call_function(_encoded_square_sums, args=(parent, seeds, ptr, total.args[4].args[0],
                                                                   total.args[9]))
            part, ids, ids_ptr, sums_of = (copy.call_function(operator.getitem, args=(found, i))
                                           for i in range(4))
        for r in rows:
            for n in list(r.users):
                n.replace_all_uses_with(ids if n.args[1] == 0 else ids_ptr)
        after[0].replace_all_uses_with(sums_of)
        for rs in row_slices:
            with copy.inserting_before(rs):
                of = [n for n in names if n.args[1] is rs.args[1] and order[rs] < order[n]]
                picked_edges = copy.call_function(_encoded_row_slice,
                                                  args=(part, *rs.args[1:3], *([ids] if of else [])))
                for n in of:
                    n.replace_all_uses_with(copy.call_function(operator.getitem, args=(picked_edges, 2)))
            rs.replace_all_uses_with(picked_edges)
        for node in regather:
            node.replace_input_with(node.args[0], node.args[0].args[0])
        _drop_dead_nodes(copy, [total])
        order = {n: i for i, n in enumerate(copy.nodes)}


def weights_of_picks(copy: fx.Graph) -> None:
    """In a copy of a graph: picks of a list by its weights, and weights[picks]  => one
    _picks_and_weights."""
    from ..ops.fused_op import _picks_and_weights
    order = {n: i for i, n in enumerate(copy.nodes)}
    names = {"_CAPI_ListSamplingWithProbs": 3, "_CAPI_BatchListSamplingWithProbs": 4}
    replaced = []
    for node in list(copy.nodes):
        if node.op != "call_function" or node.kwargs:
            continue
        name = str(getattr(node.target, "__name__", node.target)).split(".")[0]
        if len(node.args) != names.get(name) or not isinstance(node.args[0], fx.Node):
            continue
        batched = len(node.args) == 4
        if batched and any(not _call(u, operator.getitem) or u.args[1] not in (0, 1) for u in node.users):
            continue
        picks = _getitem_users(node, 0) if batched else [node]
        weights = [u for u in node.args[0].users if _call(u, operator.getitem)
                   and u.args[0] is node.args[0] and any(u.args[1] is p for p in picks)]
        if not weights or _written_between(order, [node, *weights]):
            continue
        with copy.inserting_before(node):
            both = copy.call_function(_picks_and_weights, args=node.args)
            parts = [copy.call_function(operator.getitem, args=(both, i)) for i in range(3)]
        for w in weights:
            w.replace_all_uses_with(parts[2])
        if batched:
            for i in (0, 1):
                for u in _getitem_users(node, i):
                    u.replace_all_uses_with(parts[i])
        else:
            node.replace_all_uses_with(parts[0])
        replaced += [node, *weights]
    if replaced:
        _drop_dead_nodes(copy, replaced)


def sum_slices_into_new_arrays(copy: fx.Graph) -> None:
    """In a copy of a graph: a cleared array, the squares of a column slice's values added to
    it, and the array as it is then  => one _sliced_square_sums, which need not clear it."""
    from ..ops.fused_op import _sliced_square_sums
    order = {n: i for i, n in enumerate(copy.nodes)}
    replaced = []
    for total in list(copy.nodes):
        if not _is_method(total, "_CAPI_SlicedESquareSum") or len(total.args) != 4 or total.users:
            continue
        g, cols, values, accumulator = total.args
        if not (_call(accumulator, operator.getitem) and accumulator.args[1] == 0
                and _is_wrapped(accumulator.args[0], "_before_spmm")):
            continue
        before = accumulator.args[0]
        after = [n for n in accumulator.users if _is_wrapped(n, "_after_spmm")]
        shape = before.args[1]
        if (len(before.args) != 7 or list(before.args[2:5]) != ["copy_rhs", "sum", None]
                or before.args[5] is not values or before.args[6] != 2
                or not (_is_method(before.args[0], "_CAPI_GetNumRows") and before.args[0].args[0] is g)
                or not (isinstance(shape, fx.Node) and _is_method(shape, "numel") and shape.args[0] is cols)
                or len(after) != 1 or set(accumulator.users) != {total, after[0]}
                or _written_between(order, [before, total, after[0]])):
            continue
        with copy.inserting_before(total):
            new = copy.call_function(_sliced_square_sums, args=(g, cols, values))
        after[0].replace_all_uses_with(new)
        replaced.append(total)
    if replaced:
        _drop_dead_nodes(copy, replaced)


def relabel_row_slices(copy: fx.Graph) -> None:
    """In a copy of a graph: a row slice that is relabelled by its columns and rows, whose
    edges' normalised values may be wanted, and nothing else: A[rows, cols]  => one
    _relabelled_rows, the picked rows of an encoded slice  => one _encoded_blocks, lists of
    nodes by themselves  => one _subgraph_blocks."""
    from ..ops.fused_op import (_encoded_blocks, _encoded_row_slice, _normalised, _relabelled_rows,
                                _subgraph_blocks)
    order = {n: i for i, n in enumerate(copy.nodes)}
    replaced = []
    for cut in list(copy.nodes):
        single = _is_method(cut, "_CAPI_ColRowSlicing") and len(cut.args) == 5
        picked = _call(cut, _encoded_row_slice) and len(cut.args) == 4
        square = (_is_method(cut, "_CAPI_BatchColRowSlcing") and len(cut.args) == 5
                  and cut.args[3] is cut.args[1] and cut.args[4] is cut.args[2])
        if not (single or picked or square) or cut.kwargs:
            continue
        if any(not _call(u, operator.getitem) or u.args[1] not in (0, 1, 2) for u in cut.users):
            continue
        sub, index, names = (_getitem_users(cut, i) for i in range(3))
        readers = {u for m in sub for u in m.users}
        labels = [u for u in readers
                  if _is_method(u, "_CAPI_GraphRelabel" if single else "_CAPI_BatchBlocks")]
        values = [u for u in readers if _call(u, _normalised)]
        if len(labels) != 1 or len(values) > 1 or len(readers) != len(labels) + len(values):
            continue
        label = labels[0]
        if label.kwargs or len(label.args) != 3 or label.args[0] not in sub:
            continue
        seeds, ids = label.args[1:]
        if picked:
            if ids not in names or {u for n in names for u in n.users} != {label}:
                continue
        elif seeds is not cut.args[1] or ids is not (cut.args[2] if single else cut.args[1]):
            continue
        inputs = []
        if values:
            if square or values[0].args[0] not in sub or values[0].args[2] not in index:
                continue
            inputs = [values[0].args[1], *values[0].args[3:]]
            if any(a in index or a in sub for a in inputs):
                continue
        if {u for i in index for u in i.users} != set(values):
            continue
        first = min([label, *values], key=order.get)
        # (made where the first of its readers stands: what the other one reads has to be there)
        if any(isinstance(a, fx.Node) and order.get(a, len(order)) >= order[first]
               for a in (seeds, *inputs)) or _written_between(order, [cut, label, *values]):
            continue
        with copy.inserting_before(first):
            if square:
                new = copy.call_function(_subgraph_blocks, args=cut.args[:3])
                parts = [new]
            else:
                new = (copy.call_function(_relabelled_rows, args=(*cut.args[:3], tuple(cut.args[3:]), *inputs))
                       if single else copy.call_function(_encoded_blocks, args=(*cut.args, seeds, *inputs)))
                parts = [copy.call_function(operator.getitem, args=(new, i)) for i in range(2)]
        label.replace_all_uses_with(parts[0])
        for v in values:
            v.replace_all_uses_with(parts[1])
        replaced += [cut, label, *values]
    if replaced:
        _drop_dead_nodes(copy, replaced)


def count_slices_ahead(copy: fx.Graph) -> None:
    """In a copy of a graph: the offsets of a row slice's columns, which it waits for first, are
    asked for before its rows are picked where nothing has asked for them yet."""
    from ..ops.fused_op import _picks_and_weights, _relabelled_rows
    order = {n: i for i, n in enumerate(copy.nodes)}
    for cut in list(copy.nodes):
        if not (_call(cut, _relabelled_rows) or _is_method(cut, "_CAPI_ColRowSlicing")):
            continue
        g, cols, rows = cut.args[:3]
        pick = rows.args[0] if _call(rows, operator.getitem) else rows
        name = str(getattr(pick.target, "__name__", pick.target)).split(".")[0]
        if not (_call(pick, _picks_and_weights) or pick.op == "call_function" and name in (
                "_CAPI_ListSampling", "_CAPI_ListSamplingWithProbs")):
            continue
        asked = {u for u in cols.users if g in u.all_input_nodes and order.get(u, -1) < order[cut]}
        if asked or max(order[g], order[cols]) >= order[pick]:
            continue
        with copy.inserting_before(pick):
            copy.call_method("_CAPI_PrepareSlice", args=(g, cols))


def share_leading_rows(copy: fx.Graph) -> None:
    """In a copy of a graph: the rows of a column slice are its parent's, so what is
    computed from data of all of them in one layer is what the next one computes.  Merges
    features[arange(number of rows)] and its products with a matrix, which are only read
    by operators, and reads the rows in place where products for edge operators are all that
    does (any other product may be kept for its gradient, with the rows as they were)."""
    from ..matrix_api.matrix import gen_arange
    from ..ops.fused_op import _edge_score, _leading_rows
    if any(_writes_in_place(n) for n in copy.nodes):
        return
    for node in list(copy.nodes):
        if not _is_method(node, "_CAPI_GetNumRows"):
            continue
        sliced = node.args[0]
        if (_call(sliced, operator.getitem) and sliced.args[1] == 0
                and _is_method(sliced.args[0], "_CAPI_Slicing") and sliced.args[0].args[2] == 1):
            node.args = (sliced.args[0].args[0],)

    def for_edges(node):
        return all(_call(u, _edge_score) or _is_wrapped(u, "_before_sddmm") for u in node.users)

    def only_read(node):
        return all(_call(u, torch.matmul, operator.matmul, _edge_score) or _is_wrapped(u, "_before_sddmm")
                   or (_call(u, operator.getitem) and u.args[1] is node) for u in node.users)

    seen: Dict[str, fx.Node] = {}
    for node in list(copy.nodes):
        if not (_is_method(node, "_CAPI_GetNumRows") or _call(node, gen_arange)
                or _call(node, operator.getitem, torch.matmul, operator.matmul)
                and all(isinstance(a, fx.Node) for a in node.args)):
            continue
        if not _is_method(node, "_CAPI_GetNumRows") and not only_read(node):
            continue
        key = f"{node.op}|{node.target}|{node.args}|{node.kwargs}"
        if key in seen:
            node.replace_all_uses_with(seen[key])
            copy.erase_node(node)
        else:
            seen[key] = node
    for node in list(copy.nodes):
        if (_call(node, operator.getitem) and _call(node.args[1], gen_arange) and node.users
                and all(_call(u, torch.matmul, operator.matmul) and for_edges(u) for u in node.users)
                and node.args[1].kwargs.get("dtype") is torch.int64
                and node.args[1].kwargs.get("device") == "cuda" and len(node.args[1].args) == 1):
            with copy.inserting_before(node):
                rows = copy.call_function(_leading_rows, args=(node.args[0], node.args[1].args[0]))
            node.replace_all_uses_with(rows)
    _drop_dead_nodes(copy)


# --------------------------------------------------------------- formats
# operator -> (position of on_format, position of output_format or None); positions
# count the operator object itself as argument 0 (python/gs/jit/module.py:21-31).
FORMAT_ARGS = {
    "_CAPI_Slicing": (3, 4),
    "_CAPI_Sampling": (4, 5),
    "_CAPI_SamplingProbs": (5, 6),
    "_CAPI_SlicingSampling": (5, 6),
    "_CAPI_SlicingSamplingProbs": (6, 7),
    "_CAPI_SDDMM": (7, None),
    "_CAPI_SpMM": (9, None),
    "_CAPI_FusedUOPV": (8, None),
    "_CAPI_FusedESquareSum": (9, None),
    "_CAPI_FusedEDivUSum": (9, None),
    "_CAPI_ColRowSlicing": (3, 4),
}


def _preferred(node: fx.Node) -> List[int]:
    """Formats an operator can run on, best first.  Slicing prefers the format
    whose compressed axis is the sliced one (a gather), then the other
    compressed format (a filter pass, no sort), then COO."""
    t = node.target
    if t == "_CAPI_Slicing":
        return [_CSR, _CSC, _COO] if node.args[2] == 0 else [_CSC, _CSR, _COO]
    if t in ("_CAPI_Sampling", "_CAPI_SlicingSampling"):
        return [_CSR] if node.args[1] == 0 else [_CSC]
    if t in ("_CAPI_SamplingProbs", "_CAPI_SlicingSamplingProbs"):
        return [_CSR] if node.args[1] == 0 else [_CSC]
    if t in ("_CAPI_SpMM", "_CAPI_FusedESquareSum", "_CAPI_FusedEDivUSum"):
        return [_CSR, _COO] if node.args[8] == 2 else [_CSC, _COO]
    if t == "_CAPI_SDDMM":
        return [_COO, _CSC, _CSR]
    if t == "_CAPI_ColRowSlicing":
        return [_CSC]
    return [_COO, _CSC]


def select_formats(gm: fx.GraphModule, input_formats: int = _CSC) -> fx.GraphModule:
    """Deterministic format assignment: every operator runs on the best format
    its input already holds (no conversion), and producers materialise that
    format plus COO.  Input matrices hold `input_formats`; derived matrices hold
    what their producer was told to emit.  (The reference times every plan on
    the device and keeps the fastest, python/gs/jit/module.py:306-421.)"""
    holds: Dict[fx.Node, int] = {}

    def formats_of(graph_node: fx.Node) -> int:
        if graph_node in holds:
            return holds[graph_node]
        if (graph_node.op == "call_function" and graph_node.target is operator.getitem
                and graph_node.args[0] in holds):
            return holds[graph_node.args[0]]
        return input_formats

    for node in gm.graph.nodes:
        if node.op != "call_method" or node.target not in FORMAT_ARGS:
            continue
        on_pos, out_pos = FORMAT_ARGS[node.target]
        available = formats_of(node.args[0])
        choice: Optional[int] = next((f for f in _preferred(node) if f & available), None)
        if choice is None:                      # a conversion is unavoidable
            choice = _preferred(node)[0]
        node.update_arg(on_pos, choice)
        if out_pos is not None:
            out = choice | _COO if choice != _COO else _COO
            node.update_arg(out_pos, out)
            holds[node] = out
    return _finish(gm)
