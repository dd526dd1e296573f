"""Edge scores of attention samplers: what the compiled graph runs in one kernel, what it leaves
to the operators it was written with, and that the two give the same bits -- the samples drawn by
the scores depend on every one of them."""
import math
import operator

import numpy as np
import pytest
import torch
import torch.nn.functional as F

import gsampler_amd as gs
from gsampler_amd.ops import fused_op
from tests.conftest import random_csc

DEV = "cuda:0"


def scores(A, seeds, feats, W, weights):
    sub = A[:, seeds]
    u, v = feats[sub.rows()], feats[sub.cols()]
    a = torch.sum(gs.ops.u_mul_v(sub, u @ W, v @ W), dim=1)
    b = gs.ops.v_mul_u(sub, v @ W, u @ W).sum(1)
    c = sub.div("w", sub.sum("w", axis=0), axis=0).edata["w"]
    att = F.relu(torch.stack([a, sub.edata["w"], c, b], dim=1) @ weights)
    return att + 10e-10 * torch.ones_like(att)


def two_layers(A, seeds, feats, W, weights):
    first = scores(A, seeds, feats, W, weights)
    return first, scores(A, seeds[: 5], feats, W, weights)


def plain_sum(A, seeds, feats, W, weights):
    sub = A[:, seeds]
    return torch.sum(gs.ops.u_mul_v(sub, feats[sub.rows()] @ W, feats[sub.cols()] @ W), dim=1) + 1.0


def in_place(A, seeds, feats, W, weights):
    sub = A[:, seeds]
    u = feats[sub.rows()] @ W
    a = torch.sum(gs.ops.u_mul_v(sub, u, feats[sub.cols()] @ W), dim=1)
    return a, u.add_(1.0)


def products_wanted(A, seeds, feats, W, weights):
    sub = A[:, seeds]
    p = gs.ops.u_mul_v(sub, feats[sub.rows()] @ W, feats[sub.cols()] @ W)
    return p, torch.sum(p, dim=1)


def other_sums(A, seeds, feats, W, weights):
    sub = A[:, seeds]
    u, v = feats[sub.rows()] @ W, feats[sub.cols()] @ W
    return (torch.sum(gs.ops.u_mul_v(sub, u, v), dim=0), gs.ops.u_add_v(sub, u, v).sum(1),
            gs.ops.u_mul_v(sub, u, v).sum(dim=1, keepdim=True))


def rows_escape(A, seeds, feats, W, weights):
    u = feats[A[:, seeds].rows()]
    return u, feats[A[:, seeds[:5]].rows()], u @ W


def products_of_rows(A, seeds, feats, W, weights):
    return feats[A[:, seeds].rows()] @ W, feats[A[:, seeds[:5]].rows()] @ W


def ran(compiled):
    return [n.target for n in compiled._run.__self__.graph.nodes]


def cpu_args(nodes=10):
    m = gs.Matrix(gs.Graph(nodes, nodes))
    m.edata["w"] = torch.rand(7)
    return m, torch.arange(3), torch.rand(nodes, 4), torch.rand(4, 3), torch.rand(4)


@pytest.mark.parametrize("func,kernels,sddmm", [
    (scores, 1, 0), (two_layers, 2, 0), (plain_sum, 1, 0), (in_place, 0, 1), (products_wanted, 0, 1),
    (other_sums, 0, 3), (rows_escape, 0, 0), (products_of_rows, 0, 0)])
def test_what_becomes_an_edge_score(func, kernels, sddmm):
    c = gs.jit.compile(func=func, args=cpu_args())
    t = ran(c)
    assert t.count(fused_op._edge_score) == kernels and t.count("_CAPI_SDDMM") == sddmm
    in_place_free = func not in (in_place, rows_escape, products_of_rows)
    assert t.count(fused_op._leading_rows) == (1 if in_place_free else 0)
    if func is two_layers:                   # the rows' features once for both layers
        assert t.count(torch.matmul) + t.count(operator.matmul) == 3
    assert fused_op._edge_score not in [n.target for n in c.gm.graph.nodes]


def test_operands_are_checked_without_a_gpu():
    from gsampler_amd import capi
    lib = capi.lib()
    assert lib.gs_edge_score(1, None, None, 0, 0, None, None, 1, 4, None, 0, 0.0, None, None) == 1
    assert b"terms" in lib.gs_last_error()


# ---------------------------------------------------------------------- on the GPU
def world(nodes=3000, most=40, seed=0):
    rng = np.random.default_rng(seed)
    indptr, indices = random_csc(rng, nodes, nodes, most, hub_deg=4000)
    m = gs.Matrix(gs.Graph(nodes, nodes))
    m._graph._CAPI_LoadCSC(torch.from_numpy(indptr).to(DEV), torch.from_numpy(indices).to(DEV))
    m.edata["w"] = torch.from_numpy(rng.random(indices.size).astype(np.float32) + 0.01).to(DEV)
    return m


@pytest.mark.gpu
@pytest.mark.parametrize("width", [1, 2, 3, 4, 6, 7, 8, 12, 13, 16, 17, 20, 31, 32, 33, 44, 48, 60, 63, 64])
@pytest.mark.parametrize("fmt", [gs._COO, gs._CSC, gs._CSR])
def test_kernel_gives_the_bits_of_the_operators(width, fmt, monkeypatch):
    """Also rows that are not whole 16 bytes, or begin between them; infinities and NaN; an
    edge list in an order of its own, whose compressed forms map the edges back."""
    g = torch.Generator(device=DEV).manual_seed(width)
    n, e = 700, 5001
    row, col = (torch.randint(0, n, (e,), generator=g, device=DEV) for _ in range(2))
    row[0] = col[0] = n - 1
    graph = gs.Graph(n, n)
    graph._CAPI_LoadCOO(row, col, False, False)
    store = torch.randn((4, n * width + 1), generator=g, device=DEV)
    shifted = store[:, 1:].reshape(4, n, width).unbind(0)
    aligned = [t.clone() for t in shifted]
    w, s = torch.rand(e, generator=g, device=DEV), torch.rand(n, generator=g, device=DEV)
    weights = torch.softmax(torch.randn(4, generator=g, device=DEV), 0)
    special = [t.clone() for t in aligned]
    special[0][3, 0], special[1][5, width - 1], special[2][7, 0] = float("inf"), float("-inf"), float("nan")
    P, Q, V = fused_op.PRODUCTS, fused_op.QUOTIENT, fused_op.VALUE
    for a, b, c, d in (aligned, shifted, special):
        for kinds, lhs, rhs, to in (
                ([P], [a], [b], [0, 2]), ([P, Q], [a, w], [b, s], [0, 2, 1, 0]),
                ([P, V, P], [a, w, c], [b, None, d], [2, 0, 1, 1, 0, 2]),
                ([V, P, Q, P], [w, c, w, a], [None, a, s, d], [1, 1, 0, 2, 1, 2, 2, 0])):
            for k in ({len(kinds)} if len(kinds) > 1 else {0, 1}):
                x = weights[:k].clone() if k else None
                for relu, shift in ((False, None), (True, 1e-9)):
                    args = (graph, kinds, lhs, rhs, to, x, relu, shift, fmt)
                    native = gs._library.native.edge_score(*args[:7], shift or 0.0, fmt)
                    assert (native is None) == (width > 63)
                    got = fused_op._edge_score(*args)
                    with monkeypatch.context() as patch:            # the operators
                        patch.setattr(gs._library, "native", NoKernel)
                        want = fused_op._edge_score(*args)
                    assert torch.equal(torch.nan_to_num(got, nan=7e7), torch.nan_to_num(want, nan=7e7))


class NoKernel:
    @staticmethod
    def edge_score(*args):
        return None


@pytest.mark.gpu
def test_scores_against_64_bits():
    """No further off than the operators: n products and additions in 32 bits, each rounded once."""
    m, seeds = world(), torch.arange(200, device=DEV)
    g = torch.Generator(device=DEV).manual_seed(1)
    feats, W = torch.randn((3000, 24), generator=g, device=DEV), torch.randn((24, 16), generator=g, device=DEV)
    sub = m[:, seeds]
    row, col = sub.coo[:2]
    u, v = feats @ W, feats[seeds] @ W
    got = fused_op._edge_score(sub._graph, [fused_op.PRODUCTS], [u], [v], [0, 2], None, False, None, gs._COO)
    terms = u.double()[row] * v.double()[col]
    # 16 products and log2(16) + 1 additions deep
    bound = 6 * 2.0 ** -24 * terms.abs().sum(1)
    assert ((got.double() - terms.sum(1)).abs() <= bound).all()


@pytest.mark.gpu
@pytest.mark.parametrize("func", [scores, two_layers, plain_sum, in_place, products_wanted, other_sums,
                                  rows_escape])
@pytest.mark.parametrize("kind", ["float32", "float64", "gradients", "autocast", "more rows", "wide"])
def test_compiled_equals_eager(func, kind):
    m, seeds = world(), torch.arange(0, 600, 3, device=DEV)
    g = torch.Generator(device=DEV).manual_seed(2)
    n, d, h = 3000 + 50 * (kind == "more rows"), 20, 70 if kind == "wide" else 12
    feats, W = torch.randn((n, d), generator=g, device=DEV), torch.randn((d, h), generator=g, device=DEV)
    weights = torch.softmax(torch.randn(4, generator=g, device=DEV), 0)
    if kind == "float64":
        feats, W = feats.double(), W.double()
        if func in (scores, two_layers):
            return                           # quotients are of the weights' type
    if kind == "gradients":
        weights.requires_grad_()
    args = (m, seeds, feats, W, weights)
    c = gs.jit.compile(func=func, args=args)
    with torch.autocast("cuda", enabled=kind == "autocast", dtype=torch.bfloat16):
        if kind == "autocast" and func is not rows_escape:
            for f in (func, c):              # products in bfloat16 are no operand of an SDDMM
                with pytest.raises(RuntimeError, match="BFloat16"):
                    f(*args)
            return
        want, got = func(*args), c(*args)
    want, got = (x if isinstance(x, tuple) else (x,) for x in (want, got))
    for a, b in zip(want, got):
        assert a.dtype == b.dtype and a.requires_grad == b.requires_grad and torch.equal(a, b)
    if kind == "gradients" and want[0].requires_grad:
        (dw,), (dg,) = (torch.autograd.grad(x[0].sum(), weights) for x in (want, got))
        assert torch.equal(dw, dg)


@pytest.mark.gpu
def test_features_may_change_before_the_gradient_of_their_products():
    """Rows are gathered into an array of their own, which the product keeps."""
    m, seeds = world(), torch.arange(0, 600, 3, device=DEV)
    feats, W = torch.randn((3000, 20), device=DEV), torch.randn((20, 12), device=DEV, requires_grad=True)
    args = (m, seeds, feats, W, torch.rand(4, device=DEV))
    c = gs.jit.compile(func=products_of_rows, args=args)
    out, want = c(*args), 2.0 * feats.double().sum(0)
    feats.mul_(3.0)
    (out[0].sum() + out[1].sum()).backward()
    # sums of 3000 terms in another order
    assert torch.allclose(W.grad, want.float()[:, None].expand(20, 12), rtol=1e-4, atol=1e-3)


# ------------------------------------------------- encoded slices that are not written
def layer(A, seeds, ptr, power=2, also=None, picks="listed"):
    sub = A[:, seeds::ptr]
    sub.edata["p"] = sub.edata["w"] ** power
    prob = sub.sum("p", axis=1)
    rows, rows_ptr = sub.all_rows()
    if picks == "own":
        part = sub[prob.argsort()[:4]::torch.tensor([0, 2, 4], device=prob.device), :]
        return part.edata["w"], rows
    part, index = sub.collective_sampling(3, prob, rows_ptr, False)
    out = part.div("w", prob[index], axis=1).edata["w"], rows[index]
    return out + ((sub.edata["w"],) if also == "edges" else (sub.sum("w", axis=1),) if also == "sum" else ())


@pytest.mark.parametrize("options,kernel", [
    ({}, True), (dict(power=3), False), (dict(also="edges"), False), (dict(also="sum"), False),
    (dict(picks="own"), False)])
def test_what_is_summed_in_place(options, kernel):
    bm = gs.BatchMatrix()
    m = gs.Matrix(gs.Graph(10, 10))
    m.edata["w"] = torch.rand(7)
    bm.load_from_matrix(m, True)

    def sampler(A, seeds, ptr):
        return layer(A, seeds, ptr, **options)

    t = ran(gs.jit.compile(func=sampler, args=(bm, torch.arange(6), torch.tensor([0, 3, 6]))))
    assert t.count(fused_op._encoded_square_sums) == kernel and ("_CAPI_BatchColSlicing" in t) != kernel
    assert t.count(fused_op._encoded_row_slice) == kernel and ("_CAPI_BatchRowSlicing" in t) != kernel


def written_between(A, seeds, ptr, w, scale):
    """w changes after the slice has been made and before its rows are picked."""
    A.edata["w"] = w
    sub = A[:, seeds::ptr]
    sub.edata["p"] = sub.edata["w"] ** 2
    prob = sub.sum("p", axis=1)
    _, rows_ptr = sub.all_rows()
    changed = w.mul_(scale)
    part, _ = sub.collective_sampling(3, prob, rows_ptr, False)
    return part.edata["w"], changed


def written_after(A, seeds, ptr, w, scale):
    A.edata["w"] = w
    return layer(A, seeds, ptr) + (w.mul_(scale),)


def order_of(compiled, *targets):
    return [n.target for n in compiled._run.__self__.graph.nodes if n.target in targets]


@pytest.mark.parametrize("func,kernel", [(written_between, False), (written_after, True)])
def test_slice_that_is_written_to_before_its_rows_are_read(func, kernel):
    bm = gs.BatchMatrix()
    bm.load_from_matrix(gs.Matrix(gs.Graph(10, 10)), True)
    c = gs.jit.compile(func=func, args=(bm, torch.arange(6), torch.tensor([0, 3, 6]), torch.rand(7),
                                        torch.rand(7)))
    assert order_of(c, fused_op._encoded_row_slice, "_CAPI_BatchRowSlicing", "mul_") == (
        [fused_op._encoded_row_slice, "mul_"] if kernel else ["mul_", "_CAPI_BatchRowSlicing"])


# ------------------------------------------------------------ columns normalised
def normalised(A, seeds, divisor):
    sub = A[:, seeds].div("w", divisor, axis=1)
    return sub.div("w", sub.sum("w", axis=0), axis=0).edata["w"]


def by_columns_only(A, seeds, divisor):
    sub = A[:, seeds]
    return sub.div("w", sub.sum("w", axis=0), axis=0).edata["w"], sub.edata["w"]


def quotient_kept(A, seeds, divisor):
    q = A[:, seeds].div("w", divisor, axis=1)
    return q.div("w", q.sum("w", axis=0), axis=0).edata["w"], q.edata["w"]


def sums_kept(A, seeds, divisor):
    q = A[:, seeds].div("w", divisor, axis=1)
    s = q.sum("w", axis=0)
    return q.div("w", s, axis=0).edata["w"], s


def by_rows(A, seeds, divisor):
    q = A[:, seeds].div("w", divisor, axis=1)
    return q.div("w", q.sum("w", axis=1), axis=1).edata["w"]


def divisor_written(A, seeds, divisor):
    q = A[:, seeds].div("w", divisor, axis=1)
    changed = divisor.mul_(torch.arange(1.0, 1.0 + divisor.numel(), device=divisor.device))
    return q.div("w", q.sum("w", axis=0), axis=0).edata["w"], changed


def divisor_written_after(A, seeds, divisor):
    q = A[:, seeds].div("w", divisor, axis=1)
    return q.div("w", q.sum("w", axis=0), axis=0).edata["w"], divisor.mul_(2.0)


@torch.fx.wrap
def scaled_by_ten(x):
    return x.mul_(10.0)


def by_a_function(x):
    return scaled_by_ten(x)


def by_an_overload(x):
    return torch.ops.aten.mul_.Scalar(x, 10.0)


def by_a_packet(x):
    return torch.ops.aten.mul_(x, 10.0)


def by_an_option(x):
    return F.relu(x, True)


def by_an_output(x):
    return torch.add(x, 1.0, out=x)


def not_at_all(x):
    return torch.ops.aten.mul(x, 10.0) + F.relu(x) - torch.sum(x, dim=0) * math.sqrt(2.0)


@pytest.mark.parametrize("write", [by_a_function, by_an_overload, by_a_packet, by_an_option, by_an_output,
                                   not_at_all])
def test_writes_however_they_are_spelt(write):
    def sampler(A, seeds, divisor):
        q = A[:, seeds].div("w", divisor, axis=1)
        changed = write(divisor)
        return q.div("w", q.sum("w", axis=0), axis=0).edata["w"], changed

    m = gs.Matrix(gs.Graph(10, 10))
    m.edata["w"] = torch.rand(7)
    t = ran(gs.jit.compile(func=sampler, args=(m, torch.arange(3), torch.rand(10))))
    assert (fused_op._normalised in t) == (write is not_at_all)


@pytest.mark.parametrize("func,kernels,divisions", [
    (divisor_written, 0, 2), (divisor_written_after, 1, 0), (normalised, 1, 0), (by_columns_only, 1, 0), (quotient_kept, 1, 1), (sums_kept, 0, 2), (by_rows, 0, 2)])
def test_what_is_normalised_in_one(func, kernels, divisions):
    m = gs.Matrix(gs.Graph(10, 10))
    m.edata["w"] = torch.rand(7)
    t = ran(gs.jit.compile(func=func, args=(m, torch.arange(3), torch.rand(10))))
    assert t.count(fused_op._normalised) == kernels and t.count("_CAPI_SDDMM") == divisions
    assert t.count("_CAPI_SpMM") == (kernels == 0)


@pytest.mark.gpu
@pytest.mark.parametrize("func", [normalised, by_columns_only, quotient_kept, sums_kept, by_rows])
@pytest.mark.parametrize("kind", ["float32", "float64", "gradients", "edge list"])
def test_normalised_columns_equal_eager(func, kind):
    m, seeds = world(), torch.arange(0, 900, 3, device=DEV)
    if kind == "edge list":
        row, col = m.coo[:2]
        order = torch.randperm(row.numel(), device=DEV)
        w = m.edata["w"]
        m = gs.Matrix()
        m.load_graph("COO", [row[order], col[order]])
        m.edata["w"] = w[order]
    divisor = torch.rand(m.num_rows(), device=DEV) + 0.5
    if kind == "gradients":
        m.edata["w"].requires_grad_()
        divisor.requires_grad_()
    if kind == "float64":
        m.edata["w"], divisor = m.edata["w"].double(), divisor.double()
        with pytest.raises(RuntimeError):
            func(m, seeds, divisor)
        c = gs.jit.compile(func=func, args=(m, seeds, divisor))
        with pytest.raises(RuntimeError):
            c(m, seeds, divisor)
        return
    want = func(m, seeds, divisor)
    got = gs.jit.compile(func=func, args=(m, seeds, divisor))(m, seeds, divisor)
    for a, b in zip(*((x if isinstance(x, tuple) else (x,)) for x in (want, got))):
        # the eager sums are of 32 bits, up to 4000 terms of one sign in any order
        assert a.requires_grad == b.requires_grad
        torch.testing.assert_close(a, b, rtol=1e-5, atol=0)


@pytest.mark.gpu
@pytest.mark.parametrize("func", [normalised, by_columns_only])
@pytest.mark.parametrize("length", [0, 1, 2000])
def test_edge_data_shorter_than_the_edges(func, length):
    """Edges past its end have the value 0, as the gather gives it."""
    m, seeds = world(), torch.arange(0, 900, 3, device=DEV)
    divisor = torch.rand(m.num_rows(), device=DEV) + 0.5
    m.edata["w"] = m.edata["w"][:length].clone()
    compiled = gs.jit.compile(func=func, args=(m, seeds, divisor))
    if length == 0:
        for f in (func, compiled):
            with pytest.raises(RuntimeError, match="gather_rows"):
                f(m, seeds, divisor)
        return
    want, got = func(m, seeds, divisor), compiled(m, seeds, divisor)
    for a, b in zip(*((x if isinstance(x, tuple) else (x,)) for x in (want, got))):
        torch.testing.assert_close(a, b, rtol=1e-5, atol=0, equal_nan=True)


@pytest.mark.gpu
@pytest.mark.parametrize("degrees", [[1], [2048], [2049], [2047, 1, 2048, 0, 5], [0] * 3000 + [10] + [0] * 2500 + [7],
                                     [3] * 5000, [1] * 2048 + [4100] + [0, 1] * 40, [100_000, 1]])
@pytest.mark.parametrize("select", [False, True])
@pytest.mark.parametrize("divide", [False, True])
def test_normalised_columns_against_64_bits(degrees, select, divide):
    """Tiles of one column and of thousands, columns of no edge between, over borders of tiles."""
    g = torch.Generator(device=DEV).manual_seed(len(degrees))
    deg = torch.tensor(degrees, device=DEV)
    indptr = torch.zeros(deg.numel() + 1, dtype=torch.int64, device=DEV)
    torch.cumsum(deg, 0, out=indptr[1:])
    n = int(indptr[-1])
    rows = torch.randint(0, 500, (n,), generator=g, device=DEV)
    graph = gs.Graph(500, deg.numel())
    graph._CAPI_LoadCSC(indptr, rows)
    values = torch.randn(n + 100, generator=g, device=DEV).abs()[: n + 100 * select].contiguous() + 0.01
    index = torch.randint(0, n + 100, (n,), generator=g, device=DEV) if select else None
    by = torch.rand(500, generator=g, device=DEV) + 0.1 if divide else None
    got = fused_op._normalised(graph, values, index, by, (gs._COO, gs._CSC, gs._COO))
    q = values[index] if select else values
    q = (q / by[rows] if divide else q).double()
    column = torch.repeat_interleave(torch.arange(deg.numel(), device=DEV), deg)
    sums = torch.zeros(deg.numel(), dtype=torch.float64, device=DEV).index_add_(0, column, q)
    # the sum and the quotient are rounded once each
    torch.testing.assert_close(got.double(), q / sums[column], rtol=2.5 * 2.0 ** -24, atol=0)


@pytest.mark.gpu
@pytest.mark.parametrize("degrees", [[2_500_000, 65, 1, 0, 64, 2_000_000, 17], [40] * 110_000,
                                     [2048, 2047, 2, 63, 64, 65] * 1000 + [0, 1], [300, 0, 2, 2] * 14_500])
def test_normalised_columns_of_long_runs(degrees):
    """More edges than the short runs take on: runs of one column, of a few, and of hundreds."""
    test_normalised_columns_against_64_bits(degrees, False, False)


@pytest.mark.gpu
@pytest.mark.parametrize("degrees", [[1, 0, 0, 0] * 700, [0] * 999 + [300] + [0, 0, 3] * 100 + [700] + [0] * 5000 + [1],
                                     [1] + [0] * 1023 + [511], [1] + [0] * 1022 + [511], [64, 0, 0] * 40 + [65] + [0] * 9000 + [1],
                                     ([0] * 70_000 + [40]) * 30])
def test_normalised_columns_of_which_most_are_empty(degrees):
    """Runs around two columns an edge, columns longer than a row of 64 among them."""
    for select in (False, True):
        test_normalised_columns_against_64_bits(degrees, select, select)


@pytest.mark.gpu
def test_normalised_columns_of_few_edges_take_no_time_by_the_column():
    """400 edges in two million columns: 0.05 ms, and 17 where a wavefront goes through the
    columns between them."""
    n = 2_000_000
    indptr = torch.arange(n + 1, device=DEV) // 5000
    graph = gs.Graph(500, n)
    graph._CAPI_LoadCSC(indptr, torch.zeros(400, dtype=torch.int64, device=DEV))
    values = torch.ones(400, device=DEV)
    call = lambda: fused_op._normalised(graph, values, None, None, (gs._COO, gs._CSC, gs._COO))
    assert torch.equal(call(), values)
    took = []
    for _ in range(5):  # (the host may pause inside one)
        start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        start.record()
        call()
        end.record()
        end.synchronize()
        took.append(start.elapsed_time(end))
    assert min(took) < 3.0
