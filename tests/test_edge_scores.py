"""Edge scores of attention samplers: what the compiled graph runs in one kernel, what it leaves
to the operators it was written with, and that the two give the same bits -- the samples drawn by
the scores depend on every one of them."""
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


def ran(compiled):
    return [n.target for n in compiled._run.__self__.graph.nodes]


def cpu_args(nodes=10):
    m = gs.Matrix(gs.Graph(nodes, nodes))
    m.edata["w"] = torch.rand(7)
    return m, torch.arange(3), torch.rand(nodes, 4), torch.rand(4, 3), torch.rand(4)


@pytest.mark.parametrize("func,kernels,sddmm", [
    (scores, 1, 0), (two_layers, 2, 0), (plain_sum, 1, 0), (in_place, 0, 1), (products_wanted, 0, 1),
    (other_sums, 0, 3), (rows_escape, 0, 0)])
def test_what_becomes_an_edge_score(func, kernels, sddmm):
    c = gs.jit.compile(func=func, args=cpu_args())
    t = ran(c)
    assert t.count(fused_op._edge_score) == kernels and t.count("_CAPI_SDDMM") == sddmm
    in_place_free = func is not in_place and func is not rows_escape
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
