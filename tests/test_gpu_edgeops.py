"""Edge-wise operators on the GPU: C ABI vs the oracle (fp32 within 1e-5
relative; copies and fp64 products exactly), and the gs.ops / Matrix wrappers
(broadcast tables, format selection, e_ids of converted formats)."""
import numpy as np
import pytest
import torch

import gsampler_amd as gs
from gsampler_amd import capi
from oracle import binding as orc
from tests.conftest import random_csc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
RTOL = 1e-5


def T(a):
    return None if a is None else torch.as_tensor(a, device=DEV)


def close(got, want, rtol=RTOL):
    got = got.cpu().numpy()
    assert got.shape == want.shape
    assert np.allclose(got, want, rtol=rtol, atol=1e-6), np.abs(got - want).max()


@pytest.fixture(scope="module")
def g():
    rng = np.random.default_rng(7)
    indptr, indices = random_csc(rng, 700, 500, 60, hub_deg=20000)
    col = np.repeat(np.arange(700), np.diff(indptr))
    return rng, indptr, indices, col


def views(indptr, indices, col):
    return {"coo": (("coo", indices, col), ("coo", T(indices), T(col))),
            "csc": (("csc", indptr, indices), ("csc", T(indptr), T(indices)))}


@pytest.mark.parametrize("fmt", ["coo", "csc"])
def test_sddmm_parity(g, fmt):
    rng, indptr, indices, col = g
    ov, gv = views(indptr, indices, col)[fmt]
    E = indices.size
    u = rng.random(500, dtype=np.float32) + 0.5
    v = rng.random(700, dtype=np.float32) + 0.5
    e = rng.random(E, dtype=np.float32) + 0.1
    for op in ("add", "sub", "mul", "div"):
        close(capi.sddmm(gv, op, T(u), T(v), 0, 2), orc.sddmm(ov, op, u, v, 0, 2))
    close(capi.sddmm(gv, "div", T(e), T(v), 1, 2), orc.sddmm(ov, "div", e, v, 1, 2))
    close(capi.sddmm(gv, "mul", T(e), T(u), 1, 0), orc.sddmm(ov, "mul", e, u, 1, 0))
    assert np.array_equal(capi.sddmm(gv, "copy_lhs", T(u), None, 0, 2).cpu().numpy(),
                          orc.sddmm(ov, "copy_lhs", u, None, 0, 2))
    U, V = rng.random((500, 6), dtype=np.float32), rng.random((700, 6), dtype=np.float32)
    close(capi.sddmm(gv, "dot", T(U), T(V), 0, 2), orc.sddmm(ov, "dot", U, V, 0, 2))
    close(capi.sddmm(gv, "mul", T(U), T(V), 0, 2), orc.sddmm(ov, "mul", U, V, 0, 2))
    perm = rng.permutation(E)
    e64 = rng.random(E)
    close(capi.sddmm(gv, "mul", T(e64), T(v.astype(np.float64)), 1, 2, edge_map=T(perm)),
          orc.sddmm(ov, "mul", e64, v.astype(np.float64), 1, 2, edge_map=perm), 1e-12)


@pytest.mark.parametrize("fmt", ["coo", "csc"])
def test_spmm_and_fusions_parity(g, fmt):
    rng, indptr, indices, col = g
    ov, gv = views(indptr, indices, col)[fmt]
    E = indices.size
    u = rng.random(500, dtype=np.float32) + 0.5
    e = rng.random(E, dtype=np.float32) + 0.1
    close(capi.spmm(gv, "copy_rhs", "sum", None, T(e), 0, 700),
          orc.spmm(ov, "copy_rhs", "sum", None, e, 0, 700))
    close(capi.spmm(gv, "mul", "sum", T(u), T(e), 0, 700),
          orc.spmm(ov, "mul", "sum", u, e, 0, 700))
    close(capi.e_square_sum(gv, T(e), 0, 700), orc.e_square_sum(ov, e, 0, 700))
    close(capi.e_div_u_sum(gv, T(u), T(e), 0, 700), orc.e_div_u_sum(ov, u, e, 0, 700))
    if fmt == "coo":
        close(capi.spmm(gv, "copy_rhs", "sum", None, T(e), 2, 500),
              orc.spmm(ov, "copy_rhs", "sum", None, e, 2, 500))
        close(capi.e_square_sum(gv, T(e), 2, 500), orc.e_square_sum(ov, e, 2, 500))
    F = rng.random((E, 5), dtype=np.float32)
    close(capi.spmm(gv, "copy_rhs", "sum", None, T(F), 0, 700),
          orc.spmm(ov, "copy_rhs", "sum", None, F, 0, 700))
    s = e - 0.4
    for red in ("max", "min"):
        got = capi.spmm(gv, "copy_rhs", red, None, T(s), 0, 700, want_arg=True)
        want = orc.spmm(ov, "copy_rhs", red, None, s, 0, 700, want_arg=True)
        assert np.array_equal(got[0].cpu().numpy(), want[0])
        hit = want[0] != 0
        assert np.array_equal(s[got[2].cpu().numpy()[hit]], want[0][hit])
    o1, o2 = capi.fused_u_op_v(gv, "mul", T(u), T(e[:700]), T(u * 2), T(e[:700] + 1))
    w1, w2 = orc.fused_u_op_v(ov, "mul", u, e[:700], u * 2, e[:700] + 1)
    close(o1, w1); close(o2, w2)


@pytest.mark.parametrize("shape", ["hubs", "row_ranges", "tiny_segments"])
def test_scalar_sums_on_skewed_matrices(shape):
    """The load-balanced sum kernels: a few segments that hold most of the edges
    (and rows that most edges point to), and thousands of segments with zero or
    one edge.  Sums of up to 10^6 fp32 terms are compared with a float64 sum at
    1e-5 relative (the order of additions is not fixed)."""
    rng = np.random.default_rng(31)
    if shape == "hubs":
        deg = np.full(40, 50)
        deg[[3, 17]] = [1200000, 400000]     # > 2^20 edges: per-die accumulators
        R = 3000
        w = 1.0 / np.arange(1, R + 1) ** 1.2
        indices = rng.choice(R, size=int(deg.sum()), p=w / w.sum())
    elif shape == "row_ranges":
        # several ranges of 8192 rows: one holds a hub row (many slices of one
        # range), one is empty, the last one is partial
        deg = np.full(300, 5000)
        R = 30000
        indices = rng.integers(0, R, size=int(deg.sum()))
        indices[(indices >= 8192) & (indices < 16384)] += 8192
        indices[rng.random(indices.size) < 0.4] = 20001
    else:
        deg = rng.integers(0, 2, size=9000)
        R = 500
        indices = rng.integers(0, R, size=int(deg.sum()))
    C = deg.size
    indptr = np.concatenate([[0], np.cumsum(deg)])
    col = np.repeat(np.arange(C), deg)
    e = rng.random(indices.size, dtype=np.float32) + 0.1
    u = rng.random(R, dtype=np.float32) + 0.5
    e64 = e.astype(np.float64)
    onto_cols = np.bincount(col, weights=e64, minlength=C)
    onto_rows = np.bincount(indices, weights=e64, minlength=R)
    sq_rows = np.bincount(indices, weights=e64 * e64, minlength=R)
    div_cols = np.bincount(col, weights=e64 / u[indices], minlength=C)
    coo, csc = ("coo", T(indices), T(col)), ("csc", T(indptr), T(indices))
    for view in (coo, csc):
        close(capi.spmm(view, "copy_rhs", "sum", None, T(e), 0, C), onto_cols.astype(np.float32))
        close(capi.e_div_u_sum(view, T(u), T(e), 0, C), div_cols.astype(np.float32))
    close(capi.spmm(coo, "copy_rhs", "sum", None, T(e), 2, R), onto_rows.astype(np.float32))
    close(capi.e_square_sum(coo, T(e), 2, R), sq_rows.astype(np.float32))
    # and the oracle agrees with the float64 sums as well
    assert np.allclose(orc.spmm(("csc", indptr, indices), "copy_rhs", "sum", None, e, 0, C),
                       onto_cols, rtol=1e-5)


@pytest.mark.parametrize("nnz,R,targets", [
    (1 << 20, 1, "any"),                      # one row, one range, 32 counters for it
    ((1 << 20) + 1, 8192, "any"),             # one full range; a tile with one edge
    ((1 << 20) + 8191, 8193, "sorted"),       # a range with one row; one target per wavefront
    (5_000_000, 32 * 8192, "hub"),            # most counters in use, many units of one range
    (5_000_000, 32 * 8192 + 1, "any"),        # one range more: half the counters per range
    (12_000_001, 300_000, "last"),            # every edge in the last range: the others have no unit
    (33_600_000, 1024 * 8192, "any"),         # as many ranges as there are, a few edges a run
])
def test_sums_by_row_range_at_their_borders(nnz, R, targets):
    """Against float64 sums.  A unit of at most 40 960 edges is summed in double and rounded
    once, a row's units are added in double and rounded once: well inside 2e-6, the bound of
    units added in float (153 of them for the hub, in eight shares of 20)."""
    rng = np.random.default_rng(nnz + R)
    ids = rng.integers(0, R, size=nnz)
    if targets == "sorted":
        ids.sort()
    elif targets == "hub":
        ids[rng.random(nnz) < 0.9] = 77_777
    elif targets == "last":
        ids = np.maximum(ids, R // 8192 * 8192)
    e = rng.random(nnz, dtype=np.float32) + np.float32(0.1)
    want = np.bincount(ids, weights=e.astype(np.float64), minlength=R)  # (on the host: no atomics)
    d_ids = T(ids)
    got = capi.spmm(("coo", d_ids, d_ids), "copy_rhs", "sum", None, T(e), 2, R)
    assert np.allclose(got.cpu().numpy().astype(np.float64), want, rtol=2e-6, atol=0)


@pytest.mark.parametrize("E", [1, 255, 1023, 1024, 1025, 4096, 70_001])
def test_one_value_an_edge_at_the_borders_of_a_tile(E):
    """Scalar operators on an edge list, through every target and an edge map; the same kernel
    without it reads the edge's own values."""
    rng = np.random.default_rng(E)
    row, col = rng.integers(0, 50, size=E), rng.integers(0, 70, size=E)
    u, v, e = (rng.random(n, dtype=np.float32) + 0.5 for n in (50, 70, E))
    of = {0: u, 1: e, 2: v}
    for perm in (None, rng.permutation(E)):
        for lt, rt in ((1, 0), (1, 2), (0, 2), (2, 0), (2, 1), (1, 1)):
            got = capi.sddmm(("coo", T(row), T(col)), "div", T(of[lt]), T(of[rt]), lt, rt,
                             edge_map=T(perm))
            want = orc.sddmm(("coo", row, col), "div", of[lt], of[rt], lt, rt, edge_map=perm)
            assert np.array_equal(got.cpu().numpy(), want)
        got = capi.sddmm(("coo", T(row), T(col)), "copy_rhs", None, T(v), 1, 2, edge_map=T(perm))
        assert np.array_equal(got.cpu().numpy(),
                              orc.sddmm(("coo", row, col), "copy_rhs", None, v, 1, 2, edge_map=perm))


@pytest.mark.parametrize("deg", [[2048], [2048, 2048], [1, 2047, 2049, 4095], [5000, 0, 0, 3, 9000],
                                 [70_000_000, 5_000, 0, 3_000_000]])
def test_column_sums_of_tiles_inside_one_column(deg):
    """One, and from 67 M edges four, rounds of 2048 edges a tile, most tiles inside one column."""
    rng = np.random.default_rng(len(deg))
    indptr = np.concatenate([[0], np.cumsum(deg)])
    e = rng.random(indptr[-1], dtype=np.float32) + np.float32(0.1)
    ids = torch.zeros(indptr[-1], dtype=torch.int64, device=DEV)
    want = np.array([e[a:b].astype(np.float64).sum() for a, b in zip(indptr, indptr[1:])])
    got = capi.spmm(("csc", T(indptr), ids), "copy_rhs", "sum", None, T(e), 0, len(deg))
    # a tile: 8 + 4 + 6 + 4 additions; up to 8 545 tiles of a column are added in any order,
    # whose roundings of 2^-24 are independent: sqrt(8545) of them at most half an ulp each
    assert np.allclose(got.cpu().numpy(), want, rtol=1e-5, atol=0)


def test_matrix_sum_div_and_ops_wrappers(g):
    rng, indptr, indices, col = g
    m = gs.Matrix()
    m.load_graph("CSC", [T(indptr), T(indices)])
    R = m.num_rows()
    E = indices.size
    w = rng.random(E, dtype=np.float32) + 0.1
    m.edata["w"] = T(w)
    col_sum = np.zeros(700); np.add.at(col_sum, col, w.astype(np.float64))
    row_sum = np.zeros(R); np.add.at(row_sum, indices, w.astype(np.float64))
    close(m.sum("w", 0), col_sum.astype(np.float32))
    close(m.sum("w", 1), row_sum.astype(np.float32))       # runs on a CSR built on demand
    d = rng.random(700, dtype=np.float32) + 0.5
    close(m.div("w", T(d), 0).edata["w"], w / d[col])       # div divides
    dr = rng.random(R, dtype=np.float32) + 0.5
    close(m.div("w", T(dr), 1).edata["w"], w / dr[indices])
    close(gs.ops.e_square_sum(m, "w", 1), (row_sum * 0 + np.bincount(
        indices, weights=w.astype(np.float64) ** 2, minlength=R)).astype(np.float32))
    close(gs.ops.e_square_sum(m, "w", 0), np.bincount(
        col, weights=w.astype(np.float64) ** 2, minlength=700).astype(np.float32))
    u = rng.random(R, dtype=np.float32) + 0.5
    close(gs.ops.e_div_u_sum(m, "w", T(u), 0), np.bincount(
        col, weights=(w / u[indices]).astype(np.float64), minlength=700).astype(np.float32))
    # broadcasting: [R, 3, 1] * [C, 1, 4] -> [E, 3, 4]
    A = rng.random((R, 3, 1), dtype=np.float32)
    B = rng.random((700, 1, 4), dtype=np.float32)
    close(gs.ops.u_mul_v(m, T(A), T(B)), A[indices] * B[col])
    close(gs.ops.u_add_v(m, T(A), T(B), gs._CSC), A[indices] + B[col])
    o1, o2 = gs.ops.fused_u_mul_v(m, T(u), T(d), T(u + 1), T(d + 1))
    close(o1, u[indices] * d[col]); close(o2, (u[indices] + 1) * (d[col] + 1))
    close(gs.ops.copy_e_sum(m, T(w)), col_sum.astype(np.float32))
