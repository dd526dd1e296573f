"""Encoded column slices of a super-batch (rows numbered anew per batch): the flag-byte path
against torch's sorted unique with inverse, at ranges and runs where it can go wrong."""
import numpy as np
import pytest
import torch

import gsampler_amd as gs
from tests.conftest import random_csc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("rows,cols,max_deg,hub,batches,narrow", [
    (1, 5, 3, 0, 3, False),             # one row: a range of three keys
    (63, 40, 6, 0, 2, False),           # batch border inside a rank word
    (4096, 900, 9, 0, 7, False),        # batches of exactly one group, many short columns a run
    (5001, 700, 40, 30000, 4, False),   # columns longer than a run of edges
    (5001, 4000, 800, 0, 5, True),      # above 2^20 edges: the int32 copy of the ids
    (5001, 12000, 1500, 0, 3, True),    # above 2^22 edges in the slice: four rounds a wavefront
])
def test_rows_numbered_anew(rng, rows, cols, max_deg, hub, batches, narrow):
    indptr, indices = random_csc(rng, cols, rows, max_deg, hub_deg=hub)
    assert (indices.size >= 1 << 20) == narrow
    g = gs.Graph(rows, cols)
    d_indptr, d_indices = torch.from_numpy(indptr).to(DEV), torch.from_numpy(indices).to(DEV)
    g._CAPI_LoadCSC(d_indptr, d_indices)
    seeds = torch.from_numpy(rng.integers(-2, cols + 2, size=4 * batches + cols // 2)).to(DEV)
    cuts = np.sort(rng.integers(0, seeds.numel() + 1, size=batches - 1))
    ptr = torch.tensor([0, *cuts.tolist(), seeds.numel()], device=DEV)
    sub, index = g._CAPI_BatchColSlicing(seeds, ptr, True)
    plain, plain_index = g._CAPI_BatchColSlicing(seeds, ptr, False)
    col = plain._CAPI_GetCOOCols()
    batch = torch.searchsorted(ptr[1:], col, right=True)
    keys, inverse = torch.unique(plain._CAPI_GetCOORows() + batch * rows, return_inverse=True)
    ids, row_ptr = sub._CAPI_BatchGetRows()
    assert torch.equal(index, plain_index) and torch.equal(sub._CAPI_GetCOOCols(), col)
    assert torch.equal(sub._CAPI_GetCSCIndptr(), plain._CAPI_GetCSCIndptr())
    assert torch.equal(sub._CAPI_GetCSCIndices(), inverse) and torch.equal(ids, keys % rows)
    assert torch.equal(row_ptr, torch.searchsorted(keys, torch.arange(batches + 1, device=DEV) * rows))


@pytest.mark.parametrize("rows,cols,max_deg,hub,batches,form", [
    (1, 5, 3, 0, 3, "csc"),
    (63, 40, 6, 0, 2, "csc"),           # batch border inside a rank word
    (4096, 900, 9, 0, 7, "coo"),        # an edge list in its own order: edges mapped back
    (5001, 700, 40, 30000, 4, "csc"),
    (5001, 4000, 800, 0, 5, "csc"),     # sums by ranges of rows, many columns a run
    (70_000, 200, 20_000, 0, 3, "csc"), # long columns, the int32 copy of the ids
    (5001, 12000, 1500, 0, 3, "csc"),
    (200_000, 30, 8, 0, 60, "csc"),     # too few edges for so many keys: the slice is written
])
def test_sums_of_an_encoded_slice_that_is_not_written(rng, rows, cols, max_deg, hub, batches, form):
    """Rows, picked rows' edges and edge index are those of the written slice, its sums the same
    to the rounding of their additions; rows whose values are all zero (of either sign) occur."""
    from gsampler_amd.ops import fused_op
    indptr, indices = random_csc(rng, cols, rows, max_deg, hub_deg=hub)
    g = gs.Graph(rows, cols)
    if form == "csc":
        g._CAPI_LoadCSC(torch.from_numpy(indptr).to(DEV), torch.from_numpy(indices).to(DEV))
    else:
        order = rng.permutation(indices.size)
        col = np.repeat(np.arange(cols), np.diff(indptr))
        g._CAPI_LoadCOO(torch.from_numpy(indices[order]).to(DEV), torch.from_numpy(col[order]).to(DEV),
                        False, False)
    w = rng.standard_normal(indices.size).astype(np.float32)
    w[rng.random(w.size) < 0.3] = 0.0
    w[rng.random(w.size) < 0.1] = -0.0
    w = torch.from_numpy(w).to(DEV)
    seeds = torch.from_numpy(rng.integers(-2, cols + 2, size=4 * batches + cols // 2)).to(DEV)
    cuts = np.sort(rng.integers(0, seeds.numel() + 1, size=batches - 1))
    ptr = torch.tensor([0, *cuts.tolist(), seeds.numel()], device=DEV)
    part, ids, ids_ptr, sums = fused_op._encoded_square_sums(g, seeds, ptr, w, gs._COO)
    assert len(part) == (2 if rows == 200_000 else 4)
    sub, index = g._CAPI_BatchColSlicing(seeds, ptr, True)
    want_ids, want_ptr = sub._CAPI_BatchGetRows()
    assert torch.equal(ids, want_ids) and torch.equal(ids_ptr, want_ptr)
    exact = torch.zeros(ids.numel(), dtype=torch.float64, device=DEV)
    exact.index_add_(0, sub._CAPI_GetCOORows(), w[index].double() ** 2)
    # squares rounded once, sums of up to 10^5 of them in 32 bits where no ranges are used
    torch.testing.assert_close(sums.double(), exact, rtol=1e-5, atol=0)
    picks, picks_ptr = torch.ops.gs_ops._CAPI_BatchListSampling(50, False, ids_ptr)
    got, got_index = fused_op._encoded_row_slice(part, picks, picks_ptr)
    want, want_index = sub._CAPI_BatchRowSlicing(picks, picks_ptr)
    assert torch.equal(got_index, index[want_index])
    for name in ("GetCSCIndptr", "GetCSCIndices", "GetCOORows", "GetCOOCols", "GetEdgeBptr", "GetColBptr",
                 "GetRowBptr", "GetNumRows", "GetNumCols", "GetNumEdges"):
        a, b = getattr(got, "_CAPI_" + name)(), getattr(want, "_CAPI_" + name)()
        assert torch.equal(a, b) if isinstance(a, torch.Tensor) else a == b
    (ga, gb), (wa, wb) = got._CAPI_BatchGetRows(), want._CAPI_BatchGetRows()
    assert torch.equal(ga, wa) and torch.equal(gb, wb)
    seeds_of = ids[picks]
    for a, b in zip(got._CAPI_BatchGraphRelabel(seeds, seeds_of), want._CAPI_BatchGraphRelabel(seeds, seeds_of)):
        assert (a is None and b is None) or torch.equal(a, b)


def test_values_that_are_no_plain_numbers_keep_their_row():
    """NaN, infinities and values whose square is below the smallest number."""
    from gsampler_amd.ops import fused_op
    g = gs.Graph(70, 3)
    g._CAPI_LoadCSC(torch.tensor([0, 4, 6, 7], device=DEV), torch.tensor([3, 9, 3, 64, 5, 9, 69], device=DEV))
    w = torch.tensor([float("nan"), float("inf"), 1.0, -float("inf"), 1e-30, -1e-38, -float("nan")], device=DEV)
    seeds, ptr = torch.tensor([0, 1, 2], device=DEV), torch.tensor([0, 2, 2, 3], device=DEV)
    _, ids, ids_ptr, sums = fused_op._encoded_square_sums(g, seeds, ptr, w, gs._COO)
    assert ids.tolist() == [3, 5, 9, 64, 69] and ids_ptr.tolist() == [0, 4, 4, 5]
    assert sums.isnan().tolist() == [True, False, False, False, True] and sums[1:4].tolist() == [0, float("inf")] + [float("inf")]
