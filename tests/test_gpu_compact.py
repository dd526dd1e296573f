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
