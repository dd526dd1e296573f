"""Frontier and labels of a row-sliced matrix (rows = positions in a short list
of ids) in one launch, against the oracle's unique + relabel over all edges.
Integer work: bit-exact."""
import numpy as np
import pytest
import torch

import gsampler_amd as gs
from gsampler_amd import capi
from oracle import binding as orc
from tests.conftest import random_csc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def T(a):
    return torch.as_tensor(np.asarray(a, dtype=np.int64), device=DEV)


def _case(rng, S, R, E, id_range, repeat_seeds=False, repeat_list=False, unused=0.3):
    seeds = rng.integers(0, id_range, size=S) if repeat_seeds else rng.permutation(id_range)[:S]
    list_ids = rng.integers(0, id_range, size=R) if repeat_list else rng.permutation(id_range)[:R]
    live = np.flatnonzero(rng.random(R) >= unused)          # listed ids that some edge uses
    row = rng.choice(live, size=E) if live.size and E else np.empty(0, dtype=np.int64)
    col = rng.integers(0, max(S, 1), size=row.size)
    return seeds.astype(np.int64), list_ids.astype(np.int64), row.astype(np.int64), col


def _check(seeds, list_ids, row, col):
    first = capi.first_position(T(row), list_ids.size)
    frontier, list_label, seed_label = capi.list_labels(T(seeds), T(list_ids), first)
    want = orc.unique_relabel(seeds, list_ids[row], edge_col=col if seeds.size else None)
    assert np.array_equal(frontier.cpu().numpy(), want[0])
    assert np.array_equal(list_label.cpu().numpy()[row], want[2])
    if seeds.size:
        assert np.array_equal(seed_label.cpu().numpy()[col], want[3])
        # every seed's label is the place of its first occurrence among the frontier
        assert np.array_equal(want[0][seed_label.cpu().numpy()], seeds)


@pytest.mark.parametrize("S,R,E", [(512, 512, 200_000), (1, 1, 10), (0, 700, 50_000),
                                   (1000, 1048, 300_000), (2047, 1, 5), (3, 2045, 100_000),
                                   (100, 33, 0), (700, 1025, 4000)])
@pytest.mark.parametrize("mode", ["distinct", "overlap", "repeats"])
def test_list_labels_match_unique_over_the_edges(S, R, E, mode):
    rng = np.random.default_rng(S * 7 + R * 3 + len(mode))
    id_range = {"distinct": 10**6, "overlap": S + R + 5, "repeats": max(2, (S + R) // 3)}[mode]
    seeds, list_ids, row, col = _case(rng, S, R, E, id_range, repeat_seeds=mode == "repeats",
                                      repeat_list=mode == "repeats")
    _check(seeds, list_ids, row, col)


@pytest.mark.parametrize("most", [0, 1, 63, 400, 3000])
@pytest.mark.parametrize("cols", [1, 2, 500])
def test_edge_labels_by_column_number_and_by_pointer(cols, most):
    """Runs of 512 edges inside one column, across the border of two and over many, with
    columns of no edge between; the number of edges no multiple of anything."""
    rng = np.random.default_rng(cols * 10_000 + most)
    deg = rng.integers(0, most + 1, size=cols)
    deg[rng.random(cols) < 0.2] = 0
    deg[-1] += 7
    indptr = np.concatenate([[0], np.cumsum(deg)])
    col = np.repeat(np.arange(cols), deg)
    row = rng.integers(0, 300, size=col.size)
    list_label, seed_label = rng.integers(0, 10**6, size=300), rng.integers(0, 10**6, size=cols)
    for how in (dict(col=T(col)), dict(col=None, indptr=T(indptr))):
        got = capi.list_edge_labels(T(row), list_label=T(list_label), seed_label=T(seed_label), **how)
        assert np.array_equal(got[0].cpu().numpy(), list_label[row])
        assert np.array_equal(got[1].cpu().numpy(), seed_label[col])


@pytest.mark.parametrize("short_rows,short_cols", [(0, 0), (3, 0), (0, 2), (3, 2)])
def test_lists_shorter_than_the_matrix(short_rows, short_cols):
    """Seeds and row ids may be fewer than the columns and the rows of the matrix as long as
    no edge needs the missing ones; the labels are the same by either way to them."""
    rng = np.random.default_rng(short_rows * 10 + short_cols)
    R, C = 60, 40
    indptr, indices = random_csc(rng, C, R - short_rows, 4000)
    indptr[C - short_cols:] = indptr[C - short_cols]
    indices = indices[:indptr[-1]]
    g = gs.Graph(R, C)
    g._CAPI_LoadCSC(T(indptr), T(indices))
    seeds = rng.permutation(1000)[:C - short_cols]
    row_ids = rng.permutation(1000)[:R - short_rows]
    assert indices.size >= 8 * (seeds.size + row_ids.size)
    col = np.repeat(np.arange(C), np.diff(indptr))
    want = orc.unique_relabel(seeds, row_ids[indices], edge_col=col)
    frontier, row, col, _ = g._CAPI_GraphRelabel(T(seeds), T(row_ids))
    assert np.array_equal(frontier.cpu().numpy(), want[0])
    assert np.array_equal(row.cpu().numpy(), want[2])
    assert np.array_equal(col.cpu().numpy(), want[3])


@pytest.mark.parametrize("R", [1, 4095, 4096, 4097])
@pytest.mark.parametrize("E", [1, 1024, 16_383, 16_384, 16_385, 100_003])
def test_first_positions_at_the_borders_of_a_tile(E, R):
    rng = np.random.default_rng(E + R)
    row = rng.integers(-2, R + 2, size=E)                    # ids outside are passed over
    row[-1] = R - 1
    want = np.full(R, np.iinfo(np.int64).max)
    ok = (row >= 0) & (row < R)
    np.minimum.at(want, row[ok], np.flatnonzero(ok))
    assert np.array_equal(capi.first_position(T(row), R).cpu().numpy(), want)


def test_list_labels_large_ids_and_all_used():
    rng = np.random.default_rng(5)
    seeds = rng.integers(2**40, 2**41, size=300)
    list_ids = np.concatenate([seeds[:100], rng.integers(-2**50, 2**62, size=400)])
    row = rng.integers(0, 500, size=100_000)
    row[:500] = rng.permutation(500)                          # every listed id is used
    col = rng.integers(0, 300, size=row.size)
    _check(seeds, list_ids, row, col)


def test_list_labels_refuses_what_does_not_fit():
    n = capi.LIST_LABELS_MAX_KEYS
    seeds, ids = T(np.arange(n // 2)), T(np.arange(n // 2 + 1))
    with pytest.raises(capi.GsError, match="exceed"):
        capi.list_labels(seeds, ids, torch.zeros(n // 2 + 1, dtype=torch.int64, device=DEV))


@pytest.mark.parametrize("seeds,picks", [([30, 20], [9, 40]), ([30, 2000], [9, 48]), ([30, 2000], [9, 49])])
def test_a_refused_batch_is_told_on_the_device_too(seeds, picks):
    """The last offset of the frontier is -1 in both copies where a batch has too many keys."""
    rng = np.random.default_rng(sum(picks))
    S, R = sum(seeds), sum(picks)
    sp, lp = (T(np.concatenate([[0], np.cumsum(n)])) for n in (seeds, picks))
    cols, ids, first = T(rng.permutation(5000)[:S]), T(rng.permutation(5000)[:R]), T(np.arange(R))
    frontier, labels, scratch = (torch.empty(n, dtype=torch.int64, device=DEV)
                                 for n in (S + R, S + R, S + R + 3))
    unique_ptr = torch.full((3,), -7, dtype=torch.int64, device=DEV)
    mirror = torch.full((3,), -7, dtype=torch.int64).pin_memory()
    P = lambda t: t.data_ptr()
    capi.check(capi.lib().gs_batch_list_labels(
        P(cols), P(sp), S, P(ids), P(lp), R, 10**6, 2, None, None, None, 0, P(first), P(frontier),
        P(unique_ptr), P(mirror), P(labels), P(labels) + 8 * R, None, None, P(scratch), None))
    torch.cuda.synchronize()
    assert torch.equal(unique_ptr.cpu(), mirror)
    assert (mirror[-1] == -1) == (seeds[1] + picks[1] > capi.LIST_LABELS_MAX_KEYS)


@pytest.mark.parametrize("sizes,picks,mode", [
    ([40, 1, 0, 60], [100, 30, 0, 200], "distinct"),      # a batch of one column, an empty one
    ([300] * 8, [256] * 8, "repeats"),                    # repeated seeds and repeated picks
    ([1000, 20], [1048, 20], "distinct"),                 # exactly as many keys as a batch may have
    ([1000, 20], [1049, 20], "distinct"),                 # one more: the general path
    ([60, 60], [150, 150], "swapped"),                    # picks in the other batch's segment
])
def test_batched_labels_by_way_of_the_list(sizes, picks, mode):
    """Frontier, offsets and labels of a row-sliced encoded super-batch, and all_nodes() before
    and after, against the oracle batch by batch."""
    rng = np.random.default_rng(sum(sizes) + sum(picks))
    R, C = 1500, 2500
    indptr, indices = random_csc(rng, C, R, 3000)
    g = gs.Graph(R, C)
    g._CAPI_LoadCSC(T(indptr), T(indices))
    seeds = np.concatenate([rng.integers(0, C, size=n) if mode == "repeats"
                            else rng.permutation(C)[:n] for n in sizes])
    ptr = np.concatenate([[0], np.cumsum(sizes)])
    sub, _ = g._CAPI_BatchColSlicing(T(seeds), T(ptr), True)
    ids, row_ptr = sub._CAPI_BatchGetRows()
    rp = row_ptr.cpu().numpy()
    picked = [rp[b] + (rng.integers(0, rp[b + 1] - rp[b], size=n) if mode == "repeats"
                       else rng.permutation(rp[b + 1] - rp[b])[:n]) for b, n in enumerate(picks)]
    if mode == "swapped":
        picked.reverse()
    picked_ptr = T(np.concatenate([[0], np.cumsum([p.size for p in picked])]))
    picked = T(np.concatenate(picked))
    for nodes_first in (False, True):
        part, _ = sub._CAPI_BatchRowSlicing(picked, picked_ptr)
        row_ids, d_seeds = ids[picked], T(seeds)
        if nodes_first:
            nodes, nodes_ptr = part._CAPI_BatchGetValidNodes(d_seeds, row_ids)
        frontier, uptr, row, col, _, eptr = part._CAPI_BatchGraphRelabel(d_seeds, row_ids)
        if not nodes_first:
            nodes, nodes_ptr = part._CAPI_BatchGetValidNodes(d_seeds, row_ids)
        assert torch.equal(nodes, frontier) and torch.equal(nodes_ptr, uptr)
        kept = [row.clone(), col.clone()]
        row.zero_(), col.zero_()          # the caller's own: the next call does not return them
        frontier, uptr, row, col, _, eptr = part._CAPI_BatchGraphRelabel(d_seeds, row_ids)
        assert torch.equal(row, kept[0]) and torch.equal(col, kept[1])
        keys = row_ids[part._CAPI_GetCOORows()].cpu().numpy()
        at_col = part._CAPI_GetCOOCols().cpu().numpy()
        frontier, uptr, row, col, eptr = (x.cpu().numpy() for x in (frontier, uptr, row, col, eptr))
        assert keys.size >= 8 * (picked.numel() + seeds.size) and uptr[-1] == frontier.size
        for b in range(len(sizes)):
            s, e, u = (slice(p[b], p[b + 1]) for p in (ptr, eptr, uptr))
            want = orc.unique_relabel(seeds[s], keys[e],
                                      edge_col=at_col[e] - ptr[b] if sizes[b] else None)
            assert np.array_equal(frontier[u], want[0]) and np.array_equal(row[e], want[2])
            if sizes[b]:
                assert np.array_equal(col[e], want[3])


def test_batched_labels_of_rows_that_the_caller_wrote():
    """A row in another batch's segment goes by the general path; one outside the list is read
    by nobody and refused."""
    rng = np.random.default_rng(9)
    indptr, indices = random_csc(rng, 2500, 1500, 3000)
    g = gs.Graph(1500, 2500)
    g._CAPI_LoadCSC(T(indptr), T(indices))
    seeds, ptr = T(rng.permutation(2500)[:60]), T([0, 40, 60])
    sub, _ = g._CAPI_BatchColSlicing(seeds, ptr, True)
    ids, row_ptr = sub._CAPI_BatchGetRows()
    picked, picked_ptr = T(np.concatenate([np.arange(90), int(row_ptr[1]) + np.arange(50)])), T([0, 90, 140])
    part, _ = sub._CAPI_BatchRowSlicing(picked, picked_ptr)
    assert part._CAPI_GetNumEdges() >= 8 * 200
    edge_rows = part._CAPI_GetCOORows()
    for wrong in (-1, -2**62, 140, 2**40):
        kept = edge_rows[7].item()
        edge_rows[7] = wrong
        with pytest.raises(RuntimeError, match="row of an edge lies outside"):
            part._CAPI_BatchGraphRelabel(seeds, ids[picked])
        edge_rows[7] = 139  # of the other batch
        frontier, uptr, row, _, _, _ = part._CAPI_BatchGraphRelabel(seeds, ids[picked])
        assert frontier[row[7]] == ids[picked][139] and row[7] < uptr[1]
        edge_rows[7] = kept


@pytest.mark.parametrize("sizes,picks", [
    ([64] * 8, [512] * 8),             # 4096 listed ids, the most that the list pass holds in LDS
    ([20] * 17, [241] * 17),           # 4097, few edges: by way of the list all the same
    ([100] * 10, [450] * 10),          # 4500 and several hundred thousand: the general path
])
def test_batched_labels_where_the_list_begins_or_ends_to_pay(sizes, picks):
    test_batched_labels_by_way_of_the_list(sizes, picks, "distinct")
