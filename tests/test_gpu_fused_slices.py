"""Operators that read a column slice without writing it: A[rows, cols] in one
pass over the parent matrix and the row sums of squared edge values of A[:, cols].
Checked against the CPU operators chained by hand (column slice, then row slice or
sum over the slice): what the reference computes through the intermediate slice
(src/cuda/fusion/column_row_slicing.cu:148-217, src/graph.cc:457-480)."""
import threading

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
    return None if a is None else torch.as_tensor(np.asarray(a, dtype=np.int64), device=DEV)


def same(got, want):
    for g, w in zip(got, want):
        if w is None:
            assert g is None
        else:
            assert np.array_equal(g.cpu().numpy(), w)


def chained_col_row_slice(indptr, indices, cols, rows, key_offset=None):
    """Column slice, then row slice of it, select index mapped back to the parent."""
    sub_indptr, coo_col, sub_rows, sel = orc.col_slice(indptr, indices, cols)
    if key_offset is not None:
        sub_rows = sub_rows + np.asarray(key_offset)[coo_col]
    out_indptr, major, minor, kept = orc.minor_slice(sub_rows, rows, indptr=sub_indptr)
    return out_indptr, major, minor, sel[kept]


@pytest.mark.parametrize("ncol,nrow", [(0, 5), (1, 1), (7, 0), (300, 64), (2000, 512), (512, 5000)])
def test_col_row_slice_parity(ncol, nrow):
    rng = np.random.default_rng(ncol * 7 + nrow)
    indptr, indices = random_csc(rng, 3000, 5000, 50, hub_deg=40000)
    cols = rng.integers(0, 3000, size=ncol)                 # repeats allowed
    if ncol > 5:
        cols[2] = int(np.argmax(np.diff(indptr)))           # the hub column
        cols[3] = cols[4]
    rows = rng.integers(0, 5200, size=nrow)                 # repeats and absent ids
    want = chained_col_row_slice(indptr, indices, cols, rows)
    same(capi.col_row_slice(T(indptr), T(indices), T(cols), T(rows)), want)
    # the row ids read from a 32-bit copy
    same(capi.col_row_slice(T(indptr), T(indices), T(cols), T(rows),
                            indices32=T(indices).to(torch.int32)), want)
    got = capi.col_row_slice(T(indptr), T(indices), T(cols), T(rows), with_major=False)
    assert got[1] is None
    same((got[0], got[2], got[3]), (want[0], want[2], want[3]))


@pytest.mark.parametrize("nrow", [1, 64, 65, 2048])
@pytest.mark.parametrize("nnz", [1, 300, 70_001, (1 << 23) + 5, (1 << 25) + 1])
def test_col_row_slice_tells_the_first_edge_of_every_row(nnz, nrow):
    """First edges from work-groups of every size, one to several hundred of them, beside the
    offsets and (the longest list) in a launch of their own: rows that repeat, that no edge
    has, that have one edge; row ids moved by a column's offset, and beyond 32 bits."""
    rng = np.random.default_rng(nnz + nrow)
    ids = rng.integers(0, 5000, size=nnz)
    ids[-1] = 777_777
    indptr = np.concatenate([[0], np.sort(rng.integers(0, nnz + 1, size=3)), [nnz]])
    cols = rng.permutation(4)
    rows = rng.permutation(6000)[:nrow]
    rows[-1] = 777_777
    if nrow > 2:
        rows[1] = rows[0]
    want = np.concatenate([ids[indptr[c]:indptr[c + 1]] for c in cols])
    sizes = np.diff(indptr)[cols]
    for offset in (None, np.arange(4) * 10_000, np.arange(4) * 2**33):
        keys, picked = want, rows
        if offset is not None:
            keys = want + np.repeat(offset, sizes)
            picked = rows + offset[rng.integers(0, 4, size=nrow)]
        first = torch.empty(nrow, dtype=torch.int64, device=DEV)
        got = capi.col_row_slice(T(indptr), T(ids), T(cols), T(picked), out_first=first,
                                 key_offset=T(offset) if offset is not None else None)
        expect = np.full(nrow, 2**63 - 1)
        order = np.argsort(picked, kind="stable")
        found = np.searchsorted(picked[order], keys)
        hit = (found < nrow) & (picked[order][np.minimum(found, nrow - 1)] == keys)
        np.minimum.at(expect, order[found[hit]], np.nonzero(hit)[0])
        assert np.array_equal(first.cpu().numpy(), expect)
        assert np.array_equal(got[2].cpu().numpy(), order[found[hit]])


def test_scratch_for_first_edges_where_they_are_asked_for():
    """1024 work-groups' lists of 2047 ids are 8 MB: in the workspace of the calls that tell
    first edges, in no other's, and refused where it is missing."""
    l, nnz, nrow = capi.lib(), 1 << 23, 2047
    plain = l.gs_minor_slice_workspace_bytes(nnz, nrow)
    told = l.gs_col_row_slice_first_workspace_bytes(nnz, nrow)
    assert told - plain == 4 * 1024 * nrow
    assert l.gs_col_row_slice_first_workspace_bytes(nnz, 2049) == l.gs_minor_slice_workspace_bytes(nnz, 2049)
    rng = np.random.default_rng(2)
    indptr, ids = T([0, 5000]), T(rng.integers(0, 90, size=5000))
    cols, sub, out = T([0]), T([0, 5000]), torch.empty(2, dtype=torch.int64, device=DEV)
    rows, first = T(np.arange(70)), torch.full((70,), -7, dtype=torch.int64, device=DEV)
    ws = torch.empty(l.gs_minor_slice_workspace_bytes(5000, 70), dtype=torch.uint8, device=DEV)
    P = lambda t: t.data_ptr()
    args = (P(indptr), P(ids), None, P(cols), None, 1, P(sub), 5000, P(rows), 70, P(out), None)
    assert l.gs_col_row_slice_count_first(*args, P(first), None, P(ws), ws.numel(), None) != 0
    assert l.gs_col_row_slice_count_first(*args, None, None, P(ws), ws.numel(), None) == 0
    torch.cuda.synchronize()
    assert (first == -7).all() and out[1].item() == int((ids < 70).sum())


def test_col_row_slice_of_long_columns():
    """Columns far longer than a work-group's run of edges (the layer-wise
    sampler's case), columns without edges in between, a column id outside the
    matrix (degree 0)."""
    rng = np.random.default_rng(11)
    deg = np.zeros(400, dtype=np.int64)
    deg[rng.choice(400, size=40, replace=False)] = rng.integers(20_000, 90_000, size=40)
    indptr = np.concatenate([[0], np.cumsum(deg)])
    indices = rng.integers(0, 100_000, size=int(deg.sum()))
    cols = np.concatenate([rng.integers(0, 400, size=300), [400, -1, 399]])
    rows = rng.choice(100_000, size=512, replace=False)
    same(capi.col_row_slice(T(indptr), T(indices), T(cols), T(rows)),
         chained_col_row_slice(indptr, indices, cols, rows))


def test_col_row_slice_with_per_column_key_offsets():
    """Mini-batches of a super-batch: the row ids of batch b's columns and its picked rows
    are both moved by b * stride, so a row only matches inside its own batch; ids beyond
    32 bits take the confirming look-ups."""
    rng = np.random.default_rng(5)
    indptr, indices = random_csc(rng, 2000, 3000, 40, hub_deg=9000)
    for stride in (3000, 2**33):
        col_ptr = np.array([0, 100, 100, 350, 600])
        cols = rng.integers(0, 2000, size=600)
        batch_of_col = np.repeat(np.arange(4), np.diff(col_ptr))
        key_offset = batch_of_col * stride
        picked = np.concatenate([rng.choice(3000, size=80, replace=False) + b * stride
                                 for b in range(4)])
        want = chained_col_row_slice(indptr, indices, cols, picked, key_offset)
        same(capi.col_row_slice(T(indptr), T(indices), T(cols), T(picked), T(key_offset)), want)
        same(capi.col_row_slice(T(indptr), T(indices), T(cols), T(picked), T(key_offset),
                                indices32=T(indices).to(torch.int32)), want)


@pytest.mark.parametrize("npick", [600, 5000])
@pytest.mark.parametrize("offset", [0, 70_000, 2**31 - 1, 2**31, 2**32 - 1000, -500])
def test_col_row_slice_of_columns_of_every_length(offset, npick):
    """9 M edges, for which every wave strides over runs: columns without edges, of a few, that
    end at the borders of rows, and long ones, next to each other, more than 64 of them in a
    run; the offsets of half of them at the ends of what 32-bit arithmetic can hold."""
    rng = np.random.default_rng(npick + offset % 1000)
    deg = np.concatenate([rng.integers(0, 4, size=3000), rng.integers(0, 3, size=500) * 64,
                          rng.integers(0, 900, size=500), rng.integers(50_000, 60_000, size=160),
                          rng.integers(0, 2, size=700) * rng.integers(0, 130, size=700)])
    deg[rng.choice(4000, 300)] = 1
    indptr = np.concatenate([[0], np.cumsum(deg)])
    assert 1 << 23 <= indptr[-1] < 1 << 24
    indices = rng.integers(0, 60_000, size=int(indptr[-1]))
    cols = np.arange(len(deg))
    key_offset = np.where(rng.random(len(deg)) < 0.5, offset, 0)
    picked = rng.choice(60_000, size=npick, replace=False)
    picked[npick // 2:] += offset
    want = chained_col_row_slice(indptr, indices, cols, picked, key_offset)
    narrow = T(indices).to(torch.int32)
    same(capi.col_row_slice(T(indptr), T(indices), T(cols), T(picked), T(key_offset)), want)
    same(capi.col_row_slice(T(indptr), T(indices), T(cols), T(picked), T(key_offset),
                            indices32=narrow), want)


@pytest.mark.parametrize("ncol,num_rows", [(0, 100), (3, 5000), (600, 5200), (512, 100_000)])
@pytest.mark.parametrize("use_workspace", [True, False])
def test_sliced_e_square_sum_parity(ncol, num_rows, use_workspace):
    """Row sums of w^2 over A[:, cols] against float64 sums over the written slice; the
    last case is long enough (2.8 M edges) for the sorting path when a workspace is given."""
    rng = np.random.default_rng(ncol + num_rows)
    if num_rows == 100_000:
        deg = rng.integers(3000, 8000, size=700)
        indptr = np.concatenate([[0], np.cumsum(deg)])
        indices = rng.integers(0, num_rows, size=int(deg.sum()))
        cols = rng.integers(0, 700, size=ncol)
    else:
        indptr, indices = random_csc(rng, 3000, 5000, 50, hub_deg=40000)
        cols = rng.integers(0, 3000, size=ncol)
        if ncol > 5:
            cols[1] = int(np.argmax(np.diff(indptr)))
    w = (rng.random(indices.size) + 0.05).astype(np.float32)
    _, _, sub_rows, sel = orc.col_slice(indptr, indices, cols)
    want = np.zeros(num_rows)
    ok = sub_rows < num_rows                                 # ids outside the output are skipped
    np.add.at(want, sub_rows[ok], w[sel][ok].astype(np.float64) ** 2)
    got = capi.sliced_e_square_sum(T(indptr), T(indices), T(cols),
                                   torch.as_tensor(w, device=DEV), num_rows,
                                   use_workspace=use_workspace).cpu().numpy()
    assert np.allclose(got, want, rtol=1e-5, atol=1e-30)
    got32 = capi.sliced_e_square_sum(T(indptr), T(indices), T(cols),
                                     torch.as_tensor(w, device=DEV), num_rows,
                                     use_workspace=use_workspace,
                                     indices32=T(indices).to(torch.int32)).cpu().numpy()
    assert np.allclose(got32, want, rtol=1e-5, atol=1e-30)
    # and the CPU operator over the written slice agrees with the same sums
    cpu = orc.e_square_sum(("coo", sub_rows[ok], np.zeros(int(ok.sum()), dtype=np.int64)),
                           w[sel][ok], 2, num_rows)
    assert np.allclose(cpu, want, rtol=1e-5, atol=1e-30)


@pytest.mark.parametrize("num_rows", [1, 8192, 8193, 262_144, 262_145])
@pytest.mark.parametrize("nnz", [2047, 2048, 2049, 17 * 1024, 300_001, (1 << 20) - 1])
def test_short_sliced_sums_by_ranges_of_rows(nnz, num_rows):
    """Every range of rows reads every edge: at the borders of ranges and parts, columns of no,
    one and many edges, a row of half the edges; entries keep what they hold, and -0 where no
    edge adds.  Squares are not negative, so a sum is off by its roundings alone: the square,
    a part, the parts' sum and the add, 2^-24 each."""
    rng = np.random.default_rng(nnz + num_rows)
    deg = np.concatenate([rng.integers(0, 4, size=200), [nnz // 3, 0, 0, 1, 63, 64, 65]])
    deg = np.concatenate([deg, [nnz - deg.sum()]])
    indptr = np.concatenate([[0], np.cumsum(deg)])
    indices = rng.integers(0, num_rows, size=nnz)
    indices[rng.random(nnz) < 0.5] = num_rows - 1
    cols = rng.permutation(len(deg))
    w = rng.random(nnz).astype(np.float32)
    w[rng.random(nnz) < 0.1] = 0
    e_map = rng.permutation(nnz)
    held = np.where(rng.random(num_rows) < 0.5, np.float32(-0.0), np.float32(0.25))
    want = np.zeros(num_rows)
    np.add.at(want, indices, (w[e_map] * w[e_map]).astype(np.float64))
    none = np.bincount(indices, minlength=num_rows) == 0
    lib, outs = capi.lib(), []
    need = lib.gs_sliced_e_square_sum_workspace_bytes(nnz, num_rows)
    assert (need > 0) == (nnz >= 2048 and num_rows <= 262_144)
    args = [T(indptr), T(indices), T(cols), T(e_map), torch.as_tensor(w, device=DEV)]
    sub = capi.col_count(args[0], args[2], -1, False)
    ws = torch.empty(need + 1, dtype=torch.uint8, device=DEV)
    for narrow in (None, args[1].to(torch.int32)):
        out = torch.as_tensor(held, device=DEV)
        capi.check(lib.gs_sliced_e_square_sum(
            args[0].data_ptr(), args[1].data_ptr(), None if narrow is None else narrow.data_ptr(),
            args[2].data_ptr(), len(cols), sub.data_ptr(), nnz, args[3].data_ptr(),
            args[4].data_ptr(), out.data_ptr(), num_rows, ws.data_ptr(), need,
            torch.cuda.current_stream().cuda_stream))
        got = out.cpu().numpy()
        if need:
            assert np.allclose(got, held + want, rtol=4 * 2.0**-24, atol=0)
        assert np.array_equal(got[none].view(np.int32), held[none].view(np.int32))
        assert not np.signbit(got[~none]).any()


@pytest.mark.parametrize("pinned", [False, True])
def test_threads_with_other_columns_on_one_matrix(pinned):
    """What an operator holds of a slice stays when another thread's takes its place: read in
    place, and, of a matrix in pinned host memory, the written slices of three of the threads."""
    place = (lambda a: T(a).cpu().pin_memory()) if pinned else T
    rng = np.random.default_rng(21)
    deg = rng.integers(100, 9000, size=700)
    indptr = np.concatenate([[0], np.cumsum(deg)])
    indices = rng.integers(0, 20_000, size=int(deg.sum()))
    g = gs.Graph(20_000, 700)
    g._CAPI_LoadCSC(place(indptr), place(indices))
    w = torch.as_tensor((rng.random(indices.size) + 0.05).astype(np.float32), device=DEV)
    rows = T(rng.choice(20_000, size=300, replace=False))
    cols = [T(rng.integers(0, 700, size=n)) for n in (3, 40, 300, 500)]

    def once(c):
        out = torch.zeros(20_000, device=DEV)
        g._CAPI_SlicedESquareSum(c, w, out)
        sub, index = g._CAPI_ColRowSlicing(c, rows, gs.format._CSC, gs.format._CSC)
        return out, sub._CAPI_GetCSCIndptr(), sub._CAPI_GetCSCIndices(), index

    want = [once(c) for c in cols]
    torch.cuda.synchronize()
    bad = []

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(40):
                got = once(cols[i].clone())
                same_ids = all(torch.equal(a, b) for a, b in zip(got[1:], want[i][1:]))
                # two orders of adding some hundred 32-bit terms: 1e-5 apart at most
                if not (same_ids and torch.allclose(got[0], want[i][0], rtol=1e-5)):
                    bad.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def stream_beside(first):
    """A stream whose work does not stand behind that of `first`: few of them have a queue of
    the hardware to themselves."""
    for _ in range(16):
        other, mark = torch.cuda.Stream(), torch.zeros(1, device=DEV)
        torch.cuda.synchronize()
        with torch.cuda.stream(first):
            torch.cuda._sleep(20_000_000)                   # 8 ms
        with torch.cuda.stream(other):
            mark += 1
        other.synchronize()
        if not first.query():
            torch.cuda.synchronize()
            return other
    pytest.skip("every stream stands behind the first one")


def test_a_second_stream_with_the_same_columns():
    """What one stream has queued of a slice is not read on another that does not wait for it."""
    rng = np.random.default_rng(22)
    indptr, indices = random_csc(rng, 3000, 6000, 60)
    g = gs.Graph(6000, 3000)
    g._CAPI_LoadCSC(T(indptr), T(indices))
    w = torch.as_tensor((rng.random(indices.size) + 0.05).astype(np.float32), device=DEV)
    cols, rows = rng.integers(0, 3000, size=900), rng.choice(6000, size=400, replace=False)
    want = chained_col_row_slice(indptr, indices, cols, rows, None)
    first = torch.cuda.Stream()
    second = stream_beside(first)
    c, r = T(cols), T(rows)
    sums = [torch.zeros(6000, device=DEV) for _ in range(2)]
    # (kernels are loaded at their first use)
    g._CAPI_ColRowSlicing(c.clone(), r, gs.format._CSC, gs.format._CSC)
    torch.cuda.synchronize()
    with torch.cuda.stream(first):
        g._CAPI_SlicedESquareSum(c, w, sums[0])
        torch.cuda._sleep(200_000_000)                      # 80 ms
        g._CAPI_SlicedESquareSum(c, w, sums[1])
    with torch.cuda.stream(second):
        sub, index = g._CAPI_ColRowSlicing(c, r, gs.format._CSC, gs.format._CSC)
        got = (sub._CAPI_GetCSCIndptr(), sub._CAPI_GetCSCIndices(), index)
    second.synchronize()
    assert not first.query()                                # the first one was not waited for
    same(got, (want[0], want[2], want[3]))
    first.synchronize()
    # two orders of adding at most 900 x 60 terms of 32 bits
    assert torch.allclose(*sums, rtol=1e-5)


def test_a_second_stream_beside_a_slice_being_written():
    """A slice of a matrix in pinned host memory is written, over the bus, and kept: another
    stream does not read it half done."""
    rng = np.random.default_rng(23)
    indptr, indices = random_csc(rng, 40_000, 6000, 300)
    g = gs.Graph(6000, 40_000)
    g._CAPI_LoadCSC(T(indptr).cpu().pin_memory(), T(indices).cpu().pin_memory())
    w = torch.ones(indices.size, device=DEV)
    cols, rows = rng.permutation(40_000), rng.choice(6000, size=400, replace=False)
    want = chained_col_row_slice(indptr, indices, cols, rows, None)
    first = torch.cuda.Stream()
    second = stream_beside(first)
    r, sums = T(rows), torch.zeros(6000, device=DEV)
    for c in (T(cols), T(cols)):     # (the first time kernels are loaded and memory is taken)
        torch.cuda.synchronize()
        with torch.cuda.stream(first):
            g._CAPI_SlicedESquareSum(c, w, sums)
        with torch.cuda.stream(second):
            sub, index = g._CAPI_ColRowSlicing(c, r, gs.format._CSC, gs.format._CSC)
            got = (sub._CAPI_GetCSCIndptr(), sub._CAPI_GetCSCIndices(), index)
        second.synchronize()
        same(got, (want[0], want[2], want[3]))
    torch.cuda.synchronize()
    # ones, counted exactly
    assert np.array_equal(sums.cpu().numpy(), 2.0 * np.bincount(indices, minlength=6000))


@pytest.mark.parametrize("most,ncol", [(0, 5), (1, 0), (1, 300), (3, 1), (3, 70_000), (20, 9000), (700, 1500)])
@pytest.mark.parametrize("pinned", [False, True])
def test_slices_of_short_columns(most, ncol, pinned):
    """Columns of 0 to a few hundred edges, which a matrix in device memory is read in place
    for: runs over more columns than a wavefront has lanes, slices of nothing, repeated
    columns and ids that the matrix does not have; the written slice of a pinned one."""
    rng = np.random.default_rng(most + ncol)
    indptr, indices = random_csc(rng, 4000, 6000, most, hub_deg=3000 if most == 3 else 0)
    if pinned and indices.size == 0:
        return                                               # no memory to pin
    place = (lambda a: T(a).cpu().pin_memory()) if pinned else T
    g = gs.Graph(6000, 4000)
    g._CAPI_LoadCSC(place(indptr), place(indices))
    cols = rng.integers(0, 4000, size=ncol)
    rows = rng.choice(6000, size=400, replace=False)
    want = chained_col_row_slice(indptr, indices, cols, rows, None)
    sub, index = g._CAPI_ColRowSlicing(T(cols), T(rows), gs.format._CSC, gs.format._CSC)
    same((sub._CAPI_GetCSCIndptr(), sub._CAPI_GetCSCIndices(), index), (want[0], want[2], want[3]))
    w = (rng.random(indices.size) + 0.05).astype(np.float32)
    out = torch.zeros(6000, device=DEV)
    g._CAPI_SlicedESquareSum(T(cols), torch.as_tensor(w, device=DEV), out)
    _, _, sub_rows, sel = orc.col_slice(indptr, indices, cols)
    sums = np.zeros(6000)
    np.add.at(sums, sub_rows, w[sel].astype(np.float64) ** 2)
    # at most 70 000 terms of 32 bits: rounded some sqrt(n) times 2^-24 apart
    assert np.allclose(out.cpu().numpy(), sums, rtol=2e-5, atol=1e-30)
    if ncol == 0:
        return
    ptr = np.array([0, ncol // 3, ncol // 3, ncol])
    rptr = np.array([0, 150, 250, 400])
    offset = np.repeat([0, 6000, 12000], np.diff(ptr))
    moved = rows + np.repeat([0, 6000, 12000], np.diff(rptr))
    want = chained_col_row_slice(indptr, indices, cols, moved, offset)
    sub, index = g._CAPI_BatchColRowSlcing(T(cols), T(ptr), T(rows), T(rptr))
    same((sub._CAPI_GetCSCIndptr(), sub._CAPI_GetCSCIndices(), index), (want[0], want[2], want[3]))


@pytest.mark.parametrize("n", [1, 255, 256, 257, 5000])
def test_batch_ids_moved_by_their_batch(n):
    rng = np.random.default_rng(n)
    ptr = np.concatenate([[0], np.sort(rng.integers(0, n + 1, size=300)), [n]])
    ids, out = T(rng.integers(0, 10**9, size=n)), torch.empty(n, dtype=torch.int64, device=DEV)
    batch = T(np.repeat(np.arange(301), np.diff(ptr)))
    for of in (ids, None):
        capi.check(capi.lib().gs_encode_batch_ids(of.data_ptr() if of is not None else None, T(ptr).data_ptr(),
                                                  301, n, 10**10, out.data_ptr(), None))
        torch.cuda.synchronize()
        assert torch.equal(out, batch * 10**10 + (ids if of is not None else 0))


@pytest.mark.parametrize("n", [1, 256, 257, 5000])
def test_batch_ids_picked_from_a_list(n):
    rng = np.random.default_rng(n)
    ptr = np.concatenate([[0], np.sort(rng.integers(0, n + 1, size=300)), [n]])
    ids, index = T(rng.integers(0, 10**9, size=700)), T(rng.integers(0, 700, size=n))
    batch = T(np.repeat(np.arange(301), np.diff(ptr)))
    direct, l = T(rng.integers(0, 10**9, size=n)), capi.lib()
    for source, at, name in ((ids, index, ids[index]), (direct, None, direct)):
        outs = [torch.full((n,), -7, dtype=torch.int64, device=DEV) for _ in range(3)]
        for wanted in ((0, 1, 2), (1,), (0, 2)):
            for o in outs:
                o.fill_(-7)
            capi.check(l.gs_pick_batch_ids(
                source.data_ptr(), source.numel(), at.data_ptr() if at is not None else None,
                T(ptr).data_ptr(), 301, n, 10**10,
                *(outs[i].data_ptr() if i in wanted else None for i in range(3)), None, None))
            torch.cuda.synchronize()
            for i, want in enumerate((name, name + batch * 10**10, batch * 10**10)):
                assert torch.equal(outs[i], want if i in wanted else torch.full_like(want, -7))
    # ids behind local rows, as they are and without their batch
    moved = name + batch * 10**10
    rows, out = T(rng.integers(0, n, size=3 * n + 1)), torch.empty(3 * n + 1, dtype=torch.int64, device=DEV)
    for stride, want in ((0, moved[rows]), (10**10, name[rows])):
        capi.check(l.gs_local_ids(moved.data_ptr(), n, rows.data_ptr(), rows.numel(), stride,
                                  out.data_ptr(), None, None))
        torch.cuda.synchronize()
        assert torch.equal(out, want)


@pytest.mark.parametrize("outside", [-1, 700, 2**40, -2**63])
@pytest.mark.parametrize("n", [1, 1024, 1025, 5000])
def test_places_outside_a_list_are_told(n, outside):
    rng = np.random.default_rng(n)
    ids, ptr = T(rng.integers(0, 10**9, size=700)), T([0, n])
    out = torch.empty(n, dtype=torch.int64, device=DEV)
    l, flag = capi.lib(), torch.empty(1, dtype=torch.int64, device=DEV)
    for at in (None, 0, n - 1):
        index = T(rng.integers(0, 700, size=n))
        if at is not None:
            index[at] = outside
        for call in (lambda: l.gs_pick_batch_ids(ids.data_ptr(), 700, index.data_ptr(), ptr.data_ptr(), 1, n,
                                                 10, out.data_ptr(), None, None, flag.data_ptr(), None),
                     lambda: l.gs_local_ids(ids.data_ptr(), 700, index.data_ptr(), n, 0, out.data_ptr(),
                                            flag.data_ptr(), None)):
            flag.zero_()
            capi.check(call())
            torch.cuda.synchronize()
            assert flag.item() == (at is not None)
            keep = torch.arange(n, device=DEV) != (-1 if at is None else at)
            assert torch.equal(out[keep], ids[index[keep]])


def test_rows_and_picks_that_a_list_does_not_have_are_refused():
    """Picks outside the rows of an encoded slice, edges whose rows the caller wrote outside
    the list, lists that are too short; the calls that follow are served."""
    rng = np.random.default_rng(17)
    indptr, indices = columns_of(rng.integers(1, 90, 400), rng, 400)
    g = gs.Graph(400, 400)
    g._CAPI_LoadCSC(T(indptr), T(indices))
    w = torch.ones(indices.size, device=DEV)
    seeds, ptr = batches_of(rng, 400, [20, 30])
    rows, rows_ptr, _ = g._CAPI_EncodedSquareSums(seeds, ptr, w)
    good, good_ptr = T([1, 5, int(rows_ptr[1]) + 2]), T([0, 2, 3])
    for wrong in (-1, rows.numel(), 2**40):
        bad = good.clone()
        bad[1] = wrong
        for call in (g._CAPI_EncodedPickedRows, lambda *a: g._CAPI_EncodedBlocks(*a, None, None)):
            with pytest.raises(RuntimeError, match="picked row lies outside"):
                call(seeds, ptr, rows, bad, good_ptr)
    assert g._CAPI_EncodedBlocks(seeds, ptr, rows, good, good_ptr, None, None) is not None
    sub, _, names = g._CAPI_EncodedPickedRows(seeds, ptr, rows, good, good_ptr)
    assert torch.equal(names, rows[good])

    cut, _ = g._CAPI_BatchColSlicing(seeds, ptr, True)
    ids, _ = cut._CAPI_BatchGetRows()
    want = cut._CAPI_BatchGraphRelabel(seeds, ids)
    edge_rows = cut._CAPI_GetCOORows()
    kept = edge_rows[3].item()
    for wrong in (-1, ids.numel(), 2**40):
        edge_rows[3] = wrong
        for call in (cut._CAPI_BatchGraphRelabel, cut._CAPI_BatchGetValidNodes, cut._CAPI_BatchBlocks):
            with pytest.raises(RuntimeError, match="row of an edge lies outside"):
                call(seeds, ids.clone())
    edge_rows[3] = kept
    with pytest.raises(RuntimeError, match="row of an edge lies outside"):
        cut._CAPI_BatchGraphRelabel(seeds, ids[:-1].contiguous())  # (every row has an edge)
    for a, b in zip(cut._CAPI_BatchGraphRelabel(seeds, ids.clone()), want):
        assert a is b is None or torch.equal(a, b)


@pytest.mark.parametrize("order", ["blocks", "nodes first", "edge list first", "rows written"])
@pytest.mark.parametrize("sizes", [[40], [64, 0, 300, 1], [3] * 70, [9000, 30_000]])
def test_relabel_of_the_subgraph_that_a_list_induces(sizes, order):
    """A[list, list]: the frontier from the list alone and labels by position are those that
    the general path has (a copy of the list as row ids takes it), with nodes that are in a
    batch several times, batches without nodes, few and many edges."""
    rng = np.random.default_rng(sum(sizes))
    n, degree = 12_000, 6 if sum(sizes) > 10_000 else 300
    indptr = np.arange(n + 1) * degree
    indices = rng.integers(0, 500 if sum(sizes) < 1000 else n, size=n * degree)
    g = gs.Graph(n, n)
    g._CAPI_LoadCSC(T(indptr), T(indices))
    seeds = np.concatenate([rng.integers(0, 400 if k < 1000 else n, size=k) for k in sizes])
    seeds, ptr = T(seeds), T(np.concatenate([[0], np.cumsum(sizes)]))
    results = []
    for rows in (seeds, seeds.clone()):
        sub, _ = g._CAPI_BatchColRowSlcing(seeds, ptr, seeds, ptr)
        if order == "edge list first":
            assert sub._CAPI_GetCOORows().numel() == sub._CAPI_GetNumEdges()
        elif order == "rows written":
            edge_rows = sub._CAPI_BatchGetCSCIndices()[0]
            edge_rows.copy_(torch.where(edge_rows % 2 == 0, edge_rows, torch.zeros_like(edge_rows)))
        nodes = sub._CAPI_BatchGetValidNodes(seeds, rows) if order == "nodes first" else ()
        results.append((*nodes, *sub._CAPI_BatchGraphRelabel(seeds, rows)[:4]))
        results[-1] += tuple(sub._CAPI_BatchGetValidNodes(seeds, rows))
    assert len(results[0]) == len(results[1])
    for mine, general in zip(*results):
        assert torch.equal(mine, general)


@pytest.mark.parametrize("rows", [1, 9000, 400_000])
@pytest.mark.parametrize("nnz", [0, 1, 2047, 2048, 70_001, (1 << 21) + 3])
def test_square_sums_into_an_array_that_holds_nothing(nnz, rows):
    """By ranges that are partitioned, ranges that every work-group reads and atomics: the
    same values as onto a cleared array, whatever the new one held."""
    rng = np.random.default_rng(nnz + rows)
    indices = T(np.minimum(rng.integers(0, rows, size=nnz + 5), rng.integers(0, rows, size=nnz + 5)))
    indptr, cols = T([0, nnz // 3, nnz, nnz + 5]), T([1, 0])
    w = torch.as_tensor(rng.integers(1, 3, size=nnz + 5).astype(np.float32), device=DEV)  # sums below 2^24
    want = capi.sliced_e_square_sum(indptr, indices, cols, w, rows)
    l = capi.lib()
    sub = capi.col_count(indptr, cols, -1, False)
    for size in (l.gs_sliced_e_square_sum_workspace_bytes(nnz, rows), 0):
        ws = torch.empty(max(size, 1), dtype=torch.uint8, device=DEV)
        out = torch.full((rows + 1,), 77.0, device=DEV)
        capi.check(l.gs_sliced_e_square_sums(
            indptr.data_ptr(), indices.data_ptr(), None, cols.data_ptr(), 2, sub.data_ptr(), nnz, None,
            w.data_ptr(), out.data_ptr(), rows, ws.data_ptr() if size else None, size, None))
        torch.cuda.synchronize()
        assert torch.equal(out[:-1], want) and out[-1].item() == 77.0


@pytest.mark.parametrize("nnz", [0, 5000, (1 << 25) + 1])
def test_row_slices_clear_the_sums_of_their_columns(nnz):
    indptr = T(np.sort(np.concatenate([[0, 0, nnz, nnz], np.random.default_rng(1).integers(0, nnz + 1, 700)])))
    ncol = indptr.numel() - 1
    zeros = torch.full((ncol + 1,), 5.0, dtype=torch.float64, device=DEV)
    capi.col_row_slice(indptr, torch.zeros(max(nnz, 1), dtype=torch.int64, device=DEV),
                       torch.arange(ncol, device=DEV), T([3, 0]), col_zeros=zeros)
    assert not zeros[:-1].any() and zeros[-1].item() == 5.0


def test_normalised_columns_of_one_slice_several_times():
    """The first takes the sums that the slice left cleared, the next ones clear their own."""
    rng = np.random.default_rng(4)
    indptr, indices = random_csc(rng, 300, 2000, 90)
    g = gs.Graph(2000, 300)
    g._CAPI_LoadCSC(T(indptr), T(indices))
    w = torch.as_tensor(rng.random(indices.size).astype(np.float32) + 0.1, device=DEV)
    sub, index = g._CAPI_ColRowSlicing(T(rng.permutation(300)[:200]), T(rng.permutation(2000)[:900]),
                                       gs.format._CSC, gs.format._CSC | gs.format._COO)
    got = [sub._CAPI_NormaliseColumns(w, index, None) for _ in range(3)]
    assert all(torch.allclose(g, got[0], rtol=1e-6) for g in got)
    col = torch.repeat_interleave(torch.arange(200, device=DEV), torch.diff(sub._CAPI_GetCSCIndptr()))
    sums = torch.zeros(200, dtype=torch.float64, device=DEV).index_add_(0, col, w[index].double())
    assert torch.allclose(got[0].double(), w[index].double() / sums[col], rtol=1e-6)


def sliced_for_sums(rng, num_rows=3000):
    """A row slice whose sums over columns have storage of their own (more rows than first
    edges are told of), and the normalised values it is to have."""
    indptr, indices = random_csc(rng, 300, num_rows, 90)
    g = gs.Graph(num_rows, 300)
    g._CAPI_LoadCSC(T(indptr), T(indices))
    w = torch.as_tensor(rng.random(indices.size).astype(np.float32) + 0.1, device=DEV)

    def slice_():
        return g._CAPI_ColRowSlicing(cols, rows, gs.format._CSC, gs.format._CSC | gs.format._COO)

    cols, rows = T(rng.permutation(300)[:200]), T(rng.permutation(num_rows)[:2500])
    sub, index = slice_()
    sub._CAPI_NormaliseColumns(w, index, None)            # (takes what the slice cleared)
    return slice_, w, sub._CAPI_NormaliseColumns(w, index, None)


def test_normalised_columns_on_another_stream_than_the_slice():
    """Sums that the slice's stream cleared are not used by another stream: their memory goes
    back to the first one, which may hand it out while the second still adds to it."""
    slice_, w, want = sliced_for_sums(np.random.default_rng(12))
    other = torch.cuda.Stream()
    busy = torch.rand(4096, 4096, device=DEV)
    for _ in range(3):
        sub, index = slice_()
        other.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(other):
            for _ in range(20):
                busy @ busy                               # the kernels below start after this
            got = sub._CAPI_NormaliseColumns(w, index, None)
        # what this stream gets of the size of the sums, written before they are made
        taken = [torch.full((200,), 1e30, dtype=torch.float64, device=DEV) for _ in range(64)]
        other.synchronize()
        assert torch.allclose(got, want, rtol=1e-6)
        assert all((t == 1e30).all() for t in taken)


def test_normalised_columns_recorded_behind_a_slice():
    """A graph that is recorded clears the sums itself: every replay has the eager result."""
    slice_, w, want = sliced_for_sums(np.random.default_rng(13))
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        sub, index = slice_()
        side.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            got = sub._CAPI_NormaliseColumns(w, index, None)
    torch.cuda.synchronize()
    for _ in range(4):
        got.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.allclose(got, want, rtol=1e-6)
        assert torch.allclose(sub._CAPI_NormaliseColumns(w, index, None), want, rtol=1e-6)


def test_offsets_for_the_host_while_another_thread_ages_the_caches():
    """Every load of a matrix ages what is kept of tensors' contents, from any thread, also
    between the launch of a kernel that reports to the host and the wait for its report:
    sizes, offsets and the flags of batches with repeated seeds stay what they are."""
    rng = np.random.default_rng(31)
    indptr, indices = random_csc(rng, 3000, 3000, 40)
    g = gs.Graph(3000, 3000)
    g._CAPI_LoadCSC(T(indptr), T(indices))
    seeds, ptr = T(rng.permutation(3000)[:96]), T(np.arange(0, 97, 8))
    seeds[0::16] = seeds[1::16]
    repeated = [True, False] * 6

    def step():
        gs.manual_seed(4)
        sub, _ = g._CAPI_BatchFusedSlicingSampling(seeds, ptr, 5, False)
        batch = sub._CAPI_BatchBlocks(seeds, torch.empty(0, dtype=torch.int64, device=DEV))
        parts = batch.blocks()
        assert [o is None for o in parts[2]] == repeated
        cut, index = g._CAPI_BatchColSlicing(seeds, ptr, True)
        return [*batch.offsets(), batch.row().tolist(), batch.frontier().tolist(),
                cut._CAPI_BatchGetRows()[1].tolist(), index.numel()]

    want, stop = step(), threading.Event()

    def age():
        while not stop.is_set():
            torch.ops.gs_ops._CAPI_InvalidateCaches()

    other = threading.Thread(target=age)
    other.start()
    try:
        for _ in range(100):
            assert step() == want
    finally:
        stop.set()
        other.join()


def columns_of(lengths, rng, num_rows):
    indptr = np.concatenate([[0], np.cumsum(lengths)])
    return indptr, rng.integers(0, num_rows, size=int(indptr[-1])).astype(np.int64)


@pytest.mark.parametrize("values", ["divided", "plain", None])
@pytest.mark.parametrize("shape", ["one long", "two", "some", "many", "past a run", "huge"])
def test_row_slice_that_is_only_handed_on(shape, values):
    """Labels, frontier and normalised values of a row slice that is not written are those of
    one that is: runs of edges in one column, in two, in up to 64 and in more, columns and
    rows that repeat.  Values, divisors and so the sums are exact: equal bit for bit."""
    rng = np.random.default_rng(len(shape))
    lengths = {"one long": [5000], "two": [0, 300, 0, 4100, 7], "some": rng.integers(0, 60, 400),
               "many": rng.integers(0, 9, 1700), "past a run": [3] * 5 + [0] * 90 + [2] * 400 + [20_000, 255, 257],
               "huge": rng.integers(0, 9000, 500)}[shape]
    indptr, indices = columns_of(lengths, rng, 3000)
    n, R = len(lengths), 200 if shape == "many" else 300
    if shape == "some":
        R = 100
    cols, rows = rng.permutation(n), rng.integers(0, 3100, size=R)
    if n > 20:
        cols[3], rows[7] = cols[9], rows[8]
    g = gs.Graph(3100, n)
    g._CAPI_LoadCSC(T(indptr), T(indices))
    w = torch.as_tensor(rng.integers(1, 9, size=indices.size).astype(np.float32), device=DEV)
    by = torch.as_tensor((2.0 ** rng.integers(-2, 3, size=R + 5)).astype(np.float32), device=DEV)
    cols, rows = T(cols), T(rows)
    e = w if values else None
    divisor = by if values == "divided" else None
    got = g._CAPI_RelabelledRows(cols, rows, e, divisor)
    sub, index = g._CAPI_ColRowSlicing(cols, rows, gs.format._CSC, gs.format._CSC | gs.format._COO)
    want = sub._CAPI_GraphRelabel(cols, rows)
    assert (got is None) == (shape == "many")  # more keys than one work-group takes
    if got is None:
        return
    for a, b in zip(got[:3], want):
        assert torch.equal(a, b)
    if values:
        assert torch.equal(got[3], sub._CAPI_NormaliseColumns(w, index, divisor))
    else:
        assert got[3] is None


def same_blocks(got, want):
    for part in ("frontier", "frontier_ptr", "row", "col", "indptr", "edge_ptr", "col_ptr"):
        assert torch.equal(getattr(got, part)(), getattr(want, part)()), part
    assert got.edge_ids() is None and want.edge_ids() is None and got.totals() == want.totals()


def batches_of(rng, num_ids, sizes):
    lists = [rng.choice(num_ids, size=k, replace=False) for k in sizes]
    return T(np.concatenate(lists)), T(np.concatenate([[0], np.cumsum(sizes)]))


@pytest.mark.parametrize("values", [True, False])
@pytest.mark.parametrize("seeds,picks", [([40], [90]), ([64, 0, 300, 1], [0, 90, 120, 60]), ([3] * 70, [5] * 70),
                                         ([1900, 20, 20, 20], [200, 9, 9, 9])])
def test_encoded_row_slice_that_is_only_handed_on(seeds, picks, values):
    rng = np.random.default_rng(len(seeds))
    indptr, indices = columns_of(rng.integers(0, 500, 2500), rng, 2500)
    g = gs.Graph(2500, 2500)
    g._CAPI_LoadCSC(T(indptr), T(indices))
    w = torch.as_tensor(rng.integers(1, 9, size=indices.size).astype(np.float32), device=DEV)
    refused = max(seeds) + max(picks) > 2048  # more keys in a batch than one work-group takes
    seeds, ptr = batches_of(rng, 2500, seeds)
    rows, rows_ptr, _ = g._CAPI_EncodedSquareSums(seeds, ptr, w)
    counts, starts = torch.diff(rows_ptr).tolist(), rows_ptr.tolist()
    chosen = [a + rng.choice(n, size=min(k, n), replace=False) for a, n, k in zip(starts, counts, picks)]
    row_ids, row_ptr = T(np.concatenate(chosen)), T(np.concatenate([[0], np.cumsum([len(c) for c in chosen])]))
    by = torch.as_tensor((2.0 ** rng.integers(-2, 3, size=row_ids.numel())).astype(np.float32), device=DEV)
    extra = (w, by) if values else (None, None)
    capi.profile_reset()
    capi.profile_enable(True)
    got = g._CAPI_EncodedBlocks(seeds, ptr, rows, row_ids, row_ptr, *extra)
    capi.profile_enable(False)
    launched = capi.profile_totals()
    assert (got is None) == refused
    if refused:
        assert not any(n.startswith(("member", "list")) for n in launched)  # before the slice is cut
        return
    assert "member_label" in launched
    sub, index, names = g._CAPI_EncodedPickedRows(seeds, ptr, rows, row_ids, row_ptr)
    same_blocks(got[0], sub._CAPI_BatchBlocks(seeds, names))
    assert torch.equal(got[1], sub._CAPI_NormaliseColumns(w, index, by)) if values else got[1] is None


@pytest.mark.parametrize("batches,picks", [(32, 64), (31, 65), (33, 61), (2, 900), (8, 255), (16, 65)])
def test_labels_of_batches_beside_the_offsets(batches, picks):
    """Parts of the first edges that are a batch's, or of two, or a batch's of many; one batch
    more than are labelled there.  Again and again on the same scratch memory."""
    uneven = [picks + (-1) ** b * min(b, 40) for b in range(batches)] if batches != 32 else [picks] * batches
    for _ in range(3):
        test_encoded_row_slice_that_is_only_handed_on([60] * batches, uneven, True)
    empty = [0] + [picks + picks // (batches - 1)] * (batches - 2) + [0]
    test_encoded_row_slice_that_is_only_handed_on([50] * batches, empty if batches > 2 else [0, picks], False)


@pytest.mark.parametrize("blocks", [False, True])
@pytest.mark.parametrize("square", [False, True])
def test_batches_whose_lists_have_ids_that_are_no_rows(square, blocks):
    """A matrix of fewer rows than columns: an id past its rows has no edges in any batch, in
    its own or in the one whose rows it would be taken for when moved by its batch."""
    rng = np.random.default_rng(6)
    num_rows, num_cols = 60, 100
    indptr, indices = columns_of(rng.integers(5, 40, num_cols), rng, num_rows)
    g = gs.Graph(num_rows, num_cols)
    g._CAPI_LoadCSC(T(indptr), T(indices))
    lists = [rng.permutation(num_cols)[:k] for k in (30, 0, 50, 41, 100, 7)]
    ptr = T(np.concatenate([[0], np.cumsum([len(x) for x in lists])]))
    nodes = T(np.concatenate(lists))
    rows = nodes if square else nodes.clone()
    if blocks and square:
        batch = g._CAPI_SubgraphBlocks(nodes, ptr)
    else:
        sub, _ = g._CAPI_BatchColRowSlcing(nodes, ptr, rows, ptr)
        batch = sub._CAPI_BatchBlocks(nodes, rows)
    frontier, fptr, eptr = (x().tolist() for x in (batch.frontier, batch.frontier_ptr, batch.edge_ptr))
    row, col = batch.row().cpu().numpy(), batch.col().cpu().numpy()
    for b, ids in enumerate(lists):
        assert frontier[fptr[b]:fptr[b + 1]] == ids.tolist()
        want = [(r, c) for c in ids for r in indices[indptr[c]:indptr[c + 1]] if r in ids]
        edges = slice(eptr[b], eptr[b + 1])
        assert [(ids[r], ids[c]) for r, c in zip(row[edges], col[edges])] == want


@pytest.mark.parametrize("sizes", [[40], [64, 0, 300, 1], [3] * 70, [3000, 20_000]])
def test_subgraphs_that_are_only_handed_on(sizes):
    rng = np.random.default_rng(len(sizes))
    indptr, indices = columns_of(rng.integers(0, 60, 30_000), rng, 30_000)
    g = gs.Graph(30_000, 30_000)
    g._CAPI_LoadCSC(T(indptr), T(indices))
    nodes, ptr = batches_of(rng, 30_000, sizes)
    nodes[1] = nodes[0]
    sub, _ = g._CAPI_BatchColRowSlcing(nodes, ptr, nodes, ptr)
    same_blocks(g._CAPI_SubgraphBlocks(nodes, ptr), sub._CAPI_BatchBlocks(nodes, nodes))


def test_row_slices_that_have_to_be_written():
    """No edge is kept, edge data of other types, too few edges for the pass, a parent with
    edge ids of its own; and edge data shorter than the edges."""
    rng = np.random.default_rng(8)
    indptr, indices = columns_of([2000, 3000], rng, 500)
    g = gs.Graph(900, 2)
    g._CAPI_LoadCSC(T(indptr), T(indices))
    cols, rows, w = T([1, 0]), T(rng.permutation(500)[:90]), torch.rand(5000, device=DEV)
    absent = T([600, 700])
    assert g._CAPI_RelabelledRows(cols, absent, w, None) is None
    frontier, row, col, _ = g._CAPI_RelabelledRows(cols, absent, None, None)
    assert torch.equal(frontier, cols) and row.numel() == col.numel() == 0
    assert g._CAPI_RelabelledRows(cols, rows, w.double(), None) is None
    assert g._CAPI_RelabelledRows(cols, rows, w[::2], None) is None
    assert g._CAPI_RelabelledRows(cols, rows, w, torch.ones(89, device=DEV)) is None
    assert g._CAPI_RelabelledRows(cols, T(rng.permutation(900)[:700]), w, None) is None
    assert g._CAPI_RelabelledRows(cols, rows, w, torch.ones(90, device=DEV)) is not None
    short = g._CAPI_RelabelledRows(cols, rows, w[:2500], None)[3]
    sub, index = g._CAPI_ColRowSlicing(cols, rows, gs.format._CSC, gs.format._CSC)
    assert torch.allclose(short, sub._CAPI_NormaliseColumns(w[:2500], index, None), rtol=1e-6)


def handed_on(A, seeds, k, also):
    sub = A[:, seeds]
    sub.edata["p"] = sub.edata["w"] ** 2
    prob = sub.sum("p", axis=1)
    picked, index = sub.collective_sampling(k, prob, False)
    picked = picked.div("w", prob[index], axis=1)
    picked = picked.div("w", picked.sum("w", axis=0), axis=0)
    block = picked.to_dgl_block(prefetch_edata={"w"})
    more = picked.sum("w", axis=1) if also == "sums" else index
    return picked.all_nodes(), block, more


@pytest.mark.parametrize("also", [None, "sums"])
def test_which_row_slices_are_only_handed_on(also):
    from gsampler_amd.ops.fused_op import _relabelled_rows
    rng = np.random.default_rng(21)
    indptr, indices = random_csc(rng, 500, 500, 300)
    m = gs.Matrix(gs.Graph(500, 500))
    m._graph._CAPI_LoadCSC(T(indptr), T(indices))
    m.edata["w"] = torch.as_tensor(rng.integers(1, 9, size=indices.size).astype(np.float32), device=DEV)

    def sampler(A, seeds):
        return handed_on(A, seeds, 30, also)

    seeds = T(rng.permutation(500)[:64])
    compiled = gs.jit.compile(func=sampler, args=(m, seeds))
    targets = [n.target for n in compiled._run.__self__.graph.nodes]
    assert targets.count(_relabelled_rows) == (also != "sums")
    results = []
    for run in (compiled, handed_on_by_operators(compiled)):
        gs.manual_seed(3)
        nodes, block, more = run(m, seeds)
        results.append([nodes, block.row, block.col, block.edata["w"], more])
    for a, b in zip(*results):
        assert torch.allclose(a.double(), b.double(), rtol=1e-6)


def test_offsets_asked_for_ahead():
    """Offsets of a slice whose size is on its way, by the thread that asked and by another,
    behind more requests than the host copies that are kept, and of columns changed since."""
    rng = np.random.default_rng(5)
    indptr, indices = columns_of(rng.integers(0, 200, 900), rng, 700)
    g = gs.Graph(700, 900)
    g._CAPI_LoadCSC(T(indptr), T(indices))
    rows = T(rng.permutation(700)[:64])
    lists = [T(rng.permutation(900)[:k]) for k in (1, 70, 500)]
    want = [g._CAPI_RelabelledRows(c, rows, None, None) for c in lists]

    def check(c, w):
        got = g._CAPI_RelabelledRows(c, rows, None, None)
        assert (got is None) == (w is None)
        assert w is None or all(torch.equal(a, b) for a, b in zip(got[:3], w[:3]))

    for c, w in zip(lists, want):
        g._CAPI_PrepareSlice(c)
        check(c, w)
        g._CAPI_PrepareSlice(c.clone())
        g._CAPI_PrepareSlice(c)
        for _ in range(70):
            g._CAPI_ColRowSlicing(rows, rows, gs.format._CSC, gs.format._CSC)
            other = gs.Graph(700, 900)
            other._CAPI_LoadCSC(T(indptr), T(indices))
            other._CAPI_PrepareSlice(c)
        g._CAPI_PrepareSlice(c)
        thread = threading.Thread(target=lambda: check(c, w))
        thread.start()
        thread.join()
        check(c, w)
    c = lists[1].clone()
    g._CAPI_PrepareSlice(c)
    c.copy_(lists[1].flip(0))
    check(c, g._CAPI_RelabelledRows(lists[1].flip(0), rows, None, None))
    for wrong in (c.int(), c.cpu(), c[::2], c[:0]):
        g._CAPI_PrepareSlice(wrong)  # (left to the operator that slices)


def test_which_slices_ask_for_their_offsets_ahead():
    rng = np.random.default_rng(6)
    indptr, indices = random_csc(rng, 500, 500, 200)
    m = gs.Matrix(gs.Graph(500, 500))
    m._graph._CAPI_LoadCSC(T(indptr), T(indices))
    prob = torch.rand(500, device=DEV)

    def sampler(A, seeds, prob):
        blocks = []
        for _ in range(2):
            sub, _ = A[:, seeds].collective_sampling(40, prob, False)
            seeds = sub.all_nodes()
            blocks.append(sub.to_dgl_block())
        return seeds, blocks

    seeds = T(rng.permutation(500)[:32])
    compiled = gs.jit.compile(func=sampler, args=(m, seeds, prob))
    assert [n.target for n in compiled._run.__self__.graph.nodes].count("_CAPI_PrepareSlice") == 2
    outs = []
    for run in (compiled, handed_on_by_operators(compiled)):
        gs.manual_seed(3)
        nodes, blocks = run(m, seeds, prob)
        outs.append([nodes] + [t for b in blocks for t in (b.row, b.col, b.srcdata["_ID"])])
    assert all(torch.equal(a, b) for a, b in zip(*outs))


@pytest.mark.parametrize("also", [None, "sums"])
def test_which_slices_of_batches_are_only_handed_on(also):
    from gsampler_amd.ops.fused_op import _encoded_blocks, _subgraph_blocks
    rng = np.random.default_rng(22)
    indptr, indices = random_csc(rng, 500, 500, 300)
    bm, m = gs.BatchMatrix(), gs.Matrix(gs.Graph(500, 500))
    m._graph._CAPI_LoadCSC(T(indptr), T(indices))
    m.edata["w"] = torch.as_tensor(rng.integers(1, 9, size=indices.size).astype(np.float32), device=DEV)

    def layers(A, seeds, ptr):
        sub = A[:, seeds::ptr]
        sub.edata["p"] = sub.edata["w"] ** 2
        prob = sub.sum("p", axis=1)
        _, rows_ptr = sub.all_rows()
        picked, index = sub.collective_sampling(30, prob, rows_ptr, False)
        picked = picked.div("w", prob[index], axis=1)
        picked = picked.div("w", picked.sum("w", axis=0), axis=0)
        nodes, ptr = picked.all_nodes()
        return nodes, picked.to_dgl_block(prefetch_edata={"w"}), picked.sum("w", axis=1) if also else index

    def subgraphs(A, nodes, ptr):
        sub = A[nodes::ptr, nodes::ptr]
        return sub.to_dgl_block(), sub.all_nodes()[0], sub.sum("w", axis=1) if also else ptr

    def flat(out):
        tensors = [t for t in out if isinstance(t, torch.Tensor)]
        for blocks in (b for b in out if not isinstance(b, torch.Tensor)):
            tensors += [t for b in blocks for t in (b.row, b.col, b.srcdata["_ID"], *b.edata.values())]
        return tensors

    for func, encoded, target in ((layers, True, _encoded_blocks), (subgraphs, False, _subgraph_blocks)):
        bm.load_from_matrix(m, encoded)
        args = (bm, *batches_of(rng, 500, [40, 0, 64]))
        compiled = gs.jit.compile(func=func, args=args)
        targets = [n.target for n in compiled._run.__self__.graph.nodes]
        assert targets.count(target) == (also is None), func.__name__
        results = []
        for run in (compiled, handed_on_by_operators(compiled)):
            gs.manual_seed(3)
            results.append(flat(run(*args)))
        for a, b in zip(*results):
            assert torch.allclose(a.double(), b.double(), rtol=1e-6)


def handed_on_by_operators(compiled):
    import copy
    other = copy.copy(compiled)
    other._run = None  # the operator graph itself
    return other


@pytest.mark.parametrize("lengths,picks", [([4_000_000], 300), ([4_000_000, 0, 700_001], 2048), ([1, 300, 0, 513, 2000, 90], 300),
                                           ([4_000_000, 3], 4000), ([700, 0, 255, 40], 4000)])
@pytest.mark.parametrize("narrow", [False, True])
def test_row_slices_whose_work_groups_look_up_their_runs_in_several_rounds(lengths, picks, narrow):
    """More than 67 M edges between picked columns that repeat: of a few long columns and of
    many that meet in a run, with the table in LDS and in L2, by ids of both widths."""
    g = torch.Generator(device=DEV).manual_seed(picks + len(lengths))
    deg = torch.tensor(lengths, device=DEV)
    indptr = torch.zeros(deg.numel() + 1, dtype=torch.int64, device=DEV)
    torch.cumsum(deg, 0, out=indptr[1:])
    indices = torch.randint(0, 100_000, (int(indptr[-1]),), generator=g, device=DEV)
    rows = torch.randint(0, 100_000, (picks,), generator=g, device=DEV)
    cols = torch.arange(len(lengths), device=DEV).repeat(70_000_000 // int(indptr[-1]) + 1)
    got = capi.col_row_slice(indptr, indices, cols, rows, with_major=False,
                             indices32=indices.to(torch.int32) if narrow else None)
    place = torch.full((100_000,), picks, dtype=torch.int64, device=DEV)
    place.scatter_reduce_(0, rows, torch.arange(picks, device=DEV), "amin")
    kept = torch.nonzero(place[indices] < picks).flatten()
    kept_ptr = torch.searchsorted(kept, indptr)
    count = (kept_ptr[1:] - kept_ptr[:-1])[cols]
    want_ptr = torch.zeros(cols.numel() + 1, dtype=torch.int64, device=DEV)
    torch.cumsum(count, 0, out=want_ptr[1:])
    assert torch.equal(got[0], want_ptr)
    select = kept[torch.arange(int(want_ptr[-1]), device=DEV)
                  + torch.repeat_interleave(kept_ptr[cols] - want_ptr[:-1], count)]
    assert torch.equal(got[3], select)
    assert torch.equal(got[2], place[indices[select]])


@pytest.mark.parametrize("R", [1, 63, 64, 65, 512, 1500, 2000])
@pytest.mark.parametrize("edges", [20_000, 700_000, 9_000_000])
def test_labels_beside_the_offsets(R, edges):
    """One part of the first edges and up to 32, of few and of all work-groups' lists, told by
    the last that ends; again and again on the same scratch memory."""
    rng = np.random.default_rng(R + edges)
    indptr, indices = columns_of(rng.multinomial(edges, np.ones(30) / 30), rng, 3000)
    g = gs.Graph(3100, 30)
    g._CAPI_LoadCSC(T(indptr), T(indices))
    for _ in range(5):
        cols, rows = T(rng.permutation(30)), T(rng.integers(0, 3100, size=R))
        got = g._CAPI_RelabelledRows(cols, rows, None, None)
        sub, _ = g._CAPI_ColRowSlicing(cols, rows, gs.format._CSC, gs.format._CSC | gs.format._COO)
        assert (got is None) == (edges < 8 * (R + 30))
        for a, b in zip(got[:3] if got else (), sub._CAPI_GraphRelabel(cols, rows)):
            assert torch.equal(a, b)


def test_labels_of_the_longest_slices():
    """More chunks of edges than have their offsets in one launch: labels, first edges and
    offsets in launches of their own.  (Values and so their sums are exact.)"""
    rng = np.random.default_rng(12)
    indptr, indices = columns_of(rng.integers(50_000, 150_000, 20), rng, 30_000)
    g = gs.Graph(30_000, 20)
    g._CAPI_LoadCSC(T(indptr), T(indices))
    w = torch.as_tensor(rng.integers(1, 9, size=indices.size).astype(np.float32), device=DEV)
    cols = T(np.concatenate([rng.permutation(20) for _ in range(34_000_000 // indices.size + 1)]))
    rows = T(rng.integers(0, 30_000, size=100))
    by = torch.as_tensor((2.0 ** rng.integers(-2, 3, size=100)).astype(np.float32), device=DEV)
    capi.profile_reset()
    capi.profile_enable(True)
    got = g._CAPI_RelabelledRows(cols, rows, w, by)
    capi.profile_enable(False)
    assert "member_first" in capi.profile_totals() and "list_labels" in capi.profile_totals()
    sub, index = g._CAPI_ColRowSlicing(cols, rows, gs.format._CSC, gs.format._CSC | gs.format._COO)
    for a, b in zip(got[:3], sub._CAPI_GraphRelabel(cols, rows)):
        assert torch.equal(a, b)
    assert torch.equal(got[3], sub._CAPI_NormaliseColumns(w, index, by))


def test_labels_of_batches_of_the_longest_slices():
    rng = np.random.default_rng(13)
    indptr, indices = columns_of(rng.integers(10_000, 15_000, 2500), rng, 2500)
    g = gs.Graph(2500, 2500)
    g._CAPI_LoadCSC(T(indptr), T(indices))
    w = torch.as_tensor(rng.integers(1, 9, size=indices.size).astype(np.float32), device=DEV)
    seeds, ptr = batches_of(rng, 2500, [250] * 12)
    rows, rows_ptr, _ = g._CAPI_EncodedSquareSums(seeds, ptr, w)
    counts, starts = torch.diff(rows_ptr).tolist(), rows_ptr.tolist()
    row_ids = T(np.concatenate([a + rng.choice(n, size=70, replace=False) for a, n in zip(starts, counts)]))
    row_ptr = torch.arange(13, device=DEV) * 70
    by = torch.as_tensor((2.0 ** rng.integers(-2, 3, size=row_ids.numel())).astype(np.float32), device=DEV)
    capi.profile_reset()
    capi.profile_enable(True)
    got = g._CAPI_EncodedBlocks(seeds, ptr, rows, row_ids, row_ptr, w, by)
    capi.profile_enable(False)
    assert "member_first" in capi.profile_totals() and "list_labels" in capi.profile_totals()
    sub, index, names = g._CAPI_EncodedPickedRows(seeds, ptr, rows, row_ids, row_ptr)
    same_blocks(got[0], sub._CAPI_BatchBlocks(seeds, names))
    assert torch.equal(got[1], sub._CAPI_NormaliseColumns(w, index, by))
