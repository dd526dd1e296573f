"""Tables that a matrix keeps (the int32 copy of its ids, the hop table of its walks) when
two streams share it, and when a walk is recorded into a graph."""
import numpy as np
import pytest
import torch

import gsampler_amd as gs
from oracle import binding as orc
from tests.conftest import random_csc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
NODES, P, Q = 200_000, 2.0, 0.5


@pytest.fixture(scope="module")
def arrays():
    indptr, indices = random_csc(np.random.default_rng(3), NODES, NODES, 16, empty_frac=0.05)
    assert 1 << 20 < indices.size < 1 << 24          # both tables are made
    for c in range(NODES):
        indices[indptr[c]:indptr[c + 1]].sort()
    return indptr, indices


def matrix(arrays):
    m = gs.Matrix(gs.Graph(NODES, NODES))
    m._graph._CAPI_LoadCSC(*(torch.from_numpy(a).to(DEV) for a in arrays))
    m._graph._CAPI_SortCSCIndices()
    torch.cuda.synchronize()
    return m


def traces(walk, n):
    return walk.reshape(-1, n).cpu().numpy()


@pytest.mark.parametrize("first_calls", [1, 2])      # the first makes the ids, the second the hops
def test_second_stream_waits_for_the_tables(arrays, first_calls):
    rng = np.random.default_rng(first_calls)
    n, length = 20_000, 6
    seeds = rng.integers(0, NODES, n)
    want = orc.node2vec(*arrays, seeds, length, P, Q, 5, 0).reshape(length + 1, n)
    m, d = matrix(arrays), torch.from_numpy(seeds).to(DEV)
    noise = torch.rand(1 << 26, device=DEV)
    torch.cuda.synchronize()
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.cuda.stream(a):
        noise.sort()                                 # the tables are queued behind this
        for _ in range(first_calls):
            gs.manual_seed(5)
            m.node2vec(d, length, P, Q)
    with torch.cuda.stream(b):
        for _ in range(3):
            gs.manual_seed(5)
            got = m.node2vec(d, length, P, Q)
            assert np.array_equal(traces(got, n), want)
    torch.cuda.synchronize()


def test_tables_outlive_their_matrix_on_another_stream(arrays):
    n, length = 20_000, 6
    seeds = np.random.default_rng(9).integers(0, NODES, n)
    want = orc.node2vec(*arrays, seeds, length, P, Q, 5, 0).reshape(length + 1, n)
    m, d = matrix(arrays), torch.from_numpy(seeds).to(DEV)
    noise = torch.rand(1 << 26, device=DEV)
    gs.manual_seed(5)
    m.node2vec(d, length, P, Q)                      # made on the default stream
    bytes_of_ids = 4 * arrays[1].size
    b = torch.cuda.Stream()
    b.wait_stream(torch.cuda.current_stream())
    keep = m.csc
    with torch.cuda.stream(b):
        noise.sort()
        gs.manual_seed(5)
        got = m.node2vec(d, length, P, Q)
    del m                                            # `keep` holds the arrays of the caller
    other = [torch.zeros(bytes_of_ids, dtype=torch.uint8, device=DEV) for _ in range(8)]
    torch.cuda.synchronize()
    assert np.array_equal(traces(got, n), want)
    del other, keep


@pytest.mark.parametrize("calls_before", [0, 1, 2])
def test_walks_recorded_into_a_graph(arrays, calls_before):
    n, length = 3000, 9
    seeds = np.random.default_rng(calls_before).integers(0, NODES, n)
    want_walk = orc.random_walk(*arrays, seeds, length, 13, 0).reshape(length + 1, n)
    want_n2v = orc.node2vec(*arrays, seeds, length, P, Q, 13, 1).reshape(length + 1, n)
    m, d = matrix(arrays), torch.from_numpy(seeds).to(DEV)

    def both():
        gs.manual_seed(13)
        return m.random_walk(d, length), m.node2vec(d, length, P, Q)

    for _ in range(calls_before):
        both()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        walk, n2v = both()
    for _ in range(3):                               # replays with eager calls in between
        walk.zero_(), n2v.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(traces(walk, n), want_walk)
        assert np.array_equal(traces(n2v, n), want_n2v)
        e_walk, e_n2v = both()
        assert np.array_equal(traces(e_walk, n), want_walk)
        assert np.array_equal(traces(e_n2v, n), want_n2v)
    torch.ops.gs_ops._CAPI_InvalidateCaches()        # frees what the matrix keeps
    other = torch.zeros(64 << 20, dtype=torch.uint8, device=DEV)
    graph.replay()
    torch.cuda.synchronize()
    assert np.array_equal(traces(walk, n), want_walk) and np.array_equal(traces(n2v, n), want_n2v)
    del other


def test_second_stream_waits_for_the_weights_cdf(arrays):
    weights = torch.rand(arrays[1].size, device=DEV) + 0.01
    seeds = torch.from_numpy(np.random.default_rng(4).permutation(NODES)[:5000]).to(DEV)

    def sample(m):
        gs.manual_seed(5)
        sub, index = m._graph._CAPI_SlicingSamplingProbs(1, seeds, weights, 7, False, gs.format._CSC,
                                                         gs.format._CSC)
        return sub._CAPI_GetCSCIndptr(), sub._CAPI_GetCSCIndices(), index

    want = sample(matrix(arrays))
    m = matrix(arrays)
    noise = torch.rand(1 << 26, device=DEV)
    torch.cuda.synchronize()
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.cuda.stream(a):
        noise.sort()                                 # the CDF is queued behind this
        m._graph._CAPI_SlicingSamplingProbs(1, seeds[:0], weights, 7, False, gs.format._CSC,
                                            gs.format._CSC)
    with torch.cuda.stream(b):
        for _ in range(2):
            for got, expected in zip(sample(m), want):
                assert torch.equal(got, expected)
    torch.cuda.synchronize()


def test_tables_can_be_switched_off(arrays):
    n = 1000
    seeds = torch.from_numpy(np.random.default_rng(2).integers(0, NODES, n)).to(DEV)
    want = orc.random_walk(*arrays, seeds.cpu().numpy(), 20, 13, 0).reshape(21, n)
    m = matrix(arrays)
    before = torch.cuda.memory_allocated()
    for _ in range(3):
        gs.manual_seed(13)
        assert np.array_equal(traces(m.random_walk(seeds, 20), n), want)
    assert torch.cuda.memory_allocated() - before >= 8 * arrays[1].size
    try:
        torch.ops.gs_ops._CAPI_SetNarrowIds(False)
        for _ in range(3):
            gs.manual_seed(13)
            assert np.array_equal(traces(m.random_walk(seeds, 20), n), want)
        assert torch.cuda.memory_allocated() == before
    finally:
        torch.ops.gs_ops._CAPI_SetNarrowIds(True)
