"""Walks by groups of lanes and over the hop table against the CPU oracle: call sizes on both
sides of every choice of group size, walk lengths that are no multiple of a group or of the
steps held in registers, dead ends, columns of one edge."""
import numpy as np
import pytest
import torch

import gsampler_amd as gs
from oracle import binding as orc
from tests.conftest import random_csc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def world():
    rng = np.random.default_rng(7)
    nodes = 4000
    indptr, indices = random_csc(rng, nodes, nodes, 9, empty_frac=0.02, hub_deg=70000)
    m = gs.Matrix(gs.Graph(nodes, nodes))
    m._graph._CAPI_LoadCSC(torch.from_numpy(indptr).to(DEV), torch.from_numpy(indices).to(DEV))
    m._graph._CAPI_SortCSCIndices()
    return rng, nodes, indptr, m.csc[1].cpu().numpy(), m


def traces(walk, n):
    return walk.reshape(-1, n).cpu().numpy()


# 16, 8, 4, 2 and 1 lanes a walk where candidates are often accepted; twice as many walks where not
@pytest.mark.parametrize("n,length,p,q", [
    (1, 1, 2.0, 0.5), (333, 7, 2.0, 0.5), (12501, 17, 2.0, 0.5), (25001, 9, 2.0, 0.5),
    (50001, 6, 2.0, 0.5), (100001, 5, 2.0, 0.5), (200001, 4, 2.0, 0.5),
    (1000, 33, 0.25, 4.0), (25000, 5, 0.25, 4.0), (32769, 5, 0.25, 4.0), (150000, 4, 0.5, 4.0),
])
def test_node2vec(world, n, length, p, q):
    rng, nodes, indptr, indices, m = world
    seeds = rng.integers(-1, nodes + 1, n)
    want = orc.node2vec(indptr, indices, seeds, length, p, q, 11, 0)
    d = torch.from_numpy(seeds).to(DEV)
    for _ in range(3):                       # without the hop table, then with it
        gs.manual_seed(11)
        got = traces(m.node2vec(d, length, p, q), n)
        assert np.array_equal(got, want.reshape(length + 1, n))


@pytest.mark.parametrize("n,length", [(1, 80), (65, 8), (1000, 9), (32768, 3), (32769, 3), (70000, 17)])
def test_random_walk(world, n, length):
    rng, nodes, indptr, indices, m = world
    seeds = rng.integers(-1, nodes + 1, n)
    want = orc.random_walk(indptr, indices, seeds, length, 13, 0)
    d = torch.from_numpy(seeds).to(DEV)
    for _ in range(3):
        gs.manual_seed(13)
        assert np.array_equal(traces(m.random_walk(d, length), n), want.reshape(length + 1, n))
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):            # a stream that did not make the table
        gs.manual_seed(13)
        assert np.array_equal(traces(m.random_walk(d, length), n), want.reshape(length + 1, n))


# From 2^20 edges on a walk reads the int32 copy of the ids: the same group sizes, below and
# above 2^15 walks (with and without the hop table, which a matrix up to 2^24 edges keeps).
@pytest.fixture(scope="module")
def wide_world():
    rng = np.random.default_rng(8)
    nodes = 130_000
    indptr, indices = random_csc(rng, nodes, nodes, 17, empty_frac=0.02, hub_deg=70000)
    assert 1 << 20 <= indices.size <= 1 << 24
    m = gs.Matrix(gs.Graph(nodes, nodes))
    m._graph._CAPI_LoadCSC(torch.from_numpy(indptr).to(DEV), torch.from_numpy(indices).to(DEV))
    m._graph._CAPI_SortCSCIndices()
    return rng, nodes, indptr, m.csc[1].cpu().numpy(), m


@pytest.mark.parametrize("n,length,p,q", [
    (333, 18, 2.0, 0.5), (12501, 17, 2.0, 0.5), (25001, 9, 2.0, 0.5), (50001, 6, 2.0, 0.5),
    (100001, 5, 2.0, 0.5), (200001, 4, 2.0, 0.5), (25000, 5, 0.25, 4.0), (32769, 5, 0.25, 4.0),
    (200001, 4, 1.0, 1.0),
])
def test_node2vec_on_int32_ids(wide_world, n, length, p, q):
    test_node2vec(wide_world, n, length, p, q)


@pytest.mark.parametrize("n,length", [(1000, 17), (32768, 9), (40000, 8)])
def test_random_walk_on_a_wide_matrix(wide_world, n, length):
    test_random_walk(wide_world, n, length)


@pytest.mark.parametrize("n,p,q,makes", [
    (16384, None, None, True), (16385, None, None, False),            # first order
    (2048, 2.0, 0.5, True), (2049, 2.0, 0.5, False), (8193, 0.25, 4.0, False),
])
def test_hop_table_is_made_for_calls_that_use_it_only(world, n, p, q, makes):
    _, nodes, indptr, indices, _ = world
    m = gs.Matrix(gs.Graph(nodes, nodes))
    m._graph._CAPI_LoadCSC(torch.from_numpy(indptr).to(DEV), torch.from_numpy(indices).to(DEV))
    m._graph._CAPI_SortCSCIndices()
    seeds = torch.arange(n, device=DEV) % nodes
    before = torch.cuda.memory_allocated()
    for _ in range(3):
        m.random_walk(seeds, 3) if p is None else m.node2vec(seeds, 3, p, q)
    grown = torch.cuda.memory_allocated() - before
    assert (grown >= 8 * indices.size) == makes and (makes or grown == 0)


# max(p, q) <= 1: one lane a walk takes its first candidate, by 64-bit ids below 2^16 walks
@pytest.mark.parametrize("n,length,p,q", [(1, 9, 0.5, 0.25), (2000, 17, 1.0, 0.5), (30000, 9, 0.25, 0.25),
                                          (65535, 5, 1.0, 1.0), (65536, 5, 1.0, 1.0), (65536, 5, 0.5, 1.0)])
def test_node2vec_whose_first_candidates_stand(world, wide_world, n, length, p, q):
    test_node2vec(world, n, length, p, q)
    test_node2vec(wide_world, n, length, p, q)


def test_int32_copy_is_made_once_enough_ids_were_read(wide_world):
    _, nodes, indptr, indices, _ = wide_world
    m = gs.Matrix(gs.Graph(nodes, nodes))
    m._graph._CAPI_LoadCSC(torch.from_numpy(indptr).to(DEV), torch.from_numpy(indices).to(DEV))
    m._graph._CAPI_SortCSCIndices()
    seeds = torch.arange(20_000, device=DEV) % nodes
    want = torch.from_numpy(orc.node2vec(indptr, indices, seeds.cpu().numpy(), 10, 2.0, 0.5, 3, 0))
    grown = []
    for _ in range(indices.size // 200_000 + 2):
        before = torch.cuda.memory_allocated()
        gs.manual_seed(3)
        got = m.node2vec(seeds, 10, 2.0, 0.5).reshape(11, -1).cpu()
        assert torch.equal(got, want.reshape(11, -1))
        del got
        grown.append(torch.cuda.memory_allocated() - before)
    made = [i for i, g in enumerate(grown) if g > 0]
    assert made == [-(-indices.size // 200_000) - 1] and grown[made[0]] >= 4 * indices.size


# Calls of one lane a walk go by marks of the columns once they have walked enough steps: returns
# to the previous node (every node's neighbours are near it), ids that repeat in a column, columns
# of 0 to 8 edges, a hub, and a column too long for its marks; one walk more than the border.
@pytest.fixture(scope="module")
def near_world():
    rng = np.random.default_rng(9)
    nodes, hub = 200_000, (1 << 24) + 5
    deg = rng.integers(0, 9, size=nodes)
    deg[1000], deg[2000] = 60_000, hub
    indptr = np.concatenate([[0], np.cumsum(deg)])
    col = np.repeat(np.arange(nodes), deg)
    indices = (col + rng.integers(-3, 4, size=col.size)) % nodes
    wide = (col == 1000) | (col == 2000)
    indices[wide] = rng.integers(0, nodes, size=int(wide.sum()))
    indices[rng.random(indices.size) < 0.002] = 2000
    indices[rng.random(indices.size) < 0.002] = 1000
    m = gs.Matrix(gs.Graph(nodes, nodes))
    m._graph._CAPI_LoadCSC(torch.from_numpy(indptr).to(DEV), torch.from_numpy(indices).to(DEV))
    m._graph._CAPI_SortCSCIndices()
    return rng, nodes, indptr, m.csc[1].cpu().numpy(), m


@pytest.mark.parametrize("n,length,p,q", [
    (100001, 9, 2.0, 0.5), (200001, 5, 4.0, 0.25), (200001, 4, 8.0, 1.0), (200001, 4, 0.5, 2.0),
    (200001, 4, 0.25, 4.0), (200001, 4, 4.0, 2.0), (100001, 9, 1.5, 0.5), (200002, 3, 1e9, 1e-9),
])
def test_node2vec_by_marks(near_world, n, length, p, q):
    test_node2vec(near_world, n, length, p, q)


def test_marks_are_made_once_enough_steps_were_walked(near_world):
    _, nodes, indptr, indices, _ = near_world
    m = gs.Matrix(gs.Graph(nodes, nodes))
    m._graph._CAPI_LoadCSC(torch.from_numpy(indptr).to(DEV), torch.from_numpy(indices).to(DEV))
    m._graph._CAPI_SortCSCIndices()
    seeds = torch.arange(100_001, device=DEV) % nodes
    grown = []
    for n in (100_000, 100_001, 100_001, 100_001, 100_001):
        before = torch.cuda.memory_allocated()
        m.node2vec(seeds[:n], 3, 2.0, 0.5)
        grown.append(torch.cuda.memory_allocated() - before)
    assert grown[:3] == [0, 0, 0] and grown[3] >= 32 * nodes and grown[4] == 0
