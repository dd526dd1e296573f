"""All layers of a node-wise sampler in one call (small layers: three launches each, queued
without waits) against the layers operator by operator, at sizes where the short path begins,
ends or has remainders."""
import gc
import threading

import numpy as np
import pytest
import torch

import gsampler_amd as gs
from gsampler_amd import capi
from gsampler_amd.utils.block import Block, BlockList
from tests.conftest import random_csc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def single(A, seeds, fanouts, replace):
    out = []
    for k in fanouts:
        sub = A[:, seeds]
        sub = sub.individual_sampling(k, sub.edata["w"] if "w" in A.edata else None, replace)
        seeds = sub.all_nodes()
        out.append(sub.to_dgl_block())
    return seeds, out


def batched(A, seeds, ptr, fanouts, replace):
    out = []
    for k in fanouts:
        sub = A[:, seeds::ptr]
        sub = sub.individual_sampling(k, sub.edata["w"] if "w" in A.edata else None, replace)
        seeds, ptr = sub.all_nodes()
        out.append(sub.to_dgl_block())
    return out


def both(func, m, args, layers):
    compiled = gs.jit.compile(func=func, args=(m, *args))
    called = [str(n.target) for n in compiled._run.__self__.graph.nodes]
    assert sum("sample_layers" in t for t in called) == 1 and "_CAPI_GraphRelabel" not in called
    gs.manual_seed(5)
    got = compiled(m, *args)
    assert gs.random_state() == (5, layers)
    gs.manual_seed(5)
    graph, data = [m._graph], [[m.row_ndata, m.col_ndata, m.edata]]
    run_time = tuple(a if isinstance(a, torch.Tensor) else None for a in (None, *args))
    return got, compiled.gm(run_time, graph, data)


def same(a, b):
    assert a.num_src == b.num_src and a.num_dst == b.num_dst
    assert torch.equal(a.row, b.row) and torch.equal(a.col, b.col)
    assert torch.equal(a.srcdata["_ID"], b.srcdata["_ID"])
    for x, y in zip(a.csc(), b.csc()):
        assert (x is None) == (y is None) and (x is None or torch.equal(x, y))


def matrix(rng, nodes, max_deg, hub, weighted):
    indptr, indices = random_csc(rng, nodes, nodes, max_deg, hub_deg=hub)
    indices[rng.random(indices.size) < 0.2] = nodes // 3        # a hub on the other side
    m = gs.Matrix(gs.Graph(nodes, nodes))
    m._graph._CAPI_LoadCSC(torch.from_numpy(indptr).to(DEV), torch.from_numpy(indices).to(DEV))
    if weighted:
        m.edata["w"] = torch.from_numpy(rng.random(indices.size).astype(np.float32)).to(DEV)
    return m


@pytest.mark.parametrize("nodes,count,fanouts,replace,weighted", [
    (50, 1, [1], False, False),
    (3000, 73, [15, 10, 5], False, False),       # queued layers
    (3000, 1024, [63], True, False),             # the widest column of the short path
    (3000, 200, [64, 3], False, False),          # one fanout too many for it, then short again
    (9000, 5000, [31, 31], False, False),        # second layer above the bound of queued layers
    (40000, 33000, [40, 2], False, False),       # first layer above the bound of short ones
    (3000, 65, [10, 5], False, True),
    (3000, 300, [7, 7], True, True),
])
def test_one_batch(rng, nodes, count, fanouts, replace, weighted):
    m = matrix(rng, nodes, 60, 2500, weighted)
    seeds = torch.from_numpy(rng.integers(0, nodes, count)).to(DEV)      # some repeat
    (n0, b0), (n1, b1) = both(single, m, (seeds, fanouts, replace), len(fanouts))
    assert torch.equal(n0, n1) and len(b0) == len(b1) == len(fanouts)
    for x, y in zip(b0, b1):
        same(x, y)


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("count", [7, 0])
def test_large_layer_of_a_matrix_without_edges(count, weighted):
    m = gs.Matrix(gs.Graph(50, 50))
    m._graph._CAPI_LoadCSC(torch.zeros(51, dtype=torch.int64, device=DEV),
                           torch.zeros(0, dtype=torch.int64, device=DEV))
    if weighted:
        m.edata["w"] = torch.zeros(0, device=DEV)
    seeds = torch.arange(count, device=DEV) * 3
    nodes, blocks = both(single, m, (seeds, [64], False), 1)[0]
    assert torch.equal(nodes, seeds)
    assert blocks[0].row.numel() == 0 and blocks[0].num_dst == count


@pytest.mark.parametrize("cuts,fanouts,replace,weighted", [
    ([0, 64], [5], False, False),
    ([0, 0, 7, 7, 1000, 1001], [15, 10, 5], False, False),       # empty batches, one of one seed
    ([0, 300, 300, 512], [4, 4], True, False),
    (list(range(0, 6001, 60)), [15, 10], False, False),          # second layer large
    ([0, 100, 250], [10, 5], False, True),
])
def test_super_batch(rng, cuts, fanouts, replace, weighted):
    nodes = 7000
    bm = gs.BatchMatrix()
    bm.load_from_matrix(matrix(rng, nodes, 40, 3000, weighted), False)
    seeds = torch.cat([torch.from_numpy(rng.permutation(nodes)[:hi - lo])
                       for lo, hi in zip(cuts, cuts[1:])])
    if len(cuts) == 4:
        seeds[3] = seeds[0]                                      # a batch whose seeds repeat
    ptr = torch.tensor(cuts, device=DEV)
    got, want = both(batched, bm, (seeds.to(DEV), ptr, fanouts, replace), len(fanouts))
    for layer, other in zip(got, want):
        assert layer.totals() == other.totals() and len(layer) == len(other) == len(cuts) - 1
        for name in ("frontier", "frontier_ptr", "row", "col", "edge_ptr", "indptr", "col_ptr"):
            assert torch.equal(getattr(layer.batch, name)(), getattr(other.batch, name)()), name
        for x, y in zip(layer, other):
            same(x, y)


@pytest.mark.parametrize("batches", [1, 511, 512])
@pytest.mark.parametrize("replace", [False, True])
def test_chains_of_short_layers_around_the_most_batches(rng, batches, replace):
    """Picks beside the labels of the layer before, for as many batches as they find the
    offsets of, and one more (a launch each): three layers, batches that are empty, that
    repeat one seed, whose seeds have no neighbours, and tiles without a new key."""
    nodes = 4000
    indptr, indices = random_csc(rng, nodes, nodes, 9, hub_deg=0)
    degree = np.diff(indptr)
    m = gs.Matrix(gs.Graph(nodes, nodes))
    m._graph._CAPI_LoadCSC(torch.from_numpy(indptr).to(DEV), torch.from_numpy(indices).to(DEV))
    bm = gs.BatchMatrix()
    bm.load_from_matrix(m, False)
    sizes = rng.integers(0, 6, size=batches)
    sizes[-1] = 2100                                   # two tiles of one repeated seed
    cuts = np.concatenate([[0], np.cumsum(sizes)])
    seeds = rng.integers(0, nodes, size=cuts[-1])
    seeds[cuts[-2]:] = seeds[-1]
    if (degree == 0).any():
        seeds[:3] = np.nonzero(degree == 0)[0][0]
    args = (torch.from_numpy(seeds).to(DEV), torch.from_numpy(cuts).to(DEV), [5, 3, 4], replace)
    got, want = both(batched, bm, args, 3)
    for layer, other in zip(got, want):
        for name in ("frontier", "frontier_ptr", "row", "col", "edge_ptr", "indptr", "col_ptr"):
            assert torch.equal(getattr(layer.batch, name)(), getattr(other.batch, name)()), name


@pytest.mark.parametrize("batches", [2, 62, 63, 64, 65])
def test_chains_of_short_layers_around_a_wavefront_of_batches(rng, batches):
    """As many batches as have their offsets held by the lanes of a wavefront, and more."""
    test_chains_of_short_layers_around_the_most_batches(rng, batches, False)


@pytest.mark.parametrize("cuts,fanouts,replace,weighted", [
    ([0, 8], [3, 2], False, False),
    ([0, 0, 30, 30, 64], [10, 5], False, False),         # batches without seeds
    ([0, 500, 1100], [8, 4], True, True),
    ([0, 9000, 33000], [40, 2], False, False),           # a large layer, then a short bound
    ([0, 300, 700], [64, 3], False, True),
])
def test_nodes_of_a_super_batch(rng, cuts, fanouts, replace, weighted):
    """Layers of which the sampler asks the nodes alone, and the induced subgraph behind
    them."""
    m = matrix(rng, 40000 if cuts[-1] > 5000 else 3000, 40, 700, weighted)
    bm = gs.BatchMatrix()
    bm.load_from_matrix(m, False)
    seeds = torch.from_numpy(rng.integers(0, m.num_cols(), size=cuts[-1])).to(DEV)

    def nodes(A, seeds, ptr, fanouts, replace):
        for k in fanouts:
            sub = A[:, seeds::ptr]
            sub = sub.individual_sampling(k, sub.edata["w"] if "w" in A.edata else None, replace)
            seeds, ptr = sub.all_nodes()
        return seeds, ptr, A[seeds::ptr, seeds::ptr].all_nodes()

    args = (seeds, torch.tensor(cuts, device=DEV), fanouts, replace)
    compiled = gs.jit.compile(func=nodes, args=(bm, *args))
    assert sum("batch_sample_nodes" in str(n.target) for n in compiled._run.__self__.graph.nodes) == 1
    gs.manual_seed(5)
    got = compiled(bm, *args)
    assert gs.random_state() == (5, len(fanouts))
    gs.manual_seed(5)
    run_time = tuple(a if isinstance(a, torch.Tensor) else None for a in (None, *args))
    want = compiled.gm(run_time, [bm._graph], [[bm.row_ndata, bm.col_ndata, bm.edata]])
    for a, b in zip((*got[:2], *got[2]), (*want[:2], *want[2])):
        assert torch.equal(a, b)


def test_workspaces_have_a_second_table_where_picks_run_beside_labels():
    size, most = capi.lib().gs_layer_workspace_bytes, 1 << 19
    table, drawn = 8 << 20, 8 * most
    unweighted, weighted = size(most, 0) - table, size(most, 1) - drawn
    assert 0 <= unweighted - weighted <= 256            # (the place of one draw, aligned)
    assert size(most, 1) < 19 << 20 and size(most, 0) < 23 << 20


@pytest.mark.parametrize("count,fanout,replace,weighted", [(1, 1, False, False), (73, 63, True, False),
                                                           (1100, 10, False, True), (4000, 25, False, False)])
def test_one_layer_by_the_call_of_its_own(rng, count, fanout, replace, weighted):
    """gs_sample_layer, picks and labels in one call, against the chained form."""
    m = matrix(rng, 3000, 40, 700, weighted)
    seeds = torch.from_numpy(rng.integers(0, 3000, size=count)).to(DEV)
    gs.manual_seed(5)
    w = m.edata["w"] if weighted else None
    want = m._graph._CAPI_SampleLayers(seeds, [fanout], replace, w)
    l, P = capi.lib(), lambda t: t.data_ptr()
    indptr, indices = m._graph._CAPI_GetCSCIndptr(), m._graph._CAPI_GetCSCIndices()
    cdf = capi.weight_cdf(indptr, w, indices, 3000) if weighted else None
    most = count * (fanout + 1)
    ws = torch.empty(l.gs_layer_workspace_bytes(most, int(weighted)), dtype=torch.uint8, device=DEV)
    capi.check(l.gs_layer_begin(most, int(weighted), P(ws), ws.numel(), None))
    ids = [torch.empty(n, dtype=torch.int64, device=DEV) for n in (most, 2, most, most, 2)]
    mirror = torch.empty(6, dtype=torch.int64).pin_memory()
    for call in range(2):  # (the first leaves the table as it found it)
        capi.check(l.gs_sample_layer(P(indptr), 3000, P(indices), None, P(cdf) if weighted else None, 3000,
                                     P(seeds), count, None, 1, fanout, int(replace), 5, 0,
                                     *(P(t) for t in ids), None, P(mirror), most, P(ws), ws.numel(), None))
        torch.cuda.synchronize()
        sizes = (int(mirror[1]), int(mirror[3]), int(mirror[3]))
        for got, n, expect in zip((ids[0], ids[2], ids[3]), sizes, want):
            assert torch.equal(got[:n], expect)


def test_seeds_outside_the_matrix_take_the_other_path(rng):
    m = matrix(rng, 500, 20, 0, False)
    seeds = torch.tensor([3, -1, 499, 500, 1 << 40, 7], device=DEV)
    (n0, b0), (n1, b1) = both(single, m, (seeds, [4, 3], False), 2)
    assert torch.equal(n0, n1)
    for x, y in zip(b0, b1):
        same(x, y)


def test_call_ids_of_other_threads_are_not_taken_back(rng):
    """A call that has to start over draws by the ids it took; the counter that all threads
    share never goes back (another thread's draws in between would be repeated)."""
    m = matrix(rng, 4000, 20, 0, False)
    seeds = torch.from_numpy(np.concatenate([rng.permutation(4000)[:500], [1 << 40]])).to(DEV)
    args = (m, seeds, [6, 5, 4], False)
    sampler = gs.jit.compile(func=single, args=args)
    sampler(*args)
    walks, stop, made = [], threading.Event(), []
    start = torch.zeros(64, dtype=torch.int64, device=DEV)

    def walker():
        with torch.cuda.stream(torch.cuda.Stream()):
            while not stop.is_set():
                walks.append(m.random_walk(start, 30))
        torch.cuda.synchronize()

    gs.manual_seed(5)
    other = threading.Thread(target=walker)
    other.start()
    try:
        for _ in range(300):
            sampler(*args)
            made.append(1)
    finally:
        stop.set()
        other.join()
    assert gs.random_state() == (5, 3 * len(made) + len(walks))


@pytest.mark.parametrize("count", [40, 9000])        # short layers, and large ones made ahead
def test_blocks_handed_out_twice_are_other_objects(rng, count):
    bm = gs.BatchMatrix()
    bm.load_from_matrix(matrix(rng, 30000, 20, 0, False), False)
    seeds = torch.cat([torch.from_numpy(rng.permutation(30000)[:count]) for _ in range(5)]).to(DEV)
    ptr = torch.arange(6, device=DEV) * count

    args = (bm, seeds, ptr, [12, 10, 4], False)
    sampler = gs.jit.compile(func=batched, args=args)
    for first in sampler(*args):
        second = BlockList(first.batch)
        for a, b in zip(first, second):
            same(a, b)
            a.srcdata["feat"], a.edata["w"], a.num_src = 1, 2, -1
            assert a is not b and "feat" not in b.srcdata and "w" not in b.edata and b.num_src >= 0
        assert all(x is y for x, y in zip(list(first), first))       # a list keeps its blocks


def test_no_blocks_are_made_ahead_while_another_thread_holds_the_interpreter(rng):
    """Making them would wait for it in the middle of a step, and they may never be asked for;
    a thread that sleeps changes nothing."""
    bm = gs.BatchMatrix()
    bm.load_from_matrix(matrix(rng, 30000, 20, 0, False), False)
    seeds = torch.cat([torch.from_numpy(rng.permutation(30000)[:9000]) for _ in range(5)]).to(DEV)
    args = (bm, seeds, torch.arange(6, device=DEV) * 9000, [12, 10, 4], False)
    sampler = gs.jit.compile(func=batched, args=args)
    blocks = lambda: sum(type(o) is Block for o in gc.get_objects())  # noqa: E731
    stop = threading.Event()

    def made_ahead(target):
        other = threading.Thread(target=target)
        other.start()
        try:
            gs.manual_seed(5)
            gc.collect()
            before = blocks()
            got = sampler(*args)
            return got, blocks() - before
        finally:
            stop.set()
            other.join()
            stop.clear()

    def spin():
        while not stop.is_set():
            pass

    got, ahead = made_ahead(spin)
    assert ahead == 0
    again, ahead = made_ahead(stop.wait)
    assert ahead == 10                               # two layers of five
    for layer, other in zip(got, again):
        for x, y in zip(layer, other):
            same(x, y)


def test_a_call_that_runs_out_of_memory_between_layers_leaves_nothing_behind(rng):
    """What the first layer's kernels still report must not be taken for the next call's."""
    m = matrix(rng, 30000, 20, 0, False)
    seeds = torch.from_numpy(rng.permutation(30000)[:60]).to(DEV)
    args = (m, seeds, [10, 60, 9], False)            # the second layer's buffer takes a segment
    sampler = gs.jit.compile(func=single, args=args)
    gs.manual_seed(5)
    n0, b0 = sampler(*args)
    other = (m, seeds[:31].contiguous(), [7, 3], False)
    sampler2 = gs.jit.compile(func=single, args=other)
    gs.manual_seed(5)
    n1, b1 = sampler2(*other)
    torch.cuda.synchronize()
    failed = 0
    for _ in range(3):
        torch.cuda.empty_cache()
        total = torch.cuda.get_device_properties(0).total_memory
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (1 << 20)) / total)
        try:
            sampler(*args)
        except torch.OutOfMemoryError:
            failed += 1
        finally:
            torch.cuda.set_per_process_memory_fraction(1.0)
        gs.manual_seed(5)
        n, blocks = sampler2(*other)
        assert torch.equal(n, n1)
        for x, y in zip(blocks, b1):
            same(x, y)
    assert failed > 0             # (the first time, a segment may still have room)
    gs.manual_seed(5)
    n, blocks = sampler(*args)
    assert torch.equal(n, n0)
    for x, y in zip(blocks, b0):
        same(x, y)
