"""The work that users of this framework have it do, as timed cases.

A case is a dict of plain values.  Its "kind" names the program: a sampler of the
reference's examples written against Matrix / BatchMatrix and compiled with
gs.jit.compile, the walks, or the feature fetch that follows sampling.  Graphs are
the seeded synthetic ones of gsampler_amd.utils (R-MAT and Chung-Lu power law, CSC,
int64 ids); their sizes and the samplers' are those of bench.py and of the tests,
and the ranges between them.

  listed()              the standing cases
  draw(rng)             one more case of the same ranges
  prepare(case, seed)   the state a program holds before the call
  run(state)            one pass through the public entry points
  work(case)            bytes and operations a pass cannot do without (expected values)
  tolerance(case)       how far another correct implementation may be off
"""
import math

import numpy as np
import torch
import torch.nn.functional as F

import gsampler_amd as gs
from gsampler_amd.format import _COO
from gsampler_amd.utils import batched_seeds, chung_lu_csc, rmat_csc

DEV = "cuda:0"
DTYPES = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}


# ------------------------------------------------------------------------ cases
def listed():
    return [
        # One mini-batch at a time on a small graph: what an interactive training loop
        # does per iteration.  Launches, host work and waits are the cost.
        dict(name="sage small", kind="sage", graph="rmat", nodes=100_000, edges=2_000_000,
             batches=0, batch_size=1024, fanouts="25,10", weighted=False),
        # The smallest super-batch: a few hundred seeds per batch, blocks for each of them.
        dict(name="sage tiny super-batch", kind="sage", graph="chung_lu", nodes=50_000,
             edges=1_000_000, batches=8, batch_size=256, fanouts="15,10,5", weighted=False),
        # The headline workload: 64 mini-batches per launch on a graph of ogbn-products' size.
        dict(name="sage super-batch", kind="sage", graph="chung_lu", nodes=2_450_000,
             edges=124_000_000, batches=64, batch_size=1024, fanouts="15,10,5", weighted=False),
        # The same with neighbours drawn by edge weight.
        dict(name="sage weighted super-batch", kind="sage", graph="chung_lu", nodes=2_450_000,
             edges=124_000_000, batches=64, batch_size=1024, fanouts="15,10,5", weighted=True),
        # Layer-wise sampling on a dense graph of Reddit's size: row sums over long columns,
        # a weighted pick of rows, the row slice, two normalisations.
        dict(name="ladies", kind="ladies", nodes=233_000, edges=115_000_000, seeds=512,
             fanouts="512,512"),
        # Layer-wise sampling of several mini-batches per launch, every batch with its own
        # numbering of rows (encoded slicing).
        dict(name="ladies batched", kind="batch_ladies", nodes=233_000, edges=11_500_000,
             batches=8, batch_size=128, fanouts="256,256"),
        # Layer-wise sampling by a fixed node weight: no row sums, slice and pick only.
        dict(name="fastgcn", kind="fastgcn", nodes=2_450_000, edges=124_000_000, seeds=1024,
             fanouts="400,400"),
        # Attention over node features decides the weights of the picks: products of node
        # features per edge, weighted sampling with replacement on the slice.
        dict(name="pass attention", kind="pass", nodes=100_000, edges=2_000_000, seeds=256,
             fanouts="10,5", features=64, hidden=16),
        # Neighbourhoods sampled first, then the subgraph that the sampled nodes induce.
        dict(name="shadow batched", kind="shadow", nodes=100_000, edges=2_000_000, batches=16,
             batch_size=64, fanouts="10,5"),
        # Second-order walks over the whole graph, as embeddings are trained from.
        dict(name="node2vec", kind="node2vec", nodes=2_450_000, edges=124_000_000,
             walks=1_000_000, length=80, p=2.0, q=0.5),
        # First-order walks of one mini-batch of seeds: a chain of dependent reads.
        dict(name="walk small", kind="walk", nodes=100_000, edges=2_000_000, walks=1024,
             length=80),
        # Features of the input nodes of one sampled mini-batch; rows of 400 bytes.
        dict(name="feature fetch", kind="gather", nodes=2_450_000, rows=166_000, features=100,
             dtype="float32"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["sage", "sage", "sage weighted", "ladies", "batch_ladies", "fastgcn",
                       "pass", "shadow", "node2vec", "walk", "gather"])
    if kind.startswith("sage"):
        nodes = _log(rng, 20_000, 2_450_000)
        batches = rng.choice([0, _log(rng, 1, 64), _log(rng, 1, 64)])
        return dict(kind="sage", graph=rng.choice(["rmat", "chung_lu"]), nodes=nodes,
                    edges=int(nodes * rng.uniform(10, 50)), batches=batches,
                    batch_size=_log(rng, 32, 1024),
                    fanouts=rng.choice(["25,10", "15,10,5", "10,5", "10,10,10", "5,5"]),
                    weighted=kind == "sage weighted")
    if kind == "ladies":
        nodes = _log(rng, 20_000, 233_000)
        return dict(kind="ladies", nodes=nodes, edges=int(nodes * _log(rng, 20, 490)),
                    seeds=_log(rng, 64, 512), fanouts=rng.choice(["%d,%d", "%d,%d,%d"]).replace(
                        "%d", str(_log(rng, 64, 512))))
    if kind == "batch_ladies":
        nodes = _log(rng, 20_000, 233_000)
        return dict(kind="batch_ladies", nodes=nodes, edges=int(nodes * rng.uniform(10, 49)),
                    batches=_log(rng, 2, 8), batch_size=_log(rng, 32, 128),
                    fanouts="%d,%d" % ((_log(rng, 32, 256),) * 2))
    if kind == "fastgcn":
        nodes = _log(rng, 50_000, 2_450_000)
        return dict(kind="fastgcn", nodes=nodes, edges=int(nodes * rng.uniform(10, 50)),
                    seeds=_log(rng, 128, 1024), fanouts="%d,%d" % ((_log(rng, 100, 400),) * 2))
    if kind == "pass":
        nodes = _log(rng, 10_000, 100_000)
        return dict(kind="pass", nodes=nodes, edges=int(nodes * rng.uniform(8, 20)),
                    seeds=_log(rng, 32, 256), fanouts=rng.choice(["10,5", "5,5", "10"]),
                    features=rng.randint(16, 64), hidden=rng.randint(8, 16))
    if kind == "shadow":
        nodes = _log(rng, 10_000, 100_000)
        return dict(kind="shadow", nodes=nodes, edges=int(nodes * rng.uniform(8, 20)),
                    batches=_log(rng, 2, 16), batch_size=_log(rng, 8, 64),
                    fanouts=rng.choice(["10,5", "8,4", "5,5"]))
    if kind in ("node2vec", "walk"):
        nodes = _log(rng, 50_000, 2_450_000)
        case = dict(kind=kind, nodes=nodes, edges=int(nodes * rng.uniform(10, 50)),
                    walks=_log(rng, 1000, 1_000_000), length=_log(rng, 5, 80))
        if kind == "node2vec":
            case.update(p=rng.choice([0.25, 0.5, 1.0, 2.0, 4.0]), q=rng.choice([0.25, 0.5, 2.0, 4.0]))
        return case
    return dict(kind="gather", nodes=_log(rng, 100_000, 2_450_000), rows=_log(rng, 1000, 500_000),
                features=rng.randint(16, 256), dtype=rng.choice(sorted(DTYPES)))


def _fanouts(case):
    return [int(k) for k in case["fanouts"].split(",")]


# --------------------------------------------------------------------- samplers
def sage_sampler(A, seeds, fanouts):
    blocks = []
    for k in fanouts:
        sub = A[:, seeds].individual_sampling(k, None, False)
        seeds = sub.all_nodes()
        blocks.append(sub.to_dgl_block())
    return seeds, blocks


def weighted_sage_sampler(A, seeds, fanouts):
    blocks = []
    for k in fanouts:
        sub = A[:, seeds]
        sub = sub.individual_sampling(k, sub.edata["w"], False)
        seeds = sub.all_nodes()
        blocks.append(sub.to_dgl_block())
    return seeds, blocks


def batch_sage_sampler(A, seeds, seeds_ptr, fanouts):
    layers = []
    for k in fanouts:
        sub = A[:, seeds::seeds_ptr].individual_sampling(k, None, False)
        seeds, seeds_ptr = sub.all_nodes()
        layers.append(sub.to_dgl_block())
    return layers


def batch_weighted_sage_sampler(A, seeds, seeds_ptr, fanouts):
    layers = []
    for k in fanouts:
        sub = A[:, seeds::seeds_ptr]
        sub = sub.individual_sampling(k, sub.edata["w"], False)
        seeds, seeds_ptr = sub.all_nodes()
        layers.append(sub.to_dgl_block())
    return layers


def ladies_sampler(A, seeds, fanouts):
    blocks = []
    for k in fanouts:
        sub = A[:, seeds]
        sub.edata["p"] = sub.edata["w"] ** 2
        prob = sub.sum("p", axis=1)
        picked, index = sub.collective_sampling(k, prob, False)
        picked = picked.div("w", prob[index], axis=1)
        picked = picked.div("w", picked.sum("w", axis=0), axis=0)
        seeds = picked.all_nodes()
        blocks.append(picked.to_dgl_block(prefetch_edata={"w"}))
    return seeds, blocks


def batch_ladies_sampler(A, seeds, seeds_ptr, fanouts):
    layers = []
    for k in fanouts:
        sub = A[:, seeds::seeds_ptr]
        sub.edata["p"] = sub.edata["w"] ** 2
        prob = sub.sum("p", axis=1)
        _, probs_ptr = sub.all_rows()
        picked, index = sub.collective_sampling(k, prob, probs_ptr, False)
        picked = picked.div("w", prob[index], axis=1)
        picked = picked.div("w", picked.sum("w", axis=0), axis=0)
        seeds, seeds_ptr = picked.all_nodes()
        layers.append(picked.to_dgl_block(prefetch_edata={"w"}))
    return layers


def fastgcn_sampler(A, seeds, fanouts):
    blocks = []
    for k in fanouts:
        sub = A[:, seeds]
        picked, _ = sub.collective_sampling(k, sub.row_ndata["deg"], False)
        seeds = picked.all_nodes()
        blocks.append(picked.to_dgl_block())
    return seeds, blocks


def pass_sampler(A, seeds, fanouts, features, W1, W2, W3):
    blocks = []
    for k in fanouts:
        sub = A[:, seeds]
        u_feats, v_feats = features[sub.rows()], features[sub.cols()]
        att1 = torch.sum(gs.ops.u_mul_v(sub, u_feats @ W1, v_feats @ W1, _COO), dim=1)
        att2 = torch.sum(gs.ops.u_mul_v(sub, u_feats @ W2, v_feats @ W2, _COO), dim=1)
        att3 = sub.div("w", sub.sum("w", axis=0), axis=0).edata["w"]
        att = torch.stack([att1, att2, att3], dim=1)
        att = F.relu(att @ F.softmax(W3, dim=0))
        att = att + 10e-10 * torch.ones_like(att)
        sub.edata["w"] = att
        picked = sub.individual_sampling(k, probs=att, replace=True)
        seeds = picked.all_nodes()
        blocks.append(picked.to_dgl_block(prefetch_edata={"w"}))
    return seeds, blocks


def batch_shadow_sampler(A, seeds, seeds_ptr, fanouts):
    for k in fanouts:
        seeds, seeds_ptr = A[:, seeds::seeds_ptr].individual_sampling(k, None, False).all_nodes()
    return A[seeds::seeds_ptr, seeds::seeds_ptr].to_dgl_block()


# ---------------------------------------------------------------------- prepare
# What a sampler returns has a size of its own for every graph, so a case keeps one
# graph and one random state, and the seed turns them into other inputs of the same
# shape: it numbers the nodes anew (node-wise samplers, whose picks follow positions),
# or puts the seeds and the edges of every column in another order (layer-wise
# samplers, whose picks follow row ids).
def _numbered_anew(indptr, indices, weights, shift):
    """The graph with node i called (i + shift) % nodes, its columns in the order of
    their new names; edge data moves along."""
    nodes = indptr.numel() - 1
    cut = int(indptr[nodes - shift])
    degree = torch.roll(indptr[1:] - indptr[:-1], shift)
    out = torch.zeros_like(indptr)
    torch.cumsum(degree, 0, out=out[1:])
    indices = torch.remainder(torch.cat([indices[cut:], indices[:cut]]) + shift, nodes)
    if weights is not None:
        weights = torch.cat([weights[cut:], weights[:cut]])
    return out, indices, weights


def _columns_turned(indptr, indices, weights, steps):
    """The edges of every column moved round by so many places."""
    degree = indptr[1:] - indptr[:-1]
    start = torch.repeat_interleave(indptr[:-1], degree)
    src = torch.arange(indices.numel(), device=indices.device).sub_(start).add_(steps)
    src.remainder_(torch.repeat_interleave(degree, degree)).add_(start)
    return indices[src], weights[src] if weights is not None else None


def _batch_matrix(m, encoding):
    bm = gs.BatchMatrix()
    bm.load_from_matrix(m, encoding)
    return bm


def prepare(case, seed):
    kind = case["kind"]
    g = torch.Generator(device=DEV)
    g.manual_seed(seed + 1)
    gs.manual_seed(7777)
    if kind == "gather":
        dtype = DTYPES[case["dtype"]]
        table = torch.rand((case["nodes"], case["features"]), generator=g, device=DEV).to(dtype)
        # the frontiers of mini-batches: distinct node ids in no particular order
        ids, n = [], case["rows"]
        while n > 0:
            ids.append(torch.randperm(case["nodes"], generator=g, device=DEV)[:n])
            n -= ids[-1].numel()
        return dict(kind=kind, table=table, ids=torch.cat(ids).contiguous())

    nodes, edges = case["nodes"], case["edges"]
    m = gs.Matrix()
    if kind in ("node2vec", "walk"):
        m.load_graph("CSC", list(chung_lu_csc(nodes, edges, seed=seed + 2, device=DEV)))
        if kind == "node2vec":
            m._graph._CAPI_SortCSCIndices()
        seeds = torch.randint(0, nodes, (case["walks"],), generator=g, device=DEV)
        return dict(kind=kind, m=m, seeds=seeds, length=case["length"], p=case.get("p"),
                    q=case.get("q"))

    same = torch.Generator(device=DEV)
    same.manual_seed(11)
    layer_wise = kind in ("ladies", "batch_ladies", "fastgcn")
    rmat = case.get("graph") == "rmat" or kind in ("pass", "shadow")
    indptr, indices = (rmat_csc if rmat else chung_lu_csc)(nodes, edges, seed=12, device=DEV)
    weights = ptr = None
    if case.get("weighted"):
        weights = torch.randn(edges, generator=same, device=DEV).exp_()
    elif kind in ("ladies", "batch_ladies", "pass"):
        weights = 1.0 - torch.rand(edges, generator=same, device=DEV)
    count = case.get("seeds") or case["batch_size"]
    if case.get("batches"):
        seeds, ptr = batched_seeds(nodes, case["batches"], count, seed=13, device=DEV)
    else:
        seeds = torch.randperm(nodes, generator=same, device=DEV)[:count].contiguous()
    change = torch.randint(nodes // 4, nodes // 2, (1,), generator=g, device=DEV).item()
    if layer_wise:
        indices, weights = _columns_turned(indptr, indices, weights, change)
        order = torch.argsort(torch.rand(seeds.view(-1, count).shape, generator=g, device=DEV), dim=1)
        seeds = seeds.view(-1, count).gather(1, order).flatten().contiguous()
    else:
        indptr, indices, weights = _numbered_anew(indptr, indices, weights, change)
        seeds = torch.remainder(seeds + change, nodes)
    m.load_graph("CSC", [indptr, indices])
    if weights is not None:
        m.edata["w"] = weights
    fanouts = _fanouts(case)
    if kind == "sage" and case["batches"]:
        func = batch_weighted_sage_sampler if case["weighted"] else batch_sage_sampler
        args = (_batch_matrix(m, False), seeds, ptr, fanouts)
    elif kind == "sage":
        func, args = weighted_sage_sampler if case["weighted"] else sage_sampler, (m, seeds, fanouts)
    elif kind == "ladies":
        func, args = ladies_sampler, (m, seeds, fanouts)
    elif kind == "batch_ladies":
        func, args = batch_ladies_sampler, (_batch_matrix(m, True), seeds, ptr, fanouts)
    elif kind == "fastgcn":
        m.row_ndata["deg"] = torch.bincount(indices, minlength=m.num_rows()).float() + 1.0
        func, args = fastgcn_sampler, (m, seeds, fanouts)
    elif kind == "pass":
        D, H = case["features"], case["hidden"]
        features = torch.roll(torch.randn((nodes, D), generator=same, device=DEV), change, 0)
        W1, W2 = (torch.randn((D, H), generator=same, device=DEV) for _ in range(2))
        W3 = torch.randn(3, generator=same, device=DEV)
        func, args = pass_sampler, (m, seeds, fanouts, features, W1, W2, W3)
    elif kind == "shadow":
        func, args = batch_shadow_sampler, (_batch_matrix(m, False), seeds, ptr, fanouts)
    else:
        raise ValueError("no such kind of case: %r" % kind)
    return dict(kind=kind, sampler=gs.jit.compile(func=func, args=args), args=args)


# -------------------------------------------------------------------------- run
def _of_blocks(blocks):
    """Edges (as local ids), source nodes and edge data of a list of blocks."""
    out = []
    for b in blocks:
        out.append([b.row, b.col, b.srcdata["_ID"], dict(b.edata)])
    return out


def _of_layer(layer):
    """The same for the blocks of all mini-batches of a layer: the arrays they are views of,
    and where each block begins."""
    b = layer.batch
    return [b.row(), b.col(), b.indptr(), b.frontier(), b.frontier_ptr(), b.edge_ptr()]


def run(state):
    kind = state["kind"]
    if kind == "gather":
        return gs.utils.gather_rows(state["table"], state["ids"])
    if kind == "walk":
        return state["m"].random_walk(state["seeds"], state["length"])
    if kind == "node2vec":
        return state["m"].node2vec(state["seeds"], state["length"], state["p"], state["q"])
    result = state["sampler"](*state["args"])
    if kind == "shadow":
        result = [result]
    if isinstance(state["args"][0], gs.BatchMatrix):
        minibatches = list(zip(*result))         # a training loop takes every block in turn
        out = [_of_layer(layer) for layer in result]
        if kind == "batch_ladies":
            out += [[b.edata["w"] for b in blocks] for blocks in minibatches]
        return out
    nodes, blocks = result
    return [nodes] + _of_blocks(blocks)


# ------------------------------------------------------------- work and tolerance
def _popularity(nodes):
    """Share of the edge ends that a node holds in the power-law graphs (R-MAT's is alike)."""
    w = np.arange(1, nodes + 1, dtype=np.float64) ** (-1.0 / 1.1)
    return w / w.sum()


def _met(p, draws):
    """Probability of every node to be met by so many draws of edge ends."""
    return -np.expm1(draws * np.log1p(-np.minimum(p, 0.999999)))


def _picked(p, count):
    """Probability of every node to be among `count` picks by weight p, without repeats."""
    count = min(count, 0.999 * p.size)
    lo, hi = 0.0, 1e12
    for _ in range(40):
        mid = math.sqrt(max(lo, 1e-3) * hi)
        lo, hi = (mid, hi) if _met(p, mid).sum() < count else (lo, mid)
    return _met(p, hi)


def _walked(case, p):
    """(columns, edges, frontier) of every layer of node-wise sampling, summed over the
    batches: expected values."""
    batches = max(1, case.get("batches") or 1)
    chosen = np.full(p.size, min(1.0, (case.get("batch_size") or case.get("seeds")) / p.size))
    deg = p * case["edges"]
    out = []
    for k in _fanouts(case):
        edges = float((chosen * np.minimum(deg, k)).sum())
        nxt = 1.0 - (1.0 - chosen) * (1.0 - _met(p, edges))
        out.append((batches * float(chosen.sum()), batches * edges, batches * float(nxt.sum())))
        chosen = nxt
    return out, chosen


def work(case):
    kind = case["kind"]
    if kind == "gather":
        row = case["features"] * torch.empty((), dtype=DTYPES[case["dtype"]]).element_size()
        return {"bytes": case["rows"] * (8 + 2 * row), "flops": 0}
    if kind in ("walk", "node2vec"):
        # a hop reads a column's two offsets and one id and writes one id (walks that meet
        # a node without neighbours end early; few do)
        return {"bytes": case["walks"] * (16 + 32 * case["length"]), "flops": 0}
    p = _popularity(case["nodes"])
    deg = p * case["edges"]
    nbytes = flops = 0.0
    if kind in ("sage", "pass", "shadow"):
        layers, chosen = _walked(case, p)
        for S, E, U in layers:
            # seeds, offsets and the ids behind the picks in; two labels an edge, the
            # frontier and the blocks' offsets out
            nbytes += 24 * S + 8 * E + (16 * E + 8 * U + 8 * S if kind != "shadow" else 8 * U)
        if case.get("weighted"):
            nbytes += 4 * sum(E for _, E, _ in layers)
        if kind == "shadow":
            nodes = case["batches"] * float(chosen.sum())
            slice_edges = case["batches"] * float((chosen * deg).sum())
            kept = case["batches"] * float((chosen * deg).sum() * (chosen * p).sum())
            nbytes += 24 * nodes + 8 * slice_edges + 16 * kept + 16 * nodes
        if kind == "pass":
            D, H = case["features"], case["hidden"]
            chosen = np.full(p.size, min(1.0, case["seeds"] / p.size))
            for k in _fanouts(case):
                S, E = float(chosen.sum()), float((chosen * deg).sum())
                # ids and weights of the slice and the features once
                nbytes += 12 * E + 4 * (case["nodes"] + S) * D
                flops += 4.0 * (case["nodes"] + S) * D * H + 4.0 * E * H
                chosen = 1.0 - (1.0 - chosen) * (1.0 - _met(p, S * k))
        return {"bytes": nbytes, "flops": flops}
    # layer-wise samplers
    batches = case.get("batches", 1)
    chosen = np.full(p.size, min(1.0, (case.get("batch_size") or case["seeds"]) / p.size))
    for k in _fanouts(case):
        S, E = float(chosen.sum()), float((chosen * deg).sum())
        rows = _picked(p, k)
        kept = E * float((rows * p).sum())
        nxt = 1.0 - (1.0 - chosen) * (1.0 - rows)
        value = 0 if kind == "fastgcn" else 4
        nbytes += batches * (24 * S + (8 + value) * E + (16 + value) * kept + 8 * float(nxt.sum()))
        if kind == "fastgcn":
            nbytes += 4 * case["nodes"]
        else:
            flops += batches * (2 * E + 3 * kept)
        chosen = nxt
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Ids and copied values are the same for every correct implementation.  Layer-wise
    samplers add and divide 32-bit numbers, and where two candidates' keys are equal to the
    last bits their order, and so a few local ids, may differ."""
    if case["kind"] in ("ladies", "batch_ladies"):
        return {"rel": 1e-5, "max": 1e-3, "differ": 0.005}
    if case["kind"] == "pass":
        return {"rel": 1e-5, "max": 1e-3}
    return "exact"
