"""Weighted sampling on the GPU vs the oracle: bit-exact keys and picks."""
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


def F(a):
    return torch.as_tensor(np.asarray(a, dtype=np.float32), device=DEV)


def same(got, want):
    assert len(got) == len(want)
    for g, w in zip(got, want):
        if w is None:
            assert g is None
        else:
            assert np.array_equal(g.cpu().numpy(), w)


def test_key_arithmetic_is_bit_identical():
    rng = np.random.default_rng(0)
    cases = [0, 2**64 - 1, (2**51 - 1) << 12, 1 << 12, 2**63] + \
        [int(x) for x in rng.integers(0, 2**64, size=300, dtype=np.uint64)]
    for i, r in enumerate(cases):
        w = float(np.float32(rng.random() * 3 + 1e-3))
        e, k = capi.weighted_key_probe(7, 3, 1000 + i, i, w, r)
        assert e == orc.neg_log2_unit(r)
        assert k == orc.weighted_key(7, 3, 1000 + i, i, w)
    assert np.isinf(capi.weighted_key_probe(7, 3, 1, 1, 0.0, 5)[1])
    assert np.isinf(capi.weighted_key_probe(7, 3, 1, 1, -2.0, 5)[1])


@pytest.mark.parametrize("fanout", [1, 5, 15, 32, 33, 64])
def test_column_sampling_parity(fanout):
    rng = np.random.default_rng(fanout)
    indptr, indices = random_csc(rng, 3000, 10**6, 120, hub_deg=30000)
    probs = rng.lognormal(0, 1, size=indices.size).astype(np.float32)
    probs[rng.random(indices.size) < 0.05] = 0.0
    cols = rng.integers(0, 3000, size=2000)
    same(capi.sample_weighted(T(indptr), T(indices), F(probs), T(cols), fanout, call_id=2),
         orc.sample_weighted(indptr, indices, probs, cols, fanout, call_id=2))
    same(capi.sample_weighted(T(indptr), T(indices), F(probs), None, fanout),
         orc.sample_weighted(indptr, indices, probs, None, fanout))


@pytest.mark.parametrize("fanout", [3, 70])
def test_column_sampling_with_replacement_parity(fanout):
    rng = np.random.default_rng(fanout)
    indptr, indices = random_csc(rng, 2000, 10**6, 80, hub_deg=9000)
    probs = rng.random(indices.size).astype(np.float32)
    probs[rng.random(indices.size) < 0.1] = 0.0
    probs[indptr[5]:indptr[6]] = 0.0            # a column without positive weight
    cols = rng.integers(0, 2000, size=1500)
    same(capi.sample_weighted(T(indptr), T(indices), F(probs), T(cols), fanout, True),
         orc.sample_weighted(indptr, indices, probs, cols, fanout, True))
    same(capi.sample_weighted(T(indptr), T(indices), F(probs), None, fanout, True),
         orc.sample_weighted(indptr, indices, probs, None, fanout, True))


def _weighted_case(seed, cols=3000, hub=30000):
    rng = np.random.default_rng(seed)
    indptr, indices = random_csc(rng, cols, 10**6, 120, hub_deg=hub)
    probs = rng.lognormal(0, 1, size=indices.size).astype(np.float32)
    probs[rng.random(indices.size) < 0.05] = 0.0
    probs[indptr[7]:indptr[8]] = 0.0             # a column without positive weight
    lo = indptr[11]                              # a column with a single positive weight
    probs[lo:indptr[12]] = 0.0
    if indptr[12] > lo:
        probs[lo] = 2.0
    for c in (20, 21, 22, 23):                   # nearly all mass on one or two items
        if indptr[c + 1] - indptr[c] > 2:
            probs[indptr[c]] = 1e7
            probs[indptr[c] + 2] = 3e6
    return rng, indptr, indices, probs


@pytest.mark.parametrize("num_rows", [None, 0, 2**22, 2**27, 2**32, 2**40])
def test_weight_cdf_is_bit_identical(num_rows):
    """None: no row ids packed; 0: the bits that the largest id needs; wider id spaces leave
    fewer bits to the shares; ids beyond 32 bits are not packed."""
    rng, indptr, indices, probs = _weighted_case(1)
    if num_rows is None:
        g, h = capi.weight_cdf(T(indptr), F(probs)), orc.weight_cdf(indptr, probs)
    else:
        ids = indices if num_rows == 0 else rng.integers(0, num_rows, size=indices.size)
        g = capi.weight_cdf(T(indptr), F(probs), T(ids), num_rows or None)
        h = orc.weight_cdf(indptr, probs, ids, num_rows or None)
    assert np.array_equal(g.cpu().numpy(), h)
    empty = capi.weight_cdf(T(np.zeros(4)), F(np.zeros(0)))
    assert empty.cpu().tolist() == [0]


def test_weight_cdf_of_one_long_column():
    """A column far longer than a tile: the shares of every tile refer to the same total."""
    rng = np.random.default_rng(8)
    deg = np.array([3, 300_000, 0, 5])
    indptr = np.concatenate([[0], np.cumsum(deg)])
    probs = rng.lognormal(size=int(deg.sum())).astype(np.float32)
    ids = rng.integers(0, 2_450_000, size=probs.size)
    assert np.array_equal(capi.weight_cdf(T(indptr), F(probs), T(ids), 2_450_000).cpu().numpy(),
                          orc.weight_cdf(indptr, probs, ids, 2_450_000))


@pytest.mark.parametrize("fanout", [1, 64, 65])
def test_with_replacement_at_the_borders_of_the_column_split(fanout):
    """Columns held in LDS, taken by one wavefront, taken by the work-group (several of them in
    one work-group too), and columns without weight; weights that start anywhere."""
    rng = np.random.default_rng(fanout)
    deg = np.array([0, 1, 7, 8, 9, 511, 512, 513, 2047, 2048, 2049, 4095, 4096, 4097, 20001, 0, 3,
                    600, 2500, 1, 512])
    indptr = np.concatenate([[0], np.cumsum(deg)])
    indices = rng.integers(0, 10**6, size=indptr[-1])
    probs = rng.lognormal(0, 2, size=indices.size).astype(np.float32)
    probs[rng.random(indices.size) < 0.3] = 0.0
    probs[indptr[17]:indptr[18]] = 0.0        # nothing to pick by: the last position
    probs[indptr[18]:indptr[19]] = -1.0
    cols = rng.permutation(np.concatenate([np.arange(deg.size), rng.integers(0, deg.size, 40)]))
    same(capi.sample_weighted(T(indptr), T(indices), F(probs), T(cols), fanout, True, call_id=3),
         orc.sample_weighted(indptr, indices, probs, cols, fanout, True, call_id=3))
    same(capi.sample_weighted(T(indptr), T(indices), F(probs), None, fanout, True),
         orc.sample_weighted(indptr, indices, probs, None, fanout, True))


@pytest.mark.parametrize("fanout", [1, 5, 15, 64])
@pytest.mark.parametrize("replace", [False, True])
@pytest.mark.parametrize("packed_rows", [False, True])
def test_cdf_column_sampling_parity(fanout, replace, packed_rows):
    rng, indptr, indices, probs = _weighted_case(fanout)
    cdf = orc.weight_cdf(indptr, probs, indices if packed_rows else None)
    g_cdf = capi.weight_cdf(T(indptr), F(probs), T(indices) if packed_rows else None)
    cols = np.concatenate([rng.integers(0, 3000, size=2000), [7, 11, 7, 20, 21, 22, 23, 20]])
    same(capi.sample_weighted(T(indptr), T(indices), None, T(cols), fanout, replace, call_id=4,
                              cdf=g_cdf),
         orc.sample_weighted(indptr, indices, None, cols, fanout, replace, call_id=4, cdf=cdf))
    same(capi.sample_weighted(T(indptr), T(indices), None, None, fanout, replace, cdf=g_cdf),
         orc.sample_weighted(indptr, indices, None, None, fanout, replace, cdf=cdf))


def test_cdf_sampling_with_replacement_beyond_the_register_budget():
    # fanouts above 64 are written pick by pick instead of being held in registers
    rng, indptr, indices, probs = _weighted_case(3)
    cdf = orc.weight_cdf(indptr, probs, indices)
    g_cdf = capi.weight_cdf(T(indptr), F(probs), T(indices))
    cols = rng.integers(0, 3000, size=500)
    for fanout in (65, 100):
        same(capi.sample_weighted(T(indptr), T(indices), None, T(cols), fanout, True, call_id=2,
                                  cdf=g_cdf),
             orc.sample_weighted(indptr, indices, None, cols, fanout, True, call_id=2, cdf=cdf))
    with pytest.raises(capi.GsError):
        capi.sample_weighted(T(indptr), T(indices), None, T(cols), 65, False, cdf=g_cdf)


@pytest.mark.parametrize("fanout", [1, 3, 4, 5, 6, 8, 10, 12, 16, 24, 32, 33])
def test_cdf_columns_of_every_short_length(fanout):
    """Columns of 0 to 70 entries, each at several distances from a 32-byte boundary:
    the search's windows at both ends of a column, columns no longer than a window, the
    picks of a wavefront packed whatever its columns take; weights far from a straight
    line (so that guesses miss and the search bisects), zero ones, columns of only those."""
    rng = np.random.default_rng(fanout)
    deg = np.concatenate([np.arange(71), rng.permutation(71), [4000, 1, 65537]])
    indptr = np.concatenate([[0], np.cumsum(deg)])
    indices = rng.integers(0, 10**6, size=int(indptr[-1])).astype(np.int64)
    probs = rng.lognormal(0, 4, size=indices.size).astype(np.float32)
    probs[rng.random(indices.size) < 0.1] = 0.0
    for c in (8, 20, 33, 70):
        probs[indptr[c]:indptr[c + 1]] = 0.0
    cols = np.concatenate([np.arange(deg.size), rng.integers(0, deg.size, size=333)])
    for packed in (False, True):
        cdf = orc.weight_cdf(indptr, probs, indices if packed else None)
        g_cdf = capi.weight_cdf(T(indptr), F(probs), T(indices) if packed else None)
        for replace in (False, True):
            same(capi.sample_weighted(T(indptr), T(indices), None, T(cols), fanout, replace,
                                      call_id=5, cdf=g_cdf),
                 orc.sample_weighted(indptr, indices, None, cols, fanout, replace, call_id=5,
                                     cdf=cdf))


@pytest.mark.parametrize("fanout", [1, 2, 5, 15, 16, 17])
def test_cdf_sampling_around_the_most_columns_of_a_team(fanout):
    """As many columns as go sixteen lanes each, and one more; columns of every length around
    what the lanes hold and around one and several steps of the search behind it, hubs; weights
    that leave fewer items with a share than picks, none at all, and one with all but nothing."""
    rng = np.random.default_rng(fanout)
    lengths = np.concatenate([np.arange(0, 34), [63, 64, 65, 126, 127, 128, 129, 130, 255, 256, 257, 500],
                              128 * np.array([15, 16, 17, 31, 32, 255, 256, 257]) + 1, [70_001, 300_000]])
    kinds = ["even", "zeros", "few", "none", "one"]
    lengths = np.repeat(lengths, len(kinds))
    indptr = np.concatenate([[0], np.cumsum(lengths)])
    indices = rng.integers(0, 2_450_000, size=indptr[-1])
    probs = rng.lognormal(0, 1, size=indices.size).astype(np.float32)
    for c, n in enumerate(lengths):
        w = probs[indptr[c]:indptr[c + 1]]
        kind = kinds[c % len(kinds)]
        if kind == "zeros":
            w[rng.random(n) < 0.6] = 0.0
        elif kind in ("few", "none"):
            w[:] = 0.0
            if kind == "few" and n:
                w[rng.integers(0, n, size=max(1, fanout // 2))] = 1.0
        elif kind == "one" and n:
            w[:] *= 1e-7
            w[rng.integers(0, n)] = 1.0
    cdfs = [(orc.weight_cdf(indptr, probs, ids), capi.weight_cdf(T(indptr), F(probs), T(ids) if ids is not None else None))
            for ids in (indices, None)]
    most = 1024 * fanout
    for count in (1, most, most + 1):
        cols = np.resize(np.concatenate([np.arange(lengths.size), [-1, lengths.size]]), count)
        ptr = np.array([0, count // 3, count // 3, count])
        for host, device in cdfs:
            same(capi.sample_weighted(T(indptr), T(indices), None, T(cols), fanout, call_id=5, cdf=device),
                 orc.sample_weighted(indptr, indices, None, cols, fanout, call_id=5, cdf=host))
            a, b = (capi._sample_weighted_cdf(T(indptr), T(indices), device, T(cols), fanout, False, 7, 5, True,
                                              T(ptr), spans=spans) for spans in (False, True))
            for x, y in zip(a, b):
                assert torch.equal(x, y)


@pytest.mark.parametrize("n,k", [(10, 20), (1000, 64), (233000, 512), (5000, 5000)])
def test_list_sampling_parity(n, k):
    rng = np.random.default_rng(n)
    probs = rng.random(n).astype(np.float32)
    probs[rng.random(n) < 0.2] = 0.0
    same(capi.list_sample_weighted(F(probs), k, call_id=4),
         orc.list_sample_weighted(probs, k, call_id=4))
    same(capi.list_sample_weighted(F(probs), k, replace=True, call_id=4),
         orc.list_sample_weighted(probs, k, replace=True, call_id=4))
    for replace in (False, True):
        for algo in (0, 1):
            got = capi.list_sample_uniform(n, k, replace, algo, call_id=9)
            assert np.array_equal(got.cpu().numpy(),
                                  orc.list_sample_uniform(n, k, replace, algo, call_id=9))


def test_batched_list_sampling_parity():
    rng = np.random.default_rng(5)
    sizes = np.array([0, 700, 3, 20000, 0, 512, 513])
    ranges = np.concatenate([[0], np.cumsum(sizes)])
    probs = rng.random(ranges[-1]).astype(np.float32)
    probs[rng.random(probs.size) < 0.3] = 0.0
    same(capi.list_sample_weighted(F(probs), 512, range_=T(ranges)),
         orc.list_sample_weighted(probs, 512, range_=ranges))
    same(capi.list_sample_weighted(F(probs), 100, replace=True, range_=T(ranges)),
         orc.list_sample_weighted(probs, 100, replace=True, range_=ranges))


@pytest.mark.parametrize("case", ["few_positive", "all_zero", "repeated_weights", "one_heavy",
                                  "k_limits"])
def test_list_selection_cases(case):
    """The K smallest keys by selection (up to 2048 picks): cells of equal keys far larger
    than the pick count, weights that repeat, one dominant weight, pick counts at and
    around the limit of the selection path."""
    rng = np.random.default_rng(len(case))
    n = 300_000
    probs = rng.random(n).astype(np.float32)
    ks = [512]
    if case == "few_positive":        # fewer positive weights than picks: the rest by index
        probs[rng.permutation(n)[300:]] = 0.0
    elif case == "all_zero":
        probs[:] = 0.0
    elif case == "repeated_weights":  # many equal weights (keys still differ: other draws)
        probs = rng.choice(np.array([0.25, 0.5, 1.0], dtype=np.float32), size=n)
    elif case == "one_heavy":
        probs *= 1e-6
        probs[12345] = 1e6
    else:
        ks = [1, 2047, 2048, 2049]
    for k in ks:
        same(capi.list_sample_weighted(F(probs), k, call_id=2),
             orc.list_sample_weighted(probs, k, call_id=2))


@pytest.mark.parametrize("case", ["wide", "tiny", "huge", "denormal", "not_a_number", "one_size", "hardly_more"])
@pytest.mark.parametrize("k", [1, 512, 513, 2048])
def test_list_selection_by_approximate_keys(case, k):
    """Weights over the whole range of a float: keys that overflow or vanish in 32 bits, weights
    whose reciprocal does, bins that end at infinity; lists hardly longer than the picks."""
    rng = np.random.default_rng(k + len(case))
    n = k + 3 if case == "hardly_more" else 150_000
    with np.errstate(over="ignore"):
        probs = {"wide": np.exp2(rng.uniform(-149, 128, n)), "tiny": np.exp2(rng.uniform(-126, -96, n)),
                 "huge": np.exp2(rng.uniform(96, 128, n)), "denormal": np.exp2(rng.uniform(-149, -120, n)),
                 "not_a_number": np.exp2(rng.uniform(-40, 40, n)), "one_size": np.ones(n),
                 "hardly_more": rng.lognormal(0, 20, n)}[case].astype(np.float32)
    if case == "not_a_number":               # never picked, as weights of zero
        probs[rng.random(n) < 0.01] = np.nan
    if case == "hardly_more":
        probs[::2] = 0.0
    same(capi.list_sample_weighted(F(probs), k, call_id=6), orc.list_sample_weighted(probs, k, call_id=6))


@pytest.mark.parametrize("k", [1, 300, 2048])
@pytest.mark.parametrize("positive", [0, 1, 290, 5000])
def test_batched_list_selection_that_comes_to_weights_of_zero(k, positive):
    """Items of weight zero follow in the order of their indices: found by the counts of the
    tiles before, whose borders are not the segments'."""
    rng = np.random.default_rng(k + positive)
    ranges = np.concatenate([[0], np.cumsum([5000, 61_003, 1023, 40_001, 2500])])
    probs = np.zeros(ranges[-1], dtype=np.float32)
    for lo, hi in zip(ranges, ranges[1:]):
        probs[lo + rng.permutation(hi - lo)[:positive]] = 0.5
    same(capi.list_sample_weighted(F(probs), k, range_=T(ranges), call_id=7),
         orc.list_sample_weighted(probs, k, range_=ranges, call_id=7))
    same(capi.list_sample_weighted(F(probs), k, call_id=7), orc.list_sample_weighted(probs, k, call_id=7))


@pytest.mark.parametrize("sizes", [[(1 << 19) - 1], [1 << 19], [1 << 20], [(1 << 20) + 4099],
                                   [3, 0, (1 << 21) + 77, 9000]])
@pytest.mark.parametrize("zeros", [0.0, 0.9999])
def test_list_selection_with_copies_of_the_histograms(sizes, zeros):
    """Lists around the shortest whose work-groups share eight histograms, in each of the
    items a thread takes; short and empty segments beside a long one; picks that come to
    weights of zero."""
    rng = np.random.default_rng(sum(sizes))
    ranges = np.concatenate([[0], np.cumsum(sizes)])
    probs = rng.random(ranges[-1]).astype(np.float32)
    probs[rng.random(probs.size) < zeros] = 0.0
    range_ = ranges if len(sizes) > 1 else None
    for k in (1, 400, 2048):
        same(capi.list_sample_weighted(F(probs), k, range_=T(range_) if range_ is not None else None, call_id=9),
             orc.list_sample_weighted(probs, k, range_=range_, call_id=9))


def test_batched_list_selection_parity():
    """Segments long enough for the selection path, ragged, one of them empty, one taken
    whole, one with fewer positive weights than picks."""
    rng = np.random.default_rng(8)
    sizes = np.array([60000, 0, 300, 4097, 150000, 33000])
    ranges = np.concatenate([[0], np.cumsum(sizes)])
    probs = rng.random(ranges[-1]).astype(np.float32)
    probs[rng.random(probs.size) < 0.3] = 0.0
    probs[ranges[5]:ranges[6]] = 0.0
    probs[ranges[5] + 100:ranges[5] + 200] = 0.5
    for k in (64, 512):
        same(capi.list_sample_weighted(F(probs), k, range_=T(ranges), call_id=3),
             orc.list_sample_weighted(probs, k, range_=ranges, call_id=3))


@pytest.mark.parametrize("replace", [False, True])
@pytest.mark.parametrize("k", [0, 1, 300, 2048, 2049])
@pytest.mark.parametrize("nseg", [1, 2, 255, 256])
def test_list_sampling_in_one_call(nseg, k, replace):
    """Counts and picks by one call, in a workspace that holds anything: lists that are
    selected from (the counts' launch clears what that needs), sorted and drawn with
    replacement; up to 255 segments the counts take one launch, beyond it a scan."""
    rng = np.random.default_rng(nseg + k)
    sizes = rng.integers(3000, 6000, size=nseg)
    ranges = np.concatenate([[0], np.cumsum(sizes)])
    n = int(ranges[-1])
    probs = rng.random(n).astype(np.float32)
    want, want_range = orc.list_sample_weighted(probs, k, replace, ranges if nseg > 1 else None, 7777, 3)
    l = capi.lib()
    g_probs, g_range = F(probs), T(ranges) if nseg > 1 else None
    ws = torch.full((l.gs_list_sample_workspace_bytes(n, nseg),), 0xA5, dtype=torch.uint8, device=DEV)
    out_range = torch.empty(nseg + 1, dtype=torch.int64, device=DEV)
    out = torch.empty(len(want), dtype=torch.int64, device=DEV)
    for _ in range(2):
        capi.check(l.gs_list_sample_weighted(
            g_probs.data_ptr(), g_range.data_ptr() if nseg > 1 else None, n, nseg, k, int(replace),
            7777, 3, out_range.data_ptr(), len(want), out.data_ptr() if len(want) else None,
            ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream))
        same((out, out_range), (want, want_range))


@pytest.mark.parametrize("replace", [False, True])
@pytest.mark.parametrize("n,k", [(100, 7), (100, 200), (9000, 400), (9000, 2049), (700_000, 512)])
def test_picks_come_with_their_weights(n, k, replace):
    """Selected, sorted, taken whole and drawn with replacement, from one list and from one
    cut into segments; a compiled sampler asks for both at once."""
    from gsampler_amd.ops import fused_op
    rng = np.random.default_rng(n + k)
    probs = F(rng.random(n).astype(np.float32))
    ranges = T(np.concatenate([[0], np.sort(rng.integers(0, n + 1, size=4)), [n]]))
    ops = torch.ops.gs_ops
    for r in (None, ranges):
        def run(fused):
            gs.manual_seed(11)
            if fused:
                return fused_op._picks_and_weights(probs, k, replace, r)
            if r is None:
                return (ops._CAPI_ListSamplingWithProbs(probs, k, replace),)
            return ops._CAPI_BatchListSamplingWithProbs(probs, k, replace, r)
        got, want = run(True), run(False)
        assert torch.equal(got[0], want[0]) and torch.equal(got[2], probs[want[0]])
        assert r is None or torch.equal(got[1], want[1])
    with_grad = probs.clone().requires_grad_()
    gs.manual_seed(11)
    picks, _, weights = fused_op._picks_and_weights(with_grad, k, replace)
    weights.sum().backward()
    assert torch.equal(with_grad.grad, torch.bincount(picks, minlength=n).float())


@pytest.mark.parametrize("replace", [False, True])
@pytest.mark.parametrize("k", [0, 1, 40, 5000])
def test_offsets_of_picks_are_known_to_the_host(k, replace):
    """What a split of the picks goes by is what the device has: short and empty segments."""
    ranges = T(np.concatenate([[0], np.cumsum([3, 0, 90, 40, 4500, 0])]))
    probs = F(np.random.default_rng(k).random(int(ranges[-1])).astype(np.float32))
    ops = torch.ops.gs_ops
    picks, offsets = ops._CAPI_BatchListSamplingWithProbs(probs, k, replace, ranges)
    parts = ops._CAPI_BatchSplitByOffset(picks, offsets)
    assert [p.numel() for p in parts] == torch.diff(offsets).tolist()
    for p, lo, hi in zip(parts, ranges[:-1].tolist(), ranges[1:].tolist()):
        assert ((p >= lo) & (p < hi)).all()


def picks(A, seeds, K, probs):
    sub = A[:, seeds]
    picked, index = sub.collective_sampling(K, probs, False)
    return picked.div("w", probs[index], axis=1).edata["w"], index


def picks_of_changed_weights(A, seeds, K, probs):
    probs = probs * 1.0
    sub = A[:, seeds]
    picked, index = sub.collective_sampling(K, probs, False)
    doubled = probs.mul_(2.0)
    return picked.div("w", probs[index], axis=1).edata["w"], index, doubled


@pytest.mark.parametrize("func,fused", [(picks, True), (picks_of_changed_weights, False)])
def test_compiled_samplers_read_the_weights_of_their_picks_once(func, fused):
    from gsampler_amd.ops import fused_op
    rng = np.random.default_rng(3)
    indptr, indices = random_csc(rng, 500, 400, 60)
    m = gs.Matrix()
    m.load_graph("CSC", [T(indptr), T(indices)])
    m.edata["w"] = F(rng.random(indices.size).astype(np.float32))
    args = (m, T(rng.permutation(500)[:60]), 50, F(rng.random(m.num_rows()).astype(np.float32)))
    compiled = gs.jit.compile(func=func, args=args)
    targets = [n.target for n in compiled._run.__self__.graph.nodes]
    assert (fused_op._picks_and_weights in targets) == fused
    gs.manual_seed(2)
    got = compiled(*args)
    gs.manual_seed(2)
    want = func(*args)
    # (the formats that a compiled sampler takes put the edges in another order)
    assert torch.equal(got[1], want[1]) and torch.equal(got[0].sort().values, want[0].sort().values)


def test_operators_through_the_api():
    rng = np.random.default_rng(6)
    indptr, indices = random_csc(rng, 500, 400, 60)
    indices[0] = 399
    probs = rng.random(indices.size).astype(np.float32)
    m = gs.Matrix()
    m.load_graph("CSC", [T(indptr), T(indices)])
    m.edata["w"] = F(probs)
    gs.manual_seed(99)
    s = m.individual_sampling(7, m.edata["w"], False)
    want = orc.sample_weighted(indptr, indices, probs, None, 7, seed=99, call_id=0)
    assert np.array_equal(s.csc[1].cpu().numpy(), want[2])
    assert np.array_equal(s.edata["w"].cpu().numpy(), probs[want[3]])
    p = rng.random(400).astype(np.float32)
    sub, picked = m.collective_sampling(50, F(p), False)          # call id 1
    want_idx, _ = orc.list_sample_weighted(p, 50, seed=99, call_id=1)
    assert np.array_equal(picked.cpu().numpy(), want_idx)
    assert sub.num_rows() == 50
    u = torch.ops.gs_ops._CAPI_ListSampling(400, 30, False)          # call id 2
    assert np.array_equal(u.cpu().numpy(), orc.list_sample_uniform(400, 30, seed=99, call_id=2))
    ranges = np.array([0, 100, 400])
    idx, ptr = torch.ops.gs_ops._CAPI_BatchListSamplingWithProbs(F(p), 20, False, T(ranges))
    w_idx, w_ptr = orc.list_sample_weighted(p, 20, range_=ranges, seed=99, call_id=3)
    assert np.array_equal(idx.cpu().numpy(), w_idx) and np.array_equal(ptr.cpu().numpy(), w_ptr)
    idx, ptr = torch.ops.gs_ops._CAPI_BatchListSampling(20, False, T(ranges))
    w_idx, w_ptr = orc.list_sample_weighted(np.ones(400, dtype=np.float32), 20, range_=ranges,
                                            seed=99, call_id=4)
    assert np.array_equal(idx.cpu().numpy(), w_idx)


@pytest.mark.parametrize("n", [(1 << 20) - 1, 1 << 20, (1 << 22) - 1, 1 << 22])
def test_batched_list_selection_where_the_items_a_thread_takes_change(n):
    """Nine segments, whose borders are no tile's, with one histogram each."""
    rng = np.random.default_rng(n)
    ranges = np.sort(np.concatenate([[0, n], rng.integers(n // 9, n // 9 * 8, size=8)]))
    probs = rng.random(n).astype(np.float32)
    for k in (1, 256):
        same(capi.list_sample_weighted(F(probs), k, range_=T(ranges), call_id=3),
             orc.list_sample_weighted(probs, k, range_=ranges, call_id=3))


@pytest.mark.parametrize("n", [4096, 5000, 8192, 9217, 600_000, (1 << 20) + 3])
@pytest.mark.parametrize("where", ["first", "last", "few", "all"])
def test_list_selection_of_candidates_that_lie_together(n, where):
    """All candidates in a segment's first or last tiles, in one list of them; weights of zero in
    the others; fewer tiles than lists; all of one weight, which narrows them in the end."""
    probs = np.full(n, 1e-6, dtype=np.float32)
    if where == "few":
        probs[:] = 0
    probs[{"first": slice(0, 900), "last": slice(n - 900, n), "few": slice(n // 2, n // 2 + 90),
           "all": slice(0, n)}[where]] = 1.0
    for ranges in (None, np.array([0, n // 2 + 77, n])):
        if ranges is not None and n < 9000:
            continue  # (segments too short to be selected from)
        for k in (1, 400, 2048):
            args = {} if ranges is None else {"range_": T(ranges)}
            same(capi.list_sample_weighted(F(probs), k, call_id=3, **args),
                 orc.list_sample_weighted(probs, k, range_=ranges, call_id=3))
