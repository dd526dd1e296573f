"""The generated graphs are the same graph every time: their degree law does not
depend on the order in which a device adds it up."""
import numpy as np
import pytest
import torch

from gsampler_amd.utils.synthetic import chung_lu_csc, power_law_cdf

# Of a share: the roundings of its sum, of the total and of the quotient, 2^-53 each,
# and the terms, whose powers are good to a last place (2^-52) on either side.
BOUND = 3.5 * 2.0 ** -52


def prefix_shares(num_nodes, exponent=2.1):
    """The same sums in integers of 2^-56: every term is off by at most half a unit,
    the additions are exact."""
    w = np.arange(1, num_nodes + 1, dtype=np.float64) ** (-1.0 / (exponent - 1.0))
    units = np.cumsum(np.rint(w * 2.0 ** 56).astype(np.uint64))
    return units.astype(np.longdouble) / np.longdouble(units[-1])


@pytest.mark.parametrize("num_nodes", [1, 2, 1000, 100_003])
def test_cdf_on_the_host(num_nodes):
    cdf = power_law_cdf(num_nodes)
    assert cdf.dtype == torch.float64 and cdf.numel() == num_nodes
    assert float(cdf[-1]) == 1.0 and bool((cdf[1:] >= cdf[:-1]).all())
    want = prefix_shares(num_nodes)
    assert float(np.max(np.abs(cdf.numpy() - want) / want)) <= BOUND


@pytest.mark.gpu
def test_cdf_on_the_device_is_the_same_every_time():
    dev, n = torch.device("cuda:0"), 2_450_000
    first = power_law_cdf(n, device=dev)
    for k in range(8):
        busy = torch.rand(1 << 24, device=dev).sort() if k % 2 else None
        again = power_law_cdf(n, device=dev)
        assert torch.equal(first.view(torch.int64), again.view(torch.int64))
        del busy
    want = prefix_shares(n)
    assert float(np.max(np.abs(first.cpu().numpy() - want) / want)) <= BOUND


@pytest.mark.gpu
def test_graph_is_the_same_every_time():
    dev = torch.device("cuda:0")
    indptr, indices = chung_lu_csc(2_450_000, 24_000_000, seed=12, device=dev)
    for _ in range(3):
        p, i = chung_lu_csc(2_450_000, 24_000_000, seed=12, device=dev)
        assert torch.equal(indptr, p) and torch.equal(indices, i)
