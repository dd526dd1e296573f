"""The generated graphs are the same graph every time: their degree law does not
depend on the order in which a device adds it up."""
import numpy as np
import pytest
import torch

from gsampler_amd.utils.synthetic import chung_lu_csc, power_law_cdf

def exact_shares(num_nodes, exponent=2.1):
    w = np.arange(1, num_nodes + 1, dtype=np.float64) ** (-1.0 / (exponent - 1.0))
    sums = np.cumsum(w, dtype=np.longdouble)
    return sums / sums[-1], sums


def bound(num_nodes, sums):
    """Of a share: the roundings of its sum, of the total and of the quotient (2^-53 each),
    the terms, whose powers are good to a last place (2^-52) on either side, and the
    terms' roundings to integers of 2^-56: standard deviation sqrt(k / 12) units, six of
    them, of the sum and of the total."""
    units = 6.0 * np.sqrt(np.arange(1, num_nodes + 1) / 12.0) * 2.0 ** -56
    return 3.5 * 2.0 ** -52 + units / sums + units[-1] / sums[-1]


@pytest.mark.parametrize("num_nodes", [1, 2, 1000, 100_003])
def test_cdf_on_the_host(num_nodes):
    cdf = power_law_cdf(num_nodes)
    assert cdf.dtype == torch.float64 and cdf.numel() == num_nodes
    assert float(cdf[-1]) == 1.0 and bool((cdf[1:] >= cdf[:-1]).all())
    want, sums = exact_shares(num_nodes)
    assert bool((np.abs(cdf.numpy() - want) / want <= bound(num_nodes, sums)).all())


@pytest.mark.gpu
def test_cdf_on_the_device_is_the_same_every_time():
    dev, n = torch.device("cuda:0"), 2_450_000
    first = power_law_cdf(n, device=dev)
    for k in range(8):
        busy = torch.rand(1 << 24, device=dev).sort() if k % 2 else None
        again = power_law_cdf(n, device=dev)
        assert torch.equal(first.view(torch.int64), again.view(torch.int64))
        del busy
    want, sums = exact_shares(n)
    assert bool((np.abs(first.cpu().numpy() - want) / want <= bound(n, sums)).all())


@pytest.mark.gpu
def test_graph_is_the_same_every_time():
    dev = torch.device("cuda:0")
    indptr, indices = chung_lu_csc(2_450_000, 24_000_000, seed=12, device=dev)
    for _ in range(3):
        p, i = chung_lu_csc(2_450_000, 24_000_000, seed=12, device=dev)
        assert torch.equal(indptr, p) and torch.equal(indices, i)
