"""The filter in front of a row slice's table in LDS, evaluated on the host."""
import numpy as np
import pytest

from gsampler_amd import capi


def passing(picked, ids, small):
    picked, ids = (np.ascontiguousarray(x, dtype=np.int32) for x in (picked, ids))
    return capi.lib().gs_probe_few_id_filter(picked.ctypes.data, picked.size, ids.ctypes.data,
                                             ids.size, int(small))


@pytest.mark.parametrize("small", [False, True])
@pytest.mark.parametrize("picks", [1, 512, 2048])
@pytest.mark.parametrize("step", [1, 2, 3, 5, 8, 16, 32, 64, 100, 256, 1000, 1024, 4096, 9216, 65536])
def test_ids_in_steps_spread_over_the_filter(step, picks, small):
    """Picked ids set a bit each of 32 * words, so that of others
    1 - (1 - 1 / (32 words)) ** picks pass an even spread.  Steps leave some unevenness: the
    bound is half as many again, and what ten of 233 000 ids are for a single bit."""
    rng = np.random.default_rng(step)
    ids = np.arange(min(233_000, 2**31 // step), dtype=np.int64) * step
    chosen = rng.permutation(ids.size)
    picked, others = ids[chosen[:picks]], ids[chosen[picks:]]
    assert passing(picked, picked, small) == picks
    even = 1.0 - (1.0 - 1.0 / (32 * (1024 if small else 2048))) ** picks
    assert passing(picked, others, small) <= 1.5 * even * others.size + 10


def test_nothing_picked_and_nothing_asked():
    assert passing([], [5], False) == 0
    assert passing([5], [], True) == 0
    assert capi.lib().gs_probe_few_id_filter(None, 1, None, 0, 0) == -1
