"""The wavefront helpers of pcp_wave.hpp, called directly."""
import ctypes as C
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def unit():
    return C.CDLL(os.path.join(ROOT, "picopic_amd", "_lib", "libpicopic_unit.so"))


def ptr(a):
    return a.ctypes.data_as(C.c_void_p)


def keys(lengths):
    return np.repeat(np.arange(len(lengths)), lengths)[:64].astype(np.uint32)


@pytest.mark.parametrize("lengths", [[64], [1] * 64, [2] * 32, [1, 15, 1, 31, 16], [17, 16, 31], [3, 60, 1], [63, 1],
                                     [1, 63], [16, 16, 16, 16], [5, 7, 9, 11, 13, 19]])
def test_joined_run_sums_equal_the_single_ones(lengths):
    """Three and four values at once, some of them equal to the runs' masks: bit for bit run_sum_f's, whose sums at a
    run's last lane are the run's."""
    key = keys(lengths)
    x = np.random.default_rng(len(lengths)).normal(0, 1e3, 64).astype(np.float32)
    one, three, four = (np.zeros((4, 64), np.float32) for _ in range(3))
    print("run sums", lengths, flush=True)
    for form, out in ((1, one), (3, three), (4, four)):
        assert unit().unit_run_sums(form, ptr(key), ptr(x), ptr(out)) == 0
    last = np.append(key[1:] != key[:-1], True)
    total = np.array([x[key == k].astype(np.float64).sum() for k in key])
    assert np.abs(one[3] - total)[last].max() <= 64 * 2.0 ** -24 * np.abs(x).sum()
    assert np.array_equal(four[:, last], one[:, last])
    assert np.array_equal(three[:3, last], one[:3, last])
