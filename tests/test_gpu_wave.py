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


def patterns():
    rng = np.random.default_rng(7)
    lane = np.arange(64)
    yield "one", np.zeros(64), np.ones(64)
    yield "two in turn", lane % 2, np.ones(64)
    yield "eight in turn", lane % 8, np.ones(64)
    yield "nine in turn", lane % 9, np.ones(64)
    yield "all different", lane, np.ones(64)
    yield "sorted", lane // 7, np.ones(64)
    yield "eight runs, two keys", lane // 8 % 2, np.ones(64)
    yield "two in turn, half inactive", lane % 2, lane // 2 % 2
    yield "none", lane, np.zeros(64)
    yield "last", lane, lane == 63
    for n in (3, 12, 40):
        yield "random %d" % n, rng.integers(0, n, 64), rng.random(64) < 0.8


@pytest.mark.parametrize("name,key,active", list(patterns()), ids=[p[0] for p in patterns()])
def test_reserving_lanes_form_groups(name, key, active):
    """Every active lane has a place of its own among its key's, and few lanes ask: one a run, and where there are
    more than eight runs at most one for each of eight keys."""
    key, active = key.astype(np.uint32) + 5, active.astype(np.int32)
    out = np.zeros((3, 64), np.int32)
    print("groups", name, flush=True)
    assert unit().unit_reserve_groups(ptr(key), ptr(active), ptr(out)) == 0
    head, size, rank = (a[active != 0] for a in out)
    k, lanes = key[active != 0], np.flatnonzero(active)
    for h in np.unique(head):
        g = head == h
        assert h in lanes and len(np.unique(k[g])) == 1 and k[g][0] == key[h]
        assert (size[g] == g.sum()).all() and np.array_equal(np.sort(rank[g]), np.arange(g.sum()))
    runs = int(active[0] + ((active[1:] != 0) & ((key[1:] != key[:-1]) | (active[:-1] == 0))).sum())
    asked, different = len(np.unique(head)), len(np.unique(k))
    assert asked <= runs
    if runs > 8 and different <= 8:
        assert asked == different
