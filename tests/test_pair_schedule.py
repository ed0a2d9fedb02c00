"""The unlike pairs of collision cells for every pair of counts (CPU).

The chains in closed form, which grouped and crowded cells run, against the
reference's loops (collisionsP12.cpp:420-528): particle f of the more numerous
species meets particle floor(f / (c + 1)) of the other in the 1st group and
floor(f / c) past the 1st group's in the 2nd, in the loops' order.
"""
import ctypes as C
import os

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
U = C.CDLL(os.path.join(ROOT, "picopic_amd", "_lib", "libpicopic_unit.so"))
U.unit_unlike_pairs.restype = C.c_long


def reference(nel, nion):
    lo, hi = min(nel, nion), max(nel, nion)
    if lo == hi:
        return np.arange(lo), np.arange(lo)
    ratio = np.float32(hi) / np.float32(lo)
    c = float(np.floor(ratio))
    rest = float(ratio) - c
    first, small, second = int((c + 1) * rest * lo), int(rest * lo), int(c * (1 - rest) * lo)
    f1, f2 = np.arange(first), np.arange(second)
    e1 = np.floor(f1.astype(np.float32) / np.float32(c + 1)).astype(int)
    e2 = np.floor(f2.astype(np.float32) / np.float32(c)).astype(int) + small
    near, far = np.concatenate([e1, e2]), np.concatenate([f1, f2 + first])
    keep = (near < lo) & (far < hi)
    near, far = near[keep], far[keep]
    order = np.argsort(near, kind="stable")
    return near[order], far[order]


def check(nel, nion):
    near, far = (np.full(nel + nion + 8, -7, np.int32) for _ in range(2))
    n = U.unit_unlike_pairs(nel, nion, near.ctypes.data_as(C.c_void_p), far.ctypes.data_as(C.c_void_p))
    a, b = reference(nel, nion)
    assert n == len(a), (nel, nion)
    assert np.array_equal(near[:n], a) and np.array_equal(far[:n], b), (nel, nion)
    # independent chains: a particle of the more numerous species is in one pair
    assert len(np.unique(b)) == len(b), (nel, nion)


@pytest.mark.parametrize("lo", range(1, 258, 32))
def test_every_pair_of_counts_of_grouped_cells(lo):
    for a in range(lo, min(lo + 32, 258)):
        for b in range(a, 258):
            check(a, b)
            check(b, a)


def test_counts_of_crowded_cells():
    rng = np.random.default_rng(3)
    for a, b in [(1, 100000), (2, 100001), (257, 4096), (3000, 3001), (40, 700), (99991, 100003), (1000, 999000)]:
        check(a, b)
        check(b, a)
    for _ in range(300):
        check(int(10 ** rng.uniform(0, 4.5)), int(10 ** rng.uniform(2.4, 4.5)))
