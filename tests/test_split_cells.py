"""Cells of coordinates at and beyond the edges of the grid (CPU).

The FP32 split's cell indexes the sort's counters and, through its domain, the
field grids: it may not leave the grid, for any coordinate.  A coordinate
outside is refused, also where only its FP32 offset or a beam's half cell past
the wall carries it there; one inside keeps its place to 2^-24 of a cell.
"""
import ctypes as C
import os

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
U = C.CDLL(os.path.join(ROOT, "picopic_amd", "_lib", "libpicopic_unit.so"))


def ptr(a):
    return a.ctypes.data_as(C.c_void_p)


def split(u, n):
    u = np.ascontiguousarray(u, dtype=np.float64)
    inside, cell, f = np.zeros(len(u), np.int32), np.full(len(u), -9, np.int64), np.zeros(len(u), np.float32)
    U.unit_split(C.c_long(len(u)), ptr(u), C.c_long(n), ptr(inside), ptr(cell), ptr(f))
    return inside.astype(bool), cell, f


@pytest.mark.parametrize("n", [1, 2, 12, 125, 128, 511, 1024, 4096, 8192])
def test_cells_stay_in_the_grid(n):
    rng = np.random.default_rng(n)
    edges = np.arange(0, n + 2, dtype=np.float64)
    near = np.concatenate([edges + s for s in (-2.0 ** -20, -2.0 ** -25, -1e-9, -6e-10, -2.0 ** -40, 0, 1e-12)]
                          + [np.nextafter(edges, -1), np.nextafter(edges, n + 9)])
    # a beam's injection radius reaches n + 1/2
    u = np.concatenate([near, rng.uniform(0, n + 0.5, 20000), n - rng.uniform(0, 1e-6, 20000),
                        [np.nan, np.inf, -np.inf, -1.0, -1e-300, n + 1e6, 1e300]])
    inside, cell, f = split(u, n)
    assert np.array_equal(inside, (u >= 0) & (u < n))
    c, o = cell[inside], f[inside]
    assert c.min() >= 0 and c.max() < n
    assert (o >= 0).all() and (o < 1).all()
    assert np.abs(c + o.astype(np.float64) - u[inside]).max() <= 2.0 ** -24


def test_the_ion_that_left_the_grid():
    # ion 70107315 of a 1024-row ramp plasma: its offset rounds to 1 in the last cell
    inside, cell, f = split([1023.999999999404], 1024)
    assert inside[0] and cell[0] == 1023 and f[0] < 1


@pytest.mark.parametrize("dx", [1e-3, 1e-6, 0.0375 / 128, 0.15 / 256, 1.1e-3, 0.7])
def test_the_upper_limit_of_a_cell_is_in_it(dx):
    i = np.arange(9000, dtype=np.int64)
    x = np.zeros(len(i))
    U.unit_below_edge(C.c_long(len(i)), ptr(i), C.c_double(dx), ptr(x))
    for q in (x / dx, x * (1 / dx)):
        assert np.array_equal(np.floor(q), i)
    assert np.abs(x / dx - (i + 1)).max() <= 9000 * 2.0 ** -49
    # the neighbour below the edge is not such a limit everywhere
    if dx == 1e-3:
        assert (np.floor(np.nextafter((i + 1) * dx, 0.0) / dx) > i).any()


@pytest.mark.parametrize("dr,dz,nr,nz,bin_r,bin_z", [(1, 1, 8, 16, 1, 16), (8, 8, 128, 512, 16, 32), (8, 2, 128, 512, 16, 32),
                                                    (2, 4, 64, 64, 16, 32), (1, 1, 125, 511, 5, 7), (3, 2, 5, 9, 1, 3)])
def test_sort_keys_count_every_cell_once(dr, dz, nr, nz, bin_r, bin_z):
    cr, cz = (a.ravel().astype(np.int64) for a in np.meshgrid(np.arange(dr * nr), np.arange(dz * nz), indexing="ij"))
    key = np.zeros(len(cr), np.uint32)
    U.unit_sort_keys(C.c_long(len(cr)), ptr(cr), ptr(cz), dr, dz, nr, nz, bin_r, bin_z, ptr(key))
    assert np.array_equal(np.sort(key), np.arange(len(cr)))
