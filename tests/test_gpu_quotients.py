"""FP64 quotients with shared reciprocals keep the reference's rounding.

The helpers themselves bit for bit, and one push, move and deposit of the FP64 step's own arithmetic against the oracle
(IEEE divisions) over the coordinates where a quotient decides a cell: on cell edges, one ulp beside them and in the
first and last cells.  Velocities and positions: 1e-14 relative (the device's pow and sqrt sequences differ from libm
in the last ulp at most); the current: 1e-12 of its largest value (the sums' order).
"""
import ctypes as C
import os

import numpy as np
import pytest

from oracle import oracle as O
from picopic_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ccs", ["vb", "zigzag"])
@pytest.mark.parametrize("pusher", ["boris-adaptive", "vay", "hc"])
def test_cell_edges(pusher, ccs):
    grid, domains = (12, 20), (2, 2)
    cell = (1.1e-3, 0.7e-3)
    size = (grid[0] * cell[0], grid[1] * cell[1])
    rng = np.random.default_rng(61)
    dr, dz = cell
    r, z = [], []
    for i in range(1, grid[0]):
        for k in range(1, grid[1]):
            for step in (-1, 0, 1):
                a, b = i * dr, k * dz
                r.append(np.nextafter(a, a + step) if step else a)
                z.append(np.nextafter(b, b - step) if step else b)
    r, z = np.array(r), np.array(z)
    n = len(r)
    v = rng.normal(0, 6e6, (3, n))
    w = rng.uniform(0.5, 1.5, n) * 1e6
    dt = 0.5 * dz / 3e8
    species = [(-1, 1, False)]
    orc = O.SMB(size, grid, domains, dt, species, pusher=pusher, ccs=ccs)
    gpu = capi.Context(size, grid, domains, dt, [s + (n + 8,) for s in species], pusher=pusher, ccs=ccs)
    ids = np.arange(n, dtype=np.uint64)
    orc.add_particles(0, r, z, *v, w, ids)
    gpu.upload(0, r, z, *v, w, ids)
    shape = (4, 3, grid[0] // 2 + 4, grid[1] // 2 + 4)
    for name, scale in (("E", 2e5), ("H", 300.0), ("H_at_et", 300.0)):
        F = rng.normal(0, scale, shape)
        orc.set_grid(name, F)
        gpu.set_grid(name, F)
    print("cell edges", pusher, ccs, flush=True)
    orc.step(1)
    gpu.step(1)
    a, b = orc.particles(0), gpu.particles(0)
    ia, ib = np.argsort(a["id"]), np.argsort(b["id"])
    assert np.array_equal(a["id"][ia], b["id"][ib])
    for k in ("r", "z", "vr", "vphi", "vz"):
        assert np.abs(a[k][ia] - b[k][ib]).max() <= 1e-14 * np.abs(a[k]).max(), k
    ja, jb = (s.get_grid("J")[:, :, 2:-2, 2:-2] for s in (orc, gpu))
    # a particle exactly on a ring's edge that leaves it outwards has no radial path there: 0 / 0 in both
    finite = np.isfinite(ja)
    assert finite.mean() > 0.95
    assert np.array_equal(finite, np.isfinite(jb))
    assert np.abs(ja - jb)[finite].max() <= 1e-12 * np.abs(ja[finite]).max()


ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def helpers(a, b):
    lib = C.CDLL(os.path.join(ROOT, "picopic_amd", "_lib", "libpicopic_unit.so"))
    a, b = (np.ascontiguousarray(x, dtype=np.float64) for x in (a, b))
    out = np.zeros((5, len(a)))
    rc = lib.unit_quotients(C.c_long(len(a)), *(x.ctypes.data_as(C.c_void_p) for x in (a, b, out)))
    assert rc == 0
    return out


def test_helpers_round_as_ieee_division_and_square_root():
    """Ordinary operands: every quotient, root and c^2 quotient bit for bit."""
    rng = np.random.default_rng(71)
    n = 1 << 20
    near = rng.uniform(1, 2, n)
    sets = [(rng.normal(0, 1, n), near),
            (near, np.nextafter(near, 2)),
            (rng.uniform(-1, 1, n) * 10.0 ** rng.integers(-60, 60, n), 10.0 ** rng.uniform(-80, 80, n)),
            (rng.integers(1, 1 << 20, n).astype(np.float64), rng.integers(1, 1 << 20, n).astype(np.float64)),
            (np.zeros(n), near)]
    for k, (a, b) in enumerate(sets):
        print("quotients", k, flush=True)
        q, q2, root, c2, _ = helpers(a, b)
        assert np.array_equal(q, a / b) and np.array_equal(q2, a / b), k
        assert np.array_equal(root, np.sqrt(b)), k
        assert np.array_equal(c2, a / 9e16), k


@pytest.mark.parametrize("dx", [1e-3, 1e-6, 0.0375 / 128, 0.15 / 256, 1.1e-3, 0.7e-3, 0.7, 1.0])
def test_cells_are_those_of_the_ieee_quotient(dx):
    """The cell of a coordinate is floor(x / dx) on and beside every edge, as the upload's check has it: one particle
    may not be in two cells."""
    i = np.arange(-3, 9000, dtype=np.float64)
    x = [i * dx, i / (1 / dx)]
    for _ in range(2):
        x += [np.nextafter(x[0], np.inf), np.nextafter(x[0], -np.inf)]
        x[0] = np.nextafter(x[0], np.inf)
    x = np.concatenate(x + [np.random.default_rng(72).uniform(0, 9000 * dx, 1 << 18), [1e300, -1e300]])
    cell = helpers(x, np.full(len(x), dx))[4]
    # coordinates past the range of an int stay past every grid
    assert np.array_equal(cell, np.clip(np.floor(x / dx), -2.0 ** 31, 2.0 ** 31 - 1))
