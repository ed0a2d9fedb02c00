"""Species maps of particles in any storage order.

The map deposit sums equal cells along the storage; a large species out of cell
order goes through an index list in cell order (from 65,537 particles for the
temperature and momentum maps and 131,073 for the energy, never for the
density).  The same particles before and after the sort give the same maps up to the order of the FP64 sums (every node
collects at most a few thousand like-signed terms: 1e-12 of the largest value),
and the oracle's.
"""
import numpy as np
import pytest

from oracle import oracle as O
from picopic_amd import capi

pytestmark = pytest.mark.gpu


def particles(rng, size, grid, n, order):
    dr, dz = size[0] / grid[0], size[1] / grid[1]
    r = np.sqrt(rng.uniform((0.3 * dr) ** 2, (size[0] - 0.5 * dr) ** 2, n))
    z = rng.uniform(0.5 * dz, size[1] - 0.5 * dz, n)
    # a crowded cell, more particles than a workgroup takes at once
    m = n // 3
    r[:m], z[:m] = rng.uniform(2.1, 2.9, m) * dr, rng.uniform(3.1, 3.9, m) * dz
    v = rng.normal(0, 4e7, (3, n))
    v *= np.minimum(1.0, 2.5e8 / np.maximum(np.linalg.norm(v, axis=0), 1.0))
    w = rng.uniform(0.5, 1.5, n) * 1e7
    if order == "cells":
        k = np.lexsort((np.floor(z / dz), np.floor(r / dr)))
        r, z, v, w = r[k], z[k], v[:, k], w[k]
    r, z, w = (a.astype(np.float32).astype(np.float64) for a in (r, z, w))
    return r, z, *(c.astype(np.float32).astype(np.float64) for c in v), w


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("n,order", [(1, "random"), (63, "random"), (65, "cells"), (5000, "random"), (5000, "cells"),
                                     (65537, "random"), (131073, "random"), (131073, "cells")])
def test_maps_do_not_depend_on_the_storage_order(precision, n, order):
    size, grid, domains = (12e-3, 20e-3), (12, 20), (2, 2)
    rng = np.random.default_rng(51)
    p = particles(rng, size, grid, n, order)
    species = [(-1, 1, False)]
    orc = O.SMB(size, grid, domains, 1e-13, species)
    gpu = capi.Context(size, grid, domains, 1e-13, [s + (n + 8,) for s in species], precision=precision)
    orc.add_particles(0, *p, np.arange(n, dtype=np.uint64))
    gpu.upload(0, *p)
    kinds = ("density", "energy", "temperature", "momentum")
    print("maps", precision, n, order, flush=True)
    first = {k: gpu.species_map(0, k)[:, :, 2:-2, 2:-2] for k in kinds}
    gpu.sort(0)
    ref = {k: orc.species_map(0, k)[:, :, 2:-2, 2:-2] for k in kinds}
    for k in kinds:
        again = gpu.species_map(0, k)[:, :, 2:-2, 2:-2]
        # the temperature is the difference of two energies: its error is the energies'
        scale = np.abs(ref["energy" if k == "temperature" else k]).max()
        assert np.abs(first[k] - again).max() <= 1e-12 * scale, k
        # FP32: positions rounded to 2^-24 of a cell against clouds that reach a node with 1e-3 of a cell or more
        assert np.abs(first[k] - ref[k]).max() <= (1e-12 if precision == "fp64" else 1e-4) * scale, k


@pytest.mark.parametrize("vz", [np.inf, -np.inf, 1e300, 4e8])
def test_particles_outside_the_grid_are_in_no_map(vz):
    """Between the phases "move" and "migrate" a particle may lie anywhere, also at an infinite longitude."""
    size, grid = (8e-3, 8e-3), (8, 8)
    maps = []
    for n in (2, 3):
        ctx = capi.Context(size, grid, (2, 2), 1e-10, [(-1, 1, True, 16)])
        x, zero = np.full(n, 4.2e-3), np.zeros(n)
        v = np.array([1e6, 2e6, vz])[:n]
        ctx.upload(0, x, x, zero, zero, v, zero + 1e6)
        print("outside", n, vz, flush=True)
        ctx.phase("move")
        maps.append([ctx.species_map(0, k)[:, :, 2:-2, 2:-2] for k in ("density", "energy", "momentum")])
    for a, b in zip(*maps):
        assert np.isfinite(a).all() and a.any()
        assert np.abs(a - b).max() <= 1e-12 * np.abs(a).max()
