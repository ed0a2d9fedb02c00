"""Positions next to the outer edges of the grid and past them.

A coordinate within 2^-25 of a cell below the grid's end has an FP32 in-cell
offset that rounds to 1, which must not carry it into the cell past the last
one (the sort's counters and the field grids end there).  A beam's particles
placed past the grid are removed.
"""
import numpy as np
import pytest

from oracle import oracle as O
from picopic_amd import capi

pytestmark = pytest.mark.gpu

CELL = 1e-3


def check(ctx, grid):
    p = ctx.particles(0)
    assert (p["r"] < grid[0] * CELL).all() and (p["z"] < grid[1] * CELL).all()
    return p


@pytest.mark.parametrize("domains", [(1, 1), (2, 2)])
def test_uploaded_particles_stay_in_the_last_cell(domains):
    grid = (8, 16)
    ctx = capi.Context((grid[0] * CELL, grid[1] * CELL), grid, domains, 1e-13, [(-1, 1, False, 64)], precision="fp32")
    u = np.array([[8 - 1e-9, 5.5], [7.5, 16 - 1e-9], [8 - 1e-9, 16 - 1e-9], [3 - 1e-9, 4.5], [2.25, 3.125]])
    z = np.zeros(len(u))
    ctx.upload(0, u[:, 0] * CELL, u[:, 1] * CELL, z, z, z, z + 1e6)
    print("upload", domains, flush=True)
    p = check(ctx, grid)
    # positions keep 2^-24 of a cell
    assert np.abs(p["r"] / CELL - u[:, 0]).max() <= 2.0 ** -23
    assert np.abs(p["z"] / CELL - u[:, 1]).max() <= 2.0 ** -23


def test_initial_plasma_stays_in_the_last_cell():
    # with this seed particle 40689 of the outer row lies at r / dr = 2 - 2e-8
    grid = (2, 2)
    ctx = capi.Context((grid[0] * CELL, grid[1] * CELL), grid, (1, 1), 1e-13, [(-1, 1, False, 100000)],
                       precision="fp32")
    ctx.init_plasma(0, 20000, 1e17, 1e17, 1.0, 1427)
    print("init_plasma", flush=True)
    p = check(ctx, grid)
    assert len(p["r"]) == 80000 and p["r"].max() > (2 - 1e-6) * CELL


@pytest.mark.parametrize("radius", [0.9, 1.0, 1.25])
@pytest.mark.parametrize("domains", [(1, 1), (2, 2)])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_beam_as_wide_as_the_grid(precision, domains, radius):
    """A beam's particles reach half a cell past its radius: the ones outside the grid are removed, as the oracle's
    runaway collector does, and the rest are the oracle's, before and after steps."""
    size, grid, dt = (8.0, 8.0), (8, 8), 1.0
    species = [(-1, 1, False), (-1, 1, True)]
    orc = O.SMB(size, grid, domains, dt, species)
    dev = capi.Context(size, grid, domains, dt, [s + (4096,) for s in species], precision=precision)
    print("wide beam", precision, domains, radius, flush=True)
    for s in (orc, dev):
        s.set_beam(1, 900, 0.0, radius * size[0], 1e-12, 1, 3.0, 2.0, 1.0, seed=5)
        for _ in range(3):
            s.inject()
            s.set_time(s.time() + dt)
    a, b = orc.particles(1), dev.particles(1)
    ia, ib = np.argsort(a["id"]), np.argsort(b["id"])
    assert len(ia) > 500 and np.array_equal(a["id"][ia], b["id"][ib])
    for k in ("r", "z", "vz", "w"):
        tol = 0 if precision == "fp64" else 1e-6
        assert np.abs(a[k][ia] - b[k][ib]).max() <= tol * np.abs(a[k]).max(), k
    assert b["r"].max() < size[0]
    for s in (orc, dev):
        s.step(2)
    assert orc.count(1) == dev.count(1)


@pytest.mark.parametrize("beam", [False, True])
@pytest.mark.parametrize("grid,domains", [((2, 2), (1, 1)), ((8, 16), (2, 2)), ((9, 7), (3, 1))])
@pytest.mark.parametrize("ccs", ["zigzag", "vb"])
def test_moves_next_to_the_walls_stay_in_the_grid(ccs, grid, domains, beam):
    """FP32 steps of particles within 2^-26 .. 2^-2 of a cell of walls and corners, at all speeds: every stored cell is
    one of the grid's, before and after a sort, and the maps of the particles are finite."""
    n = 4000
    rng = np.random.default_rng(grid[0] + 10 * beam)
    dt = 0.5 * CELL / 3e8
    edge = 2.0 ** -rng.uniform(2, 26, (2, n))
    # plasma is mirrored half a cell inside the walls, a beam only at the axis
    low, high = (0.5, 0.5) if not beam else (0.5, 0.0)
    u = np.where(rng.random(n) < 0.5, low + edge[0], grid[0] - high - edge[0])
    w = np.where(rng.random(n) < 0.5, (0.0 if beam else 0.5) + edge[1], grid[1] - high - edge[1])
    v = rng.normal(size=(3, n))
    v *= 10.0 ** rng.uniform(-6, 8.4, n) / np.linalg.norm(v, axis=0)
    ctx = capi.Context((grid[0] * CELL, grid[1] * CELL), grid, domains, dt, [(-1, 1, beam, n)], ccs=ccs,
                       precision="fp32")
    ctx.upload(0, u * CELL, w * CELL, *v, np.full(n, 1e3))
    print("walls", ccs, grid, domains, beam, flush=True)
    for _ in range(3):
        ctx.step(1)
        p = check(ctx, grid)
        assert len(p["r"]) and (p["r"] >= 0).all() and (p["z"] >= 0).all()
        assert beam or len(p["r"]) == n
        ctx.sort(0)
        assert ctx.count(0) == len(p["r"])
        assert all(np.isfinite(ctx.species_map(0, k)).all() for k in ("density", "momentum"))
