"""FP32 currents of wavefronts whose run sums take the bounded and the general form.

Particles in cell order, `ppc` a cell: from one run a wavefront to a run a lane.  A heavy particle's contributions pass
the bound that the multiply-add form needs and must not reach the cells beside its own.  Against the FP64 oracle; a
node's FP32 sum of up to a few hundred terms errs by at most 2e-5 of the largest current of its kind (heavy or not).
"""
import numpy as np
import pytest

from oracle import oracle as O
from picopic_amd import capi

pytestmark = pytest.mark.gpu

GRID = (8, 24)


def current(make, heavy, ccs, domains, ppc):
    cell = 1e-6
    dt = 0.25 * cell / 3e8
    rng = np.random.default_rng(5 + ppc)
    cr, cz = (a.repeat(ppc) for a in np.divmod(np.arange(3 * 18) , 18))
    n = len(cr)
    # offsets of 8 bits: exact in FP32; moves of about a sixth of a cell, so that some particles change cells
    r = (cr + 3 + rng.integers(20, 236, n) / 256) * cell
    z = (cz + 3 + rng.integers(20, 236, n) / 256) * cell
    v = np.clip(rng.normal(0, 6e7, (3, n)), -1.5e8, 1.5e8).astype(np.float32).astype(np.float64)
    w = np.full(n, 1e6)
    if heavy:
        w[n // 2] = 2e31
    s = make((GRID[0] * cell, GRID[1] * cell), GRID, domains, dt, [(-1, 1, False)], ccs, n)
    s[1](0, r, z, *v, w, np.arange(n, dtype=np.uint64))
    s[0].step(1)
    return s[0].get_grid("J")[:, :, 2:-2, 2:-2]


def oracle(size, grid, domains, dt, species, ccs, n):
    s = O.SMB(size, grid, domains, dt, species, pusher="vay", ccs=ccs)
    return s, s.add_particles


def device(size, grid, domains, dt, species, ccs, n):
    s = capi.Context(size, grid, domains, dt, [x + (n,) for x in species], pusher="vay", ccs=ccs, precision="fp32")
    return s, s.upload


@pytest.mark.parametrize("ppc", [1, 3, 7, 70])
@pytest.mark.parametrize("ccs,domains", [("zigzag", (1, 1)), ("zigzag", (2, 2)), ("vb", (2, 2))])
def test_run_sums(ccs, domains, ppc):
    light = current(oracle, False, ccs, domains, ppc)
    mixed = current(oracle, True, ccs, domains, ppc)
    print("run sums", ccs, domains, ppc, flush=True)
    got = current(device, False, ccs, domains, ppc)
    assert np.abs(got - light).max() <= 2e-5 * np.abs(light).max()
    got = current(device, True, ccs, domains, ppc)
    hit = mixed != light
    assert hit.any() and np.abs(mixed).max() > 2.0 ** 120
    assert np.abs(got - mixed)[~hit].max() <= 2e-5 * np.abs(light).max()
    assert np.abs(got - mixed)[hit].max() <= 2e-5 * np.abs(mixed).max()


@pytest.mark.parametrize("ccs,domains", [("zigzag", (1, 1)), ("zigzag", (2, 2)), ("vb", (2, 2))])
def test_particles_at_rest_deposit_nothing(ccs, domains):
    """Wavefronts of particles at rest skip the sums; with one moving particle among them its current is the oracle's."""
    cell = 1e-6
    n = 150
    size = (GRID[0] * cell, GRID[1] * cell)
    r, z = np.full(n, 3.375 * cell), np.full(n, 5.625 * cell)
    w, ids = np.full(n, 1e6), np.arange(n, dtype=np.uint64)
    for moving in (0, 1):
        v = np.zeros((3, n))
        v[:, 70] = moving * np.array([3e7, 2e7, -4e7])
        out = []
        print("rest", ccs, domains, moving, flush=True)
        for make in (oracle, device):
            s, add = make(size, GRID, domains, 0.25 * cell / 3e8, [(-1, 1, False)], ccs, n)
            add(0, r, z, *v, w, ids)
            s.step(1)
            out.append(s.get_grid("J")[:, :, 2:-2, 2:-2])
        if ccs == "zigzag" and not moving:
            assert not out[1].any()
        assert np.abs(out[1] - out[0]).max() <= 2e-5 * np.abs(out[0]).max()
