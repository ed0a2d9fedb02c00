"""Grouped collision cells at the edges of their size classes.

Cells are collided in groups of one size class (at most 16, 32, 64, 128 or 256
particles of either species), their pairs as dense lists over the group.  One
pass against the oracle's keyed pass, for cells at and next to every class
edge, odd and even, equal and unequal counts, and with more cells than one
group holds.  Tolerances: P12, whose like pairs' relative speed is a round-off,
as reasoned below; TA77S and SK98, whose operations are the oracle's one by one,
last-ulp library differences.
"""
import numpy as np
import pytest

from picopic_amd import capi
from tests.test_gpu_collisions import build, compare, plasma

pytestmark = pytest.mark.gpu

EDGES = [(1, 1), (1, 2), (2, 1), (3, 3), (4, 9), (15, 16), (16, 16), (17, 5), (16, 17), (31, 32), (32, 33), (63, 64),
         (64, 65), (65, 2), (127, 128), (128, 129), (129, 31), (255, 256), (256, 256), (256, 3), (2, 255), (257, 40)]


@pytest.mark.parametrize("scheme", ["p12", "ta77s", "sk98"])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_class_edges_match_the_oracle(scheme, precision):
    rng = np.random.default_rng(41)
    grid = (2, len(EDGES))
    ce, ci = np.array([[e for e, _ in EDGES]] * 2), np.array([[i for _, i in EDGES]] * 2)
    ce[1], ci[1] = ci[0].copy(), ce[0].copy()
    if scheme == "ta77s":
        # single particles divide round-off by round-off in the energy correction
        ce, ci = np.maximum(ce, 2), np.maximum(ci, 2)
    fp32 = precision == "fp32"
    data = plasma(rng, grid, (grid[0] * 1e-4, grid[1] * 1e-4), ce, ci, fp32=fp32,
                  weights="mixed" if scheme == "ta77s" else "equal")
    orc, gpu = build(grid, (1, 1), data, precision)
    print("class edges", scheme, precision, flush=True)
    orc.collide(scheme, 0, 1, seed=13, step=1)
    gpu.collide(scheme, 0, 1, 13, 1)
    # a like pair's round-off turns its velocity by up to sqrt(2 eps) = 2.1e-8 of the pair's speed
    print(compare(orc, gpu, 1e-6 if fp32 else 2.2e-8 if scheme == "p12" else 1e-12))


def test_many_groups_match_the_oracle():
    rng = np.random.default_rng(42)
    grid = (20, 30)
    ce, ci = rng.integers(0, 40, grid), rng.integers(0, 40, grid)
    ce[ce < 2], ci[ci < 2] = 2, 2
    data = plasma(rng, grid, (grid[0] * 1e-4, grid[1] * 1e-4), ce, ci, weights="mixed")
    orc, gpu = build(grid, (2, 3), data, "fp64")
    print("many groups", flush=True)
    orc.collide("ta77s", 0, 1, seed=3, step=5)
    gpu.collide("ta77s", 0, 1, 3, 5)
    print(compare(orc, gpu, 1e-12))


def test_equal_shuffle_keys_keep_every_particle():
    """Particles with one id draw one shuffle key: every one still takes a place of its own, so each pair's momentum
    and energy (equal weights) stay with the cell."""
    rng = np.random.default_rng(43)
    grid = (2, 3)
    size = (grid[0] * 1e-4, grid[1] * 1e-4)
    c = np.full(grid, 24)
    data = [d[:6] + (np.zeros(len(d[0]), dtype=np.uint64),) for d in plasma(rng, grid, size, c, c)]
    species = [(-1, 1, False, 512), (1, 1836, False, 512)]
    gpu = capi.Context(size, grid, (1, 1), 1e-10, species)
    for sp, d in enumerate(data):
        gpu.upload(sp, *d)
    print("equal keys", flush=True)
    gpu.collide("p12", 0, 1, 3, 0)
    after = [gpu.particles(s) for s in (0, 1)]

    def momentum(v):
        return v / np.sqrt(1.0 - (v ** 2).sum(0) / 9e16)

    p0 = [m * momentum(np.stack(data[s][2:5])) for s, m in enumerate((9.1e-31, 1836 * 9.1e-31))]
    p1 = [m * momentum(np.stack([after[s][k] for k in ("vr", "vphi", "vz")]))
          for s, m in enumerate((9.1e-31, 1836 * 9.1e-31))]
    assert not any(np.array_equal(a, b) for a, b in zip(p0, p1))
    # 144 pairs a species, a few ulp of the pair's momentum each
    drift = np.abs(sum(p.sum(1) for p in p1) - sum(p.sum(1) for p in p0))
    assert (drift <= 1e-12 * sum(np.abs(p).sum() for p in p0)).all(), drift
