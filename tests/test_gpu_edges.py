"""Edge cases of the step on the device against the oracle: a species with
no particles, species whose counts are not multiples of a wavefront (1, 63,
65, 129 particles: partial trips, partial 4-particle fix-up groups), in one
and in four domains (the single-domain specialisation and the general
kernel), both precisions and both deposition schemes.  Three steps from
random fields; particles are compared by id, fields over the interior."""
import numpy as np
import pytest

from oracle import oracle as O
from tests import helpers as Hh

pytestmark = pytest.mark.gpu


def _pair(precision, ccs, domains, counts, seed=5):
    from picopic_amd import capi
    size, grid = Hh.geometry(16, 32)
    dt = 0.5 * (size[1] / grid[1]) / 3e8
    species = Hh.species_list(True)
    orc = O.SMB(size, grid, domains, dt, species, pusher="boris-adaptive", ccs=ccs)
    gpu = capi.Context(size, grid, domains, dt, [s + (max(4 * n, 16),) for s, n in zip(species, counts)],
                       pusher="boris-adaptive", ccs=ccs, precision=precision)
    rng = np.random.default_rng(seed)
    dr, dz = size[0] / grid[0], size[1] / grid[1]
    for sp, ((q, m, b), n) in enumerate(zip(species, counts)):
        if n == 0:
            continue
        r, z, vr, vp, vz, w = Hh.make_particles(rng, size, grid, n, m, fast_fraction=0.3, special=False,
                                                temp_ev=1.0 if m == 1 else 0.1)
        if precision == "fp32":
            # both sides start from the FP32-representable state
            ir, iz = np.floor(r / dr), np.floor(z / dz)
            r = (ir + (r / dr - ir).astype(np.float32).astype(np.float64)) * dr
            z = (iz + (z / dz - iz).astype(np.float32).astype(np.float64)) * dz
            vr, vp, vz, w = (a.astype(np.float32).astype(np.float64) for a in (vr, vp, vz, w))
        ids = np.arange(n, dtype=np.uint64) + np.uint64(sp * 10 ** 6)
        orc.add_particles(sp, r, z, vr, vp, vz, w, ids)
        gpu.upload(sp, r, z, vr, vp, vz, w, ids)
    E, H, Hat = Hh.random_fields(rng, orc.n_domains, orc.nr_d, orc.nz_d)
    if precision == "fp32":
        E, H, Hat = (a.astype(np.float32).astype(np.float64) for a in (E, H, Hat))
    for name, arr in (("E", E), ("H", H), ("H_at_et", Hat)):
        orc.set_grid(name, arr)
        gpu.set_grid(name, arr)
    return orc, gpu, species


def _by_id(p):
    o = np.argsort(p["id"])
    return {k: v[o] for k, v in p.items()}


@pytest.mark.parametrize("counts", [(0, 65, 1), (63, 0, 129)])
@pytest.mark.parametrize("domains", [(1, 1), (2, 2)])
@pytest.mark.parametrize("ccs", ["zigzag", "vb"])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_empty_and_ragged_species(precision, ccs, domains, counts):
    print("case", precision, ccs, domains, counts, flush=True)
    orc, gpu, species = _pair(precision, ccs, domains, counts)
    tol_p, tol_f = (1e-12, 1e-12) if precision == "fp64" else (1e-5, 1e-4)
    orc.step(3)
    gpu.step(3)
    for sp in range(len(species)):
        a, b = _by_id(orc.particles(sp)), _by_id(gpu.particles(sp))
        assert len(a["id"]) == len(b["id"]) == gpu.count(sp)
        if counts[sp] == 0 or len(a["id"]) == 0:
            assert len(b["id"]) == len(a["id"])
            continue
        assert np.array_equal(a["id"], b["id"])
        for k in ("r", "z", "vr", "vphi", "vz"):
            e = Hh.relerr(b[k], a[k])
            assert e <= tol_p, (sp, k, e)
    for nm in ("E", "H", "J"):
        e = Hh.relerr(gpu.get_grid(nm)[:, :, 2:-2, 2:-2], orc.get_grid(nm)[:, :, 2:-2, 2:-2])
        print(nm, e)
        assert e <= tol_f, (nm, e)


@pytest.mark.parametrize("speed", [3.1e8, 1e200, np.inf])
@pytest.mark.parametrize("pusher", ["boris-adaptive", "vay", "hc"])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_faster_than_light_is_an_error(precision, pusher, speed):
    """Also where v^2 / c^2 overflows: the step reports it rather than dropping the particle in silence."""
    from picopic_amd import capi
    ctx = capi.Context((8e-3, 8e-3), (8, 8), (1, 1), 1e-13, [(-1, 1, False, 64)], pusher=pusher, precision=precision)
    x, zero = np.full(3, 4.2e-3), np.zeros(3)
    print("beta", precision, pusher, speed, flush=True)
    with np.errstate(over="ignore"):
        ctx.upload(0, x, x, zero, zero, np.array([1e6, speed, 2e6]), zero + 1e6)
        with pytest.raises(capi.PcpError, match="0x2|0x3"):
            ctx.step(1)
            ctx.sync()


@pytest.mark.parametrize("ccs", ["zigzag", "vb"])
def test_phases_before_the_collector_leave_out_particles_past_the_grid(ccs):
    """Deposit and push between the phases "move" and "migrate": particles past the walls have no cell; the others'
    current and velocities are those of a run without them."""
    from picopic_amd import capi
    size, grid, dt = (8e-3, 8e-3), (8, 8), 2e-12
    rng = np.random.default_rng(4)
    n, m = 40, 10
    r, z = rng.uniform(1e-3, 6e-3, n + m), rng.uniform(1e-3, 6e-3, n + m)
    vr, vz, zero = rng.normal(0, 1e7, n + m), rng.normal(0, 1e7, n + m), np.zeros(n + m)
    r[n:n + m // 2], vr[n:n + m // 2] = 7.9e-3, 2e8
    z[n + m // 2:], vz[n + m // 2:] = 7.9e-3, 2e8
    out = []
    print("before the collector", ccs, flush=True)
    for k in (n, n + m):
        ctx = capi.Context(size, grid, (2, 2), dt, [(-1, 1, True, 64)], ccs=ccs)
        ctx.upload(0, r[:k], z[:k], vr[:k], zero[:k], vz[:k], zero[:k] + 1e6, np.arange(k, dtype=np.uint64))
        E, H, Hat = Hh.random_fields(np.random.default_rng(5), 4, 4, 4)
        for name, a in (("E", E), ("H", H), ("H_at_et", Hat)):
            ctx.set_grid(name, a)
        for ph in ("move", "deposit", "push", "migrate"):
            ctx.phase(ph)
        p = _by_id(ctx.particles(0))
        out.append((ctx.get_grid("J"), p))
        assert len(p["id"]) == n
    (ja, a), (jb, b) = out
    assert np.abs(ja).max() > 0 and np.abs(ja - jb).max() <= 1e-12 * np.abs(ja).max()
    for k in ("r", "z", "vr", "vz"):
        assert np.array_equal(a[k], b[k]), k
