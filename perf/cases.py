"""The calls a user of picopic_amd makes, as cases with inputs, a pass and a tolerance.

Every case goes through ``picopic_amd.capi.Context`` (or ``picopic_amd.config``, which builds one) the way the
package's own main loop, benchmark and configurations do.  The kinds:

``functional``  a JSON configuration of the reference's functional test (PML, several domains, an injected beam,
                FP64, no graph): the smallest calls, where launches and latency count.
``step``        one dump interval of a plasma or beam-plasma run on the device-generated plasma: ``steps`` calls'
                worth of the particle loop with the step graph on, then the E, H and J frames.  Both precisions, both
                current schemes, the three pushers in use, with and without collisions in the step.
``upload``      the same on particles the caller made (single domain, ZigZag), where plain torch gives the result.
``phases``      the phase entry points one by one, as a driver does that keeps its own time loop, then the particles.
``relax``       collision passes alone (velocity relaxation of a plasma), then the temperature and momentum maps.
``maps``        a diagnostics frame: the species maps and the energies.
``train``       the collision surrogate's network: a gradient batch and the forward pass of the same rows.
"""
import math

import numpy as np
import torch

from picopic_amd import capi, config

C_LIGHT = 3e8
EL_CHARGE = 1.6e-19
EL_MASS = 9.1e-31
EPSILON0 = 8.85e-12
MAGN_CONST = 1.26e-6
PI = 3.1415926535897932
CELL = 1e-3
BUNCH = dict(n_peak=1e16, sigma_r=2e-3, sigma_z=5e-3, z0=0.1, gamma=5.0)
# normalisation of a surrogate network fitted on n = 2e16..5e17 m^-3, Te 0.3..3 eV, Ti 0.03..0.3 eV: feature
# means and deviations, target scales (the weights themselves are random)
NORM = ([17.0, 17.0, -0.05, -0.04, -1.03, math.log10(0.5 * CELL / C_LIGHT)], [0.41, 0.41, 0.31, 0.30, 0.29, 1e-4],
        [0.5, 0.5, 0.5, 0.5])
NPARAM = 64 * 32 + 64 + 64 * 64 + 64 + 16 * 64 + 16


def listed():
    step = dict(kind="step", density_left=1.0, bunch=0, collisions="none")
    return [
        # the reference's functional test: 81-step runs of a small beam-plasma case, dumped every 20 steps
        dict(name="functional", kind="functional", nr=128, nz=256, dom_r=2, dom_z=4, macro=210000, steps=20),
        # the committed uniform configuration: FP64, Villasenor-Buneman, 2 x 4 domains
        dict(step, name="uniform_fp64", nr=128, nz=512, dom_r=2, dom_z=4, ppc=16, precision="fp64", ccs="vb",
             pusher="boris-adaptive", steps=20),
        # a small beam-plasma run from the caller's own particles, odd sizes
        dict(name="beam_upload", kind="upload", nr=125, nz=511, ppc=15, bunch=30001, precision="fp32",
             pusher="boris-adaptive", steps=20),
        # the beam-plasma wakefield
        dict(step, name="wakefield", nr=512, nz=4096, dom_r=1, dom_z=1, ppc=64, precision="fp32", ccs="zigzag",
             pusher="boris-adaptive", bunch=1 << 20, steps=20),
        # uneven domains: a density ramp 0.1 n -> n over 8 x 8 domains
        dict(step, name="ramp_fp32", nr=1024, nz=4096, dom_r=8, dom_z=8, ppc=32, precision="fp32", ccs="vb",
             pusher="vay", density_left=0.1, steps=20),
        # the same in double precision, a quarter of the length
        dict(step, name="ramp_fp64", nr=1024, nz=1024, dom_r=8, dom_z=2, ppc=32, precision="fp64", ccs="vb",
             pusher="vay", density_left=0.1, steps=20),
        # the benchmark's full form: surrogate collisions in every step, the largest case
        dict(step, name="full", nr=1024, nz=8192, dom_r=8, dom_z=8, ppc=32, precision="fp32", ccs="zigzag",
             pusher="hc", bunch=1 << 20, collisions="surrogate", steps=20),
        # the full form's physics without a surrogate: double precision, P12 pairs in every step
        dict(step, name="full_p12", nr=512, nz=2048, dom_r=4, dom_z=2, ppc=32, precision="fp64", ccs="zigzag",
             pusher="hc", bunch=1 << 18, collisions="p12", steps=5),
        # a driver with its own time loop
        dict(name="phases", kind="phases", nr=128, nz=256, dom_r=2, dom_z=2, ppc=8, ccs="vb", pusher="boris-adaptive",
             steps=10),
        # velocity relaxation, cells from sparse (axis) to 128 per species
        dict(name="relax_p12", kind="relax", nr=256, nz=512, ppc=64, precision="fp32", scheme="p12", passes=4),
        # a diagnostics frame of every species map
        dict(name="maps", kind="maps", nr=128, nz=512, ppc=24, precision="fp64"),
        # a training batch of the surrogate
        dict(name="train", kind="train", rows=200000),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["functional", "step", "step", "step", "step", "step", "upload", "phases", "relax", "relax",
                       "maps", "train"])
    prec = rng.choice(["fp32", "fp64"])
    pusher = rng.choice(["boris-adaptive", "vay", "hc"])
    if kind == "functional":
        dr, dz = rng.choice([1, 2, 4]), rng.choice([1, 2, 4, 8])
        nr, nz = dr * rng.randint(24, 256 // dr), dz * rng.randint(32, 512 // dz)
        return dict(kind=kind, nr=nr, nz=nz, dom_r=dr, dom_z=dz, macro=int(_log(rng, 3e4, 1e6)),
                    steps=rng.randint(5, 30))
    if kind == "train":
        return dict(kind=kind, rows=int(_log(rng, 3000, 1000000)))
    if kind == "upload":
        return dict(kind=kind, nr=rng.randint(40, 200), nz=rng.randint(160, 600), ppc=rng.randint(4, 20),
                    bunch=int(_log(rng, 2000, 50000)), precision=prec, pusher=pusher, steps=rng.randint(6, 24))
    if kind == "phases":
        dr, dz = rng.choice([1, 2, 4]), rng.choice([1, 2, 4])
        return dict(kind=kind, nr=dr * rng.randint(16, 128 // dr), nz=dz * rng.randint(32, 320 // dz), dom_r=dr,
                    dom_z=dz, ppc=rng.randint(2, 12), ccs=rng.choice(["vb", "zigzag"]), pusher=pusher,
                    steps=rng.randint(5, 15))
    if kind == "maps":
        return dict(kind=kind, nr=rng.randint(32, 160), nz=rng.randint(100, 600), ppc=rng.randint(4, 24),
                    precision=prec)
    if kind == "relax":
        ppc = int(_log(rng, 6, 130))
        cells = _log(rng, 2e5, 1.5e7) / ppc
        nr = rng.randint(24, 200)
        return dict(kind=kind, nr=nr, nz=max(17, int(cells / nr)), ppc=ppc, precision=prec,
                    scheme=rng.choice(["p12", "ta77s", "sk98"]), passes=rng.randint(2, 5))
    coll = rng.choice(["none", "none", "p12", "surrogate"]) if prec == "fp32" else rng.choice(["none", "none", "p12"])
    ppc = int(_log(rng, 6, 80))
    cells = _log(rng, 6e5, 6e7 if coll != "p12" else 1.5e7) / ppc
    dr, dz = rng.choice([1, 2, 4]), rng.choice([1, 2, 4])
    nr = dr * max(12, int(math.sqrt(cells / rng.uniform(2, 9)) / dr))
    nz = dz * max(128 // dz + 1, int(cells / nr / dz))
    return dict(kind="step", nr=nr, nz=nz, dom_r=dr, dom_z=dz, ppc=ppc, precision=prec,
                ccs=rng.choice(["vb", "zigzag"]), pusher=pusher, density_left=rng.choice([1.0, 1.0, 0.1]),
                bunch=rng.choice([0, int(_log(rng, 3000, 300000))]), collisions=coll, steps=rng.randint(5, 20))


def _divisor(n, want):
    """The largest divisor of n that is at most `want`."""
    return max(d for d in range(1, want + 1) if n % d == 0)


def _tune(ctx, case, fp32):
    """The sort bin and plasma sort interval a user keeps from an autotuned run."""
    bin_r, bin_z = _divisor(case["nr"] // case["dom_r"], 16), _divisor(case["nz"] // case["dom_z"], 32)
    if bin_r * bin_z >= 64:
        ctx.set_sort_bin(bin_r, bin_z)
    if fp32:
        ctx.set_launch(512 if case["collisions"] != "none" or case["ccs"] == "vb" else 256, 0)
    for s in range(2):
        ctx.set_sort_interval(s, 16)


def _species(n_plasma, bunch):
    cap = n_plasma + n_plasma // 50 + 1024
    return [(-1, 1, False, cap), (1, 1836, False, cap)] + ([(-1, 1, True, bunch)] if bunch else [])


def _seeds(seed, n):
    return [int(x) for x in np.random.default_rng(seed).integers(1, 1 << 31, n)]


def _round32(x):
    return x.astype(np.float32).astype(np.float64)


def _particles(case, seed):
    """Particles on the host, uniform in r^2, with in-cell offsets, velocities and weights that FP32 holds."""
    rng = np.random.default_rng(seed)
    nr, nz = case["nr"], case["nz"]
    n = case["ppc"] * nr * nz
    out = []

    def place(r, z):
        ir, iz = np.floor(r), np.floor(z)
        return (ir + np.minimum(_round32(r - ir), 1 - 2.0 ** -24)) * CELL, (iz + np.minimum(_round32(z - iz), 1 - 2.0 ** -24)) * CELL

    for mass, temp in ((1.0, 1.0), (1836.0, 0.1)):
        r, z = place(np.sqrt(rng.uniform(0.36, (nr - 0.6) ** 2, n)), rng.uniform(0.6, nz - 0.6, n))
        v = rng.standard_normal((3, n), dtype=np.float32).astype(np.float64) * math.sqrt(temp * EL_CHARGE / (mass * EL_MASS))
        w = np.full(n, 1e17 * PI * (nr * CELL) ** 2 * nz * CELL / n)
        out.append((r, z, _round32(v[0]), _round32(v[1]), _round32(v[2]), _round32(w)))
    m = case.get("bunch", 0)
    if m:
        x = rng.normal(0, BUNCH["sigma_r"] / CELL, (2, m))
        r, z = place(np.clip(np.hypot(x[0], x[1]), 0.6, nr - 0.6),
                     np.clip(rng.normal(BUNCH["z0"] / CELL, BUNCH["sigma_z"] / CELL, m), 0.6, nz - 20.0))
        vz = np.full(m, C_LIGHT * math.sqrt(1 - BUNCH["gamma"] ** -2))
        w = np.full(m, BUNCH["n_peak"] * (2 * PI) ** 1.5 * BUNCH["sigma_r"] ** 2 * BUNCH["sigma_z"] / m)
        out.append((r, z, np.zeros(m), np.zeros(m), _round32(vz), _round32(w)))
    return out


def _batch(case, seed):
    rng = np.random.default_rng(seed)
    x = np.zeros((case["rows"], 8), dtype=np.float32)
    x[:, :6] = rng.uniform(-1.7, 1.7, (case["rows"], 6))
    t = rng.standard_normal((case["rows"], 4), dtype=np.float32)
    p = np.zeros(NPARAM, dtype=np.float32)
    o = 0
    for rows, used, cols, cused in ((64, 64, 32, 6), (64, 64, 64, 64), (16, 4, 64, 64)):
        a = math.sqrt(6.0 / (cused + used))
        m = np.zeros((rows, cols), dtype=np.float32)
        m[:used, :cused] = rng.uniform(-a, a, (used, cused))
        p[o:o + rows * cols] = m.ravel()
        o += rows * cols
        p[o:o + used] = rng.normal(0, 0.1, used)
        o += rows
    return x, t, p


def prepare(case, seed):
    kind = case["kind"]
    if kind == "functional":
        cfg = {
            "macro_amount": case["macro"], "beam_plasma_macro_size_ratio": 2,
            "geometry": {"size": {"radius": 0.0375, "longitude": 0.15},
                         "grid": {"radius": case["nr"], "longitude": case["nz"]},
                         "domains_amount": {"radius": case["dom_r"], "longitude": case["dom_z"]},
                         "pml": {"left_wall": 0, "right_wall": 0.05, "outer_wall": 0.2, "sigma_1": 1e-5,
                                 "sigma_2": 7e-2}},
            "time": {"start": 0, "end": 1e-11, "step": 1e-13},
            "particles": [{"name": "electrons", "charge": -1, "mass": 1, "density": 1e17, "temperature": 1},
                          {"name": "ions", "charge": 1, "mass": 1836, "density": 1e17, "temperature": 0.1}],
            "beams": [{"name": "electrons", "charge": -1, "mass": 1, "velocity": 2.8e8, "start_time": 0,
                       "bunch": {"amount": 2, "distance": 0.0914, "length": 0.0056, "radius": 0.005,
                                 "density": 1e16}}],
        }
        ctx, _ = config.context(cfg, seed=_seeds(seed, 1)[0])
        return dict(case=case, ctx=ctx)
    if kind == "train":
        x, t, p = _batch(case, seed)
        ctx = capi.Context((16 * CELL, 16 * CELL), (16, 16), (1, 1), 0.5 * CELL / C_LIGHT, [(-1, 1, False, 64)])
        ctx.mlp_set_params(p)
        return dict(case=case, ctx=ctx, x=x, t=t)
    nr, nz = case["nr"], case["nz"]
    size, grid = (nr * CELL, nz * CELL), (nr, nz)
    domains = (case.get("dom_r", 1), case.get("dom_z", 1))
    dt = 0.5 * CELL / C_LIGHT
    n = case["ppc"] * nr * nz
    s = _seeds(seed, 6)
    if kind == "relax":
        # dense enough for the passes to change the temperatures, as in a relaxation study
        ctx = capi.Context(size, grid, domains, 2e-10, _species(n, 0), precision=case["precision"])
        ctx.init_plasma(0, case["ppc"], 1e20, 1e20, 10.0, s[0])
        ctx.init_plasma(1, case["ppc"], 1e20, 1e20, 1.0, s[1])
        return dict(case=case, ctx=ctx, seed=s[2], n=0)
    fp32 = case.get("precision", "fp64") == "fp32"
    ctx = capi.Context(size, grid, domains, dt, _species(n, case.get("bunch", 0)),
                       pusher=case.get("pusher", "boris-adaptive"),
                       ccs=case.get("ccs", "zigzag"), precision="fp32" if fp32 else "fp64")
    if kind in ("upload", "maps"):
        for sp, p in enumerate(_particles(case, seed)):
            ctx.upload(sp, *p)
        if kind == "upload":
            _tune(ctx, dict(case, dom_r=1, dom_z=1, ccs="zigzag", collisions="none"), fp32)
            ctx.set_graph(True)
        return dict(case=case, ctx=ctx)
    left = 1e17 * case.get("density_left", 1.0)
    ctx.init_plasma(0, case["ppc"], left, 1e17, 1.0, s[0])
    ctx.init_plasma(1, case["ppc"], left, 1e17, 0.1, s[1])
    if kind == "phases":
        return dict(case=case, ctx=ctx)
    if case["bunch"]:
        z0 = min(BUNCH["z0"], 0.4 * size[1])
        ctx.init_bunch(2, case["bunch"], BUNCH["n_peak"], BUNCH["sigma_r"], BUNCH["sigma_z"], z0, BUNCH["gamma"], s[2])
    if case["collisions"] == "surrogate":
        ctx.mlp_init(7)
        ctx.surrogate_set_norm(np.concatenate(NORM))
    if case["collisions"] != "none":
        ctx.set_collisions(case["collisions"], 0, 1, seed=s[3])
    _tune(ctx, case, fp32)
    ctx.set_graph(True)
    return dict(case=case, ctx=ctx)


def _frames(ctx):
    # J's halo is scratch after a step: the interior is what it defines
    return {"E": ctx.get_grid("E"), "H": ctx.get_grid("H"), "J": ctx.get_grid("J")[:, :, 2:-2, 2:-2]}


def run(state):
    case, ctx = state["case"], state["ctx"]
    kind = case["kind"]
    if kind in ("functional", "step", "upload"):
        ctx.step(case["steps"])
        return _frames(ctx)
    if kind == "phases":
        for _ in range(case["steps"]):
            for ph in ("yee_e", "overlay_e", "yee_h", "overlay_h", "push", "move", "migrate", "deposit", "overlay_j"):
                ctx.phase(ph)
        out = _frames(ctx)
        for sp in range(2):
            p = ctx.particles(sp)
            out["species%d" % sp] = {k: p[k] for k in ("r", "z", "vr", "vphi", "vz", "w")}
        return out
    if kind == "relax":
        for _ in range(case["passes"]):
            ctx.collide(case["scheme"], 0, 1, state["seed"], state["n"])
            state["n"] += 1
        return {"%s%d" % (m, sp): ctx.species_map(sp, m)[:, :, 2:-2, 2:-2] for sp in (0, 1)
                for m in ("energy", "momentum")}
    if kind == "maps":
        out = {"%s%d" % (m, sp): ctx.species_map(sp, m)[:, :, 2:-2, 2:-2] for sp in (0, 1)
               for m in ("density", "energy", "temperature", "momentum")}
        out["kinetic"] = [ctx.kinetic_energy(0), ctx.kinetic_energy(1)]
        return out
    g, loss = ctx.mlp_grad(state["x"], state["t"])
    return {"grad": g, "loss": loss, "y": ctx.mlp_forward(state["x"])}


def work(case):
    kind = case["kind"]
    if kind == "train":
        # rows in (x twice, t), y out; forward twice, backward twice a forward
        net = 2 * (6 * 64 + 64 * 64 + 64 * 4)
        return {"bytes": case["rows"] * (2 * 32 + 16 + 16), "flops": case["rows"] * net * 4}
    cells = case["nr"] * case["nz"]
    real = 4 if case.get("precision", "fp64") == "fp32" else 8
    if kind == "functional":
        n = case["macro"]
    else:
        n = 2 * case["ppc"] * cells * 0.5 * (1 + case.get("density_left", 1.0)) + case.get("bunch", 0)
    if kind == "maps":
        # 8 maps and 2 energies: position, weight and (but for the density) velocity of a species' particles
        return {"bytes": 0.5 * n * real * 2 * (3 + 3 * 6 + 4) + 12 * cells * 8, "flops": n * 400}
    if kind == "relax":
        # velocities in and out, weight and cell; about 250 operations a pair, and 1.5 pairs a particle
        return {"bytes": case["passes"] * n * (7 * real + 4) + 8 * 8 * cells, "flops": case["passes"] * n * 1.5 * 250}
    # per step: position, velocity, weight in, position and velocity out (FP32: the packed cell as well), and the
    # grids' 41 values a cell; then the frames
    step = n * (13 if real == 4 else 11) * real + 41 * real * cells
    flops = n * 300
    if case.get("collisions", "none") == "p12":
        step += n * (7 * real + 4)
        flops += n * 1.5 * 250
    if case.get("collisions", "none") == "surrogate":
        step += n * 6 * real
        flops += cells * 9500
    out = 9 * 8 * cells + (n * 6 * 8 if kind == "phases" else 0)
    return {"bytes": case["steps"] * step + out, "flops": case["steps"] * flops}


def tolerance(case):
    """About four times what the same sources give when the compiler contracts products and sums into FMAs (every
    rounding changes, nothing else), or what the result is off the 64-bit one where that is more."""
    kind = case["kind"]
    if kind == "train":
        # BF16 products: 0.004 off 64 bits
        return {"rel": 1e-2}
    if kind == "maps":
        # FP64 sums in another order: 5e-14
        return {"rel": 1e-12}
    if kind == "relax":
        # like-particle pairs have round-off relative speeds: sk98 4e-11, p12 2e-6 (5e-4); ta77s' correction divides
        # differences of a cell's nearly equal energies (rounding alone moves its maps by 0.1)
        return {"rel": 1e-5, "max": 2e-3} if case["scheme"] != "ta77s" else {"rel": 0.03, "max": 0.99}
    fp32 = case.get("precision", "fp64") == "fp32"
    if case.get("ccs", "vb" if kind == "functional" else "zigzag") == "vb":
        # a move shorter than 1e-15 m along r or z takes the strict branch, which clears J_r nodes: which particles do
        # is a matter of rounding (FP64 2e-4 and 0.2 at the worst node, FP32 0.1)
        return {"rel": 0.03, "max": 0.99} if fp32 else {"rel": 1e-3, "max": 0.9}
    if fp32:
        # 1.3e-4 off 64 bits after 20 steps; single nodes where a fast particle crossed a cell edge 0.3
        return {"rel": 6e-4, "max": 0.99}
    # FP64: 3e-11 (4e-9), with like-particle pairs 4e-9 (1e-6)
    return {"rel": 2e-8, "max": 4e-6} if case.get("collisions", "none") != "none" else {"rel": 1e-10, "max": 2e-8}


# ---- what plain torch gives in 64 bits ----

def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _exact_train(case, seed):
    x, t, p = (torch.from_numpy(a).double().to(_dev()) for a in _batch(case, seed))
    w, o = [], 0
    for rows, cols in ((64, 32), (64, 64), (16, 64)):
        w.append(p[o:o + rows * cols].reshape(rows, cols))
        o += rows * cols
        w.append(p[o:o + rows])
        o += rows
    for a in w:
        a.requires_grad_(True)
    n = case["rows"]
    xp = torch.zeros(n, 32, dtype=torch.float64, device=x.device)
    xp[:, :6] = x[:, :6]
    h = torch.tanh(xp @ w[0].T + w[1])
    h = torch.tanh(h @ w[2].T + w[3])
    y = (h @ w[4].T + w[5])[:, :4]
    loss = ((y - t) ** 2).sum() / n
    g = torch.autograd.grad(loss, w)
    return {"grad": torch.cat([a.reshape(-1) for a in g]).cpu(), "loss": float(loss.detach()), "y": y.detach().cpu()}


def _gather(F, i, k, wr1, wr2, wz1, wz2):
    return (F[i, k] * wr1 + F[i + 1, k] * wr2) * wz1, F[i, k + 1] * wr1 * wz2, F[i + 1, k + 1] * wr2 * wz2


def _weights(x, u, half_r, half_z):
    """Cell, ring-area and axial weights of the cloud at radius x, longitude u (cell units) on nodes at integer
    (half 0) or half-integer (half 1: the node row below is the cell's own) places."""
    a = x if half_r else x - 0.5
    i = torch.floor(a)
    r2 = i + (0.5 if half_r else 1.0)
    c1, c2 = (2 * i + 1, 2 * i + 3) if half_r else (2 * i + 2, 2 * i + 4)
    wr1 = (r2 ** 2 - (x - 0.5) ** 2) / c1
    wr2 = ((x + 0.5) ** 2 - r2 ** 2) / c2
    b = u - 0.5 if half_z else u
    k = torch.floor(b)
    wz2 = b - k
    return i.long() + 2, k.long() + 2, wr1, wr2, 1 - wz2, wz2


def _push(pusher, q, m, dt, e, h, v):
    c2 = C_LIGHT ** 2
    dot = lambda a, b: a[0] * b[0] + a[1] * b[1] + a[2] * b[2]  # noqa: E731
    inv = lambda a: 1 / torch.sqrt(1 + dot(a, a) / c2)  # noqa: E731
    f = q * dt / (2 * m)
    gam = 1 / torch.sqrt(1 - dot(v, v) / c2)
    u = [a * gam for a in v]
    b = [f * MAGN_CONST * a for a in h]
    if pusher == "vay":
        up = [a + 2 * f * c for a, c in zip(u, e)]
        g = inv(u)
        up = [up[0] + g * (u[1] * b[2] - u[2] * b[1]), up[1] + g * (u[2] * b[0] - u[0] * b[2]),
              up[2] + g * (u[0] * b[1] - u[1] * b[0])]
        bb = dot(b, b)
        s = 1 + dot(up, up) - bb
        al = 1 / torch.sqrt(0.5 * (s + torch.sqrt(s * s + 4 * (bb + dot(up, b) ** 2))))
        b = [a * al for a in b]
        s = 1 / (1 + dot(b, b))
        al = dot(up, b)
        p = [s * (up[0] + al * b[0] + b[2] * up[1] - b[1] * up[2]), s * (up[1] + al * b[1] + b[0] * up[2] - b[2] * up[0]),
             s * (up[2] + al * b[2] + b[1] * up[0] - b[0] * up[1])]
    elif pusher == "hc":
        um = [a + f * c for a, c in zip(u, e)]
        bb = dot(b, b)
        s = 1 + dot(um, um) - bb
        g = 1 / torch.sqrt(0.5 * (s + torch.sqrt(s * s + 4 * (bb + dot(b, um) ** 2))))
        b = [a * g for a in b]
        x, y, z = (a * a for a in b)
        c0, c1, cc = b[0] * b[1], b[1] * b[2], b[2] * b[0]
        det = 1 / (1 + x + y + x)
        up = [((1 + x - y - z) * um[0] + 2 * (c0 + b[2]) * um[1] + 2 * (cc - b[2]) * um[2]) * det,
              (2 * (c0 - b[2]) * um[0] + (1 - x + y - z) * um[1] + 2 * (c1 + b[0]) * um[2]) * det,
              (2 * (cc + b[1]) * um[0] + 2 * (c1 - b[0]) * um[1] + (1 - x - y + z) * um[2]) * det]
        p = [a + f * c for a, c in zip(up, e)]
    else:
        t = [a + f * c for a, c in zip(u, e)]
        g = inv(t)
        b = [a * g for a in b]
        k = 2 / (1 + dot(b, b))
        x = t[0] + t[1] * b[2] - t[2] * b[1]
        y = t[1] - t[0] * b[2] + t[2] * b[0]
        z = t[2] + t[0] * b[1] - t[1] * b[0]
        p = [t[0] + k * (y * b[2] - z * b[1]) + f * e[0], t[1] + k * (z * b[0] - x * b[2]) + f * e[1],
             t[2] + k * (x * b[1] - y * b[0]) + f * e[2]]
    g = inv(p)
    return [a * g for a in p]


def _reflect(r, z, r0, z0, vr, vz, R, L):
    h = CELL / 2
    r0, z0, ddr, ddz = r0.clone(), z0.clone(), r - r0, z - z0
    for _ in range(4):
        m = r > R - h
        small = (R - h) - r0
        sz = small * ddz / ddr
        vr, r = torch.where(m, -vr, vr), torch.where(m, 2 * (R - h) - r, r)
        ddr, ddz = torch.where(m, ddr - small, ddr), torch.where(m, ddz - sz, ddz)
        r0, z0 = torch.where(m, torch.full_like(r0, R - h), r0), torch.where(m, z0 - sz, z0)
        m = z > L - h
        small = (L - h) - z0
        sr = small * ddr / ddz
        vz, z = torch.where(m, -vz, vz), torch.where(m, 2 * (L - h) - z, z)
        ddr, ddz = torch.where(m, ddr - sr, ddr), torch.where(m, ddz - small, ddz)
        z0, r0 = torch.where(m, torch.full_like(z0, L - h), z0), torch.where(m, r0 - sr, r0)
        m = r < h
        small = h - r0
        sz = small * ddz / ddr
        vr, r = torch.where(m, -vr, vr), torch.where(m, torch.clamp(CELL - r, min=h), r)
        ddr, ddz = torch.where(m, ddr - small, ddr), torch.where(m, ddz - sz, ddz)
        r0, z0 = torch.where(m, torch.full_like(r0, h), r0), torch.where(m, z0 - sz, z0)
        m = z < h
        small = h - z0
        sr = small * ddr / ddz
        vz, z = torch.where(m, -vz, vz), torch.where(m, torch.clamp(CELL - z, min=h), z)
        ddr, ddz = torch.where(m, ddr - sr, ddr), torch.where(m, ddz - small, ddz)
        z0, r0 = torch.where(m, torch.full_like(z0, CELL), z0), torch.where(m, r0 - sr, r0)
    return r, z, vr, vz


def _exact_upload(case, seed):
    """The particle loop of one domain between conducting walls, ZigZag deposition, in torch."""
    nr, nz, dt = case["nr"], case["nz"], 0.5 * CELL / C_LIGHT
    R, L = nr * CELL, nz * CELL
    dev = _dev()
    new = lambda: torch.zeros(3, nr + 4, nz + 4, dtype=torch.float64, device=dev)  # noqa: E731
    E, H, Ht, J = new(), new(), new(), new()
    I, K = slice(2, nr + 2), slice(2, nz + 2)
    sp = []
    for (q, m, beam), p in zip(((-1, 1.0, 0), (1, 1836.0, 0), (-1, 1.0, 1)), _particles(case, seed)):
        sp.append([q * EL_CHARGE, m * EL_MASS, beam] + [torch.from_numpy(a).to(dev) for a in p])
    ring = torch.arange(nr, dtype=torch.float64, device=dev)[:, None]

    def shift(F, di=0, dk=0, a=0, b=0, c=0, d=0):
        """F on rows a .. nr - b, columns c .. nz - d of the interior, displaced."""
        return F[2 + a + di:nr + 2 - b + di, 2 + c + dk:nz + 2 - d + dk]

    def halo0(F):
        F[:, :2], F[:, -2:], F[:, :, :2], F[:, :, -2:] = 0, 0, 0, 0

    kh = 2 * dt / (2 * EPSILON0)
    for _ in range(case["steps"]):
        halo0(E)
        e_r = lambda **s: kh * (shift(J[0], **s) + (shift(Ht[1], **s) - shift(Ht[1], dk=-1, **s)) / CELL)  # noqa: E731
        s = dict(a=0, b=nr - 1, c=1, d=1)
        shift(E[0], **s).sub_(e_r(**s))
        shift(E[2], **s).sub_(kh * (shift(J[2], **s) - shift(Ht[1], **s) * 4 / CELL))
        s = dict(a=1, b=1, c=0, d=1)
        rr = ring[1:nr - 1]
        shift(E[2], **s).sub_(kh * (shift(J[2], **s) - (shift(Ht[1], **s) - shift(Ht[1], di=-1, **s)) / CELL
                                    - (shift(Ht[1], **s) + shift(Ht[1], di=-1, **s)) / (2 * CELL * rr)))
        s = dict(a=1, b=1, c=1, d=1)
        shift(E[0], **s).sub_(e_r(**s))
        shift(E[1], **s).sub_(kh * (shift(J[1], **s) - (shift(Ht[0], **s) - shift(Ht[0], dk=-1, **s)) / CELL
                                    + (shift(Ht[2], **s) - shift(Ht[2], di=-1, **s)) / CELL))
        halo0(Ht)
        H.zero_()
        al = dt * (shift(E[1], dk=1) - shift(E[1])) / (CELL * MAGN_CONST)
        Ht[0, nr + 1, K] += al[-1]
        H[0, I, K] = Ht[0, I, K] + al / 2
        Ht[0, I, K] += al
        al = dt * ((shift(E[2], di=1) - shift(E[2])) / CELL - (shift(E[0], dk=1) - shift(E[0])) / CELL) / MAGN_CONST
        H[1, I, K] = Ht[1, I, K] + al / 2
        Ht[1, I, K] += al
        al = dt * ((shift(E[1], di=1) + shift(E[1])) / (2 * CELL * (ring + 0.5))
                   + (shift(E[1], di=1) - shift(E[1])) / CELL) / MAGN_CONST
        H[2, I, K] = Ht[2, I, K] - al / 2
        Ht[2, I, K] -= al
        J.zero_()
        for s in sp:
            q, m, beam, r, z, vr, vp, vz, w = s
            x, u = r / CELL, z / CELL
            full = lambda F, hr, hz: sum(_gather(F, *_weights(x, u, hr, hz)))  # noqa: E731
            ep = _gather(E[1], *_weights(x, u, True, False))
            # the gather's last E_phi term goes to E_z
            e = [full(E[0], False, False), ep[0] + ep[1], full(E[2], True, True) + ep[2]]
            h = [full(H[0], True, True), full(H[1], False, True), full(H[2], False, False)]
            vr, vp, vz = _push(case["pusher"], q, m, dt, e, h, [vr, vp, vz])
            a, b, zn = r + vr * dt, vp * dt, z + vz * dt
            rn = torch.sqrt(a * a + b * b)
            sn = b / rn
            cs = torch.sqrt(1 - sn * sn)
            if beam:
                low = rn < CELL / 2
                vr, rn = torch.where(low, -vr, vr), torch.where(low, CELL - rn, rn)
            else:
                rn, zn, vr, vz = _reflect(rn, zn, r, z, vr, vz, R, L)
            vr, vp = cs * vr - sn * vp, sn * vr + cs * vp
            # ZigZag: two segments through the relay point
            io, ko, i1, k1 = (torch.floor(c / CELL) for c in (r, z, rn, zn))
            mid = torch.floor((rn + r) / 2 / CELL)
            vol = 1 / (PI * CELL ** 3 * (2 * mid + 1))

            def relay(c, d, y, t):
                low = torch.minimum(c, d) * CELL + CELL
                return torch.minimum(low, torch.maximum(torch.maximum(c, d) * CELL, (y + t) / 2))

            rr_, zr_ = relay(io, i1, r, rn), relay(ko, k1, z, zn)
            g = q * w / dt * vol
            fp = q * w * vp * vol
            segs = ((io, ko, g * (rr_ - r), g * (zr_ - z), (r + rr_) / 2 - io * CELL, (z + zr_) / 2 - ko * CELL),
                    (i1, k1, g * (rn - rr_), g * (zn - zr_), (rn + rr_) / 2 - i1 * CELL, (zn + zr_) / 2 - k1 * CELL))

            def add(c, i, k, val):
                J[c].view(-1).index_add_(0, ((i.long() + 2) * (nz + 4) + k.long() + 2), val)

            for i, k, fr, fz, wr, wz in segs:
                add(0, i, k, fr * (1 - wz))
                add(0, i, k + 1, fr * wz)
                add(2, i, k, fz * (1 - wr))
                add(2, i + 1, k, fz * wr)
            wr2, wz1, wz2 = segs[1][4], segs[0][5], segs[1][5]
            add(1, i1, k1, fp * (1 - wr2) * (1 - wz2))
            add(1, i1, k1 + 1, fp * (1 - wr2) * wz1)
            add(1, i1 + 1, k1, fp * wr2 * (1 - wz2))
            add(1, i1 + 1, k1 + 1, fp * wr2 * wz2)
            s[3:8] = rn, zn, vr, vp, vz
    return {"E": E[None].cpu(), "H": H[None].cpu(), "J": J[None, :, I, K].cpu()}


def _exact_maps(case, seed):
    nr, nz = case["nr"], case["nz"]
    dev = _dev()
    out = {"kinetic": []}
    c2, lim2 = C_LIGHT ** 2, 5e7 ** 2
    for sp, p in enumerate(_particles(dict(case, bunch=0), seed)):
        m = (1.0, 1836.0)[sp] * EL_MASS
        r, z, vr, vp, vz, w = (torch.from_numpy(a).to(dev) for a in p)
        x, u = r / CELL, z / CELL
        i, k = torch.floor(x), torch.floor(u)
        v1 = torch.where(x > 1, 2 * i + 1, torch.ones_like(x))
        # the ring below the node's half radius; on the axis the cloud folds over it
        fold = x <= 0.5
        low = torch.where(fold, 0.5 - x + x * x, (i + 0.5) ** 2 - (x - 0.5) ** 2) / v1
        high = ((x + 0.5) ** 2 - (i + 0.5) ** 2) / (2 * i + 2)
        v0 = torch.where(fold, 2 * x * x + 0.5, 2 * x) * PI * CELL ** 3
        top = u - k
        v2 = vr * vr + vp * vp + vz * vz
        gam = torch.where(v2 < lim2, 1 / torch.sqrt(1 - v2 / c2), torch.ones_like(v2))

        def node(val):
            F = torch.zeros(nr + 4, nz + 4, dtype=torch.float64, device=dev)
            for di, a in ((0, low), (1, high)):
                for dk, b in ((0, 1 - top), (1, top)):
                    F.view(-1).index_add_(0, (i.long() + 2 + di) * (nz + 4) + k.long() + 2 + dk, val / v0 * a * b)
            return F[2:-2, 2:-2]

        n = node(w)
        pw = [node(m * w * c * gam) for c in (vr, vp, vz)]
        pa = node(m * w * torch.sqrt(v2) * gam)

        def energy(p2):
            p2 = p2 / n ** 2
            rest = m * c2
            e = torch.where(p2 > lim2 * m * m, torch.sqrt(p2 * c2 + rest ** 2) - rest, 0.5 * p2 / m) / EL_CHARGE
            return torch.where(n == 0, torch.zeros_like(e), e)[None, None].cpu()

        out["density%d" % sp] = n[None, None].cpu()
        out["energy%d" % sp] = energy(pa ** 2)
        out["temperature%d" % sp] = energy(pa ** 2 - pw[0] ** 2 - pw[1] ** 2 - pw[2] ** 2)
        out["momentum%d" % sp] = torch.stack([torch.where(n == 0, torch.zeros_like(c), c / n) for c in pw])[None].cpu()
        g = 1 / torch.sqrt(1 - v2 / c2)
        out["kinetic"].append(float((w * m * v2 * g * g / (g + 1)).sum()))
    return out


def exact(case, seed):
    """Plain torch in 64 bits; None where the result hangs on the package's own random draws and plasma
    (device-generated particles, keyed collision pairs)."""
    if case["kind"] == "train":
        return _exact_train(case, seed)
    if case["kind"] == "upload":
        return _exact_upload(case, seed)
    if case["kind"] == "maps":
        return _exact_maps(case, seed)
    return None
