"""Performance cases of the library: the calls a simulation spends its time in.

A case is one call sequence of a public entry point on one size:

  rhs      ampe_rhs_eval: the right-hand side of the integrator callbacks, full
           (Newton) or lagged (difference-quotient Jv), on one or several
           patches;
  precond  ampe_precond_setup and then ampe_precond_solve on a few Krylov
           vectors: FP64 red-black or FP32 multigrid blocks;
  steps    ampe_sim: a state loaded, advanced by some BDF steps and read back;
  amr      ampe_sim on a patch hierarchy: the same over several levels;
  kks      ampe_kks_batch: phase concentrations of independent cells with a
           temperature each, from the default or the surrogate start.

The physics are the workloads of ampe_amd.params (two-grain quadratic wells,
binary CALPHAD polycrystal, dilute anisotropic dendrite, three-phase ternary
grains).  prepare() holds what a program holds before the call: the handle with
its state, and device vectors in the level's layout.  Cell vectors come back
as views of each patch's interior cells (the entry points define no ghost
values of their results), one output per field.
"""
import ctypes as C
import math

import numpy as np
import torch
import torch.nn.functional as F

from ampe_amd import hip as H
from ampe_amd import params as P
from ampe_amd import surrogate as SG

DEV = "cuda:0"
RGAS = 8.314472
SOLVES = 4  # Krylov vectors per preconditioner setup


# --------------------------------------------------------------------- cases
def listed():
    return [
        # the 128^2 two-grain regression size: a call of launches only
        dict(name="rhs_2d_two_grain_128", kind="rhs", model="quadratic", nx=128, ny=128, nz=1,
             patches=1, lagged=False),
        # a 2-D dendrite (anisotropic flux, dilute alloy, bounded domain) on
        # uneven patches, as a clustered level has
        dict(name="rhs_2d_dendrite", kind="rhs", model="dilute", nx=1500, ny=1130, nz=1,
             patches=6, lagged=False),
        # the Jv evaluation of a 3-D polycrystal on odd, uneven patches
        dict(name="jv_3d_polycrystal_odd", kind="rhs", model="calphad", nx=151, ny=93, nz=67,
             patches=3, lagged=True),
        # the largest single-level workload of the benchmark: 256^3
        dict(name="rhs_3d_polycrystal_256", kind="rhs", model="calphad", nx=256, ny=256, nz=256,
             patches=1, lagged=False),
        # the plain FP64 preconditioner on an odd 3-D level
        dict(name="precond_f64_redblack", kind="precond", model="calphad", nx=131, ny=95, nz=77,
             patches=2, fp32=False, mg=False),
        # the benchmark's preconditioner at its size
        dict(name="precond_f32_mg_256", kind="precond", model="calphad", nx=256, ny=256, nz=256,
             patches=1, fp32=True, mg=True),
        # a 2-D regression-size run with the default solver (FP64, red-black,
        # modified Gram-Schmidt): host loop, launches and reductions
        dict(name="steps_2d_two_grain", kind="steps", model="quadratic", nx=128, ny=128, nz=1,
             fp32=False, mg=False, cgs=False, nsteps=4),
        # the benchmark's integrator form on a medium level
        dict(name="steps_3d_polycrystal_128", kind="steps", model="calphad", nx=128, ny=128,
             nz=128, fp32=True, mg=True, cgs=True, nsteps=8),
        # three-level 2-D dendrite: many small patches, FAC over the levels
        dict(name="amr_2d_dendrite", kind="amr", model="dendrite", n0=256, fp32=False, nsteps=4),
        # two-level 3-D ternary grains, nine orders and two species
        dict(name="amr_3d_ternary", kind="amr", model="ternary", n0=96, fp32=True, nsteps=2),
        # a patch's worth of cells with a temperature field
        dict(name="kks_batch", kind="kks", n=3000001, guess=False),
        # the same physics started from the trained network
        dict(name="kks_batch_surrogate", kind="kks", n=500009, guess=True),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["rhs", "rhs", "rhs", "precond", "precond", "steps", "steps", "amr",
                       "kks"])
    if kind == "kks":
        return dict(kind="kks", n=_logint(rng, 2000, 3000000), guess=rng.random() < 0.5)
    if kind == "amr":
        if rng.random() < 0.5:
            return dict(kind="amr", model="dendrite", n0=8 * rng.randint(12, 32),
                        fp32=rng.random() < 0.5, nsteps=rng.randint(1, 4))
        return dict(kind="amr", model="ternary", n0=4 * rng.randint(8, 20),
                    fp32=rng.random() < 0.5, nsteps=rng.randint(1, 2))
    if kind == "steps":
        if rng.random() < 0.5:
            n = 8 * rng.randint(6, 24)
            return dict(kind="steps", model="quadratic", nx=n, ny=n, nz=1, fp32=False, mg=False,
                        cgs=rng.random() < 0.5, nsteps=rng.randint(1, 4))
        mg = rng.random() < 0.7
        e = 8 if mg else 1
        n = [e * rng.randint(32 // e, 112 // e) for _ in range(3)]
        return dict(kind="steps", model="calphad", nx=n[0], ny=n[1], nz=n[2], fp32=mg, mg=mg,
                    cgs=True, nsteps=rng.randint(2, 8))
    model = rng.choice(["quadratic", "dilute", "calphad", "calphad"])
    if kind == "rhs":
        if model == "calphad" and rng.random() < 0.7:
            n = [_logint(rng, 17, 220) for _ in range(3)]
        else:
            n = [_logint(rng, 65, 1400), _logint(rng, 65, 1400), 1]
        return dict(kind="rhs", model=model, nx=n[0], ny=n[1], nz=n[2],
                    patches=rng.choice([1, 1, 2, 5]), lagged=rng.random() < 0.6)
    mg = rng.random() < 0.6
    if model == "dilute":
        model = "quadratic"
    if mg:
        e = rng.choice([4, 8, 16])
        d3 = rng.random() < 0.7
        n = [e * rng.randint(max(2, 32 // e), (176 if d3 else 640) // e) for _ in range(3)]
    else:
        d3 = rng.random() < 0.7
        n = [_logint(rng, 21, 140 if d3 else 600) for _ in range(3)]
    return dict(kind="precond", model=model, nx=n[0], ny=n[1], nz=n[2] if d3 else 1,
                patches=1 if mg else rng.choice([1, 2, 3]), fp32=mg, mg=mg)


# ------------------------------------------------------------------- physics
def _model(case):
    nd = 3 if case["nz"] > 1 else 2
    if case["model"] == "quadratic":
        p = P.two_grain_params(ndim=nd)
    elif case["model"] == "calphad":
        p = P.polycrystal_params(ndim=nd)
    else:
        p = P.dilute_params(ndim=nd, dilute_keq=0.14)
        if nd == 2:
            p.flux_type, p.aniso_nu, p.aniso_knumber = P.FLUX_ANISOTROPIC, 0.05, 4
    return p


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _rand(g, *shape):
    return torch.rand(shape, generator=g, dtype=torch.float64, device=DEV)


def _centres(case):
    """Cell centre coordinates (z, y, x) as broadcastable tensors."""
    n = (case["nz"], case["ny"], case["nx"])
    out = []
    for a in range(3):
        sh = [1, 1, 1]
        sh[a] = n[a]
        out.append((torch.arange(n[a], dtype=torch.float64, device=DEV) + 0.5).view(sh))
    return out


def _state(case, p, seed, smooth):
    """phi, c, q on the domain ([nz, ny, nx]); smooth: compositions of a
    relaxed state (equal diffusion potential, noise 1e-3) in place of noise
    over the whole range."""
    g = _gen(seed)
    n = (case["nz"], case["ny"], case["nx"])
    nd = p.ndim
    x = _centres(case)
    u = _rand(g, 3, 16)
    quat = lambda k: torch.stack([  # noqa: E731
        torch.sqrt(1 - u[0, k]) * torch.sin(2 * math.pi * u[1, k]),
        torch.sqrt(1 - u[0, k]) * torch.cos(2 * math.pi * u[1, k]),
        torch.sqrt(u[0, k]) * torch.sin(2 * math.pi * u[2, k]),
        torch.sqrt(u[0, k]) * torch.cos(2 * math.pi * u[2, k])])
    if case["model"] == "calphad":
        # Voronoi grains with liquid pockets far from the seeds
        pos = _rand(g, 16, 3)
        best = torch.full(n, 1e300, dtype=torch.float64, device=DEV)
        lab = torch.zeros(n, dtype=torch.int64, device=DEV)
        for k in range(16):
            d2 = torch.zeros((1, 1, 1), dtype=torch.float64, device=DEV)
            for a in range(3 - nd, 3):
                d = (x[a] - pos[k, a] * n[a]).abs()
                d = torch.minimum(d, n[a] - d)
                d2 = d2 + d * d
            lab = torch.where(d2 < best, torch.full_like(lab, k), lab)
            best = torch.minimum(best, d2)
        dist = best.sqrt_()
        thr = torch.kthvalue(dist.view(-1)[::7], int(0.7 * (dist.numel() // 7 + 1)))[0]
        phi = 0.5 * (1.0 - torch.tanh((dist - thr) / 1.5))
        q = torch.stack([quat(k) for k in range(16)], 1)[:, lab]
        del best, lab, dist
        if smooth:
            cl = torch.full(n, 0.40, dtype=torch.float64, device=DEV)
            cs = torch.full((1,), 0.40, dtype=torch.float64, device=DEV)
            mu = _mu(p, cl.view(-1)[:1], 0)
            for _ in range(60):
                cs = (cs - (_mu(p, cs, 1) - mu) / _d2f(p, cs, 1)).clamp(1e-6, 1 - 1e-6)
            h = _interp(phi, p.conc_interp)
            c = (1 - h) * cl + h * cs + 1e-3 * (_rand(g, *n) - 0.5)
        else:
            c = 0.3 + 0.2 * _rand(g, *n)
    else:
        r0 = 0.25 * min(n[3 - nd:])
        d2 = sum((x[a] - 0.5 * n[a] - 0.3 * _rand(g, 1)[0]) ** 2 for a in range(3 - nd, 3))
        phi = 0.5 * (1.0 - torch.tanh((d2.sqrt() - r0) / 2.0))
        if case["model"] == "quadratic":
            c = torch.where(phi >= 0.5, 0.45, 0.40) + 0.01 * (_rand(g, *n) - 0.5)
            if smooth:
                h = _interp(phi, p.conc_interp)
                c = (1 - h) * 0.40 + h * 0.45 + 1e-3 * (_rand(g, *n) - 0.5)
            q = torch.where((phi >= 0.5)[None], quat(0)[:, None, None, None],
                            quat(1)[:, None, None, None])
        else:
            c = 0.05 + 0.004 * (_rand(g, *n) - 0.5)
            phi = (phi + 0.01 * torch.randn(n, generator=g, dtype=torch.float64, device=DEV)
                   * ((phi > 0.05) & (phi < 0.95))).clamp(0.0, 1.0)
            q = quat(0)[:, None, None, None].expand(4, *n)
    return phi.contiguous(), c.contiguous(), q.contiguous()


# ------------------------------------------------------------------- layout
def _boxes(case):
    """The domain cut along x (and y from five patches on) at uneven places;
    even places for the multigrid and the 2-D checkerboard."""
    n = (case["nx"], case["ny"], case["nz"])
    k = case.get("patches", 1)
    ky = 2 if k >= 5 else 1
    kx = (k + ky - 1) // ky
    cuts = []
    for m, parts in ((n[0], kx), (n[1], ky)):
        w = [1.0 + 0.35 * (i % 3) for i in range(parts)]
        e = [0] + [2 * int(m * sum(w[:i + 1]) / sum(w) / 2) for i in range(parts)]
        e[-1] = m
        cuts.append(e)
    out = []
    for j in range(ky):
        for i in range(kx):
            b = P.Box()
            b.lo[:] = [cuts[0][i], cuts[1][j], 0]
            b.hi[:] = [cuts[0][i + 1] - 1, cuts[1][j + 1] - 1, n[2] - 1 if n[2] > 1 else 0]
            out.append(b)
    return out


def _domain(case):
    """Periodic domain box; None: zero-slope boundaries (the dendrite)."""
    if case["model"] == "dilute":
        return None
    b = P.Box()
    b.lo[:] = [0, 0, 0]
    b.hi[:] = [case["nx"] - 1, case["ny"] - 1, case["nz"] - 1 if case["nz"] > 1 else 0]
    return b


def _cut(a, b):
    """Box b of domain arrays [..., nz, ny, nx]."""
    return a[..., b.lo[2]:b.hi[2] + 1, b.lo[1]:b.hi[1] + 1, b.lo[0]:b.hi[0] + 1]


def _views(lev, v, nc):
    """Interior cells of every patch of a vector of nc component blocks."""
    out = []
    g, gz = lev.ghost, lev.ghost if lev.ndim == 3 else 0
    for k, b in enumerate(lev.boxes):
        n = [b.hi[a] - b.lo[a] + 1 for a in range(3)]
        off = lev.cell_off[k] + g + g * lev.sy[k] + gz * lev.sz[k]
        out.append(torch.as_strided(v, (nc, n[2], n[1], n[0]),
                                    (lev.ncg, lev.sz[k], lev.sy[k], 1), off))
    return out


def _fields(blocks):
    """Per patch: phase, composition and orientation."""
    return [[b[:1], b[1:2], b[2:]] for b in blocks]


def _vector(lev, parts):
    v = torch.zeros(sum(a.shape[0] for a in parts) * lev.ncg, dtype=torch.float64, device=DEV)
    a = torch.cat([t for t in parts])
    for b, w in zip(lev.boxes, _views(lev, v, a.shape[0])):
        w.copy_(_cut(a, b))
    return v


def _host(a, boxes):
    return np.concatenate([_cut(a, b).reshape(*a.shape[:-3], -1).cpu().numpy() for b in boxes], -1)


def _solver(case):
    # the first step a state of this kind is started with; it doubles up to dt
    kw = dict(dt=5e-6, dt_init=6e-7) if case["model"] == "calphad" else dict(dt=1e-3, dt_init=1.5e-5)
    if case["model"] == "calphad":
        kw.update(maxl=10, max_newton=5, atol=3e-7, rtol=3e-9)
    else:
        kw.update(maxl=10, max_newton=5)
    if case.get("fp32"):
        kw.update(precision=P.FAC_FP32)
    if case.get("mg"):
        kw.update(precond=P.PRECOND_MG, fac_sweeps=1, quat_sweeps=1, mg_max_levels=4,
                  mg_coarse_sweeps=2)
    if case.get("cgs") or case.get("mg"):
        kw.update(gstype=P.GS_CLASSICAL)
    return P.solver_defaults(**kw)


def _ptr(t):
    return C.c_void_p(t.data_ptr())


class _Held:
    pass


# ------------------------------------------------------------------- prepare
def prepare(case, seed):
    kind = case["kind"]
    if kind == "kks":
        return _prepare_kks(case, seed)
    if kind == "amr":
        return _prepare_amr(case, seed)
    s = _Held()
    s.kind, s.case = kind, case
    s.p, s.s = _model(case), _solver(case)
    boxes, dom = _boxes(case), _domain(case)
    phi, c, q = _state(case, s.p, seed, kind == "steps")
    s.host = (_host(phi, boxes), _host(c, boxes), _host(q, boxes))
    s.sim = H.Sim(s.p, s.s, boxes, periodic=dom)
    if kind == "steps":
        s.shape = (case["ny"], case["nx"]) if s.p.ndim == 2 else (case["nz"], case["ny"],
                                                                  case["nx"])
        return s
    s.lev = H.Level(s.p.ndim, boxes, 1, periodic=dom)
    s.sim.set_state(*s.host)
    del s.host
    s.nc = 6
    s.y = _vector(s.lev, [phi[None], c[None], q])
    s.out = torch.zeros_like(s.y)
    g = _gen(seed + 1)
    torch.cuda.synchronize()
    if kind == "rhs":
        if case["lagged"]:
            # the face data of a full evaluation, then a displaced state
            H.check(H.lib().ampe_rhs_eval(s.sim.h, 0.0, _ptr(s.y), _ptr(s.out), 0))
            torch.cuda.synchronize()
            d = _displaced(case, seed, phi, c, q)
            s.y = _vector(s.lev, [d[0][None], d[1][None], d[2]])
    else:
        H.check(H.lib().ampe_rhs_eval(s.sim.h, 0.0, _ptr(s.y), _ptr(s.out), 0))
        s.gamma = _gamma(s.s)
        s.r = [_vector(s.lev, [torch.randn((6,) + phi.shape, generator=g, dtype=torch.float64,
                                           device=DEV)]) for _ in range(SOLVES)]
        s.z = [torch.zeros_like(s.y) for _ in range(SOLVES)]
    torch.cuda.synchronize()
    return s


def _gamma(sol):
    return sol.dt * 2.0 / 3.0


def _displaced(case, seed, phi, c, q):
    g = _gen(seed + 2)
    return (phi + 1e-4 * (_rand(g, *phi.shape) - 0.5), c + 1e-4 * (_rand(g, *c.shape) - 0.5),
            q + 1e-4 * (_rand(g, *q.shape) - 0.5))


_NETS = {}


def _network():
    """The trained network: a program trains it once, at start-up."""
    if "net" not in _NETS:
        p = P.polycrystal_params(ndim=3)
        _NETS["net"] = SG.train_kks_surrogate(p, P.auni_tdep(P.seeded_rk()), DEV,
                                              n_samples=1000000, steps=4000)[0]
    return _NETS["net"]


def _prepare_kks(case, seed):
    s = _Held()
    s.kind, s.case = "kks", case
    s.p, s.tab = P.polycrystal_params(ndim=3), P.auni_tdep(P.seeded_rk())
    g = _gen(seed)
    n = case["n"]
    s.c, s.phi, s.T = (0.05 + 0.9 * _rand(g, n), _rand(g, n), 1200.0 + 400.0 * _rand(g, n))
    s.cl, s.cs = torch.zeros_like(s.c), torch.zeros_like(s.c)
    s.it = torch.zeros(n, dtype=torch.int32, device=DEV)
    s.net = _network() if case["guess"] else None
    return s


def _dendrite(case):
    """Levels and fields of a three-level 2-D dendrite: level 0 in 5 x 5 uneven
    patches, level 1 over the middle half in 2 x 2 patches, level 2 over the
    seed in 3 x 2 patches."""
    n0 = case["n0"]
    p = P.dilute_params(ndim=2, dilute_keq=0.14)
    p.flux_type, p.aniso_nu, p.aniso_knumber = P.FLUX_ANISOTROPIC, 0.05, 4
    e = [0] + [2 * int(n0 * f / 2) for f in (0.21, 0.36, 0.6, 0.78)] + [n0]

    def grid(ex, ey):
        return [((ex[i], ey[j]), (ex[i + 1] - 1, ey[j + 1] - 1))
                for j in range(len(ey) - 1) for i in range(len(ex) - 1)]
    h = 2 * (n0 // 4)
    l1 = [h, 2 * (n0 // 2) - 2 * (n0 // 16), 2 * n0 - h]
    m = 4 * (n0 // 2) - 4 * (n0 // 12)
    w = 8 * (n0 // 12)
    l2x = [m, m + 4 * (w // 12), m + 8 * (w // 12), m + w]
    l2y = [m, m + 4 * (w // 8), m + w]
    return p, [grid(e, e), grid(l1, l1), grid(l2x, l2y)]


def _ternary(case):
    """Eight grains of two solids in liquid on two levels, the fine one over
    the middle of the domain in 2 x 2 x 2 patches (the Sintering deck's
    interface energy and mobilities)."""
    n0 = case["n0"]
    p = P.sintering_deck()[0]
    p.ndim, p.norderp, p.norderp_A = 3, 9, 4
    for a, (cur, ceq) in enumerate((((3e3, 5e3), (0.2, 0.2)), ((6e3, 4e3), (0.45, 0.15)),
                                    ((5e3, 8e3), (0.15, 0.4)))):
        for k in range(2):
            p.tern_A[a][k], p.tern_ceq[a][k] = cur[k], ceq[k]
    h = n0 // 2
    fine = [((h + i * h, h + j * h, h + k * h),
             (h + i * h + h - 1, h + j * h + h - 1, h + k * h + h - 1))
            for k in range(2) for j in range(2) for i in range(2)]
    return p, [[((0, 0, 0), (n0 - 1,) * 3)], fine]


def _prepare_amr(case, seed):
    s = _Held()
    s.kind, s.case = "amr", case
    n0 = case["n0"]
    dend = case["model"] == "dendrite"
    s.p, levels = (_dendrite if dend else _ternary)(case)
    nd = s.p.ndim
    s.hier = H.Hier(nd, levels, (n0,) * nd, tuple(s.p.dx), not dend)
    kw = dict(maxl=10, max_newton=5, gstype=P.GS_CLASSICAL,
              precision=P.FAC_FP32 if case["fp32"] else P.FP64)
    kw.update(dict(dt=1e-7, atol=1e-6, rtol=1e-8) if dend else
              dict(dt=1e-5, dt_init=1e-6, atol=1e-4, rtol=1e-6))
    s.s = P.solver_defaults(**kw)
    s.sim = H.HierSim(s.p, s.s, s.hier)
    s.y0 = np.zeros(s.sim.nc * s.hier.ncg)
    g = _gen(seed)
    pos, comp = _rand(g, 8, 3), 0.05 + 0.5 * _rand(g, 9, 2)
    blocks = [s.hier.patch_blocks(s.y0, m) for m in range(s.sim.nc)]

    def put(m, b, v):
        blocks[m][b][3][...] = v.cpu().numpy()

    thr = None
    for b, (lev, lo, hi, _) in enumerate(blocks[0]):
        r = 0.5 ** lev
        ax = [(torch.arange(lo[d], hi[d] + 1, dtype=torch.float64, device=DEV) + 0.5) * r
              for d in range(nd)]
        x = torch.meshgrid(*ax[::-1], indexing="ij")[::-1]
        if dend:
            d = torch.sqrt((x[0] - 0.5 * n0) ** 2 + (x[1] - 0.5 * n0) ** 2) * 4.0
            phi = 0.5 * (1.0 - torch.tanh((d - 0.25 * n0) / 2.0))
            noise = torch.randn(phi.shape, generator=g, dtype=torch.float64, device=DEV)
            put(0, b, (phi + 0.01 * noise * ((phi > 0.05) & (phi < 0.95))).clamp(0, 1))
            put(1, b, 0.05 + 0.002 * (2 * _rand(g, *phi.shape) - 1))
            for m in range(4):
                put(2 + m, b, torch.full_like(phi, 1.0 if m == 0 else 0.0))
            continue
        best = torch.full(x[0].shape, 1e300, dtype=torch.float64, device=DEV)
        lab = torch.zeros(best.shape, dtype=torch.int64, device=DEV)
        for k in range(8):
            d2 = 0
            for a in range(3):
                d = (x[a] - pos[k, a] * n0).abs()
                d = torch.minimum(d, n0 - d)
                d2 = d2 + d * d
            lab = torch.where(d2 < best, torch.full_like(lab, k), lab)
            best = torch.minimum(best, d2)
        dist = best.sqrt()
        if thr is None:
            thr = torch.kthvalue(dist.view(-1), int(0.7 * dist.numel()))[0]
        solid = 0.5 * (1.0 - torch.tanh((dist - thr) / 1.5))
        tot = torch.zeros_like(solid)
        c = [torch.zeros_like(solid) for _ in range(2)]
        for k in range(8):
            v = torch.where(lab == k, solid, torch.zeros_like(solid))
            put(k, b, v)
            tot += v
            for a in range(2):
                c[a] += v * comp[k, a]
        put(8, b, 1.0 - tot)
        for a in range(2):
            put(9 + a, b, c[a] + (1.0 - tot) * comp[8, a])
    return s


# ----------------------------------------------------------------------- run
def run(s):
    L = H.lib()
    if s.kind == "rhs":
        H.check(L.ampe_rhs_eval(s.sim.h, 0.0, _ptr(s.y), _ptr(s.out), int(s.case["lagged"])))
        return _fields(_views(s.lev, s.out, s.nc))
    if s.kind == "precond":
        j = C.c_int()
        H.check(L.ampe_precond_setup(s.sim.h, 0.0, _ptr(s.y), s.gamma, C.byref(j)))
        for r, z in zip(s.r, s.z):
            H.check(L.ampe_precond_solve(s.sim.h, 0.0, _ptr(r), _ptr(z), s.gamma, 1e-3))
        return [_fields(_views(s.lev, z, s.nc)) for z in s.z]
    if s.kind == "steps":
        s.sim.set_state(*s.host)
        rc, st = s.sim.advance(s.case["nsteps"])
        if rc:
            raise RuntimeError("the integrator gave up: %s" % st)
        return s.sim.get_state(s.shape)
    if s.kind == "amr":
        s.sim.set_state(s.y0)
        rc, st = s.sim.advance(s.case["nsteps"])
        if rc:
            raise RuntimeError("the integrator gave up: %s" % st)
        y = s.sim.get_state()
        return [np.concatenate([v.ravel() for *_, v in s.hier.patch_blocks(y, m)])
                for m in range(s.sim.nc)]
    H.kks_batch(s.p, s.tab, s.c, s.phi, s.T, s.cl, s.cs, iters=s.it, guess=s.net)
    return [s.cl, s.cs, s.it]


# ---------------------------------------------------------------------- work
def _cells(case):
    if case["kind"] == "amr":
        if case["model"] == "dendrite":
            lv = _dendrite(case)[1]
        else:
            lv = _ternary(case)[1]
        return sum(math.prod(hi[d] - lo[d] + 1 for d in range(len(lo))) for v in lv for lo, hi in v)
    return case["nx"] * case["ny"] * case["nz"]


def work(case):
    """Bytes: inputs read once, results written once.  The right-hand side of
    a full evaluation also leaves the phase concentrations and the face data
    of the lagged evaluations behind it; a lagged one reads them.  Integrator
    steps: per Newton iteration (two a step) and per Krylov iteration (three a
    Newton iteration) one state read and one written, the least the method
    can do.  Flops: a KKS Newton update is about 230, an energy 60."""
    kind = case["kind"]
    if kind == "kks":
        return dict(bytes=case["n"] * 44.0, flops=case["n"] * (1000.0 + (9000 if case["guess"] else 600)))
    n = float(_cells(case))
    nd = 2 if kind == "amr" and case["model"] == "dendrite" else 3
    if kind != "amr":
        nd = 3 if case["nz"] > 1 else 2
    nc = 11 if case.get("model") == "ternary" else 6
    kks = 700.0 if case.get("model") == "calphad" else 30.0
    if kind == "rhs":
        per = 8.0 * (2 * nc + 2 + 3 * nd + (0 if case["lagged"] else 2))
        return dict(bytes=n * per, flops=n * (kks + 60.0 * nd + 150.0))
    if kind == "precond":
        e = 4.0 if case["fp32"] else 8.0
        sweeps = 2.0
        setup = 8.0 * (nc + 2 + nd) + e * (2 + 2 * nd)
        solve = 16.0 * nc + e * (2 + 2 * nd)
        return dict(bytes=n * (setup + SOLVES * solve),
                    flops=n * (kks + SOLVES * sweeps * nc * (6 * nd + 4) * (8.0 / 7 if case["mg"] else 1)))
    its = case["nsteps"] * 2 * (1 + 3)
    return dict(bytes=n * 16.0 * nc * its, flops=n * its * (kks + nc * 40.0))


def tolerance(case):
    """Four times what was measured: rhs, precond and kks against exact();
    integrator runs with the Gram-Schmidt sums in the other order (classical,
    modified), and with the preconditioner in the other precision where it is
    FP32 (another rounding of a solve that only steers the Krylov loop)."""
    kind = case["kind"]
    if kind == "kks":
        return dict(rel=1.3e-13, max=2.2e-12, differ=2e-3)
    if kind == "rhs":
        # CALPHAD energies cancel in the driving force
        return dict(rel=3.2e-13, max=1.5e-11) if case["model"] == "calphad" else dict(rel=4e-15, max=1.2e-13)
    if kind == "precond":
        return dict(rel=5e-7, max=5e-6) if case["fp32"] else dict(rel=4e-15, max=1e-14)
    if kind == "amr":
        return dict(rel=2e-9, max=4e-8) if case["model"] == "ternary" else dict(rel=6e-11, max=3e-9)
    return dict(rel=1e-11, max=4e-10) if case["fp32"] else dict(rel=1e-12, max=1e-10)


# --------------------------------------------------------------------- exact
# Plain torch in 64 bits on domain arrays padded by one cell (periodic images,
# or the nearest cell on a bounded domain).  x, y, z are directions 0, 1, 2.
def _pad(a, nd, per):
    mode = "circular" if per else "replicate"
    if nd == 2:
        return F.pad(a.transpose(0, 1), (1, 1, 1, 1), mode=mode).transpose(0, 1)
    return F.pad(a[None], (1, 1, 1, 1, 1, 1), mode=mode)[0]


def _at(ap, nd, off, face=-1, side=0):
    """The padded array [k, nz, ny, nx] at offset off (x, y, z); face d: at
    the n + 1 faces of that direction, the cell below (side 0) or above."""
    sl = [slice(None)]
    for a in (2, 1, 0):
        m = ap.shape[3 - a]
        if a >= nd:
            sl.append(slice(None))
        elif a == face:
            sl.append(slice(0, m - 1) if side == 0 else slice(1, m))
        else:
            sl.append(slice(1 + off[a], m - 1 + off[a]))
    return ap[tuple(sl)]


def _lohi(f, d):
    """Values of a face array at the low and the high faces of the cells."""
    ax = 3 - d
    m = f.shape[ax]
    return f.narrow(ax, 0, m - 1), f.narrow(ax, 1, m - 1)


def _unit(d, s=1):
    o = [0, 0, 0]
    o[d] = s
    return o


def _interp(x, t):
    t = t.decode() if isinstance(t, bytes) else t
    if t == "q":
        return x.clamp(min=0.0) ** 2
    if t == "c":
        return torch.ones_like(x)
    x = x.clamp(0.0, 1.0)
    if t == "p":
        return x ** 3 * (10 - 15 * x + 6 * x * x)
    return x * x * (3 - 2 * x) if t == "h" else x


def _dinterp(x, t):
    t = t.decode() if isinstance(t, bytes) else t
    if t == "q":
        return 2 * x.clamp(min=0.0)
    if t == "c":
        return torch.zeros_like(x)
    if t == "l":
        return torch.ones_like(x)
    x = x.clamp(0.0, 1.0)
    return 30 * x * x * (1 - x) ** 2 if t == "p" else 6 * x * (1 - x)


def _f(p, c, k):
    if p.fe_model == P.FE_QUADRATIC:
        return p.quad_A[k] * (c - p.quad_ceq[k] - p.quad_m[k] * (p.temperature - p.quad_Tref)) ** 2
    rt = RGAS * p.temperature
    if p.fe_model == P.FE_KKS_DILUTE:
        f = rt * (c * torch.log(c) - c)
        if k == 1:
            f = f - rt * math.log(p.dilute_keq) * c + rt * (p.dilute_keq - 1.0) * (
                p.temperature - p.dilute_Tm) / p.dilute_m
        return f
    m = p.calphad[k]
    x = 2 * c - 1
    ex = m.L[0] + x * (m.L[1] + x * (m.L[2] + x * m.L[3]))
    return c * m.gA + (1 - c) * m.gB + rt * (c * torch.log(c) + (1 - c) * torch.log(1 - c)) \
        + c * (1 - c) * ex


def _mu_of(c, gA, gB, L, rt):
    x = 2 * c - 1
    ex = L[0] + x * (L[1] + x * (L[2] + x * L[3]))
    dx = L[1] + x * (2 * L[2] + x * 3 * L[3])
    return gA - gB + rt * torch.log(c / (1 - c)) + (1 - 2 * c) * ex + 2 * c * (1 - c) * dx


def _d2_of(c, L, rt):
    x = 2 * c - 1
    ex = L[0] + x * (L[1] + x * (L[2] + x * L[3]))
    dx = L[1] + x * (2 * L[2] + x * 3 * L[3])
    return rt / (c * (1 - c)) - 2 * ex + 4 * (1 - 2 * c) * dx + 4 * c * (1 - c) * (
        2 * L[2] + x * 6 * L[3])


def _mu(p, c, k):
    if p.fe_model == P.FE_QUADRATIC:
        return 2 * p.quad_A[k] * (c - p.quad_ceq[k] - p.quad_m[k] * (p.temperature - p.quad_Tref))
    rt = RGAS * p.temperature
    if p.fe_model == P.FE_KKS_DILUTE:
        return rt * torch.log(c) - (rt * math.log(p.dilute_keq) if k == 1 else 0.0)
    m = p.calphad[k]
    return _mu_of(c, m.gA, m.gB, m.L, rt)


def _d2f(p, c, k):
    return _d2_of(c, p.calphad[k].L, RGAS * p.temperature)


def _newton(c, h, cl, cs, ph, rt):
    """mu_L(cL) = mu_S(cS), (1 - h) cL + h cS = c from (cl, cs); ph: per phase
    (gA, gB, L), numbers or tensors."""
    for _ in range(40):
        f1 = (_mu_of(cl, *ph[0], rt) - _mu_of(cs, *ph[1], rt)) / rt
        f2 = (1 - h) * cl + h * cs - c
        a, b = _d2_of(cl, ph[0][2], rt) / rt, -_d2_of(cs, ph[1][2], rt) / rt
        det = a * h - b * (1 - h)
        dl, ds = -(h * f1 - b * f2) / det, -(a * f2 - (1 - h) * f1) / det
        al = torch.ones_like(c)
        for _ in range(30):
            out = (cl + al * dl <= 0) | (cl + al * dl >= 1) | (cs + al * ds <= 0) | (cs + al * ds >= 1)
            if not bool(out.any()):
                break
            al = torch.where(out, 0.5 * al, al)
        cl, cs = cl + al * dl, cs + al * ds
        if float(torch.maximum((al * dl).abs().max(), (al * ds).abs().max())) < 1e-14:
            break
    return cl, cs


def _phases(p, c, phi):
    """Phase concentrations of the level's solve."""
    h = _interp(phi, p.conc_interp)
    if p.fe_model == P.FE_QUADRATIC:
        e = [p.quad_ceq[k] + p.quad_m[k] * (p.temperature - p.quad_Tref) for k in range(2)]
        r = p.quad_A[0] / p.quad_A[1]
        cl = (c - h * (e[1] - r * e[0])) / (1 - h + h * r)
        return cl, e[1] + r * (cl - e[0])
    if p.fe_model == P.FE_KKS_DILUTE:
        cl = c / (1 - h + h * p.dilute_keq)
        return cl, p.dilute_keq * cl
    ph = [(p.calphad[k].gA, p.calphad[k].gB, p.calphad[k].L) for k in range(2)]
    return _newton(c, h, c.clone(), c.clone(), ph, RGAS * p.temperature)


def _norm2(p, qp, nd, d):
    """|grad q|^2 at the faces of direction d."""
    s = 0.0
    for n in range(nd):
        if n == d:
            g = (_at(qp, nd, [0] * 3, d, 1) - _at(qp, nd, [0] * 3, d, 0)) / p.dx[n]
        else:
            g = 0.25 / p.dx[n] * (_at(qp, nd, _unit(n), d, 0) - _at(qp, nd, _unit(n, -1), d, 0)
                                  + _at(qp, nd, _unit(n), d, 1) - _at(qp, nd, _unit(n, -1), d, 1))
        s = s + (g * g).sum(0, keepdim=True)
    return s


def _face_coef(p, pp, n2, nd, d):
    a = 0.5 * (_at(pp, nd, [0] * 3, d, 0) + _at(pp, nd, [0] * 3, d, 1))
    gni = torch.where(n2 > p.gradient_floor ** 2, n2.clamp(min=1e-300) ** -0.5,
                      torch.full_like(n2, 1.0 / p.gradient_floor))
    return -gni * 2.0 * p.H_parameter * p.temperature * _interp(a, p.orient_interp1) \
        - p.epsilon_q ** 2 * _interp(a, p.orient_interp2)


def _quat_mobility(p, phi):
    x = phi.clamp(0.0, 1.0)
    return p.min_quat_mobility + (p.quat_mobility - p.min_quat_mobility) * (
        1 - x ** 3 * (10 - 15 * x + 6 * x * x))


def _flux(p, pp, qp, nd, d):
    lo, hi = _at(pp, nd, [0] * 3, d, 0), _at(pp, nd, [0] * 3, d, 1)
    if p.flux_type != P.FLUX_ANISOTROPIC:
        return p.epsilon_phi ** 2 / p.dx[d] * (hi - lo)
    t = 1 - d
    gn = (hi - lo) / p.dx[d]
    gt = 0.25 / p.dx[t] * (_at(pp, nd, _unit(t), d, 0) - _at(pp, nd, _unit(t, -1), d, 0)
                           + _at(pp, nd, _unit(t), d, 1) - _at(pp, nd, _unit(t, -1), d, 1))
    gx, gy = (gn, gt) if d == 0 else (gt, gn)
    big = gx.abs() > float(np.float32(1e-12))
    th = torch.where(big, torch.atan(gy / torch.where(big, gx, torch.ones_like(gx))),
                     torch.full_like(gx, 0.5 * math.pi))
    qa = (0.5 * (_at(qp[:1], nd, [0] * 3, d, 0) + _at(qp[:1], nd, [0] * 3, d, 1))).clamp(-1.0, 1.0)
    w = p.aniso_knumber * (th - 2 * torch.acos(qa))
    e = p.epsilon_phi * (1 + p.aniso_nu * torch.cos(w))
    de = -p.aniso_knumber * p.epsilon_phi * p.aniso_nu * torch.sin(w)
    return e * e * gx - e * de * gy if d == 0 else e * e * gy + e * de * gx


def _diffusivities(p, pp, clp, csp, nd):
    rt = RGAS * p.temperature
    dl, ds = (p.D_liquid * math.exp(-p.Q0_liquid / rt), p.D_solid * math.exp(-p.Q0_solid / rt))
    out = []
    for d in range(nd):
        m = lambda a: 0.5 * (_at(a, nd, [0] * 3, d, 0) + _at(a, nd, [0] * 3, d, 1))  # noqa: E731
        f = m(pp)
        h = _interp(f, p.energy_interp)
        dd = (1 - h) * dl + h * ds
        out.append((dd, dd * _dinterp(f, p.energy_interp) * (m(clp) - m(csp))))
    return out


def _face_data(p, phi, c, q, nd, per):
    """The lagged face data: |grad q|^2 and the diffusivities."""
    pp, qp = _pad(phi, nd, per), _pad(q, nd, per)
    cl, cs = _phases(p, c, phi)
    return ([_norm2(p, qp, nd, d) for d in range(nd)],
            _diffusivities(p, pp, _pad(cl, nd, per), _pad(cs, nd, per), nd))


def _rhs(p, phi, c, q, data, nd, per):
    n2, dif = data
    pp, cp, qp = _pad(phi, nd, per), _pad(c, nd, per), _pad(q, nd, per)
    cl, cs = _phases(p, c, phi)
    zero = [0, 0, 0]
    r = 0.0
    for d in range(nd):
        lo, hi = _lohi(_flux(p, pp, qp, nd, d), d)
        r = r + (hi - lo) / p.dx[d]
    r = r - p.phi_well_scale * 32.0 * phi * (1 - phi) * (1 - 2 * phi)
    gm2 = 0.0
    for d in range(nd):
        g = 0.5 / p.dx[d] * (_at(qp, nd, _unit(d)) - _at(qp, nd, _unit(d, -1)))
        gm2 = gm2 + (g * g).sum(0, keepdim=True)
    r = r - 2 * p.H_parameter * p.temperature * _dinterp(phi, p.orient_interp1) * gm2.sqrt() \
        - 0.5 * p.epsilon_q ** 2 * _dinterp(phi, p.orient_interp2) * gm2
    kl, ka = 1e-6 / p.vm_L, 1e-6 / p.vm_A
    mu = _mu(p, cl, 0) * kl if p.fe_model == P.FE_QUADRATIC else _mu(p, cs, 1) * ka
    r = r + _dinterp(phi, p.energy_interp) * (_f(p, cl, 0) * kl - _f(p, cs, 1) * ka - mu * (cl - cs))
    rphi = p.phi_mobility * r
    rc = 0.0
    for d in range(nd):
        j = (dif[d][0] * (_at(cp, nd, zero, d, 1) - _at(cp, nd, zero, d, 0))
             + dif[d][1] * (_at(pp, nd, zero, d, 1) - _at(pp, nd, zero, d, 0))) / p.dx[d]
        lo, hi = _lohi(j, d)
        rc = rc + (hi - lo) / p.dx[d]
    div, lam = 0.0, 0.0
    for d in range(nd):
        f = _face_coef(p, pp, n2[d], nd, d) * (_at(qp, nd, zero, d, 1) - _at(qp, nd, zero, d, 0)) / p.dx[d]
        lo, hi = _lohi(f, d)
        div = div + (hi - lo) / p.dx[d]
        lam = lam - (q * (hi - lo)).sum(0, keepdim=True) * 0.5 / p.dx[d]
    lam = lam / (q * q).sum(0, keepdim=True)
    return torch.cat([rphi, p.conc_mobility * rc, -_quat_mobility(p, phi) * (div + 2 * q * lam)])


class _Grid:
    """One multigrid level: the three operators in 64 bits."""

    def __init__(self, nd, dx, gamma, p, cphi, dc, fc, sm, masks):
        self.nd, self.dx, self.gamma, self.p = nd, dx, gamma, p
        self.cphi, self.dc, self.fc, self.sm, self.masks = cphi, dc, fc, sm, masks

    def parts(self, x, block):
        """A x and its diagonal."""
        nd, z = self.nd, [0, 0, 0]
        xp = _pad(x, nd, True)
        if block == "q":
            sp = _pad(self.sm, nd, True)
            ax, dg = 0.0, 0.0
            for d in range(nd):
                lo, hi = (f / self.dx[d] ** 2 for f in _lohi(self.fc[d], d))
                dg = dg - lo - hi
                ax = ax + lo * _at(sp, nd, _unit(d, -1)) * _at(xp, nd, _unit(d, -1)) \
                    + hi * _at(sp, nd, _unit(d)) * _at(xp, nd, _unit(d))
            dg = self.gamma * self.sm ** 2 * dg + 1.0
            return dg * x + self.gamma * self.sm * ax, dg
        m = self.p.phi_mobility if block == "p" else self.p.conc_mobility
        cc = self.cphi if block == "p" else 1.0
        ax, dg = cc * x, cc
        for d in range(nd):
            if block == "p":
                lo = hi = -self.gamma * self.p.epsilon_phi ** 2
            else:
                lo, hi = _lohi(self.dc[d], d)
            w = m / self.dx[d] ** 2
            ax = ax + w * (hi * (_at(xp, nd, _unit(d)) - x) - lo * (x - _at(xp, nd, _unit(d, -1))))
            dg = dg - w * (hi + lo)
        return ax, dg

    def smooth(self, b, x, block, n):
        for _ in range(n):
            for m in self.masks:
                ax, dg = self.parts(x, block)
                x = torch.where(m, x + (b - ax) / dg, x)
        return x

    def mean(self, a):
        """Coarse cells: the mean of their children."""
        for d in range(self.nd):
            lo, hi = a.unfold(3 - d, 2, 2).unbind(-1)
            a = 0.5 * (lo + hi)
        return a

    def coarse(self):
        nd = self.nd

        def side(f, d):
            for e in range(nd):
                if e == d:
                    f = f.index_select(3 - e, torch.arange(0, f.shape[3 - e], 2, device=f.device))
                else:
                    lo, hi = f.unfold(3 - e, 2, 2).unbind(-1)
                    f = 0.5 * (lo + hi)
            return f
        sm = self.mean(self.sm)
        return _Grid(nd, [2 * h for h in self.dx], self.gamma, self.p, self.mean(self.cphi),
                     [side(f, d) for d, f in enumerate(self.dc)],
                     [side(f, d) for d, f in enumerate(self.fc)], sm, _colours(sm.shape[1:]))

    def prolong(self, e):
        nd = self.nd
        for d in range(nd):
            ax = 3 - d
            dn, up = torch.roll(e, 1, ax), torch.roll(e, -1, ax)
            e = torch.stack([0.75 * e + 0.25 * dn, 0.75 * e + 0.25 * up], ax + 1).flatten(ax, ax + 1)
        return e


def _colours(shape):
    k = [torch.arange(m, device=DEV) for m in shape]
    par = (k[0].view(-1, 1, 1) + k[1].view(1, -1, 1) + k[2].view(1, 1, -1)) % 2
    return [(par == col)[None] for col in range(2)]


def _vcycle(grids, b, block, sol, l=0):
    g = grids[l]
    x = torch.zeros_like(b)
    nu = sol.quat_sweeps if block == "q" else sol.fac_sweeps
    if l == len(grids) - 1:
        return g.smooth(b, x, block, sol.mg_coarse_sweeps)
    x = g.smooth(b, x, block, nu)
    r = b - g.parts(x, block)[0]
    x = x + g.prolong(_vcycle(grids, g.mean(r), block, sol, l + 1))
    return g.smooth(b, x, block, nu)


def _precond(case, p, sol, phi, c, q, rs):
    nd = p.ndim
    gamma = _gamma(sol)
    n2, dif = _face_data(p, phi, c, q, nd, True)
    pp = _pad(phi, nd, True)
    sm = _quat_mobility(p, phi).sqrt()
    cphi = 1 + gamma * p.phi_mobility * p.phi_well_scale * 32.0 * (1 + 6 * phi * (phi - 1))
    grids = [_Grid(nd, list(p.dx), gamma, p, cphi, [-gamma * a for a, _ in dif],
                   [_face_coef(p, pp, n2[d], nd, d) for d in range(nd)], sm,
                   _colours(phi.shape[1:]))]
    out = []
    if case["mg"]:
        ext = [m for m in phi.shape[1:] if m > 1]
        while len(grids) < sol.mg_max_levels and all(m % 2 == 0 and m // 2 >= 2 for m in ext):
            grids.append(grids[-1].coarse())
            ext = [m // 2 for m in ext]
    for r in rs:
        z = []
        for block, b in (("p", r[:1]), ("c", r[1:2]), ("q", r[2:] / sm)):
            if case["mg"]:
                x = _vcycle(grids, b, block, sol)
            else:
                x = grids[0].smooth(b, torch.zeros_like(b), block,
                                    sol.quat_sweeps if block == "q" else sol.fac_sweeps)
            z.append(x * sm if block == "q" else x)
        out.append(torch.cat(z))
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "kks":
        s = prepare(dict(case, guess=False), seed)
        ph = []
        for k in range(2):
            g = []
            for sp in range(2):
                f = s.tab.g[k][sp]
                v = torch.zeros_like(s.T)
                for j in range(f.nrange):
                    a = f.coef[j]
                    w = a[0] + a[1] * s.T + a[2] * s.T * torch.log(s.T) + a[3] * s.T ** 2 \
                        + a[4] * s.T ** 3 + a[5] * s.T ** 7 + a[6] / s.T + a[7] / s.T ** 9
                    v = w if j == 0 else torch.where(s.T >= f.Tc[j], w, v)
                g.append(v)
            ph.append((g[0], g[1], [s.tab.L[k][i][0] + s.tab.L[k][i][1] * s.T for i in range(4)]))
        h = _interp(s.phi, s.p.conc_interp)
        half = torch.full_like(s.c, 0.5)
        cl, cs = _newton(s.c, h, half, half.clone(), ph, RGAS * s.T)
        return [cl, cs, None]
    if kind in ("steps", "amr"):
        # where an implicit step stops depends on its Newton and Krylov
        # tolerances: no value of its own
        return None
    p, sol = _model(case), _solver(case)
    nd = p.ndim
    per = _domain(case) is not None
    phi, c, q = _state(case, p, seed, False)
    data = _face_data(p, phi[None], c[None], q, nd, per) if kind == "rhs" else None
    boxes = _boxes(case)
    if kind == "rhs":
        if case["lagged"]:
            phi, c, q = _displaced(case, seed, phi, c, q)
        r = _rhs(p, phi[None], c[None], q, data, nd, per)
        return _fields([_cut(r, b) for b in boxes])
    g = _gen(seed + 1)
    rs = [torch.randn((6,) + phi.shape, generator=g, dtype=torch.float64, device=DEV)
          for _ in range(SOLVES)]
    return [_fields([_cut(z, b) for b in boxes]) for z in _precond(case, p, sol, phi[None], c[None], q, rs)]
