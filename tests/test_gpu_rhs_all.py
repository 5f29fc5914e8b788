"""The integrator's right-hand side, formed for all fields in one launch, against
the separate entry points: gradients, face coefficients, phase, orientation and
composition one after the other on the same fields.  A full evaluation, then a
lagged one at another state (face gradients and composition coefficients of the
first).  Levels of one and several patches, odd extents with remainder tiles,
columns longer and shorter than the planes a workgroup of the gradient kernel
marches over, bounded levels; each flux, energy, interpolation, average, floor
and mobility type; without orientation, without composition.

The operations and their order are the same, and so are the values.  The 3-D
gradient kernel for four components (a column of planes in LDS) is compared with
the general one (one component per call, the squares added): their transverse
gradients sum the same differences in another order, each within 8 roundings of
values <= 1, of gradients <= 2 / h, so |grad q|^2 of 12 squares differs by at most
12 * 2 * (2 / h) * 8 * 2^-53 / h."""
import ctypes as C

import numpy as np
import pytest

from ampe_amd import params as P

pytestmark = pytest.mark.gpu

# name: (extents, cuts along x, periodic)
LEVELS = {"tile3": ((64, 4, 16), (), True), "odd3": ((67, 9, 35), (), True),
          "thin3": ((5, 3, 2), (), True), "two3": ((70, 7, 18), (65,), True),
          "bounded3": ((12, 9, 17), (4,), False), "tile2": ((128, 8, 1), (), True),
          "odd2": ((67, 13, 1), (33,), True), "bounded2": ((9, 6, 1), (), False)}
INTERP = [b"q", b"p", b"h", b"w", b"l", b"m", b"3", b"s", b"c"]


def _check(level, p):
    import torch
    from ampe_amd import hip as H
    n, cuts, periodic = LEVELS[level]
    nd = p.ndim
    edges = [0, *cuts, n[0]]
    boxes = []
    for a, b in zip(edges, edges[1:]):
        box = P.Box()
        box.hi[:] = [b - 1, n[1] - 1, n[2] - 1]
        box.lo[:] = [a, 0, 0]
        boxes.append(box)
    dom = P.Box()
    dom.hi[:] = [n[0] - 1, n[1] - 1, n[2] - 1]
    dom = dom if periodic else None
    sim = H.Sim(p, P.solver_defaults(dt=1e-3), boxes, periodic=dom)
    lev = H.Level(nd, boxes, 1, periodic=dom)
    rng = np.random.Generator(np.random.Philox(5))
    shape = (n[2], n[1], n[0]) if nd == 3 else (n[1], n[0])
    nq = 4 if p.evolve_quat else 0

    def fields():
        phi, c = rng.uniform(0.02, 0.98, shape), rng.uniform(0.3, 0.5, shape)
        q = rng.normal(size=(4,) + shape)
        q /= np.sqrt((q ** 2).sum(0))
        return phi, c, q

    def vec(phi, c, q):
        f = [phi] + ([c] if p.with_conc else []) + [q[m] for m in range(nq)]
        return torch.from_numpy(np.concatenate([lev.to_ghosted(a, 1) for a in f])).to("cuda:0")

    cut = lambda a: np.concatenate([a[..., b.lo[0]:b.hi[0] + 1].reshape(*a.shape[:a.ndim - nd], -1)  # noqa: E731
                                    for b in boxes], -1)
    f0 = fields()
    sim.set_state(cut(f0[0]), cut(f0[1]) if p.with_conc else None, cut(f0[2]) if nq else None)
    L = H.lib()
    ptr = lambda t: C.c_void_p(t.data_ptr()) if t is not None else None  # noqa: E731
    dev = lambda k: torch.zeros(k, dtype=torch.float64, device="cuda:0")  # noqa: E731
    lagged = None
    for fd in (0, 1):
        y = vec(*(f0 if fd == 0 else fields()))
        nc = 1 + p.with_conc + nq
        ng = y.numel() // nc
        got = torch.zeros_like(y)
        torch.cuda.synchronize()
        H.check(L.ampe_rhs_eval(sim.h, 0.0, ptr(y), ptr(got), fd))
        # y's ghosts are filled now
        part = [y[m * ng:(m + 1) * ng].clone() for m in range(nc)]
        phi, c = part[0], part[1] if p.with_conc else None
        q = y[(nc - nq) * ng:].clone() if nq else None
        ref = torch.zeros_like(y)
        cl = cs = None
        if c is not None:
            cl, cs = dev(ng), dev(ng)
            if fd == 0:
                start = c  # the state's composition
            H.check(L.ampe_kks_solve(lev.h, C.byref(p), ptr(phi), ptr(c), ptr(start), ptr(start),
                                     ptr(cl), ptr(cs), C.byref(C.c_int()), None))
        ns = lev.nside_tot
        if lagged is None:
            lagged = [dev(ns) for _ in range(3)]
        n2, Dc, Dp = lagged
        rp = dev(ng)
        H.check(L.ampe_phase_rhs(lev.h, C.byref(p), ptr(phi), ptr(q), ptr(cl), ptr(cs), ptr(rp),
                                 None))
        ref[:ng] = rp
        if nq:
            fc, rq = dev(ns), dev(4 * ng)
            if not fd:
                H.check(L.ampe_quat_grad(lev.h, C.byref(p), ptr(q), None, ptr(n2), None))
                one, each = type(p).from_buffer_copy(p), dev(ns)
                one.evolve_quat, one.qlen = 0, 1
                tot = dev(ns)
                for m in range(4):
                    H.check(L.ampe_quat_grad(lev.h, C.byref(one), ptr(part[nc - nq + m]), None,
                                             ptr(each), None))
                    torch.cuda.synchronize()
                    tot += each
                    torch.cuda.synchronize()
                bound = 12 * 2 * 2 * 8 * 2.0 ** -53 / p.dx[0] ** 2
                assert float((n2 - tot).abs().max()) <= bound
            H.check(L.ampe_quat_face_coefs(lev.h, C.byref(p), ptr(phi), ptr(n2), ptr(fc), None))
            H.check(L.ampe_quat_rhs_fc(lev.h, C.byref(p), ptr(phi), ptr(q), ptr(fc), ptr(rq), None))
            ref[(nc - nq) * ng:] = rq
        if p.with_conc:
            rc = dev(ng)
            if not fd:
                H.check(L.ampe_conc_coeffs(lev.h, C.byref(p), ptr(phi), ptr(cl), ptr(cs), ptr(Dc),
                                           ptr(Dp), None))
            H.check(L.ampe_conc_rhs(lev.h, C.byref(p), ptr(c), ptr(phi), ptr(Dc), ptr(Dp), ptr(rc),
                                    None))
            ref[ng:2 * ng] = rc
        torch.cuda.synchronize()
        for m in range(nc):
            a, b = got[m * ng:(m + 1) * ng].cpu().numpy(), ref[m * ng:(m + 1) * ng].cpu().numpy()
            for k in range(len(boxes)):
                sl = (slice(1, -1),) * nd
                u, v = lev.ghost_view(a, k)[sl], lev.ghost_view(b, k)[sl]
                assert np.all(np.isfinite(u)), (fd, m)
                assert np.array_equal(u, v), (fd, m, k, float(np.max(np.abs(u - v))),
                                              float(np.max(np.abs(v))))


@pytest.mark.parametrize("level", list(LEVELS))
@pytest.mark.parametrize("make,flux", [
    (P.two_grain_params, P.FLUX_SIMPLE), (P.two_grain_params, P.FLUX_ISOTROPIC),
    (P.polycrystal_params, P.FLUX_SIMPLE), (P.dilute_params, P.FLUX_ANISOTROPIC)])
def test_levels(dev, level, make, flux):
    nd = 3 if LEVELS[level][0][2] > 1 else 2
    _check(level, make(ndim=nd, flux_type=flux, aniso_nu=0.04))


@pytest.mark.parametrize("kw", [
    dict(evolve_quat=0), dict(with_conc=0), dict(evolve_quat=0, with_conc=0),
    dict(avg_type=b"h"), dict(floor_type=b"t"), dict(floor_type=b"s"), dict(phi_well_type=b"s"),
    dict(quat_mobility_type=b"e"), dict(quat_mobility_type=b"i")]
    + [dict(energy_interp=t, orient_interp1=INTERP[-1 - i], orient_interp2=INTERP[i - 3])
       for i, t in enumerate(INTERP)])
def test_types(dev, kw):
    for level in ("odd2", "two3"):
        nd = 3 if level == "two3" else 2
        _check(level, P.two_grain_params(ndim=nd, **kw))


@pytest.mark.parametrize("nd,floor", [(2, b"m"), (3, b"t"), (3, b"s")])
def test_lagged_before_any_full(dev, nd, floor):
    """A lagged evaluation of a new integrator takes no face gradients: the
    orientation's right-hand side is the separate entry point's with |grad q|^2 = 0
    on every face (the floor's coefficient)."""
    import torch
    from ampe_amd import hip as H
    shape = (9, 12, 70)[3 - nd:]
    box = H.boxes_of(shape, nd)
    p = P.two_grain_params(ndim=nd, with_conc=0, floor_type=floor)
    sim = H.Sim(p, P.solver_defaults(dt=1e-3), [box], periodic=box)
    lev = H.Level(nd, [box], 1, periodic=box)
    rng = np.random.Generator(np.random.Philox(6))
    phi, q = rng.uniform(0.1, 0.9, shape), rng.normal(size=(4,) + shape)
    q /= np.sqrt((q ** 2).sum(0))
    y = torch.from_numpy(np.concatenate([lev.to_ghosted(a) for a in [phi, *q]])).to(dev)
    got = torch.zeros_like(y)
    n2 = torch.zeros(lev.nside_tot, dtype=torch.float64, device=dev)
    want = torch.zeros(4 * lev.ncg, dtype=torch.float64, device=dev)
    ptr = lambda t: C.c_void_p(t.data_ptr())  # noqa: E731
    torch.cuda.synchronize()
    H.check(H.lib().ampe_rhs_eval(sim.h, 0.0, ptr(y), ptr(got), 1))  # fills y's ghosts
    torch.cuda.synchronize()
    H.check(H.lib().ampe_quat_rhs(lev.h, C.byref(p), ptr(y), ptr(y[lev.ncg:]), ptr(n2), ptr(want),
                                  None))
    a, b = got.cpu().numpy()[lev.ncg:].reshape(4, -1), want.cpu().numpy().reshape(4, -1)
    for m in range(4):
        u, v = (lev.ghost_view(x[m], 0)[(slice(1, -1),) * nd] for x in (a, b))
        assert np.abs(v).max() > 0 and np.array_equal(u, v)
