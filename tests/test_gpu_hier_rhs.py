"""The integrator's right-hand side on a hierarchy (coarsening and ghosts of all
fields together, every level's cells in the same launches, one correction launch)
against the level-by-level, field-by-field entry points on the same state: a full
evaluation, then a lagged one at another state.  The state afterwards (covered
cells, all ghosts) and the right-hand side on the uncovered cells agree to the
last bit: the operations and their order are the same."""
import ctypes as C

import numpy as np
import pytest

from ampe_amd import params as P
from test_gpu_amr import HIERS

pytestmark = pytest.mark.gpu

MODELS = {
    "quadratic": lambda nd: P.two_grain_params(ndim=nd),
    "isotropic": lambda nd: P.two_grain_params(ndim=nd, flux_type=P.FLUX_ISOTROPIC),
    "calphad": lambda nd: P.polycrystal_params(ndim=nd),
    "dilute": lambda nd: P.dilute_params(ndim=nd, flux_type=P.FLUX_ANISOTROPIC, aniso_nu=0.04),
    "no_quat": lambda nd: P.two_grain_params(ndim=nd, evolve_quat=0),
    "no_conc": lambda nd: P.two_grain_params(ndim=nd, with_conc=0),
    "phase": lambda nd: P.two_grain_params(ndim=nd, with_conc=0, evolve_quat=0),
}


@pytest.mark.parametrize("model", list(MODELS))
@pytest.mark.parametrize("name", list(HIERS))
def test_matches_separate(dev, name, model):
    import torch
    from ampe_amd import hip as H
    nd, levels, dom0, periodic = HIERS[name]
    p = MODELS[model](nd)
    h = H.Hier(nd, levels, dom0, (p.dx[0],) * 3, periodic)
    s = P.solver_defaults(dt=1e-3, precision=P.FP64)
    sim = H.HierSim(p, s, h)
    L, ng, ns = H.lib(), h.ncg, h.nside_tot
    nq, nc = (4 if p.evolve_quat else 0), sim.nc
    rng = np.random.Generator(np.random.Philox(9))

    def state():
        y = rng.uniform(0.05, 0.95, (nc, ng))
        if p.with_conc:
            y[1] = rng.uniform(0.3, 0.5, ng)
        if nq:
            q = rng.normal(size=(4, ng))
            y[nc - 4:] = q / np.sqrt((q ** 2).sum(0))
        return torch.from_numpy(y).to(dev)

    ptr = lambda t: C.c_void_p(t.data_ptr()) if t is not None else None  # noqa: E731
    z = lambda n: torch.zeros(n, dtype=torch.float64, device=dev)  # noqa: E731
    unc = torch.from_numpy(np.zeros(ng)).to(dev)
    H.check(L.ampe_hier_weights(h.h, ptr(unc), None))
    torch.cuda.synchronize()
    unc = unc > 0
    comp = C.c_void_p()
    H.check(L.ampe_hier_composite(h.h, C.byref(comp)))
    side = [z(ns) for _ in range(3)]
    start = None
    for fd in (0, 1):
        y = state()
        if fd == 0:
            sim.set_state(y.cpu().numpy().ravel())
        ref, got = y.clone(), torch.zeros_like(y)
        torch.cuda.synchronize()
        H.check(L.ampe_hier_coarsen(h.h, ptr(ref[0]), 1, 0, None))
        if p.with_conc:
            H.check(L.ampe_hier_coarsen(h.h, ptr(ref[1]), 1, 0, None))
        if nq:
            H.check(L.ampe_hier_coarsen(h.h, ptr(ref[nc - 4:]), 4, 1, None))
        H.check(L.ampe_hier_ghost_fill(h.h, ptr(ref), nc, 2, None))
        H.check(L.ampe_rhs_eval(sim.h, 0.0, ptr(y), ptr(got), fd))
        torch.cuda.synchronize()
        assert torch.equal(y, ref)
        phi = ref[0]
        c = ref[1] if p.with_conc else None
        q = ref[nc - 4:] if nq else None
        cl = cs = None
        if c is not None:
            start = c.clone() if start is None else start
            cl, cs = z(ng), z(ng)
            torch.cuda.synchronize()
            H.check(L.ampe_kks_solve(comp, C.byref(p), ptr(phi), ptr(c), ptr(start), ptr(start),
                                     ptr(cl), ptr(cs), C.byref(C.c_int()), None))
        out = torch.zeros_like(ref)
        n2, Dc, Dp = side
        torch.cuda.synchronize()
        H.check(L.ampe_hier_phase_rhs(h.h, C.byref(p), ptr(phi), ptr(q), ptr(cl), ptr(cs),
                                      ptr(out[0]), None))
        if nq:
            fc = z(ns)
            torch.cuda.synchronize()
            if not fd:
                H.check(L.ampe_hier_quat_face_norm2(h.h, C.byref(p), ptr(q), ptr(n2), None))
            H.check(L.ampe_hier_quat_rhs(h.h, C.byref(p), ptr(phi), ptr(q), ptr(n2), ptr(fc),
                                         ptr(out[nc - 4:]), None))
        if c is not None:
            if not fd:
                H.check(L.ampe_hier_conc_coeffs(h.h, C.byref(p), ptr(phi), ptr(cl), ptr(cs),
                                                ptr(Dc), ptr(Dp), None))
            H.check(L.ampe_hier_conc_rhs(h.h, C.byref(p), ptr(c), ptr(phi), ptr(Dc), ptr(Dp),
                                         ptr(out[1]), None))
        torch.cuda.synchronize()
        a, b = got[:, unc], out[:, unc]
        assert bool(torch.isfinite(a).all()) and torch.equal(a, b), \
            (fd, [float((a[m] - b[m]).abs().max()) for m in range(nc)])
