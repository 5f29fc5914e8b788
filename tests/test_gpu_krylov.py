"""SPGMR's fused vector kernels.  Long Krylov spaces (a compiled count of basis
vectors up to ten, a loop above) against the oracle's integrator, both
orthogonalisations; and classical against modified Gram-Schmidt, which share the
solution up to rounding, where their kernels differ in form: levels of one tile,
of few (each pass sums the products of the one before) and of more than 1024 (a
reduction in between), odd numbers of components, FP32 solutions read in the
row parity-split layout and in the plain one, FP64 ones, patch hierarchies are in
the hierarchy tests.

Tolerances: the fields of the first steps agree with the oracle to 1e-10 as with
short spaces.  Both orthogonalisations give the same vectors in exact
arithmetic; the solutions differ by the rounding of vectors of the state's size in
the WRMS norm (difference quotients: 2^-53 each, FP32 solves 2^-24) times the
condition of the preconditioned operator, 100 at most here (spectrum within
[0.02, 2])."""
import numpy as np
import pytest

from ampe_amd import params as P

pytestmark = pytest.mark.gpu


def _boxes(n, cuts):
    edges = [0, *cuts, n[0]]
    out = []
    for a, b in zip(edges, edges[1:]):
        box = P.Box()
        box.hi[:] = [b - 1, n[1] - 1, n[2] - 1]
        box.lo[:] = [a, 0, 0]
        out.append(box)
    dom = P.Box()
    dom.hi[:] = [n[0] - 1, n[1] - 1, n[2] - 1]
    return out, dom


@pytest.mark.parametrize("gstype,maxl,eplifac,model", [
    (P.GS_MODIFIED, 14, 1e-5, {}), (P.GS_CLASSICAL, 14, 1e-5, {}),
    # two vectors a pass: both remainders up to the longest space, odd component counts
    (P.GS_MODIFIED, 30, 1e-11, {}), (P.GS_MODIFIED, 29, 1e-11, dict(with_conc=0))])
def test_long_spaces_match_oracle(dev, gstype, maxl, eplifac, model):
    from oracle import oracle as O
    from ampe_amd import hip as H
    n = 48
    p = P.two_grain_params(ndim=2, **model)
    p.quad_ceq[0], p.quad_ceq[1] = 0.40, 0.45
    phi, c, q = P.two_grain_state(n=n, radius=n / 4, ndim=2)
    c = c if p.with_conc else None
    s = P.solver_defaults(maxl=maxl, max_newton=5, gstype=gstype, eplifac=eplifac)
    osim = O.Sim(p, s, n)
    osim.set_state(phi, c, q)
    box = H.boxes_of((n, n), 2)
    gsim = H.Sim(p, s, [box], periodic=box)
    gsim.set_state(phi, c, q)
    for _ in range(2):
        ro, _ = osim.advance(1)
        rg, st = gsim.advance(1)
        assert ro == rg == 0
    assert st["nli"] > (10 if maxl == 14 else 20) * st["nni"], st  # long spaces occurred
    for a, b in zip(gsim.get_state((n, n))[:3], osim.get_state()[:3]):
        if not b.any():
            continue  # a field the model does not have
        assert np.max(np.abs(a - b)) <= 1e-10 * np.max(np.abs(b))


@pytest.mark.parametrize("n,cuts,fp32,mg,model", [
    ((48, 4, 1), (), False, False, {}), ((64, 48, 1), (), False, True, {}),
    ((544, 512, 1), (), False, False, {}), ((544, 512, 1), (), True, True, {}),
    ((66, 34, 1), (33,), True, False, {}), ((128, 64, 1), (), True, True, dict(evolve_quat=0)),
    ((48, 40, 1), (), False, False, dict(with_conc=0)),
    ((48, 40, 1), (), False, False, dict(with_conc=0, evolve_quat=0)),
    ((32, 16, 16), (), True, True, {}), ((33, 15, 17), (10,), False, False, {})])
def test_classical_matches_modified(dev, n, cuts, fp32, mg, model):
    from ampe_amd import hip as H
    nd = 3 if n[2] > 1 else 2
    shape = (n[2], n[1], n[0]) if nd == 3 else (n[1], n[0])
    rng = np.random.Generator(np.random.Philox(3))
    x = [np.arange(k) for k in shape]
    wave = np.ones(shape)
    for a, k in enumerate(shape):
        wave = wave * (0.6 + 0.4 * np.cos(2 * np.pi * x[a] / k).reshape(
            [-1 if b == a else 1 for b in range(nd)]))
    phi = 0.1 + 0.8 * wave
    c = 0.42 + 0.01 * rng.uniform(-1, 1, shape)
    q = np.stack([wave, 1 - 0.5 * wave, 0.3 * wave, 0.2 + 0 * wave])
    q /= np.sqrt((q ** 2).sum(0))
    p = P.two_grain_params(ndim=nd, **model)
    p.quad_ceq[0], p.quad_ceq[1] = 0.40, 0.45
    boxes, dom = _boxes(n, cuts)
    cut = lambda a: np.concatenate([a[..., b.lo[0]:b.hi[0] + 1].reshape(*a.shape[:a.ndim - nd], -1)  # noqa: E731
                                    for b in boxes], -1)
    res, eplifac = [], 1e-4
    for gs in (P.GS_MODIFIED, P.GS_CLASSICAL):
        s = P.solver_defaults(maxl=13, max_newton=5, gstype=gs, eplifac=eplifac, dt=1e-3,
                              precision=P.FAC_FP32 if fp32 else P.FP64,
                              precond=P.PRECOND_MG if mg else P.PRECOND_REDBLACK)
        sim = H.Sim(p, s, boxes, periodic=dom)
        sim.set_state(cut(phi), cut(c) if p.with_conc else None, cut(q) if p.evolve_quat else None)
        rc, st = sim.advance(2)
        assert rc == 0 and st["nli"] >= 2 * st["nni"], st
        f = sim.get_state((sim.ncell,))[:3]
        res.append([f[0]] + ([f[1]] if p.with_conc else []) +
                   (list(f[2]) if p.evolve_quat else []))
    assert all(np.all(np.isfinite(a)) for a in res[0])
    ew = np.concatenate([(a - b) / (s.rtol * np.abs(b) + s.atol) for a, b in zip(*res)])
    moved = np.concatenate([(a - b) / (s.rtol * np.abs(b) + s.atol)
                            for a, b in zip(res[0][:1], [cut(phi)])])
    assert np.sqrt(np.mean(moved ** 2)) > 1.0  # the steps did something
    size = np.concatenate([b / (s.rtol * np.abs(b) + s.atol) for b in res[1]])
    bound = 100 * np.sqrt(np.mean(size ** 2)) * 2.0 ** (-24 if fp32 else -53)
    assert np.sqrt(np.mean(ew ** 2)) <= bound, (np.sqrt(np.mean(ew ** 2)), bound)


@pytest.mark.parametrize("n,cuts,fp32,mg", [((48, 40, 1), (), False, False),
                                            ((66, 34, 1), (33,), True, False),
                                            ((64, 32, 1), (), True, True),
                                            ((16, 12, 8), (), True, True),
                                            ((17, 6, 5), (9,), False, False)])
@pytest.mark.parametrize("make,kw", [
    (P.two_grain_params, {}), (P.two_grain_params, dict(evolve_quat=0)),
    (P.two_grain_params, dict(with_conc=0)), (P.two_grain_params, dict(with_conc=0, evolve_quat=0)),
    (P.two_grain_params, dict(flux_type=P.FLUX_ISOTROPIC)),
    (P.dilute_params, dict(flux_type=P.FLUX_ANISOTROPIC, aniso_nu=0.03))])
def test_values_passed_on_match_stored(dev, n, cuts, fp32, mg, make, kw):
    """A lagged evaluation passes its values on to the preconditioner's input, an
    unlagged one stores them for a launch of their own.  Where nothing that is
    lagged varies (gradients below the floor, equal phases) the two take the same
    steps to the last bit."""
    from ampe_amd import hip as H
    nd = 3 if n[2] > 1 else 2
    shape = (n[2], n[1], n[0]) if nd == 3 else (n[1], n[0])
    rng = np.random.Generator(np.random.Philox(8))
    p = make(ndim=nd, **kw)
    p.gradient_floor = 1e6
    p.D_solid, p.Q0_solid = p.D_liquid, p.Q0_liquid
    p.quad_ceq[0] = p.quad_ceq[1] = 0.4
    p.dilute_keq = 1.0
    phi, c = rng.uniform(0.3, 0.7, shape), rng.uniform(0.35, 0.45, shape)
    q = rng.normal(size=(4,) + shape) * 0.1 + 1.0
    q /= np.sqrt((q ** 2).sum(0))
    boxes, dom = _boxes(n, cuts)
    cut = lambda a: np.concatenate([a[..., b.lo[0]:b.hi[0] + 1].reshape(*a.shape[:a.ndim - nd], -1)  # noqa: E731
                                    for b in boxes], -1)
    res = []
    for lag in (0, 1):
        s = P.solver_defaults(maxl=5, max_newton=5, dt=1e-8, lag_quat_sidegrad=lag,
                              gstype=P.GS_CLASSICAL if fp32 else P.GS_MODIFIED,
                              precision=P.FAC_FP32 if fp32 else P.FP64,
                              precond=P.PRECOND_MG if mg else P.PRECOND_REDBLACK)
        sim = H.Sim(p, s, boxes, periodic=dom)
        sim.set_state(cut(phi), cut(c) if p.with_conc else None, cut(q) if p.evolve_quat else None)
        rc, st = sim.advance(2)
        assert rc == 0 and st["nli"] > 0, (rc, st)
        f = sim.get_state((sim.ncell,))
        res.append([f[0]] + ([f[1], f[3], f[4]] if p.with_conc else []) +
                   ([f[2]] if p.evolve_quat else []))
    for a, b in zip(*res):
        assert np.all(np.isfinite(a)) and np.array_equal(a, b), float(np.max(np.abs(a - b)))
