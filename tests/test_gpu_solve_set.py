"""The one-level preconditioner solve with every block in the same launches
(one cycle per block) against the block-by-block solve: with two cycles allowed
and a tolerance no residual exceeds, the latter stops after the same first
cycle, so the solutions are identical to the last bit.  Levels that wrap (one
periodic patch of even extents: neighbours read across the boundary, a start
from zero that clears nothing), patches whose colours meet (ghost fills, the
same start), odd extents, odd patch corners and bounded levels (cleared start,
full residual), a V-cycle whose coarse levels turn odd, the smallest extents,
two ghost cells, no orientation, no composition, and unequal sweep counts (two
sets).  The same solves on one patch and on several agree as well where the
colouring does not depend on the patches."""
import ctypes as C

import numpy as np
import pytest

from ampe_amd import params as P

pytestmark = pytest.mark.gpu

# name: (extents, cuts along x, periodic)
LEVELS = {"wrap3": ((16, 12, 8), (), True), "wrap3_small": ((4, 4, 4), (), True),
          "wrap2": ((70, 12, 1), (), True), "two3": ((16, 12, 8), (6,), True),
          "halves3": ((16, 12, 8), (8,), True),
          "odd3": ((15, 12, 9), (), True), "odd_corner3": ((16, 12, 8), (5,), True),
          "odd2": ((33, 17, 1), (), True), "bounded3": ((12, 8, 10), (4,), False),
          "turns_odd2": ((140, 36, 1), (), True), "wide3": ((136, 6, 4), (64,), True)}


def _solve(level, cycles, fp32, mg, sweeps=(1, 1), **model):
    import torch
    from ampe_amd import hip as H
    n, cuts, periodic = LEVELS[level]
    nd = 3 if n[2] > 1 else 2
    p = P.two_grain_params(ndim=nd)
    for k, v in model.items():
        setattr(p, k, v)
    ghost = 2 if p.conc_rhs_form == P.CONC_RHS_EBS and p.ebs_stencil == P.EBS_ORDER4 else 1
    s = P.solver_defaults(dt=1e-3, fac_sweeps=sweeps[0], quat_sweeps=sweeps[1],
                          fac_max_cycles=cycles, quat_max_cycles=cycles, mg_coarse_sweeps=2,
                          precision=P.FAC_FP32 if fp32 else P.FP64,
                          precond=P.PRECOND_MG if mg else P.PRECOND_REDBLACK)
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
    sim = H.Sim(p, s, boxes, periodic=dom)
    lev = H.Level(nd, boxes, ghost, periodic=dom)
    rng = np.random.Generator(np.random.Philox(17))
    shape = (n[2], n[1], n[0]) if nd == 3 else (n[1], n[0])
    nq = 4 if p.evolve_quat else 0
    phi, c = rng.uniform(0.05, 0.95, shape), rng.uniform(0.3, 0.5, shape)
    q = rng.normal(size=(4,) + shape)
    q /= np.sqrt((q ** 2).sum(0))
    cut = lambda a: np.concatenate([a[..., b.lo[0]:b.hi[0] + 1].reshape(*a.shape[:a.ndim - nd], -1)  # noqa: E731
                                    for b in boxes], -1)
    sim.set_state(cut(phi), cut(c) if p.with_conc else None, cut(q) if nq else None)
    fields = [phi] + ([c] if p.with_conc else []) + [q[m] for m in range(nq)]
    nc = len(fields)
    vec = lambda f: torch.from_numpy(np.concatenate(  # noqa: E731
        [lev.to_ghosted(a, ghost) for a in f])).to("cuda:0")
    y, r = vec(fields), vec(list(rng.normal(size=(nc,) + shape)))
    out, z = torch.zeros_like(y), torch.full_like(y, float("nan"))
    ptr = lambda t: C.c_void_p(t.data_ptr())  # noqa: E731
    L = H.lib()
    torch.cuda.synchronize()
    H.check(L.ampe_rhs_eval(sim.h, 0.0, ptr(y), ptr(out), 0))
    j = C.c_int()
    H.check(L.ampe_precond_setup(sim.h, 0.0, ptr(y), 7e-4, C.byref(j)))
    for _ in range(2):  # the second solve starts from what the first left behind
        H.check(L.ampe_precond_solve(sim.h, 0.0, ptr(r), ptr(z), 7e-4, 1e30))
    torch.cuda.synchronize()
    got = z.cpu().numpy().reshape(nc, -1)
    res = []
    for m in range(nc):
        a = np.zeros(shape)
        for k, b in enumerate(boxes):
            v = lev.ghost_view(got[m], k)
            sl = (slice(ghost, -ghost),) * nd
            a[..., b.lo[0]:b.hi[0] + 1] = v[sl]
        res.append(a)
    return np.array(res)


@pytest.mark.parametrize("fp32,mg", [(False, False), (True, False), (False, True), (True, True)])
@pytest.mark.parametrize("level", list(LEVELS))
def test_set_solve_matches_block_by_block(dev, level, fp32, mg):
    a = _solve(level, 1, fp32, mg)
    b = _solve(level, 2, fp32, mg)
    assert np.all(np.isfinite(a)) and np.array_equal(a, b), float(np.max(np.abs(a - b)))


@pytest.mark.parametrize("mg", [False, True])
@pytest.mark.parametrize("model,sweeps", [
    (dict(evolve_quat=0), (2, 1)), (dict(with_conc=0), (2, 2)), (dict(), (2, 1)),
    (dict(), (1, 3)), (dict(), (0, 2)),
    (dict(conc_rhs_form=P.CONC_RHS_EBS, ebs_stencil=P.EBS_ORDER4), (1, 1))])
def test_models_and_sweeps(dev, model, sweeps, mg):
    for level in ("wrap3", "two3", "odd2"):
        for fp32 in (False, True):
            a = _solve(level, 1, fp32, mg, sweeps, **model)
            b = _solve(level, 2, fp32, mg, sweeps, **model)
            assert np.all(np.isfinite(a)) and np.array_equal(a, b), (level, fp32)


@pytest.mark.parametrize("fp32,mg", [(False, False), (True, False), (False, True), (True, True)])
def test_wrapped_patch_matches_several(dev, fp32, mg):
    # (halves: the same multigrid levels as the whole)
    assert np.array_equal(_solve("wrap3", 1, fp32, mg), _solve("halves3", 1, fp32, mg))
