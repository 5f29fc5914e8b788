"""The one-level preconditioner solve, every block in the same launches (one
cycle per block).

test_matches_host_cycle compares it with red-black sweeps and V-cycles written
out on whole-domain arrays on the host (every colour from the values before it,
neighbours by padding the domain, full residuals restricted, cleared starts): a
form that starts from zero without clearing, reads across the boundary, restricts
the red residuals alone or stores rows by parity has to give the same values to
rounding.  The block operators' coefficients come from their own entry points
and formulas.

The other tests compare the solve with itself, bit for bit: against the
block-by-block solve (with two cycles allowed and a tolerance no residual exceeds
it stops after the same first cycle; the same sweeps on sets of one block: what
is compared is how the blocks share launches, vectors and layouts), and one patch
against two halves.

Levels that wrap (one periodic patch of even extents), patches whose colours
meet, odd extents, odd patch corners and bounded levels, a V-cycle whose coarse
levels turn odd, the smallest extents, two ghost cells, no orientation, no
composition, and unequal sweep counts (two sets)."""
import ctypes as C

import numpy as np
import pytest

from ampe_amd import params as P

pytestmark = pytest.mark.gpu

GAMMA = 7e-4
# name: (extents, cuts along x, periodic)
LEVELS = {"wrap3": ((16, 12, 8), (), True), "wrap3_small": ((4, 4, 4), (), True),
          "wrap2": ((70, 12, 1), (), True), "two3": ((16, 12, 8), (6,), True),
          "halves3": ((16, 12, 8), (8,), True),
          "odd3": ((15, 12, 9), (), True), "odd_corner3": ((16, 12, 8), (5,), True),
          "odd2": ((33, 17, 1), (), True), "bounded3": ((12, 8, 10), (4,), False),
          "turns_odd2": ((140, 36, 1), (), True), "wide3": ((136, 6, 4), (64,), True)}


def _solve(level, cycles, fp32, mg, sweeps=(1, 1), operators=None, **model):
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
    H.check(L.ampe_precond_setup(sim.h, 0.0, ptr(y), GAMMA, C.byref(j)))
    for _ in range(2):  # the second solve starts from what the first left behind
        H.check(L.ampe_precond_solve(sim.h, 0.0, ptr(r), ptr(z), GAMMA, 1e30))
    torch.cuda.synchronize()
    if operators is not None:  # (y's ghosts are filled)
        operators.update(p=p, lev=lev, periodic=periodic, boxes=boxes, phi=phi,
                         r=_domain(lev, r.cpu().numpy(), nc, shape, ghost))
        side = lambda: torch.zeros(lev.nside_tot, dtype=torch.float64, device="cuda:0")  # noqa: E731
        n2, fc, Dc, Dp = side(), side(), side(), side()
        f, g = [y[m * lev.ncg:] for m in (0, 1, 2)], C.byref(p)
        H.check(L.ampe_quat_grad(lev.h, g, ptr(f[2]), None, ptr(n2), None))
        H.check(L.ampe_quat_face_coefs(lev.h, g, ptr(f[0]), ptr(n2), ptr(fc), None))
        H.check(L.ampe_conc_coeffs(lev.h, g, ptr(f[0]), ptr(f[1]), ptr(f[1]), ptr(Dc), ptr(Dp), None))
        operators.update(fc=fc.cpu().numpy(), Dc=Dc.cpu().numpy())
    return _domain(lev, z.cpu().numpy(), nc, shape, ghost)


def _domain(lev, v, nc, shape, ghost):
    """Domain arrays of nc component blocks."""
    out = np.zeros((nc,) + shape)
    for m, a in enumerate(v.reshape(nc, -1)):
        for k, b in enumerate(lev.boxes):
            out[m][..., b.lo[0]:b.hi[0] + 1] = lev.ghost_view(a, k)[(slice(ghost, -ghost),) * lev.ndim]
    return out


# ------------------------------------------------------------------ host cycle
def _near(a, d, periodic):
    """Neighbours' values below and above along d."""
    ax, n = a.ndim - 1 - d, a.shape[-1 - d]
    w = [(1, 1) if e == ax else (0, 0) for e in range(a.ndim)]
    ap = np.pad(a, w, mode="wrap" if periodic else "edge")
    return np.take(ap, range(n), ax), np.take(ap, range(2, n + 2), ax)


class _Grid:
    """One level's operators on domain arrays; direction d is axis -1 - d; cuts:
    the patches' corners along x."""

    def __init__(self, periodic, dx, cuts, C0, D, F, sm):
        self.periodic, self.dx, self.cuts = periodic, dx, cuts
        self.C, self.D, self.F, self.sm = C0, D, F, sm  # D, F: (low, high) per direction

    def rows(self, block, x, op):
        """A x and its diagonal."""
        nd = self.sm.ndim
        if block == "q":
            dg, ax = 0.0, 0.0
            for d in range(nd):
                (lo, hi), (xl, xh) = self.F[d], _near(self.sm * x, d, self.periodic)
                ax = ax + (lo * xl + hi * xh) / self.dx[d] ** 2
                dg = dg - (lo + hi) / self.dx[d] ** 2
            dg = 1.0 + op["gamma"] * self.sm ** 2 * dg
            return dg * x + op["gamma"] * self.sm * ax, dg
        c, m = (self.C, op["Mphi"]) if block == "p" else (1.0, op["Mc"])
        ax, dg = c * x, c
        for d in range(nd):
            lo, hi = (op["Dphi"],) * 2 if block == "p" else self.D[d]
            xl, xh = _near(x, d, self.periodic)
            ax = ax + m * (hi * (xh - x) - lo * (x - xl)) / self.dx[d] ** 2
            dg = dg - m * (lo + hi) / self.dx[d] ** 2
        return ax, dg

    def smooth(self, block, x, b, n, op):
        nd = self.sm.ndim
        idx = np.indices(self.sm.shape)
        par = idx.sum(0)
        if nd == 2:  # colours count from the patch's corner along x
            par = par - np.array([max(c for c in self.cuts if c <= i)
                                  for i in range(self.sm.shape[-1])])
        for _ in range(n):
            for colour in (0, 1):
                ax, dg = self.rows(block, x, op)
                x = np.where(par % 2 == colour, x + (b - ax) / dg, x)
        return x

    def coarse(self):
        nd = self.sm.ndim

        def side(pair, d):  # the mean of the fine faces covering a coarse one
            out = []
            for high, f in enumerate(pair):
                f = np.take(f, range(high, f.shape[-1 - d], 2), -1 - d)
                for e in range(nd):
                    f = f if e == d else _halve(f, e)
                out.append(f)
            return tuple(out)
        return _Grid(self.periodic, [2 * h for h in self.dx], [c // 2 for c in self.cuts],
                     _mean(self.C, nd), [side(f, d) for d, f in enumerate(self.D)],
                     [side(f, d) for d, f in enumerate(self.F)], _mean(self.sm, nd))

    def prolong(self, e):
        for d in range(self.sm.ndim):
            lo, hi = _near(e, d, self.periodic)
            ax = e.ndim - 1 - d
            sh = e.shape[:ax] + (2 * e.shape[ax],) + e.shape[ax + 1:]
            e = np.stack([0.75 * e + 0.25 * lo, 0.75 * e + 0.25 * hi], ax + 1).reshape(sh)
        return e


def _halve(a, d):
    n = a.shape[-1 - d]
    return 0.5 * (np.take(a, range(0, n, 2), -1 - d) + np.take(a, range(1, n, 2), -1 - d))


def _mean(a, nd):
    for d in range(nd):
        a = _halve(a, d)
    return a


def _cycle(grids, block, b, nu, ncoarse, op):
    g = grids[0]
    if len(grids) == 1:
        return g.smooth(block, np.zeros_like(b), b, ncoarse, op)
    x = g.smooth(block, np.zeros_like(b), b, nu, op)
    e = _cycle(grids[1:], block, _mean(b - g.rows(block, x, op)[0], g.sm.ndim), nu, ncoarse, op)
    return g.smooth(block, x + grids[1].prolong(e), b, nu, op)


def _faces(o, field):
    """(low, high) face values of every cell per direction from a side field."""
    lev, out = o["lev"], []
    nd = lev.ndim
    for d in range(nd):
        lo, hi = np.zeros(o["phi"].shape), np.zeros(o["phi"].shape)
        for k, b in enumerate(o["boxes"]):
            n = [b.hi[a] - b.lo[a] + 1 + (a == d) for a in range(nd)]
            f = field[lev.side_off[k][d]:][:int(np.prod(n))].reshape(n[::-1])
            sl = (..., slice(b.lo[0], b.hi[0] + 1))
            m = f.shape[-1 - d]
            lo[sl] = np.take(f, range(m - 1), -1 - d)
            hi[sl] = np.take(f, range(1, m), -1 - d)
        out.append((lo, hi))
    return out


@pytest.mark.parametrize("fp32,mg", [(False, False), (True, False), (False, True), (True, True)])
@pytest.mark.parametrize("sweeps", [(1, 1), (2, 1)])
@pytest.mark.parametrize("level", list(LEVELS))
def test_matches_host_cycle(dev, level, fp32, mg, sweeps):
    o = {}
    got = _solve(level, 1, fp32, mg, sweeps, operators=o)
    p, phi, nd = o["p"], o["phi"], o["lev"].ndim
    op = dict(gamma=GAMMA, Mphi=p.phi_mobility, Mc=p.conc_mobility, Dphi=-GAMMA * p.epsilon_phi ** 2)
    assert p.phi_well_type == b"d" and p.quat_mobility_type == b"p"
    sm = np.sqrt(p.min_quat_mobility + (p.quat_mobility - p.min_quat_mobility) *
                 (1 - phi ** 3 * (10 - 15 * phi + 6 * phi ** 2)))
    grids = [_Grid(o["periodic"], list(p.dx), [b.lo[0] for b in o["boxes"]],
                   1 + GAMMA * p.phi_mobility * p.phi_well_scale * 32 * (1 + 6 * phi * (phi - 1)),
                   [tuple(-GAMMA * a for a in f) for f in _faces(o, o["Dc"])],
                   _faces(o, o["fc"]), sm)]
    if mg:
        ends = lambda g: list(zip(g.cuts, g.cuts[1:] + [g.sm.shape[-1]]))  # noqa: E731
        while all(n % 2 == 0 and n >= 4 for n in list(grids[-1].sm.shape[:-1]) +
                  [e - c for c, e in ends(grids[-1])]) and all(c % 2 == 0 for c in grids[-1].cuts):
            grids.append(grids[-1].coarse())
    colours = 0
    for block, m, k, nu in (("p", 0, 1, sweeps[0]), ("c", 1, 1, sweeps[0]), ("q", 2, 4, sweeps[1])):
        b = o["r"][m:m + k] / (sm if block == "q" else 1.0)
        x = _cycle(grids, block, b, nu, 2 if mg else nu, op) * (sm if block == "q" else 1.0)
        colours = 2 * (2 if mg else nu) + 4 * nu * (len(grids) - 1)
        # a colour's update is some thirty roundings of terms of its row's size, the
        # rows are diagonally dominant, and an error passes on through later colours
        # and levels without growing
        u = 2.0 ** (-24 if fp32 else -53)
        err = np.linalg.norm(got[m:m + k] - x) / np.linalg.norm(x)
        assert err <= 30 * colours * u, (block, err, colours)


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
