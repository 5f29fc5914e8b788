"""The hierarchy preconditioner with every block in the same launches against
the block-by-block FAC solve: same operations on the same values, so the
integrator's states and counters are identical to the last bit.  The
block-by-block form is the one with a coarse-solve tolerance (fac_tol = 0 is
never met, so its sweeps are the same).  Three bounded 2-D levels of uneven
patches with the orientation block, with equal and unequal sweep counts
(one set, or the orientation after the elliptic blocks), nine orders and two
species on two periodic 3-D levels (slots of four, four and one component)
and fifty orders in 2-D (thirteen slots), in FP64 and FP32."""
import ctypes as C

import numpy as np
import pytest

from ampe_amd import params as P

pytestmark = pytest.mark.gpu


def _fill(hier, y, nc, f):
    blocks = [hier.patch_blocks(y, m) for m in range(nc)]
    for b, (lev, lo, hi, _) in enumerate(blocks[0]):
        ax = [(np.arange(lo[d], hi[d] + 1) + 0.5) * 0.5 ** lev for d in range(hier.ndim)]
        x = np.meshgrid(*ax[::-1], indexing="ij")[::-1]
        for m, v in enumerate(f(x)):
            blocks[m][b][3][...] = v


def _dendrite(H):
    p = P.dilute_params(ndim=2, dilute_keq=0.14)
    p.flux_type, p.aniso_nu, p.aniso_knumber = P.FLUX_ANISOTROPIC, 0.05, 4
    levels = [[((0, 0), (10, 23)), ((11, 0), (23, 23))],
              [((12, 12), (25, 35)), ((26, 12), (35, 35))], [((30, 28), (41, 43))]]
    h = H.Hier(2, levels, (24, 24), tuple(p.dx), False)

    def f(x):
        d = np.sqrt((x[0] - 12.3) ** 2 + (x[1] - 11.8) ** 2) * 4.0
        phi = 0.5 * (1.0 - np.tanh((d - 8.0) / 2.0))
        a = 0.3 * np.sin(0.4 * x[0]) * np.cos(0.3 * x[1])
        return [phi, 0.05 + 0.002 * np.sin(x[0] + 2 * x[1]), np.cos(a), np.sin(a), 0 * a, 0 * a]
    return p, h, f, dict(dt=1e-7, atol=1e-6, rtol=1e-8)


def _orders(H, ndim, n0, nord, tern):
    p = P.sintering_deck()[0]
    p.ndim, p.norderp, p.norderp_A = ndim, nord, nord // 2
    if not tern:
        p.with_conc, p.fe_model = 0, P.FE_QUADRATIC
    h0 = n0 // 2
    fine = [((h0,) * ndim, (h0 + 7,) * ndim), ((h0 + 8,) + (h0,) * (ndim - 1),
                                               (h0 + 13,) + (h0 + 5,) * (ndim - 1))]
    h = H.Hier(ndim, [[((0,) * ndim, (n0 - 1,) * ndim)], fine], (n0,) * ndim, tuple(p.dx), True)
    rng = np.random.Generator(np.random.Philox(8))
    pos = rng.uniform(0, n0, (nord - 1, ndim))

    def f(x):
        out, tot = [], 0.0
        for s in pos:
            d = np.sqrt(sum((a - b) ** 2 for a, b in zip(x, s)))
            v = 0.5 * (1.0 - np.tanh((d - 0.2 * n0) / 1.5)) / (nord - 1)
            out.append(v)
            tot = tot + v
        out.append(1.0 - tot)
        return out + ([0.3 + 0.2 * out[0], 0.4 - 0.3 * out[1]] if tern else [])
    return p, h, f, dict(dt=1e-6, atol=1e-4, rtol=1e-6)


CASES = {"dendrite_equal": (lambda H: _dendrite(H), 2, 2),
         "dendrite_more_orientation": (lambda H: _dendrite(H), 1, 3),
         "dendrite_fewer_orientation": (lambda H: _dendrite(H), 3, 1),
         "ternary_3d": (lambda H: _orders(H, 3, 16, 9, True), 2, 2),
         "fifty_orders_2d": (lambda H: _orders(H, 2, 20, 50, False), 2, 1)}


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("case", list(CASES))
def test_set_solve_matches_block_by_block(dev, case, fp32):
    from ampe_amd import hip as H
    make, fac, quat = CASES[case]
    p, h, f, kw = make(H)
    got = []
    for tol in (-1.0, 0.0):
        s = P.solver_defaults(maxl=8, max_newton=5, fac_sweeps=fac, quat_sweeps=quat, fac_tol=tol,
                              precision=P.FAC_FP32 if fp32 else P.FP64, **kw)
        sim = H.HierSim(p, s, h)
        y = np.zeros(sim.nc * h.ncg)
        _fill(h, y, sim.nc, f)
        sim.set_state(y)
        rc, st = sim.advance(2)
        assert rc == 0, st
        got.append((sim.get_state(), {k: st[k] for k in ("nst", "nni", "nli", "nps", "ncfn")}))
    assert got[0][1] == got[1][1], (got[0][1], got[1][1])
    for m in range(sim.nc):
        for (*_, a), (*_, b) in zip(h.patch_blocks(got[0][0], m), h.patch_blocks(got[1][0], m)):
            assert np.array_equal(a, b), (case, m, float(np.max(np.abs(a - b))))


def test_state_after_steps_is_averaged(dev):
    """The integrator's solve leaves covered cells undefined: both state outputs
    hold the averages there, and the steps do not depend on what was there."""
    from ampe_amd import hip as H
    nd, levels, dom0, periodic = 2, [[((0, 0), (15, 15))], [((8, 8), (23, 23))]], (16, 16), True
    p = P.two_grain_params(ndim=nd)
    p.quad_ceq[0], p.quad_ceq[1] = 0.40, 0.45
    h = H.Hier(nd, levels, dom0, (1.0,) * 3, periodic)
    sim = H.HierSim(p, P.solver_defaults(dt=1e-3), h)
    rng = np.random.Generator(np.random.Philox(2))
    y = rng.uniform(0.4, 0.6, (sim.nc, h.ncg))
    y[sim.nc - 4:] /= np.sqrt((y[sim.nc - 4:] ** 2).sum(0))
    sim.set_state(y.ravel())
    rc, _ = sim.advance(2)
    assert rc == 0
    a = sim.get_state().reshape(sim.nc, -1)
    ncell = 16 * 16 + 16 * 16
    f = [np.zeros(ncell), np.zeros(ncell), np.zeros((4, ncell))]
    ptr = lambda v: v.ctypes.data_as(C.c_void_p)  # noqa: E731
    H.check(H.lib().ampe_sim_get_state(sim.h, ptr(f[0]), ptr(f[1]), ptr(f[2]), None, None))
    # level 0's interior of the composite layout, cells 4..11 covered
    for m, v in enumerate([f[0], f[1], *f[2]]):
        c = a[m, :18 * 18].reshape(18, 18)[1:-1, 1:-1]
        fine = a[m, 18 * 18:].reshape(18, 18)[1:-1, 1:-1]
        assert np.array_equal(v[:256].reshape(16, 16), c)
        assert np.array_equal(v[256:].reshape(16, 16), fine)
        if m < 2:
            avg = 0.25 * (fine[::2, ::2] + fine[1::2, ::2] + fine[::2, 1::2] + fine[1::2, 1::2])
            assert np.max(np.abs(c[4:12, 4:12] - avg)) <= 8 * 2.0 ** -53
