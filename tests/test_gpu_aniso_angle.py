"""The 2-D anisotropic phase flux, whose angle terms are formed algebraically,
against the oracle's angle form: several symmetries (also zero and negative),
directions along both axes, phase gradients at and below the threshold where the
direction is taken as pi/2, orientations at and beyond the ends of acos, one and
four orientation components.

Bound: the angle form's cosine and sine are within kn 16 2^-53 of the exact ones,
the algebraic ones within kn 8 2^-53; a face's flux changes by at most
2 nu (1 + |kn|) of that relative to its size, a cell has four faces; 1e-13 for the
other terms, as for the simple flux."""
import ctypes as C

import numpy as np
import pytest

from ampe_amd import params as P
from test_gpu_parity import _dev, _fields, _p, _rel, _setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kn", [4, 6, 1, 2, 3, 8, 0, -4])
@pytest.mark.parametrize("kind", ["random", "axes", "flat", "ends", "one"])
def test_matches_angle_form(dev, kn, kind):
    nu = 0.05
    p = P.two_grain_params(ndim=2, flux_type=P.FLUX_ANISOTROPIC, aniso_nu=nu, aniso_knumber=kn,
                           with_conc=0)
    O, H, pt, lev = _setup(2, p)
    phi, q, _, _, _ = _fields(pt, seed=3)
    f, rng = phi.reshape(pt.ny + 2, -1), np.random.Generator(np.random.Philox(4))
    if kind == "axes":
        f[:] = np.cos(0.3 * np.arange(f.shape[1]))[None, :]  # gy = 0
        f[: f.shape[0] // 2] = np.sin(0.4 * np.arange(f.shape[0] // 2))[:, None]  # gx = 0
    elif kind == "flat":
        f[:] = 0.5 + 10.0 ** rng.uniform(-14, -9, f.shape) * rng.choice([-1, 1], f.shape)
    elif kind == "ends":
        q[:] = rng.choice([1.0, -1.0, 1.0 + 2.0 ** -52, 1.0 - 2.0 ** -53, 0.0], q.shape)
    elif kind == "one":
        p.evolve_quat, p.qlen = 0, 1
    r_o = pt.cells()
    O.lib().o_phase_rhs(C.byref(pt.G), C.byref(p), O.ptr(phi), O.ptr(q), None, None, O.ptr(r_o))
    ds = [_dev(a, dev) for a in (phi, q)]
    r = _dev(np.zeros_like(r_o), dev)
    H.check(H.lib().ampe_phase_rhs(lev.h, C.byref(p), _p(ds[0]), _p(ds[1]), None, None, _p(r),
                                   None))
    a, b = pt.interior(r.cpu().numpy()), pt.interior(r_o)
    assert np.all(np.isfinite(a))
    assert _rel(a, b) < 1e-13 + 4 * 2 * nu * (1 + abs(kn)) * abs(kn) * 24 * 2.0 ** -53
