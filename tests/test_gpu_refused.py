"""Models no kernel forms and fields a kernel would read that are not there:
refused with an error, on one level and on a hierarchy, before anything is
launched."""
import ctypes as C

import pytest

from ampe_amd import params as P

pytestmark = pytest.mark.gpu


def _make(p, hier):
    from ampe_amd import hip as H
    s = P.solver_defaults()
    box = H.boxes_of((8, 8), 2)
    if not hier:
        return H.Sim(p, s, [box], periodic=box)
    h = H.Hier(2, [[((0, 0), (7, 7))], [((4, 4), (11, 11))]], (8, 8), tuple(p.dx), True)
    return H.HierSim(p, s, h)


@pytest.mark.parametrize("hier", [False, True])
def test_unknown_free_energy(dev, hier):
    from ampe_amd import hip as H
    p = P.two_grain_params(ndim=2)
    p.fe_model = 7
    with pytest.raises(H.AmpeError, match="free-energy"):
        _make(p, hier)
    p.with_conc = 0  # no composition field, no energy: as before
    _make(p, hier)


@pytest.mark.parametrize("hier", [False, True])
def test_anisotropy_without_orientation(dev, hier):
    from ampe_amd import hip as H
    p = P.dilute_params(ndim=2, flux_type=P.FLUX_ANISOTROPIC, aniso_nu=0.05, evolve_quat=0)
    with pytest.raises(H.AmpeError, match="orientation"):
        _make(p, hier)
    p.flux_type = P.FLUX_SIMPLE
    _make(p, hier)


@pytest.mark.parametrize("missing", ["orientation", "anisotropy", "concentrations"])
def test_hierarchy_phase_rhs_fields(dev, missing):
    import torch
    from ampe_amd import hip as H
    h = H.Hier(2, [[((0, 0), (7, 7))], [((4, 4), (11, 11))]], (8, 8), (1.0, 1.0, 1.0), True)
    p = P.dilute_params(ndim=2)
    if missing == "anisotropy":
        p.evolve_quat, p.flux_type = 0, P.FLUX_ANISOTROPIC
    x = torch.zeros(4 * h.ncg, dtype=torch.float64, device=dev)
    ptr = C.c_void_p(x.data_ptr())
    q, cl = (ptr, None) if missing == "concentrations" else (None, ptr)
    rc = H.lib().ampe_hier_phase_rhs(h.h, C.cast(C.pointer(p), C.c_void_p), ptr, q, cl, cl, ptr,
                                     None)
    assert rc < 0 and missing.encode() in H.lib().ampe_last_error()
