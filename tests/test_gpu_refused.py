"""Models no kernel forms: refused with an error when the integrator is made, on
one level and on a hierarchy."""
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
