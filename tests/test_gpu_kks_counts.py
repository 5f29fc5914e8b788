"""Counts of ampe_kks_solve from the workgroups' slots: a level of one
workgroup, one of a few, and one whose workgroups walk several strides; a call
with a failing cell, whose slots leave nothing behind for the next.  The
iterations returned are the largest over the cells, and equal what the same
cells take on another level."""
import ctypes as C

import numpy as np
import pytest

from ampe_amd import params as P

pytestmark = pytest.mark.gpu


def _solve(lev, p, x):
    import torch
    from ampe_amd import hip as H
    d = [torch.from_numpy(lev.to_ghosted(a)).to("cuda:0") for a in x]
    for t in d:
        H.check(H.lib().ampe_ghost_fill(lev.h, C.c_void_p(t.data_ptr()), 1, None))
    out = [torch.zeros_like(d[0]) for _ in range(2)]
    it = C.c_int(-7)
    ptr = lambda t: C.c_void_p(t.data_ptr())  # noqa: E731
    rc = H.lib().ampe_kks_solve(lev.h, C.byref(p), ptr(d[0]), ptr(d[1]), ptr(d[1]), ptr(d[1]),
                                ptr(out[0]), ptr(out[1]), C.byref(it), None)
    torch.cuda.synchronize()
    return rc, it.value, np.array([lev.ghost_view(o.cpu().numpy(), 0) for o in out])


@pytest.mark.parametrize("n", [(5, 3), (61, 33), (1100, 1010)])
def test_counts(dev, n):
    from ampe_amd import hip as H
    rng = np.random.Generator(np.random.Philox(4))
    p = P.polycrystal_params(ndim=2)
    shape = n[::-1]
    lev = H.Level(2, [H.boxes_of(shape, 2)], 1, periodic=H.boxes_of(shape, 2))
    hard = (rng.uniform(0.05, 0.95, shape), rng.uniform(0.2, 0.6, shape))
    # every cell the same: the count of that cell alone, however many there are
    easy = (np.full(shape, 0.5), np.full(shape, 0.4))
    rc, it, v = _solve(lev, p, hard)
    one = H.Level(2, [H.boxes_of((1, 1), 2)], 1, periodic=H.boxes_of((1, 1), 2))
    rc1, it1, v1 = _solve(one, p, (np.full((1, 1), 0.5), np.full((1, 1), 0.4)))
    assert rc >= 0 and rc1 >= 0 and it >= it1 > 0
    for _ in range(2):
        rc2, it2, v2 = _solve(lev, p, easy)
        assert rc2 == rc1 and it2 == it1
        assert np.array_equal(v2, np.broadcast_to(v1[:, :1, :1], v2.shape))
        bad = p.newton_max_its
        p.newton_max_its = 1  # one update is not enough: the call reports it
        rc3, it3, _ = _solve(lev, p, easy)
        p.newton_max_its = bad
        assert rc3 != rc1 or it3 != it1
    rc4, it4, v4 = _solve(lev, p, hard)
    assert (rc4, it4) == (rc, it) and np.array_equal(v4, v)
