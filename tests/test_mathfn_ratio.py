"""CPU check of the logarithm of a quotient used by the KKS solve and the
driving force (ampe_amd/csrc/mathfn.h: log_ratio), compiled with the host
compiler and compared with extended precision over quotients near one, across
the switch points sqrt(1/2) and sqrt(2), far apart, and subnormal; NaN outside
positive finite arguments."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

HDR = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "ampe_amd", "csrc", "mathfn.h")


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("ratio")
    src, so = d / "r.cpp", d / "r.so"
    src.write_text(f'#include "{os.path.abspath(HDR)}"\n'
                   'extern "C" void ratio(const double* a, const double* b, double* y, long n)\n'
                   '{ for (long i = 0; i < n; i++) y[i] = ampe::log_ratio(a[i], b[i]); }\n')
    subprocess.run(["g++", "-O2", "-ffp-contract=off", "-shared", "-fPIC", "-o", str(so),
                    str(src)], check=True)
    return C.CDLL(str(so))


def _ratio(L, a, b):
    a, b = (np.ascontiguousarray(v, dtype=np.float64) for v in (a, b))
    y = np.empty_like(a)
    L.ratio(*(v.ctypes.data_as(C.c_void_p) for v in (a, b, y)), C.c_long(a.size))
    return y


@pytest.mark.parametrize("spread", [1e-15, 1e-9, 1e-3, 0.7, 30.0, 600.0])
def test_rounding_bound(lib, spread):
    """The sum and the quotient in s and the final addition round once each (the
    difference is exact), the series and the exponent's tail add a fraction:
    3.6 units of 2^-53 relative."""
    rng = np.random.default_rng(3)
    a = np.exp(rng.uniform(-2.0, 2.0, 200_000))
    b = a * np.exp(rng.uniform(-spread, spread, a.size))
    # extended precision: log1p of the exact difference near one
    x, z = a.astype(np.longdouble), b.astype(np.longdouble)
    ref = np.where(np.abs(x - z) < 0.3 * z, np.log1p((x - z) / z), np.log(x) - np.log(z))
    err = np.abs(_ratio(lib, a, b) - ref)
    assert np.all(err <= 3.6 * 2.0 ** -53 * np.abs(ref))


def test_special_values(lib):
    a = np.array([1.0, 3.0, 5e-324, 1e308, 0.0, 1.0, -1.0, np.nan, np.inf, -1.0])
    b = np.array([1.0, 3.0, 1e-310, 1e-308, 1.0, 0.0, 1.0, 1.0, 1.0, -1.0])
    y = _ratio(lib, a, b)
    assert y[0] == 0.0 and y[1] == 0.0
    assert abs(y[2] - (np.log(5e-324) - np.log(1e-310))) < 1e-11
    assert abs(y[3] - 616 * np.log(10.0)) < 1e-12 * 1420
    assert np.all(np.isnan(y[4:]))
