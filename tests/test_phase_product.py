"""CPU check of the tile phasors' sin and cos of a product (mwa_hyperdrive_amd/csrc/sm_math.h), against
the product reduced in exact rational arithmetic."""

import ctypes as C
import math
import subprocess
from fractions import Fraction
from pathlib import Path

import numpy as np
import pytest

ROOT = Path(__file__).resolve().parent.parent
SRC = r"""
#include "sm_math.h"
static const double kTab[128] = {SM_SINCOS32_TABLE};
extern "C" void run(int n, const double *x, const double *f, double c, double *s, double *co) {
    for (int i = 0; i < n; ++i) sm::table_sincos_product(x[i], sm::two_quotient(f[i], c), kTab, s[i], co[i]);
}
extern "C" void quotient(double a, double b, double *out) {
    const sm::TwoDouble q = sm::two_quotient(a, b);
    out[0] = q.hi;
    out[1] = q.lo;
}
"""
# pi to 60 digits
PI = Fraction(3141592653589793238462643383279502884197169399375105820974945, 10 ** 60)


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("phase")
    (d / "t.cpp").write_text(SRC)
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", f"-I{ROOT / 'mwa_hyperdrive_amd' / 'csrc'}",
                    "-o", str(d / "t.so"), str(d / "t.cpp")], check=True)
    L = C.CDLL(str(d / "t.so"))
    L.run.argtypes = [C.c_int, C.c_void_p, C.c_void_p, C.c_double, C.c_void_p, C.c_void_p]
    L.quotient.argtypes = [C.c_double, C.c_double, C.c_void_p]
    return L


def test_quotient_in_two_doubles(lib):
    rng = np.random.default_rng(0)
    out = np.empty(2)
    for a in np.concatenate([[0.0, 1.0, -167e6], rng.uniform(-1e9, 1e9, 200)]):
        lib.quotient(float(a), 299792458.0, out.ctypes.data)
        exact = Fraction(float(a)) / 299792458
        assert out[0] == float(exact)
        assert abs(Fraction(out[0]) + Fraction(out[1]) - exact) <= abs(exact) * Fraction(1, 2 ** 104)


def test_phases_of_long_baselines(lib):
    """The bound of the sine alone (4e-16 for an exact argument); the phase rounded to one double
    is off by up to half a spacing, 9e-13 at 1e4 rad."""
    rng = np.random.default_rng(1)
    n = 3000
    x = rng.uniform(-2e4, 2e4, n)
    f = rng.choice([40e3, 1.28e6, 100e6, 167e6, 2.7e9], n) + rng.integers(0, 10 ** 6, n)
    x[0], f[1] = 0.0, 0.0
    s, c = np.empty(n), np.empty(n)
    lib.run(n, x.ctypes.data, f.ctypes.data, 299792458.0, s.ctypes.data, c.ctypes.data)
    worst = rounded = 0.0
    for i in range(n):
        p = Fraction(float(x[i])) * Fraction(float(f[i])) / 299792458
        r = float(p - 2 * PI * round(p / (2 * PI)))
        # (1.5 eps of r <= pi: the reduced argument and the library's own sine are rounded too.)
        worst = max(worst, abs(s[i] - math.sin(r)), abs(c[i] - math.cos(r)))
        rounded = max(rounded, abs(math.sin(x[i] * (f[i] / 299792458.0)) - math.sin(r)))
    assert worst <= 4e-16 + 1.5 * math.pi * 2.0 ** -53
    assert rounded > 1e-12  # what one double would have lost
