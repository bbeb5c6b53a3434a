"""CPU check of the kernels' FP64 exponentials (mwa_hyperdrive_amd/csrc/sm_math.h), compiled for
the host with g++ and compared with a 30-digit evaluation."""

import ctypes as C
import subprocess
from decimal import Decimal, getcontext
from pathlib import Path

import numpy as np
import pytest

ROOT = Path(__file__).resolve().parent.parent
SRC = r"""
#include "sm_math.h"
static const double kTab[64] = {SM_EXP64_TABLE};
extern "C" void run_table(int n, const double *x, double *y) {
    for (int i = 0; i < n; ++i) y[i] = sm::table_exp(x[i], kTab);
}
extern "C" void run_small(int n, const double *x, double *y) {
    for (int i = 0; i < n; ++i) y[i] = sm::small_exp(x[i]);
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("exp")
    (d / "t.cpp").write_text(SRC)
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", f"-I{ROOT / 'mwa_hyperdrive_amd' / 'csrc'}",
                    "-o", str(d / "t.so"), str(d / "t.cpp")], check=True)
    return C.CDLL(str(d / "t.so"))


def run(fn, x):
    x = np.ascontiguousarray(x, np.float64)
    y = np.empty_like(x)
    fn(x.size, C.c_void_p(x.ctypes.data), C.c_void_p(y.ctypes.data))
    return y


def exact(x):
    getcontext().prec = 30
    return [Decimal(float(v)).exp() for v in x]


# Table entry and final rounding half an ulp each, the series' roundings on |e^r - 1| < 0.006:
# 1.1 ulp, i.e. 2.5e-16 relative.
@pytest.mark.parametrize("lo,hi", [(-700.0, 0.0), (-1.7, 1.7), (-1e-3, 1e-3), (0.0, 700.0)])
def test_table_exp(lib, lo, hi):
    x = np.random.default_rng(1).uniform(lo, hi, size=4000)
    rel = max(abs(float((Decimal(float(g)) - w) / w)) for g, w in zip(run(lib.run_table, x), exact(x)))
    assert rel <= 2.5e-16, rel


def test_table_exp_edges(lib):
    y = run(lib.run_table, [0.0, -0.0, -745.2, -800.0, -1e5, np.nan])
    assert y[0] == 1.0 and y[1] == 1.0 and np.all(y[2:5] == 0.0) and np.isnan(y[5])
    # The reduction's switch points between table cells.
    x = (np.arange(-2000, 2000) + 0.5) * np.log(2.0) / 64.0
    rel = max(abs(float((Decimal(float(g)) - w) / w)) for g, w in zip(run(lib.run_table, x), exact(x)))
    assert rel <= 2.5e-16, rel


def test_small_exp(lib):
    x = np.random.default_rng(2).uniform(-2e-3, 2e-3, size=4000)
    rel = max(abs(float((Decimal(float(g)) - w) / w)) for g, w in zip(run(lib.run_small, x), exact(x)))
    assert rel <= 1.2e-16 and np.isnan(run(lib.run_small, [np.nan])[0]), rel
