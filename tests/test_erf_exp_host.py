"""erf_exp.h on the CPU: the ends of the range.

The header is compiled for the host (its device keywords defined away, one
thread filling the table) and run over arguments that no table covers: exp of
anything below the range of doubles is 0, of anything above it infinity, erf is
+-1 from 6 on, infinities included, and a NaN stays one.
"""

import ctypes as C
import math
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

STUB = """
#pragma once
#include <cmath>
struct double2 { double x, y; };
inline double2 make_double2(double x, double y) { return {x, y}; }
struct Dim { unsigned x; };
static const Dim threadIdx = {0}, blockDim = {1};
inline void __syncthreads() {}
using std::fma;
"""
SHIM = """
#define __device__
#define __forceinline__ inline
#define __shared__ static
#define asm(...)
#include "%s/3d-mfcfd_amd/csrc/erf_exp.h"
extern "C" double series(double x) { return mfcfd::exp_series(x); }
extern "C" void erf_exp(double x, double* er, double* ex) {
    mfcfd::load_erf_nodes();
    mfcfd::erf_exp(x, *er, *ex);
}
""" % ROOT


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ is not available")
    d = tmp_path_factory.mktemp("erf_exp")
    os.makedirs(d / "hip")
    (d / "hip" / "hip_runtime.h").write_text(STUB)
    (d / "shim.cpp").write_text(SHIM)
    subprocess.run(["g++", "-O1", "-fPIC", "-std=gnu++17", "-ffp-contract=off", "-shared", "-I", str(d),
                    "-o", str(d / "liberfexp.so"), str(d / "shim.cpp")], check=True)
    L = C.CDLL(str(d / "liberfexp.so"))
    L.series.restype = C.c_double
    L.series.argtypes = [C.c_double]
    L.erf_exp.argtypes = [C.c_double, C.POINTER(C.c_double), C.POINTER(C.c_double)]
    return L


def both(lib, x):
    er, ex = C.c_double(), C.c_double()
    lib.erf_exp(x, C.byref(er), C.byref(ex))
    return er.value, ex.value


@pytest.mark.parametrize("x", [-746.0, -1455.0, -1456.0, -1499.9, -1500.0, -1500.1, -1e4, -1e12, -2.9e24, -4e24, -1e30,
                               -1e200, -1.7e308, -math.inf])
def test_exp_below_the_range_is_zero(lib, x):
    v = lib.series(x)
    assert v == 0.0 and math.copysign(1.0, v) == 1.0


@pytest.mark.parametrize("x", [710.0, 1455.0, 1456.0, 1e4, 1e25, 1e200, math.inf])
def test_exp_above_the_range_is_infinite(lib, x):
    assert lib.series(x) == math.inf


@pytest.mark.parametrize("s", [28.0, 30.0, 1e6, 1.6e12, 2e12, 1e13, 1.4e154, 1e200, math.inf])
def test_erf_and_exp_beyond_the_table(lib, s):
    assert both(lib, s) == (1.0, 0.0)
    assert both(lib, -s) == (-1.0, 0.0)


def test_nan_stays(lib):
    assert math.isnan(lib.series(math.nan))
    assert all(math.isnan(v) for v in both(lib, math.nan))
