"""The ERI kernels' Boys function (gtfock_amd/csrc/boys.h) built for the host:
its exp(-T) on both sides of the asymptotic limit T = 36, where the orders are
joined by recursions that add or subtract it."""
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gtfock_amd", "csrc")

# what boys.h and gtf_internal.h take from the HIP headers
HIP = """
#pragma once
#include <cmath>
#define __host__
#define __device__
#define __global__
#define __forceinline__ inline
struct double2 { double x, y; };
struct double4 { double x, y, z, w; };
struct int2 { int x, y; };
struct int4 { int x, y, z, w; };
inline double __builtin_amdgcn_rsq(double x) { return 1.0 / std::sqrt(x); }
inline float __builtin_amdgcn_rsqf(float x) { return 1.0f / std::sqrt(x); }
inline float __builtin_amdgcn_exp2f(float x) { return std::exp2(x); }
using std::fma;
"""

# the table slabs of one order as the kernels hold them (rows), and as the
# columns of an LDS copy; F_0..F_M of n arguments
SRC = """
#include "boys.h"
#include "basis_internal.h"
#include <vector>
template <int M>
static void eval(int cols, const std::vector<double>& t8, long n, const double* T, double* F)
{
    std::vector<double> lds(BOYS8_SLAB + BOYS8_EXP);
    const double2* src = (const double2*)(t8.data() + (size_t)M * BOYS8_SLAB);
    for (int k = 0; k < BOYS8_SLAB / 2; k++)
        ((double2*)lds.data())[(k % (BOYS8_NTERM / 2)) * BOYS8_NGRID + k / (BOYS8_NTERM / 2)] = src[k];
    for (int k = 0; k < BOYS8_EXP; k++) lds[BOYS8_SLAB + k] = t8[(size_t)BOYS8_NM * BOYS8_SLAB + k];
    for (long k = 0; k < n; k++)
        if (cols) boys_eval8<M, true>(T[k], F + 9 * k, lds.data());
        else boys_eval8<M, false>(T[k], F + 9 * k, (const double*)src);
}
// the upward recursion of T >= BOYS_TMAX with libm's exp
extern "C" void boys_upward(int M, long n, const double* T, double* F)
{
    for (long k = 0; k < n; k++, F += 9) {
        const double rt = rsqrt_nr(T[k]), h = 0.5 * rt * rt, e = std::exp(-T[k]);
        F[0] = 0.88622692545275801365 * rt;
        for (int m = 1; m <= M; m++) F[m] = ((2 * m - 1) * F[m - 1] - e) * h;
    }
}
extern "C" void boys(int M, int cols, long n, const double* T, double* F)
{
    std::vector<double> t8((size_t)BOYS8_TOTAL);
    gtf_boys_taylor_tables(t8.data());
    switch (M) {
    case 0: eval<0>(cols, t8, n, T, F); break;
    case 1: eval<1>(cols, t8, n, T, F); break;
    case 4: eval<4>(cols, t8, n, T, F); break;
    case 5: eval<5>(cols, t8, n, T, F); break;
    default: eval<8>(cols, t8, n, T, F); break;
    }
}
"""


@pytest.fixture(scope="module")
def boys(tmp_path_factory):
    import ctypes
    d = tmp_path_factory.mktemp("boys")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text(HIP)
    (d / "boys_host.cpp").write_text(SRC)
    out = str(d / "libboys.so")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-I", str(d), "-I", CSRC, "-o", out,
                           str(d / "boys_host.cpp"), os.path.join(CSRC, "basis.cpp")])
    L = ctypes.CDLL(out)
    dp = ctypes.POINTER(ctypes.c_double)

    def f(M, cols, T):
        T = np.ascontiguousarray(T)
        F = np.zeros((len(T), 9))
        a = ctypes.c_long(len(T)), T.ctypes.data_as(dp), F.ctypes.data_as(dp)
        if cols is None:
            L.boys_upward(M, *a)
        else:
            L.boys(M, cols, *a)
        return F[:, :M + 1]
    return f


@pytest.mark.parametrize("cols", [0, 1])
@pytest.mark.parametrize("M", [1, 4, 5, 8])
def test_boys_exponential_is_fp64(boys, M, cols):
    rng = np.random.default_rng(M)
    eps = np.finfo(float).eps
    # beyond the limit: the upward recursion with libm's exp.  exp(-T) is at
    # most 1e-8 of (2m - 1) F_(m-1), so an exponential good to 1e-14 leaves the
    # same numbers but for a rounding that falls on a tie.
    T = np.concatenate([[36.0, 40.0, 71.99, 72.0, 100.0, 700.0, 1e4, 1e7], rng.uniform(36.0, 38.0, 4000),
                        rng.uniform(36.0, 90.0, 4000)])
    err = np.abs(boys(M, cols, T) / boys(M, None, T) - 1.0).max()
    print("M = %d: %.2g eps above the limit" % (M, err / eps))
    assert err <= eps
    # below: F_(m-1) = (2T F_m + exp(-T)) / (2m - 1) from the kernel's own F_m
    T = np.concatenate([[0.0, 1e-8, 0.05, 35.95, np.nextafter(36.0, 0.0)], rng.uniform(0.0, 36.0, 8000)])
    F = boys(M, cols, T)
    for m in range(1, M + 1):
        r = (2.0 * T * F[:, m] + np.exp(-T)) / (2 * m - 1)
        assert np.abs(F[:, m - 1] / r - 1.0).max() <= 8 * eps


def test_boys_order_zero(boys):
    T = np.concatenate([[0.0, 35.99, 36.0, 50.0, 80.0, 1e6], np.random.default_rng(0).uniform(0.0, 80.0, 4000)])
    import math
    ref = np.array([1.0 if t == 0.0 else 0.5 * math.sqrt(math.pi / t) * math.erf(math.sqrt(t)) for t in T])
    for cols in (0, 1):
        assert np.abs(boys(0, cols, T)[:, 0] / ref - 1.0).max() < 1e-14
