// boys.h -- Boys function F_m(T) = int_0^1 t^(2m) exp(-T t^2) dt on the GPU.
//
// T < BOYS_TMAX: Taylor expansion of the highest order around the nearest
//   grid point, F_M(T) = sum_k F_{M+k}(T0) (T0 - T)^k / k!
//   (dF_m/dT = -F_{m+1}), then the stable downward recursion
//   F_m = (2T F_{m+1} + exp(-T)) / (2m + 1).
// T >= BOYS_TMAX: F_0 = sqrt(pi/T)/2 (erfc(6) ~ 2e-17) and the upward
//   recursion F_m = ((2m - 1) F_{m-1} - exp(-T)) / (2T).
// The grid values are made on the host from the convergent series
//   F_m(T) = exp(-T) sum_k (2T)^k / ((2m+1)(2m+3)...(2m+2k+1))
// in long double (gtf_boys_table in basis.cpp).
#pragma once
#include "gtf_internal.h"

// F_0..F_M(T) for the ERI kernels from the compact Taylor table: slab holds,
// for grid points T0 = i * BOYS8_DELTA (i = 0 .. BOYS8_NGRID - 1), the
// BOYS8_NTERM = 8 coefficients c_k = F_{M+k}(T0) / k! of order M, one 64-byte
// row per point, so that
//   F_M(T) = sum_k c_k (T0 - T)^k,  |T0 - T| <= BOYS8_DELTA / 2
// (truncation below 1e-15 relative).  FP64 in every kernel, the FP32 tiles
// included.  A class touches one slab (23 KB), small enough to stay in the
// vector L1 cache or in LDS.  COLS: the slab is an LDS copy stored as four
// columns of BOYS8_NGRID double2 -- rows of 64 bytes would put the same part
// of every row on 4 of the 16 bank groups of a 16-byte read.
//
// The recursions' exp(-T): exp(-T0), tabulated after the slabs, times the
// exponential series of T0 - T (8 terms beyond 1: the next is below 1e-17).  The
// library's exp costs 30 instructions and a dozen constants in registers, a
// third of a low-L primitive quartet.
// Beyond BOYS_TMAX it corrects F_m by exp(-T) / ((2m - 1) F_(m-1)) of itself:
// 2e-15, 3e-13, 6e-12 and 8e-9 at most for m = 1, 3, 4 and 8.
//   M <= BOYS_FAST_M: 2^n times the hardware's 2^f in FP32, good to 1e-7, which
//     is 1e-18 of F_m, a hundredth of its last bit (largest error over 36..45
//     the same as with libm's exp).
//   above: 2^n times the series of exp(r), |r| <= ln 2 / 2, to r^9 in FP64, good
//     to 1e-11.  (FP32: 3.0e-15 of F_8, FP64 2.8e-15.)  The table for T -
//     BOYS_TMAX instead cost (dd|dd) 11 %: its one wavefront per SIMD waits for
//     the load.
#define BOYS_FAST_M 4
template <int M, bool COLS = false>
__device__ __forceinline__ void boys_eval8(double T, double* F, const double* __restrict__ slab)
{
    if (T < BOYS_TMAX) {
        const int i = (int)(T * BOYS8_INV_DELTA + 0.5);
        const double dt = fma((double)i, BOYS8_DELTA, -T);
        const double2* r = reinterpret_cast<const double2*>(slab) + i * (COLS ? 1 : BOYS8_NTERM / 2);
        constexpr int S = COLS ? BOYS8_NGRID : 1;
        const double2 c01 = r[0], c23 = r[S], c45 = r[2 * S], c67 = r[3 * S];
        double f = fma(c67.y, dt, c67.x);
        f = fma(f, dt, c45.y);
        f = fma(f, dt, c45.x);
        f = fma(f, dt, c23.y);
        f = fma(f, dt, c23.x);
        f = fma(f, dt, c01.y);
        f = fma(f, dt, c01.x);
        F[M] = f;
        if constexpr (M > 0) {
            const double e0 = slab[(COLS ? 1 : BOYS8_NM - M) * BOYS8_SLAB + i];
            double x = fma(dt, 1.0 / 40320.0, 1.0 / 5040.0);
            x = fma(x, dt, 1.0 / 720.0);
            x = fma(x, dt, 1.0 / 120.0);
            x = fma(x, dt, 1.0 / 24.0);
            x = fma(x, dt, 1.0 / 6.0);
            x = fma(x, dt, 0.5);
            x = fma(x, dt, 1.0);
            const double e = fma(e0 * x, dt, e0);
            const double t2 = T + T;
            static_for<0, M>([&](auto k) {
                constexpr int m = M - 1 - decltype(k)::value;
                F[m] = (t2 * F[m + 1] + e) * (1.0 / (2 * m + 1));
            });
        }
    } else {
        const double rt = rsqrt_nr(T);
        F[0] = 0.88622692545275801365 * rt;  // sqrt(pi)/2
        if constexpr (M > 0) {
            const double y = T * -1.4426950408889634074;  // -log2(e)
            const double n = rint(y);
            double x;
            if constexpr (M <= BOYS_FAST_M) {
                x = (double)__builtin_amdgcn_exp2f((float)(y - n));
            } else {
                const double r = fma(n, -0.69314718055994530942, -T);  // -ln(2)
                x = fma(r, 1.0 / 362880.0, 1.0 / 40320.0);
                x = fma(x, r, 1.0 / 5040.0);
                x = fma(x, r, 1.0 / 720.0);
                x = fma(x, r, 1.0 / 120.0);
                x = fma(x, r, 1.0 / 24.0);
                x = fma(x, r, 1.0 / 6.0);
                x = fma(x, r, 0.5);
                x = fma(x, r, 1.0);
                x = fma(x, r, 1.0);
            }
            const double e = ldexp(x, (int)n);
            const double h = 0.5 * rt * rt;
            static_for<1, M + 1>([&](auto k) {
                constexpr int m = decltype(k)::value;
                F[m] = ((2 * m - 1) * F[m - 1] - e) * h;
            });
        }
    }
}

// F_0..F_M(T) for the one-electron kernels (M <= 8) from the full table
template <int M>
__device__ __forceinline__ void boys_eval(double T, double* F, const double* __restrict__ tab)
{
    const double e = M > 0 ? exp(-T) : 0.0;
    if (T < BOYS_TMAX) {
        const int i = (int)(T * BOYS_INV_DELTA + 0.5);
        const double dt = i * BOYS_DELTA - T;
        const double* row = tab + i * BOYS_NCOL + M;
        double f = row[6];
        f = row[5] + dt * (1.0 / 6.0) * f;
        f = row[4] + dt * (1.0 / 5.0) * f;
        f = row[3] + dt * (1.0 / 4.0) * f;
        f = row[2] + dt * (1.0 / 3.0) * f;
        f = row[1] + dt * (1.0 / 2.0) * f;
        f = row[0] + dt * f;
        F[M] = f;
        static_for<0, M>([&](auto k) {
            constexpr int m = M - 1 - decltype(k)::value;
            F[m] = (2.0 * T * F[m + 1] + e) / (2 * m + 1);
        });
    } else {
        F[0] = 0.88622692545275801365 / sqrt(T);
        static_for<1, M + 1>([&](auto k) {
            constexpr int m = decltype(k)::value;
            F[m] = ((2 * m - 1) * F[m - 1] - e) / (2.0 * T);
        });
    }
}
