// oneel.hip -- overlap, kinetic and nuclear-attraction matrices by the
// McMurchie-Davidson scheme (setup work, replaces
// pfock/one_electron.c:28-119 and the closed OED library):
//   S_ab = s^x_ab s^y_ab s^z_ab, s the one-dimensional overlaps
//   T_ab = sum over directions of  -2b^2 s_{i,j+2} + b(2j+1) s_{ij} - j(j-1)/2 s_{i,j-2}
//   V_ab = -sum_C Z_C (2 pi / p) sum_tuv E^{ab}_{tuv} R_{tuv}(p, P - C)
//
// One wavefront per unordered shell pair, in code compiled for its two angular
// momenta.  Its lanes are PP primitive pairs x 64 / PP shares of the nuclei
// (PP the power of two that holds the pair's primitive pairs, at most 64); a
// lane sums R over its nuclei, contracts once, and the 64 partial blocks are
// added with lane shuffles.  Bound by latency: few wavefronts live (the d
// blocks take most of the registers) and little work in each.  One thread per
// ordered pair with sizes known at run time had its tables in scratch memory,
// and a wavefront waited for the pair with the most primitives: 13.3 ms of the
// 35.2 ms set-up of C24H12 (180 shells, 36 nuclei); now 0.14 ms of 21.1 ms.
#include "boys.h"
#include "eri_md.h"
#include "gtf_internal.h"
#include "oneel.h"

namespace {

// cartesian exponents of component c of order l
__host__ __device__ constexpr int cart_x(int l, int c) { return herm_t((l == 0 ? 0 : nherm(l - 1)) + c); }
__host__ __device__ constexpr int cart_y(int l, int c) { return herm_u((l == 0 ? 0 : nherm(l - 1)) + c); }
__host__ __device__ constexpr int cart_z(int l, int c) { return herm_v((l == 0 ? 0 : nherm(l - 1)) + c); }

// a primitive pair of the two shells
struct PrimPair {
    double a, b, p, cc;
    double P[3], PA[3], PB[3], K[3];  // K: exp(-mu AB_d^2)
};

__device__ __forceinline__ PrimPair prim_pair(const BasisView& b, int A, int B, int k)
{
    const int nb = b.nprim[B], i = k / nb, j = k - i * nb;
    PrimPair q;
    q.a = b.alpha[b.poff[A] + i];
    q.b = b.alpha[b.poff[B] + j];
    q.p = q.a + q.b;
    q.cc = b.coef[b.poff[A] + i] * b.coef[b.poff[B] + j];
    const double mu = q.a * q.b / q.p;
    for (int d = 0; d < 3; d++) {
        const double ca = b.center[3 * A + d], cb = b.center[3 * B + d];
        q.P[d] = (q.a * ca + q.b * cb) / q.p;
        q.PA[d] = q.P[d] - ca;
        q.PB[d] = q.P[d] - cb;
        q.K[d] = exp(-mu * (ca - cb) * (ca - cb));
    }
    return q;
}

// cartesian block -> spherical, summed over the wavefront; lane e of the
// first ones returns element e
template <int LA, int LB>
__device__ __forceinline__ double sph_sum(const double (&cart)[ncart(LA) * ncart(LB)], int lane)
{
    double mine = 0.0;
    static_for<0, nsph(LA)>([&](auto as_) {
        static_for<0, nsph(LB)>([&](auto bs_) {
            constexpr int as = decltype(as_)::value, bs = decltype(bs_)::value;
            double v = 0.0;
            static_for<0, ncart(LA)>([&](auto ia_) {
                static_for<0, ncart(LB)>([&](auto ib_) {
                    constexpr int ia = decltype(ia_)::value, ib = decltype(ib_)::value;
                    constexpr double w = sph_coef(LA, as, ia) * sph_coef(LB, bs, ib);
                    if constexpr (w != 0.0) v += w * cart[ia * ncart(LB) + ib];
                });
            });
            for (int m = 32; m; m >>= 1) v += __shfl_xor(v, m);
            if (lane == as * nsph(LB) + bs) mine = v;
        });
    });
    return mine;
}

// S, T, V of shells A, B (LA >= LB), both triangles
template <int LA, int LB>
__device__ __forceinline__ void oneel_block(const BasisView& b, const double* __restrict__ boys, int ld,
                                            double* __restrict__ S, double* __restrict__ Tk, double* __restrict__ V,
                                            int A, int B)
{
    constexpr int NCA = ncart(LA), NCB = ncart(LB), L = LA + LB, HL = nherm(L);
    const int lane = threadIdx.x & 63;
    const int np = b.nprim[A] * b.nprim[B];
    int lp = 0;
    while (lp < 6 && (1 << lp) < np) lp++;
    const int pp = 1 << lp, share = lane >> lp, nshare = 64 >> lp;
    const bool writes = lane < nsph(LA) * nsph(LB);
    const int as = lane / nsph(LB), bs = lane - as * nsph(LB);
    const long k1 = (long)(b.fstart[A] + as) * ld + b.fstart[B] + bs;
    const long k2 = (long)(b.fstart[B] + bs) * ld + b.fstart[A] + as;
    {
        double vc[NCA * NCB];
        static_for<0, NCA * NCB>([&](auto e_) { vc[decltype(e_)::value] = 0.0; });
        for (int k = lane & (pp - 1); k < np; k += pp) {
            const PrimPair q = prim_pair(b, A, B, k);
            // Hermite Coulomb R_{tuv}(p, P - C), summed with -Z_C
            double Rs[HL];
            static_for<0, HL>([&](auto h_) { Rs[decltype(h_)::value] = 0.0; });
            for (int c = share; c < b.natoms; c += nshare) {
                const double X = q.P[0] - b.atom_xyz[3 * c], Y = q.P[1] - b.atom_xyz[3 * c + 1],
                             Z = q.P[2] - b.atom_xyz[3 * c + 2], z = b.atom_Z[c];
                double F[L + 1], R[HL];
                boys_eval<L>(q.p * (X * X + Y * Y + Z * Z), F, boys);
                hermite_R<L, double>(R, F, 1.0, -2.0 * q.p, X, Y, Z);
                static_for<0, HL>([&](auto h_) { Rs[decltype(h_)::value] -= z * R[decltype(h_)::value]; });
            }
            // E[d][x][y][t], x <= LA, y <= LB
            double E[3][LA + 1][LB + 1][L + 1];
            const double h = 0.5 / q.p;
            static_for<0, 3>([&](auto d_) {
                constexpr int d = decltype(d_)::value;
                E[d][0][0][0] = q.K[d];
                static_for<0, LA>([&](auto x_) {
                    constexpr int x = decltype(x_)::value;
                    static_for<0, x + 2>([&](auto t_) {
                        constexpr int t = decltype(t_)::value;
                        double v = 0.0;
                        if constexpr (t <= x) v += q.PA[d] * E[d][x][0][t];
                        if constexpr (t + 1 <= x) v += (t + 1) * E[d][x][0][t + 1];
                        if constexpr (t > 0) v += h * E[d][x][0][t - 1];
                        E[d][x + 1][0][t] = v;
                    });
                });
                static_for<0, LB>([&](auto y_) {
                    constexpr int y = decltype(y_)::value;
                    static_for<0, LA + 1>([&](auto x_) {
                        constexpr int x = decltype(x_)::value;
                        static_for<0, x + y + 2>([&](auto t_) {
                            constexpr int t = decltype(t_)::value;
                            double v = 0.0;
                            if constexpr (t <= x + y) v += q.PB[d] * E[d][x][y][t];
                            if constexpr (t + 1 <= x + y) v += (t + 1) * E[d][x][y][t + 1];
                            if constexpr (t > 0) v += h * E[d][x][y][t - 1];
                            E[d][x][y + 1][t] = v;
                        });
                    });
                });
            });
            const double w = q.cc * 2.0 * M_PI / q.p;
            static_for<0, NCA>([&](auto ia_) {
                static_for<0, NCB>([&](auto ib_) {
                    constexpr int ia = decltype(ia_)::value, ib = decltype(ib_)::value;
                    constexpr int ax = cart_x(LA, ia), ay = cart_y(LA, ia), az = cart_z(LA, ia);
                    constexpr int bx = cart_x(LB, ib), by = cart_y(LB, ib), bz = cart_z(LB, ib);
                    double v = 0.0;
                    static_for<0, ax + bx + 1>([&](auto t_) {
                        static_for<0, ay + by + 1>([&](auto u_) {
                            constexpr int t = decltype(t_)::value, u = decltype(u_)::value;
                            double r = 0.0;
                            static_for<0, az + bz + 1>([&](auto z_) {
                                constexpr int zz = decltype(z_)::value;
                                r += E[2][az][bz][zz] * Rs[hidx(t, u, zz)];
                            });
                            v += E[0][ax][bx][t] * E[1][ay][by][u] * r;
                        });
                    });
                    vc[ia * NCB + ib] += w * v;
                });
            });
        }
        const double v = sph_sum<LA, LB>(vc, lane);
        if (writes) {
            V[k1] = v;
            if (A != B) V[k2] = v;
        }
    }
    double sc[NCA * NCB], tc[NCA * NCB];
    static_for<0, NCA * NCB>([&](auto e_) { sc[decltype(e_)::value] = tc[decltype(e_)::value] = 0.0; });
    // no nuclei here: the primitive pairs are over all 64 lanes
    for (int k = lane; k < np; k += 64) {
        const PrimPair q = prim_pair(b, A, B, k);
        const double sq = sqrt(M_PI / q.p), h = 0.5 / q.p;
        // one-dimensional overlaps s[d][x][y], x <= LA, y <= LB + 2, and
        // kinetic factors t[d][x][y], y <= LB
        double s[3][LA + 1][LB + 3], t[3][LA + 1][LB + 1];
        static_for<0, 3>([&](auto d_) {
            constexpr int d = decltype(d_)::value;
            s[d][0][0] = q.K[d] * sq;
            static_for<0, LA>([&](auto x_) {
                constexpr int x = decltype(x_)::value;
                double v = q.PA[d] * s[d][x][0];
                if constexpr (x > 0) v += x * h * s[d][x - 1][0];
                s[d][x + 1][0] = v;
            });
            static_for<0, LB + 2>([&](auto y_) {
                constexpr int y = decltype(y_)::value;
                static_for<0, LA + 1>([&](auto x_) {
                    constexpr int x = decltype(x_)::value;
                    double v = q.PB[d] * s[d][x][y];
                    if constexpr (x > 0) v += x * h * s[d][x - 1][y];
                    if constexpr (y > 0) v += y * h * s[d][x][y - 1];
                    s[d][x][y + 1] = v;
                });
            });
            static_for<0, LA + 1>([&](auto x_) {
                static_for<0, LB + 1>([&](auto y_) {
                    constexpr int x = decltype(x_)::value, y = decltype(y_)::value;
                    double v = -2.0 * q.b * q.b * s[d][x][y + 2] + q.b * (2 * y + 1) * s[d][x][y];
                    if constexpr (y >= 2) v -= 0.5 * y * (y - 1) * s[d][x][y - 2];
                    t[d][x][y] = v;
                });
            });
        });
        static_for<0, NCA>([&](auto ia_) {
            static_for<0, NCB>([&](auto ib_) {
                constexpr int ia = decltype(ia_)::value, ib = decltype(ib_)::value;
                constexpr int ax = cart_x(LA, ia), ay = cart_y(LA, ia), az = cart_z(LA, ia);
                constexpr int bx = cart_x(LB, ib), by = cart_y(LB, ib), bz = cart_z(LB, ib);
                const double sx = s[0][ax][bx], sy = s[1][ay][by], sz = s[2][az][bz];
                sc[ia * NCB + ib] += q.cc * sx * sy * sz;
                tc[ia * NCB + ib] += q.cc * (t[0][ax][bx] * sy * sz + sx * t[1][ay][by] * sz + sx * sy * t[2][az][bz]);
            });
        });
    }
    const double s = sph_sum<LA, LB>(sc, lane), t = sph_sum<LA, LB>(tc, lane);
    if (writes) {
        S[k1] = s;
        Tk[k1] = t;
        if (A != B) {
            S[k2] = s;
            Tk[k2] = t;
        }
    }
}

// the pairs blk, blk + nblk, ... of one molecule
__device__ __forceinline__ void oneel_pairs(const BasisView& b, const double* __restrict__ boys, int ld,
                                            double* __restrict__ S, double* __restrict__ Tk, double* __restrict__ V,
                                            int blk, int nblk)
{
    const long npair = (long)b.nshells * (b.nshells + 1) / 2;
    for (long k = blk; k < npair; k += nblk) {
        long i = (long)((sqrt(8.0 * (double)k + 1.0) - 1.0) * 0.5);
        while (i * (i + 1) / 2 > k) i--;
        while ((i + 1) * (i + 2) / 2 <= k) i++;
        int A = (int)i, B = (int)(k - i * (i + 1) / 2);
        if (b.L[A] < b.L[B]) {
            const int t = A;
            A = B;
            B = t;
        }
        switch (b.L[A] * (b.L[A] + 1) / 2 + b.L[B]) {
        case 0: oneel_block<0, 0>(b, boys, ld, S, Tk, V, A, B); break;
        case 1: oneel_block<1, 0>(b, boys, ld, S, Tk, V, A, B); break;
        case 2: oneel_block<1, 1>(b, boys, ld, S, Tk, V, A, B); break;
        case 3: oneel_block<2, 0>(b, boys, ld, S, Tk, V, A, B); break;
        case 4: oneel_block<2, 1>(b, boys, ld, S, Tk, V, A, B); break;
        default: oneel_block<2, 2>(b, boys, ld, S, Tk, V, A, B); break;
        }
    }
}
static_assert(GTF_LMAX == 2, "oneel_pairs lists the pairs of l = 0..2");

}  // namespace

__global__ __launch_bounds__(64) void oneel_kernel(BasisView b, const double* __restrict__ boys, int ld,
                                                   double* __restrict__ S, double* __restrict__ Tk,
                                                   double* __restrict__ V)
{
    oneel_pairs(b, boys, ld, S, Tk, V, blockIdx.x, gridDim.x);
}

// Many molecules in one launch: molecule k owns the workgroups
// [mol[k].blk0, mol[k + 1].blk0) (mol[nmol].blk0 = the grid) and views the
// shared basis arrays from its own shell and atom offsets.  A pair's sums do
// not depend on the grid: each molecule's matrices are those of oneel_kernel.
__global__ __launch_bounds__(64) void oneel_batch_kernel(BasisView b, const double* __restrict__ boys,
                                                         const OneelMol* __restrict__ mol, int nmol,
                                                         double* __restrict__ S, double* __restrict__ Tk,
                                                         double* __restrict__ V)
{
    const int blk = blockIdx.x;
    int lo = 0, hi = nmol - 1;  // last k with mol[k].blk0 <= blk
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (mol[mid].blk0 <= blk) lo = mid;
        else hi = mid - 1;
    }
    const OneelMol m = mol[lo];
    const BasisView v{m.nshells,           b.nbf,          m.natoms,
                      b.L + m.shell_off,   b.nprim + m.shell_off, b.poff + m.shell_off,
                      b.fstart + m.shell_off, b.atom + m.shell_off, b.alpha,
                      b.coef,              b.center + 3 * m.shell_off, b.atom_xyz + 3 * m.atom_off,
                      b.atom_Z + m.atom_off};
    oneel_pairs(v, boys, m.ld, S + m.moff, Tk + m.moff, V + m.moff, blk - m.blk0, mol[lo + 1].blk0 - m.blk0);
}

// a workgroup per pair; where the launch would hold more than a million of
// them, fewer that each take several
int gtf_oneel_blocks(int nshells, int nmol)
{
    const long pairs = (long)nshells * (nshells + 1) / 2, cap = (1L << 20) / (nmol > 0 ? nmol : 1);
    return (int)(pairs < cap ? pairs : cap < 64 ? (pairs < 64 ? pairs : 64) : cap);
}

int gtf_oneel_batch(hipStream_t st, const BasisView& b, const double* boys, const OneelMol* d_mol, int nmol,
                    int nblocks, double* S, double* T, double* V)
{
    if (nmol <= 0 || nblocks <= 0) return 0;
    oneel_batch_kernel<<<nblocks, 64, 0, st>>>(b, boys, d_mol, nmol, S, T, V);
    GTF_CHECK(hipGetLastError());
    return 0;
}

int gtf_oneel(hipStream_t st, const BasisView& b, const double* boys, int ld, double* S, double* T, double* V)
{
    oneel_kernel<<<gtf_oneel_blocks(b.nshells, 1), 64, 0, st>>>(b, boys, ld, S, T, V);
    GTF_CHECK(hipGetLastError());
    return 0;
}
