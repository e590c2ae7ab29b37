// eri_md.h -- McMurchie-Davidson electron-repulsion integrals for one shell
// quartet class, fully unrolled at compile time.
//
//   (ab|cd) = 2 pi^(5/2) / (p q sqrt(p+q))
//             sum_{tuv} E^{ab}_{tuv} sum_{t'u'v'} (-1)^{t'+u'+v'} E^{cd}_{t'u'v'}
//             R_{t+t',u+u',v+v'}(alpha, P - Q),   alpha = p q / (p + q)
//
// (McMurchie and Davidson, J. Comput. Phys. 26, 218 (1978)).  The Hermite
// coefficients E are stored per primitive pair already contracted with the
// spherical transform, the contraction coefficients, exp(-mu |AB|^2) and 1/p,
// so a primitive quartet costs the Boys function, the R recursion and two
// small matrix products.  A thread owns NC consecutive bra components of one
// contracted quartet and all ket components.
#pragma once
#include "boys.h"
#include "gtf_internal.h"

#define GTF_TWO_PI_2_5 34.986836655249725693  // 2 pi^(5/2)

// R^{0}_{tuv} for t+u+v <= L, in place (stage n = L .. 0):
//   R^n_{000} = pref (-2 alpha)^n F_n(T)
//   R^n_{t+1,u,v} = t R^{n+1}_{t-1,u,v} + X R^{n+1}_{t,u,v}   (same for u/Y, v/Z)
template <int L, typename Real>
__device__ __forceinline__ void hermite_R(Real* R, const Real* F, Real pref, Real m2a, Real X, Real Y,
                                          Real Z)
{
    Real pw[L + 1];
    pw[0] = pref;
    static_for<1, L + 1>([&](auto n_) {
        constexpr int n = decltype(n_)::value;
        pw[n] = pw[n - 1] * m2a;
    });
    R[0] = pw[L] * F[L];
    static_for<0, L>([&](auto s_) {
        constexpr int n = L - 1 - decltype(s_)::value;
        constexpr int top = nherm(L - n);
        static_for<0, top - 1>([&](auto i_) {
            constexpr int h = top - 1 - decltype(i_)::value;
            constexpr int t = herm_t(h), u = herm_u(h), v = herm_v(h);
            if constexpr (t > 0) {
                Real r = X * R[hidx(t - 1, u, v)];
                if constexpr (t > 1) r += Real(t - 1) * R[hidx(t - 2, u, v)];
                R[h] = r;
            } else if constexpr (u > 0) {
                Real r = Y * R[hidx(t, u - 1, v)];
                if constexpr (u > 1) r += Real(u - 1) * R[hidx(t, u - 2, v)];
                R[h] = r;
            } else {
                Real r = Z * R[hidx(t, u, v - 1)];
                if constexpr (v > 1) r += Real(v - 1) * R[hidx(t, u, v - 2)];
                R[h] = r;
            }
        });
        R[0] = pw[n] * F[n];
    });
}

template <int h1, int h2>
__host__ __device__ constexpr int hsum()
{
    return hidx(herm_t(h1) + herm_t(h2), herm_u(h1) + herm_u(h2), herm_v(h1) + herm_v(h2));
}

template <int LA, int LB, int LC, int LD>
struct EriShape {
    static constexpr int LAB = LA + LB, LCD = LC + LD, L = LAB + LCD;
    static constexpr int HAB = nherm(LAB), HCD = nherm(LCD), HL = nherm(L);
    static constexpr int NA = nsph(LA), NB = nsph(LB), NCc = nsph(LC), ND = nsph(LD);
    static constexpr int NAB = NA * NB, NCD = NCc * ND;
    static constexpr int ESZ_AB = NAB * HAB, ESZ_CD = NCD * HCD;
};

// Register budget heuristic: the largest divisor NC of NAB whose live set
// R + NC*(Ebra + V + acc) stays within ~128 doubles.
template <int LA, int LB, int LC, int LD>
__host__ __device__ constexpr int default_nc()
{
    using S = EriShape<LA, LB, LC, LD>;
    int best = 1;
    for (int nc = 1; nc <= S::NAB; ++nc) {
        if (S::NAB % nc) continue;
        int reg = S::HL + nc * (S::HAB + S::HCD + S::NCD) + S::L + 8;
        if (reg <= 128) best = nc;
    }
    return best;
}

// Components per thread of the tile kernels (eri_kernels.h), as the fewest
// near-equal chunks of the split side whose live doubles (R, the partial
// contraction and the integrals of a chunk) stay within TILE_REGS: with about
// 40 registers of addresses and temporaries that is 256 VGPRs, two waves per
// SIMD.  A class that needs one component per thread may exceed it.
#define TILE_REGS 104
#define TILE_STATIC_SPLITS 3
__host__ __device__ constexpr int tile_chunk(int total, int per, int fixed)
{
    int nc = (TILE_REGS - fixed) / per;
    if (nc < 1) nc = 1;
    if (nc > total) nc = total;
    const int ns = (total + nc - 1) / nc;
    // each compile-time chunk is its own code; beyond a few, one component per
    // thread with the chunk known at run time
    return ns <= TILE_STATIC_SPLITS ? (total + ns - 1) / ns : 1;
}
// bra components per thread, the ket side whole
template <int LA, int LB, int LC, int LD>
__host__ __device__ constexpr int tile_nc()
{
    using S = EriShape<LA, LB, LC, LD>;
    return tile_chunk(S::NAB, S::HCD + S::NCD, S::HL);
}
// ket components per thread, the bra side whole (exchanged contraction)
template <int LA, int LB, int LC, int LD>
__host__ __device__ constexpr int tile_nct()
{
    using S = EriShape<LA, LB, LC, LD>;
    return tile_chunk(S::NCD, S::NAB + (NzTab<LC, LD>::data.nnz + S::NCD - 1) / S::NCD, S::HL);
}
// a chunk known at compile time (see tile_chunk)
__host__ __device__ constexpr bool tile_static(int total, int nc) { return (total + nc - 1) / nc <= TILE_STATIC_SPLITS; }

// log2 of the lanes of a wavefront that hold one ket, each with another bra
// component, in the standard tile kernels of run-time components.  (dd|dd) is
// bound by the ket coefficients, 200 KB from L2 for every component of 64 kets;
// with four components of 16 kets a load serves four lanes.  The bra's
// coefficients are then the lane's own, vector loads of four lines, and the
// seventh group of 25 components has three lanes without one.  C54H18's class
// 4.1 -> 3.2 ms, 60 d shells 2.8 -> 2.35 ms; C96H24's, which has no J_PQ buffers,
// 13.7 -> 14.4 ms.
template <int LA, int LB, int LC, int LD>
__host__ __device__ constexpr int comp_lanes()
{
    return LA + LB + LC + LD >= 8 ? 2 : 0;
}

// classes whose kernels apply the primitive screening of eri_block (by
// total angular momentum L)
__host__ __device__ constexpr bool prim_screened_l(int L) { return L <= 3; }
template <int LA, int LB, int LC, int LD>
__host__ __device__ constexpr bool prim_screened()
{
    return prim_screened_l(LA + LB + LC + LD);
}

// Contracted integrals (bra components c0..c0+NC-1, all ket components) of
// the quartet (bra pair | ket pair), summed over the bra primitive pairs
// i0, i0 + istep, ... and, in the classes of prim_screened, the
// primitive quartets whose Schwarz bound q_bra q_ket is at least pv.peps.  acc[c][cd], cd = c_sph * nsph(LD) + d_sph.
// The ket coefficients are read in the compact nonzero-only layout and the
// structurally zero terms are skipped at compile time; when a thread owns the
// whole bra pair (NC == NAB, c0 == 0) the bra side is treated the same way.
template <int LA, int LB, int LC, int LD, int NC, typename Real>
__device__ __forceinline__ void eri_block(const PairView& pv, int bra, int ket, int c0,
                                          const double* __restrict__ boys_slab,
                                          Real (&acc)[NC][EriShape<LA, LB, LC, LD>::NCD], int i0, int istep)
{
    using S = EriShape<LA, LB, LC, LD>;
    constexpr int L = S::L, HAB = S::HAB, HCD = S::HCD, HL = S::HL, NCD = S::NCD;
    constexpr bool BRA_FULL = (NC == S::NAB);
    using TA = NzTab<LA, LB>;
    using TC = NzTab<LC, LD>;
    constexpr int NZAB = TA::data.nnz, NZCD = TC::data.nnz;
    static_for<0, NC>([&](auto c_) {
        static_for<0, NCD>([&](auto d_) { acc[decltype(c_)::value][decltype(d_)::value] = Real(0); });
    });
    const int nb = pv.nprim[bra], nk = pv.nprim[ket];
    const double4* __restrict__ pb = pv.prim + pv.poff[bra];
    const double4* __restrict__ pk = pv.prim + pv.poff[ket];
    const double* __restrict__ Eb = BRA_FULL ? pv.Ez + pv.zoff[bra] : pv.E + pv.eoff[bra] + (long)c0 * HAB;
    const double* __restrict__ Ek0 = pv.Ez + pv.zoff[ket];
    // primitive screening (classes of total angular momentum <= 3, whose
    // s and p shells carry the long contractions; the higher classes would
    // pay for it in registers): a pair's primitives are stored by
    // descending Schwarz bound, so the kets of bra primitive i that pass
    // q_i q_j >= peps are a prefix, found by bisection once per i, and once
    // one bra primitive has none the later ones have none either
    constexpr bool PSCREEN = prim_screened<LA, LB, LC, LD>();
    for (int i = i0; i < nb; i += istep) {
        int nke = nk;
        if constexpr (PSCREEN) {
            if (pv.peps > 0.0) {
                const double qi = pv.q[pv.poff[bra] + i];
                const double* __restrict__ qk = pv.q + pv.poff[ket];
                int lo = 0, hi = nk;
                while (lo < hi) {
                    const int mid = (lo + hi) >> 1;
                    if (qi * qk[mid] >= pv.peps) lo = mid + 1;
                    else hi = mid;
                }
                nke = lo;
                if (nke == 0) break;
            }
        }
        const double4 B = pb[i];
        Real eb[NC][HAB];
        static_for<0, NC>([&](auto c_) {
            constexpr int c = decltype(c_)::value;
            static_for<0, HAB>([&](auto h_) {
                constexpr int h = decltype(h_)::value;
                if constexpr (BRA_FULL) {
                    if constexpr (TA::data.nz[c][h]) eb[c][h] = Real(Eb[(long)i * NZAB + TA::data.pos[c][h]]);
                } else {
                    eb[c][h] = Real(Eb[(long)i * S::ESZ_AB + c * HAB + h]);
                }
            });
        });
        for (int j = 0; j < nke; ++j) {
            const double4 K = pk[j];
            // T = alpha |PQ|^2 and F_0..F_L(T) in FP64 for both precisions;
            // an FP32 tile rounds them for the R recursion and contractions
            const double Xd = B.y - K.y, Yd = B.z - K.z, Zd = B.w - K.w;
            const double rd = rsqrt_nr(B.x + K.x);
            const double alphad = B.x * K.x * (rd * rd);
            const double Td = alphad * (Xd * Xd + Yd * Yd + Zd * Zd);
            double Fd[L + 1];
            boys_eval8<L>(Td, Fd, boys_slab);
            Real F[L + 1];
            static_for<0, L + 1>([&](auto m_) {
                constexpr int m = decltype(m_)::value;
                F[m] = Real(Fd[m]);
            });
            const Real pref = Real(GTF_TWO_PI_2_5 * rd);
            Real R[HL];
            hermite_R<L, Real>(R, F, pref, Real(-2.0 * alphad), Real(Xd), Real(Yd), Real(Zd));
            Real V[NC][HCD];
            static_for<0, HCD>([&](auto h2_) {
                constexpr int h2 = decltype(h2_)::value;
                constexpr bool neg = (horder(h2) & 1) != 0;
                static_for<0, NC>([&](auto c_) {
                    constexpr int c = decltype(c_)::value;
                    Real v = Real(0);
                    static_for<0, HAB>([&](auto h1_) {
                        constexpr int h1 = decltype(h1_)::value;
                        if constexpr (!BRA_FULL || TA::data.nz[c][h1])
                            v += eb[c][h1] * R[hsum<h1, h2>()];
                    });
                    V[c][h2] = neg ? -v : v;
                });
            });
            const double* __restrict__ ek = Ek0 + (long)j * NZCD;
            static_for<0, NCD>([&](auto cd_) {
                constexpr int cd = decltype(cd_)::value;
                static_for<0, HCD>([&](auto h2_) {
                    constexpr int h2 = decltype(h2_)::value;
                    if constexpr (TC::data.nz[cd][h2]) {
                        const Real e = Real(ek[TC::data.pos[cd][h2]]);
                        static_for<0, NC>([&](auto c_) {
                            constexpr int c = decltype(c_)::value;
                            acc[c][cd] += e * V[c][h2];
                        });
                    }
                });
            });
        }
    }
}

// ---- the tile kernels' evaluators -------------------------------------------
//
// A wavefront's lanes hold 64 kets and share one bra pair.  Everything of the
// bra (p, P, q, E) is the same for every lane and comes through the scalar
// cache into SGPRs; a ket's data come from KetView, whose 64-ket blocks are
// stored component by component, so a load instruction of the wavefront
// reads one or a few contiguous lines.  Loads of one pair's record per lane
// (64 lines per instruction) kept the L1 tag lookups busy for 65-80 % of the
// (ss|ss), (ps|ss) and (dp|ss) kernels' cycles and the VALU for 28-39 %.
// The ket primitive is the outer loop, so its data are loaded once and the
// inner loop over the bra primitives touches no vector memory but the Boys
// table.

// memory that no kernel writes while it is read: uniform loads become scalar
template <typename T>
using const_as = const T __attribute__((address_space(4)));
template <typename T>
__device__ __forceinline__ const_as<T>* as_const(const T* p)
{
    return (const_as<T>*)(uintptr_t)p;
}

// the bra pair of a tile (wave-uniform); Coef: the type its coefficients are
// read in (the FP32 form has a rounded copy of the compact ones; the full ones,
// which only a run-time component of a d-p or d-d bra reads, it rounds as it
// reads them)
template <typename Coef>
struct BraRef {
    const_as<double>* prim;  // (p, Px, Py, Pz) per primitive pair
    const_as<double>* q;
    const_as<Coef>* E;       // compact, or full from component c0 (the chunk's rows)
    int n;                   // primitive pairs
    double peps;
    const Coef* lane_E;      // full, from this lane's component (comp_lanes)
};

// the ket of a lane: its first record (see KetView), its primitive pairs
struct KetRef {
    const double2* d;
    const double* q;
    int n;
};

// p, P, alpha, F_0..F_L of one primitive quartet, then R (as eri_block: the
// FP32 form rounds after the Boys function); zero where on is false
template <int L, typename Real, bool BLDS>
__device__ __forceinline__ void prim_quartet_R(const_as<double>* B, const double2& k0, const double2& k1, bool on,
                                               const double* __restrict__ boys_slab, Real (&R)[nherm(L)])
{
    const double Xd = B[1] - k0.y, Yd = B[2] - k1.x, Zd = B[3] - k1.y;
    const double rd = rsqrt_nr(B[0] + k0.x);
    const double alphad = B[0] * k0.x * (rd * rd);
    const double Td = alphad * (Xd * Xd + Yd * Yd + Zd * Zd);
    double Fd[L + 1];
    boys_eval8<L, BLDS>(Td, Fd, boys_slab);
    Real F[L + 1];
    static_for<0, L + 1>([&](auto m_) GTF_INLINE {
        constexpr int m = decltype(m_)::value;
        F[m] = Real(Fd[m]);
    });
    hermite_R<L, Real>(R, F, Real(on ? GTF_TWO_PI_2_5 * rd : 0.0), Real(-2.0 * alphad), Real(Xd), Real(Yd), Real(Zd));
}

#define PAIR_MAX_L 1
// Runs body(i, R) over the bra primitives of one ket primitive.  With
// primitive screening the wavefront goes on while any lane's bound passes (the
// bounds fall with i) and a lane that has ended adds zeros.  The classes of L
// <= PAIR_MAX_L form R of two bra primitives at a time: a primitive quartet is
// a chain of about 70 dependent operations, and their 3-4 wavefronts per SIMD
// do not fill its gaps (with L = 2 too, (ps|ps) took 197 registers and gained
// nothing).
template <int L, bool PSCREEN, typename Real, bool BLDS, typename Coef, typename Body>
__device__ __forceinline__ void bra_loop(const BraRef<Coef>& b, const double2& k0, const double2& k1, double qj, bool on,
                                         const double* __restrict__ boys_slab, Body&& body)
{
    auto passes = [&](int i) GTF_INLINE { return on && (!PSCREEN || !(b.peps > 0.0) || b.q[i] * qj >= b.peps); };
    int i = 0;
    if constexpr (L <= PAIR_MAX_L) {
        for (; i + 1 < b.n; i += 2) {
            const bool p0 = passes(i), p1 = passes(i + 1);
            if (__ballot(p0) == 0) return;
            Real R0[nherm(L)], R1[nherm(L)];
            prim_quartet_R<L, Real, BLDS>(b.prim + 4 * i, k0, k1, p0, boys_slab, R0);
            prim_quartet_R<L, Real, BLDS>(b.prim + 4 * i + 4, k0, k1, p1, boys_slab, R1);
            body(i, R0);
            body(i + 1, R1);
        }
    }
    for (; i < b.n; i++) {
        const bool p = passes(i);
        if constexpr (PSCREEN)
            if (__ballot(p) == 0) return;
        Real R[nherm(L)];
        prim_quartet_R<L, Real, BLDS>(b.prim + 4 * i, k0, k1, p, boys_slab, R);
        body(i, R);
    }
}

// Runs body(record, k0, k1, q, lane takes part) over a lane's ket primitives
// j0, j0 + js, ...; the next primitive's (p, P) and bound are loaded before
// the body, which would otherwise wait for L2 every time.
template <int KREC, bool PSCREEN, typename Body>
__device__ __forceinline__ void ket_loop(const KetRef& k, int j0, int js, Body&& body)
{
    // the record of a lane that has ended: any that exists
    const double2* kr = k.d + (long)j0 * (KREC * 64);
    const double* kq = k.q + (long)j0 * 64;
    double2 n0 = make_double2(1.0, 0.0), n1 = make_double2(0.0, 0.0);
    double nq = 0.0;
    if (j0 < k.n) {
        n0 = kr[0];
        n1 = kr[64];
        if constexpr (PSCREEN) nq = kq[0];
    }
    for (int j = j0; __ballot(j < k.n) != 0; j += js) {
        const double2 k0 = n0, k1 = n1;
        const double qj = nq;
        const double2* rec = kr;
        kr += (long)js * (KREC * 64);
        kq += (long)js * 64;
        if (j + js < k.n) {
            n0 = kr[0];
            n1 = kr[64];
            if constexpr (PSCREEN) nq = kq[0];
        }
        body(rec, j, k0, k1, qj, j < k.n);
    }
}

// Integrals of bra components A0 .. A0 + NC - 1 (all ket components) of a
// lane's quartet, over the ket primitives j0, j0 + js, .. and every bra
// primitive.  A0 >= 0: the compact E of the whole pair, its structural zeros
// skipped at compile time; A0 < 0: one component (NC = 1) whose rows b.E
// points at in the full layout.  The bra contraction is summed over the bra
// primitives before the ket coefficients are applied: of (dd|dd) they are 200 KB
// a wavefront, from L2, and applied within the loop over the bra primitives they
// took C54H18's class 7.6 ms, now 4.1, and 24 d shells of four primitives 67 ms,
// now 14.  Not for (dd|ss), where one coefficient a component is applied and the
// sum only holds registers (2.9 ms instead of 2.2).
template <int LA, int LB, int LC, int LD, int A0, int NC, typename Real, bool BLDS, bool LANE_E = false, typename Coef>
__device__ __forceinline__ void eri_lane(const BraRef<Coef>& b, const KetRef& k, int j0, int js,
                                         const double* __restrict__ boys_slab,
                                         Real (&acc)[NC][EriShape<LA, LB, LC, LD>::NCD])
{
    using S = EriShape<LA, LB, LC, LD>;
    using TA = NzTab<LA, LB>;
    using TC = NzTab<LC, LD>;
    constexpr int L = S::L, HAB = S::HAB, HCD = S::HCD, NCD = S::NCD, NZC = TC::data.nnz;
    constexpr int ESTRIDE = A0 >= 0 ? TA::data.nnz : S::ESZ_AB;
    constexpr bool SUM_BRA = LA + LB < 4 || LC + LD > 0;
    constexpr bool PSCREEN = prim_screened<LA, LB, LC, LD>();
    // small ket blocks are loaded ahead of the bra loop
    constexpr bool EARLY = NZC <= 6;
    static_for<0, NC>([&](auto c_) GTF_INLINE {
        static_for<0, NCD>([&](auto d_) GTF_INLINE { acc[decltype(c_)::value][decltype(d_)::value] = Real(0); });
    });
    ket_loop<KetView::rec(NZC), PSCREEN>(k, j0, js, [&](const double2* rec, int, const double2& k0, const double2& k1,
                                                        double qj, bool on) GTF_INLINE {
        double2 e2[EARLY ? (NZC + 1) / 2 : 1];
        if constexpr (EARLY)
            if (on)
                static_for<0, (NZC + 1) / 2>([&](auto p_) GTF_INLINE { e2[decltype(p_)::value] = rec[(2 + decltype(p_)::value) * 64]; });
        Real W[NC][HCD];
        if constexpr (SUM_BRA)
            static_for<0, NC>([&](auto c_) GTF_INLINE {
                static_for<0, HCD>([&](auto h_) GTF_INLINE { W[decltype(c_)::value][decltype(h_)::value] = Real(0); });
            });
        // acc[c] += the ket coefficients of h2 times w
        auto apply_ket = [&](auto c_, auto h2_, Real w) GTF_INLINE {
            constexpr int c = decltype(c_)::value, h2 = decltype(h2_)::value;
            constexpr bool neg = (horder(h2) & 1) != 0;
            static_for<0, NCD>([&](auto cd_) GTF_INLINE {
                constexpr int cd = decltype(cd_)::value;
                if constexpr (TC::data.nz[cd][h2]) {
                    constexpr int pos = TC::data.pos[cd][h2];
                    const double2 v = EARLY ? e2[EARLY ? pos / 2 : 0] : rec[(2 + pos / 2) * 64];
                    const Real e = Real(pos % 2 ? v.y : v.x);
                    acc[c][cd] += neg ? -e * w : e * w;
                }
            });
        };
        bra_loop<L, PSCREEN, Real, BLDS>(b, k0, k1, qj, on, boys_slab, [&](int i, const Real (&R)[S::HL]) GTF_INLINE {
            if constexpr (LANE_E) {
                const Coef* E = b.lane_E + (long)i * ESTRIDE;
                static_for<0, HAB>([&](auto h1_) GTF_INLINE {
                    constexpr int h1 = decltype(h1_)::value;
                    const Real e = Real(E[h1]);
                    static_for<0, HCD>([&](auto h2_) GTF_INLINE {
                        constexpr int h2 = decltype(h2_)::value;
                        W[0][h2] += e * R[hsum<h1, h2>()];
                    });
                });
                return;
            }
            // component by component: a row of E is in SGPRs once and used for
            // every h2
            static_for<0, NC>([&](auto c_) GTF_INLINE {
                constexpr int c = decltype(c_)::value;
                const_as<Coef>* E = b.E + (long)i * ESTRIDE;
                static_for<0, HCD>([&](auto h2_) GTF_INLINE {
                    constexpr int h2 = decltype(h2_)::value;
                    Real v = SUM_BRA ? W[c][h2] : Real(0);
                    static_for<0, HAB>([&](auto h1_) GTF_INLINE {
                        constexpr int h1 = decltype(h1_)::value;
                        if constexpr (A0 < 0) v += Real(E[h1]) * R[hsum<h1, h2>()];
                        else if constexpr (TA::data.nz[A0 < 0 ? 0 : A0 + c][h1])
                            v += E[TA::data.pos[A0 < 0 ? 0 : A0 + c][h1]] * R[hsum<h1, h2>()];
                    });
                    if constexpr (SUM_BRA) W[c][h2] = v;
                    else if (on) apply_ket(c_, h2_, v);
                });
            });
        });
        if constexpr (SUM_BRA)
            if (on)
                static_for<0, HCD>([&](auto h2_) GTF_INLINE {
                    static_for<0, NC>([&](auto c_) GTF_INLINE { apply_ket(c_, h2_, W[decltype(c_)::value][decltype(h2_)::value]); });
                });
    });
}

// The same with the contractions exchanged: ket components C0 .. C0 + NCT - 1
// and every bra component, acc[d][ab].  The ket side of R is contracted first
// (its coefficients stay in registers over the bra loop), then the bra's
// coefficients are applied from SGPRs.  C0 < 0: one component (NCT = 1), kfull
// its rows in the full layout (KetView::f) from the first primitive pair on.
template <int LA, int LB, int LC, int LD, int C0, int NCT, typename Real, bool BLDS>
__device__ __forceinline__ void eri_lane_t(const BraRef<Real>& b, const KetRef& k, int j0, int js,
                                           const double* __restrict__ kfull, const double* __restrict__ boys_slab,
                                           Real (&acc)[NCT][EriShape<LA, LB, LC, LD>::NAB])
{
    using S = EriShape<LA, LB, LC, LD>;
    using TA = NzTab<LA, LB>;
    using TC = NzTab<LC, LD>;
    constexpr int L = S::L, HAB = S::HAB, HCD = S::HCD, NAB = S::NAB;
    constexpr bool PSCREEN = prim_screened<LA, LB, LC, LD>();
    static_for<0, NCT>([&](auto c_) GTF_INLINE {
        static_for<0, NAB>([&](auto d_) GTF_INLINE { acc[decltype(c_)::value][decltype(d_)::value] = Real(0); });
    });
    ket_loop<KetView::rec(TC::data.nnz), PSCREEN>(k, j0, js, [&](const double2* rec, int j, const double2& k0,
                                                                 const double2& k1, double qj, bool on) GTF_INLINE {
        Real ek[NCT][HCD];
        static_for<0, NCT>([&](auto d_) GTF_INLINE {
            constexpr int d = decltype(d_)::value;
            static_for<0, HCD>([&](auto h2_) GTF_INLINE {
                constexpr int h2 = decltype(h2_)::value;
                double v = 0.0;
                if constexpr (C0 < 0) {
                    if (on) v = kfull[((long)j * S::ESZ_CD + h2) * 64];
                    ek[d][h2] = Real((horder(h2) & 1) != 0 ? -v : v);
                } else if constexpr (TC::data.nz[C0 < 0 ? 0 : C0 + d][h2]) {
                    constexpr int pos = TC::data.pos[C0 < 0 ? 0 : C0 + d][h2];
                    if (on) {
                        const double2 e = rec[(2 + pos / 2) * 64];
                        v = pos % 2 ? e.y : e.x;
                    }
                    ek[d][h2] = Real((horder(h2) & 1) != 0 ? -v : v);
                }
            });
        });
        bra_loop<L, PSCREEN, Real, BLDS>(b, k0, k1, qj, on, boys_slab, [&](int i, const Real (&R)[S::HL]) GTF_INLINE {
            const_as<Real>* E = b.E + (long)i * TA::data.nnz;
            Real U[NCT][HAB];
            static_for<0, NCT>([&](auto d_) GTF_INLINE {
                constexpr int d = decltype(d_)::value;
                static_for<0, HAB>([&](auto h1_) GTF_INLINE {
                    constexpr int h1 = decltype(h1_)::value;
                    Real v = Real(0);
                    static_for<0, HCD>([&](auto h2_) GTF_INLINE {
                        constexpr int h2 = decltype(h2_)::value;
                        if constexpr (C0 < 0 || TC::data.nz[C0 < 0 ? 0 : C0 + d][h2]) v += ek[d][h2] * R[hsum<h1, h2>()];
                    });
                    U[d][h1] = v;
                });
            });
            // the bra's rows in their order in memory: a row is in SGPRs once
            static_for<0, NAB>([&](auto ab_) GTF_INLINE {
                constexpr int ab = decltype(ab_)::value;
                static_for<0, HAB>([&](auto h1_) GTF_INLINE {
                    constexpr int h1 = decltype(h1_)::value;
                    if constexpr (TA::data.nz[ab][h1]) {
                        const Real e = E[TA::data.pos[ab][h1]];
                        static_for<0, NCT>([&](auto d_) GTF_INLINE {
                            constexpr int d = decltype(d_)::value;
                            acc[d][ab] += e * U[d][h1];
                        });
                    }
                });
            });
        });
    });
}
