// eri_kernels.h -- per-class ERI kernels with their epilogues.
//
//  EPI_JK    fused J/K digestion of the screened unique quartets; the
//            multiplicities are those of update_F (pfock/fock_task.c:29-117),
//            the accumulators hold 2J and -K before symmetrisation.
//  EPI_DIAG  Schwarz values max |(mn|mn)| of a shell pair
//            (pfock/screening.c:63-89).
//  EPI_STORE write the contracted integrals in the caller's order (for CInt_computeShellQuartet).
//
// Work is handed out by a device-wide atomic task counter (the GPU form of
// taskq_next, pfock/taskq.c:55-62): each workgroup takes 256 consecutive work
// units (unit = quartet * NSPLIT + bra-component chunk) until none are left.
#pragma once
#include "eri_md.h"

#ifndef GTF_ATOMIC_ADD
#define GTF_ATOMIC_ADD(p, v) atomicAdd((p), (v))
#endif

enum { EPI_JK = 0, EPI_DIAG = 1, EPI_STORE = 2 };

// flags of a quartet of EPI_STORE: how the caller's order of its shells
// differs from the canonical one
enum { GTF_STORE_SWAPPED = 1, GTF_STORE_FLIP_BRA = 2, GTF_STORE_FLIP_KET = 4 };

struct EriArgs {
    // work decode: either bra rows (row_off over bra_list x ket_list) or qlist
    long nunits;
    const long* row_off;
    int nrows;
    const int* bra_list;
    const int* ket_list;
    const int2* qlist;
    int* counter;   // task counter (reset to 0 before the launch)
    int ntasks;
    PairView pv;
    const int* fstart;
    const double* boys8;  // compact Taylor tables, BOYS8_NM slabs of BOYS8_SLAB, exp(-T0)
    // EPI_JK: nd densities (and their J, K) dstride elements apart, all
    // digested from each integral (pfock/fock_task.c:46 loops num_dmat)
    const double* D;
    double* J;
    double* K;
    int nd;
    long dstride;
    // EPI_DIAG
    unsigned long long* vbits;
    // EPI_STORE: (bra, ket, first double, GTF_STORE_* flags) per quartet
    const int4* slist;
    double* out;
    // EPI_DIAG, EPI_STORE: 2^llane lanes share a quartet's bra primitive pairs
    int llane;
    // tiles of the LDS-strip J/K kernel and their runs of kets (gtf_internal.h)
    const TileHead* tiles;
    const int4* runs;
    // per density and ket component, by position in the ket list: the density
    // elements of the kets, and the accumulators of their J_PQ (JkList)
    const double* dk;
    double* jk;
    long nket;  // list length
    KetView kv;  // the ket list, for the tile kernels
    int ntiles;
    int nbf;  // LDS strip capacity (largest molecule)
    int jpq_lds;  // the wavefronts have J_PQ buffers in LDS (TileLaunch::buffered)
    // exact screening of the block-padded rows
    const double* vbra;
    const double* vket;
    const int* rank_bra;
    const int* rank_ket;
    double tol2;
    int same;
    // mixed precision: FP64 quartets have v_bra * v_ket >= tau2, FP32 the rest
    double tau2;
    // packed per-molecule matrices: block offset and leading dimension per shell
    const long* mbase;
    const int* mld;
    // global-atomic path: bra pair (index into bra_list) and absolute first
    // ket of each row
    const int* row_bra;
    const int* row_kstart;
    // batches: molecule of each shell and, per molecule, whether its J/K are
    // built (0: its quartets are skipped; a molecule whose SCF has ended)
    const int* shell_mol;
    const int* mol_active;
    // tile kernels (optional): per workgroup {clock at start, clock at exit,
    // tiles taken}, three entries at 3 * blockIdx.x -- the load balance of a
    // launch (pfock/pfock.c:1918-2010 reports it across processes)
    long long* wg_stat;
};

// one workgroup's record of its part in a tile launch
__device__ __forceinline__ void record_workgroup(const EriArgs& a, long long t_begin, int taken)
{
    if (a.wg_stat && threadIdx.x == 0) {
        long long* w = a.wg_stat + 3L * blockIdx.x;
        w[0] = t_begin;
        w[1] = (long long)wall_clock64();
        w[2] = taken;
    }
}

// the bra pair's molecule takes part in this build
__device__ __forceinline__ bool bra_active(const EriArgs& a, int bra)
{
    return !a.mol_active || a.mol_active[a.shell_mol[a.pv.s1[bra]]];
}

// the Schwarz test of pfock/fock_task.c:192 and, for a diagonal class, the
// one-orientation rule, for bra row r and ket slot j
__device__ __forceinline__ bool quartet_valid(const EriArgs& a, int r, int j)
{
    return a.vbra[r] * a.vket[j] >= a.tol2 && (!a.same || a.rank_ket[j] <= a.rank_bra[r]);
}

__device__ __forceinline__ int find_row(const long* __restrict__ off, int nrows, long q)
{
    int lo = 0, hi = nrows;  // off[lo] <= q < off[hi]
    while (hi - lo > 1) {
        int mid = (lo + hi) >> 1;
        if (off[mid] <= q) lo = mid;
        else hi = mid;
    }
    return lo;
}

template <int LA, int LB, int LC, int LD, int NC>
__device__ __forceinline__ void digest(const EriArgs& a, int bra, int ket, int c0,
                                       const double (&acc)[NC][EriShape<LA, LB, LC, LD>::NCD], long doff);

// One component chunk of one quartet.  EPI_DIAG and EPI_STORE, whose lists hold
// a pair's or a quartet's whole primitive work, deal the bra primitive pairs to
// 2^llane lanes that add their integrals with lane shuffles: in one thread, a
// pair of 8-primitive shells took 4096 primitive quartets one after another
// while the wavefronts were too few to fill the chip.  Schwarz values of
// C24H12's pairs 2.5 -> 0.5 ms, of water's 1.8 -> 0.3 ms.
template <int LA, int LB, int LC, int LD, int NC, int EPI>
__device__ __forceinline__ void eri_unit(const EriArgs& a, long u)
{
    using S = EriShape<LA, LB, LC, LD>;
    constexpr int NSPLIT = S::NAB / NC;
    constexpr int NCD = S::NCD, ND = S::ND, NB = S::NB;
    int li = 0, nl = 1;
    if constexpr (EPI != EPI_JK) {
        nl = 1 << a.llane;
        li = (int)u & (nl - 1);
        u >>= a.llane;
    }
    const long q = u / NSPLIT;
    const int c0 = (int)(u - q * NSPLIT) * NC;
    int bra, ket;
    int4 dst;
    if constexpr (EPI == EPI_STORE) {
        dst = a.slist[q];
        bra = dst.x;
        ket = dst.y;
    } else if (a.qlist) {
        const int2 bk = a.qlist[q];
        bra = bk.x;
        ket = bk.y;
    } else {
        const int row = find_row(a.row_off, a.nrows, q);
        const int r = a.row_bra[row];
        const int j = a.row_kstart[row] + (int)(q - a.row_off[row]);
        if (!quartet_valid(a, r, j)) return;
        bra = a.bra_list[r];
        ket = a.ket_list[j];
    }
    if constexpr (EPI == EPI_JK) {
        if (!bra_active(a, bra)) return;
    }
    double acc[NC][NCD];
    eri_block<LA, LB, LC, LD, NC, double>(a.pv, bra, ket, c0, a.boys8 + (LA + LB + LC + LD) * BOYS8_SLAB, acc, li, nl);
    if constexpr (EPI != EPI_JK) {
        for (int m = nl >> 1; m; m >>= 1)
            static_for<0, NC>([&](auto c_) {
                static_for<0, NCD>([&](auto d_) {
                    double& x = acc[decltype(c_)::value][decltype(d_)::value];
                    x += __shfl_xor(x, m);
                });
            });
    }

    if constexpr (EPI == EPI_STORE) {
        // strides of the components in the caller's order: a flipped pair has
        // its second shell first, a swapped quartet its ket pair first
        const int f = dst.w;
        const int sb = f & GTF_STORE_SWAPPED ? NCD : 1, sk = f & GTF_STORE_SWAPPED ? 1 : S::NAB;
        const int sa_ = f & GTF_STORE_FLIP_BRA ? sb * NB : sb, sb_ = f & GTF_STORE_FLIP_BRA ? sb : sb * (S::NAB / NB);
        const int sc_ = f & GTF_STORE_FLIP_KET ? sk * ND : sk, sd_ = f & GTF_STORE_FLIP_KET ? sk : sk * S::NCc;
        double* o = a.out + (unsigned)dst.z;
        static_for<0, NC>([&](auto c_) {
            constexpr int c = decltype(c_)::value;
            const int ia = (c0 + c) / NB, ib = (c0 + c) - ia * NB;
            const int ob = ia * sa_ + ib * sb_;
            static_for<0, NCD>([&](auto d_) {
                constexpr int cd = decltype(d_)::value;
                constexpr int e = c * NCD + cd;
                if ((e & (nl - 1)) == li) o[ob + (cd / ND) * sc_ + (cd % ND) * sd_] = acc[c][cd];
            });
        });
    } else if constexpr (EPI == EPI_DIAG) {
        double mx = 0.0;
        static_for<0, NC>([&](auto c_) {
            constexpr int c = decltype(c_)::value;
            static_for<0, NCD>([&](auto d_) {
                constexpr int cd = decltype(d_)::value;
                if (cd == c0 + c) mx = fmax(mx, fabs(acc[c][cd]));
            });
        });
        if (li == 0) atomicMax(a.vbits + bra, (unsigned long long)__double_as_longlong(mx));
    } else {
        for (int d = 0; d < a.nd; d++)
            digest<LA, LB, LC, LD, NC>(a, bra, ket, c0, acc, d * a.dstride);
    }
}

// update_F digestion of one thread's NC bra components of quartet (bra|ket)
// by FP64 atomics straight into J and K (the classes whose LDS strips do not
// fit).
template <int LA, int LB, int LC, int LD, int NC>
__device__ __forceinline__ void digest(const EriArgs& a, int bra, int ket, int c0,
                                       const double (&acc)[NC][EriShape<LA, LB, LC, LD>::NCD], long doff)
{
    using S = EriShape<LA, LB, LC, LD>;
    constexpr int NCD = S::NCD, ND = S::ND, NB = S::NB;
    const int M = a.pv.s1[bra], N = a.pv.s2[bra], P = a.pv.s1[ket], Q = a.pv.s2[ket];
    const int f1 = (M != N), f2 = (P != Q), f3 = (bra != ket);
    const double cJ1 = 2.0 * (1 + f1) * (1 + f2);
    const double cJ2 = 2.0 * f3 * (1 + f1) * (1 + f2);
    const double cMP = (1 + f3), cNP = f1 * (1 + f3), cMQ = f2 * (1 + f3), cNQ = f1 * f2 * (1 + f3);
    const int ld = a.mld[M];
    const long base = a.mbase[M];
    const int oM = a.fstart[M], oN = a.fstart[N], oP = a.fstart[P], oQ = a.fstart[Q];
    const double* __restrict__ D = a.D + doff + base;
    double* J = a.J + doff + base;
    double* K = a.K + doff + base;
    int mloc[NC], nloc[NC];
    double dmn[NC];
    static_for<0, NC>([&](auto c_) {
        constexpr int c = decltype(c_)::value;
        const int ab = c0 + c;
        mloc[c] = ab / NB;
        nloc[c] = ab % NB;
        dmn[c] = D[(long)(oM + mloc[c]) * ld + oN + nloc[c]];
    });
    // J_MN += cJ1 * sum_pq D_pq I   and   J_PQ += cJ2 * sum_mn D_mn I
    static_for<0, NC>([&](auto c_) {
        constexpr int c = decltype(c_)::value;
        double s = 0.0;
        static_for<0, NCD>([&](auto d_) {
            constexpr int cd = decltype(d_)::value;
            s += D[(long)(oP + cd / ND) * ld + oQ + cd % ND] * acc[c][cd];
        });
        GTF_ATOMIC_ADD(&J[(long)(oM + mloc[c]) * ld + oN + nloc[c]], cJ1 * s);
    });
    if (f3) {
        static_for<0, NCD>([&](auto d_) {
            constexpr int cd = decltype(d_)::value;
            double s = 0.0;
            static_for<0, NC>([&](auto c_) {
                constexpr int c = decltype(c_)::value;
                s += dmn[c] * acc[c][cd];
            });
            GTF_ATOMIC_ADD(&J[(long)(oP + cd / ND) * ld + oQ + cd % ND], cJ2 * s);
        });
    }
    // K_MP -= cMP sum_q D_nq I,  K_NP -= cNP sum_q D_mq I
    // K_MQ -= cMQ sum_p D_np I,  K_NQ -= cNQ sum_p D_mp I
    static_for<0, NC>([&](auto c_) {
        constexpr int c = decltype(c_)::value;
        const long rm = (long)(oM + mloc[c]) * ld, rn = (long)(oN + nloc[c]) * ld;
        static_for<0, S::NCc>([&](auto p_) {
            constexpr int p = decltype(p_)::value;
            double smp = 0.0, snp = 0.0;
            static_for<0, ND>([&](auto q_) {
                constexpr int qq = decltype(q_)::value;
                const double x = acc[c][p * ND + qq];
                smp += D[rn + oQ + qq] * x;
                snp += D[rm + oQ + qq] * x;
            });
            GTF_ATOMIC_ADD(&K[rm + oP + p], -cMP * smp);
            if (f1) GTF_ATOMIC_ADD(&K[rn + oP + p], -cNP * snp);
        });
        if (f2) {
            static_for<0, ND>([&](auto q_) {
                constexpr int qq = decltype(q_)::value;
                double smq = 0.0, snq = 0.0;
                static_for<0, S::NCc>([&](auto p_) {
                    constexpr int p = decltype(p_)::value;
                    const double x = acc[c][p * ND + qq];
                    smq += D[rn + oP + p] * x;
                    snq += D[rm + oP + p] * x;
                });
                GTF_ATOMIC_ADD(&K[rm + oQ + qq], -cMQ * smq);
                if (f1) GTF_ATOMIC_ADD(&K[rn + oQ + qq], -cNQ * snq);
            });
        }
    });
}

template <int LA, int LB, int LC, int LD, int NC, int EPI>
__global__ __launch_bounds__(256) void eri_kernel(EriArgs a)
{
    if (a.counter) {
        __shared__ int s_task;
        for (;;) {
            if (threadIdx.x == 0) s_task = atomicAdd(a.counter, 1);
            __syncthreads();
            const int task = s_task;
            __syncthreads();
            if (task >= a.ntasks) break;
            const long u = (long)task * 256 + threadIdx.x;
            if (u < a.nunits) eri_unit<LA, LB, LC, LD, NC, EPI>(a, u);
        }
    } else {
        const long u = (long)blockIdx.x * 256 + threadIdx.x;
        if (u < a.nunits) eri_unit<LA, LB, LC, LD, NC, EPI>(a, u);
    }
}

// Fused ERI + J/K digestion over bra-row tiles.  A workgroup takes a tile --
// one bra pair and runs of its kets -- and accumulates J_MN and the exchange
// blocks of the bra shells in LDS, flushed with one HBM atomic per touched
// element when the tile is done.  The flush was half of the (ps|ps) kernel on
// C54H18 when a tile held at most 320 kets (21.7 ms, 13.1 without digestion),
// so a tile takes as much of its bra's row as the balance allows.  Dynamic
// LDS: the Boys slab (BLDS only) + per density tile_work() doubles, and with
// BLDS the density rows, (NA + NB) * nbf.
//
// The tile's work is cut into wavefront units: 64 lanes over (ket, ket
// primitive class), one chunk of the ket primitives, one chunk of the split
// side's components.  The bra pair and the component chunk are the same for
// all lanes of a unit (but see comp_lanes); the kets are consecutive in their list.  2^lic chunks
// of the ket primitives (primitives ic, ic + 2^lic, ...: the primitives are
// ordered by their bound, so an interleaved chunk holds its share of the ones
// that screening drops) keep a unit near unit_pq primitive quartets per lane;
// chunks of the ket's rather than the bra's primitives, so that a ket record
// is read by one unit only.  Where a run has few kets, 2^ljc lanes share a ket
// and take every 2^ljc-th of the chunk; they add their integrals with lane
// shuffles and the first one digests.  Digestion is linear in the integrals,
// so every unit digests its partial sum on its own.
//
// A wavefront takes all units of a run's 64 kets one after another, from a
// counter in LDS (their costs differ; dealt in turn, the wavefronts waited
// for the slowest at the tile's end).  It sums J_PQ of those kets in a buffer
// of its own and adds it to the list's accumulators with one coalesced atomic
// per component: scattered into the matrix it was 64 cache lines each.
#define GTF_TILE_UNITS 1024
#define GTF_UNIT_PQ 64
#define GTF_TILE_PQ 1048576
// J_MN is the same few addresses for every lane of a unit: 16 copies, picked
// by lane, leave 4 lanes to an address (64 lanes adding to one are served
// one after another)
#define GTF_JMN_COPIES 16

// The Boys Taylor slab of order L copied from HBM into the first
// GTF_BOYS_LDS doubles of dynamic LDS, as columns (boys_eval8).  A persistent
// workgroup copies it once; every primitive quartet of every tile it takes
// then reads its Taylor row from LDS instead of from up to 64 lines per load.
// The barrier before the first tile orders the copy before the first
// read.  It costs 26 KB of LDS per workgroup, which
// lowers the occupancy of classes whose strips are already large, so it is a
// per-class choice (the tile shape's boys_lds).  FP32 tiles use the same FP64
// slab: the Boys function is FP64 in both precisions.
#define GTF_BOYS_LDS (BOYS8_SLAB + BOYS8_EXP)
template <int L>
__device__ __forceinline__ const double* boys_to_lds(const EriArgs& a, double* smem)
{
    const double2* src = reinterpret_cast<const double2*>(a.boys8 + L * BOYS8_SLAB);
    double2* dst = reinterpret_cast<double2*>(smem);
    constexpr int C = BOYS8_NTERM / 2;
    for (int k = threadIdx.x; k < BOYS8_SLAB / 2; k += blockDim.x) dst[(k % C) * BOYS8_NGRID + k / C] = src[k];
    const double2* ex = reinterpret_cast<const double2*>(a.boys8 + BOYS8_NM * BOYS8_SLAB);
    for (int k = threadIdx.x; k < BOYS8_EXP / 2; k += blockDim.x) dst[BOYS8_SLAB / 2 + k] = ex[k];
    return smem;
}

// Boys slab of a tile kernel: in LDS (BLDS; the work area then starts after
// it) or read in place from HBM through the caches (the work area starts at
// the LDS base)
template <int L, bool BLDS>
__device__ __forceinline__ const double* tile_boys(const EriArgs& a, double* smem, double*& work)
{
    if constexpr (BLDS) {
        work = smem + GTF_BOYS_LDS;
        return boys_to_lds<L>(a, smem);
    } else {
        work = smem;
        return a.boys8 + L * BOYS8_SLAB;
    }
}

// f(std::integral_constant<int, s>) for the run-time s in [0, N)
template <int N, int S = 0, typename F>
__device__ __forceinline__ void split_switch(int s, F&& f)
{
    if constexpr (S + 1 == N) {
        f(std::integral_constant<int, S>{});
    } else {
        if (s == S) f(std::integral_constant<int, S>{});
        else split_switch<N, S + 1>(s, f);
    }
}

// what a unit's digestion reads and writes
struct DigestCtx {
    const_as<double>* Dm;  // rows of shell M, uniform reads (D_mn)
    const double *rm, *rn;  // D rows of shells M and N
    int ld, oN, oP, oQ;
    int f1, f2, f3;
    double* strip;          // LDS: row r < NA is function M + r, row NA + r is N + r
    int nbf;
    double* jmn;            // LDS: this lane's copy of J_MN
    const double* dk;       // the ket's density elements, a component every nk
    long nk;
    double* jpq;            // LDS: the ket's J_PQ, a component every 64; null: in jk
    double* jk;             // the list's J_PQ, a component every nk
    int clane;              // comp_lanes: distance of a ket's lanes
    bool lead;              // and the first of them
};

// update_F digestion (pfock/fock_task.c:29-117) of bra components A0 .. A0 +
// NAr - 1 and ket components C0 .. C0 + NCr - 1 of a lane's quartet; get(ab,
// cd) reads an integral.  With jreg (the thread owns every bra component of
// its quartets) J_MN is summed there over the tile.  Contributions to the
// same element of the strip are summed over the thread's components first.
// crt: the run-time component of a kernel that has one bra component (A0 < 0)
// or one ket component (C0 < 0) per thread.
template <int LA, int LB, int LC, int LD, int A0, int NAr, int C0, int NCr, bool JREG, int CL, typename Get>
__device__ __forceinline__ void digest_unit(const DigestCtx& x, int crt, Get&& get, double* jreg)
{
    using S = EriShape<LA, LB, LC, LD>;
    constexpr int NA = S::NA, NB = S::NB, ND = S::ND;
    constexpr bool RT = A0 < 0, KRT = C0 < 0;
    constexpr int AB0 = RT ? 0 : A0, CD0 = KRT ? 0 : C0;
    constexpr int M0 = AB0 / NB, M1 = (AB0 + NAr - 1) / NB + 1;
    constexpr int P0 = KRT ? 0 : CD0 / ND, P1 = KRT ? 1 : (CD0 + NCr - 1) / ND + 1, QN = KRT ? 1 : ND;
    const int mrt = RT ? crt / NB : 0, nrt = RT ? crt - mrt * NB : 0;
    const int prt = KRT ? crt / ND : 0, qrt = KRT ? crt - prt * ND : 0;
    const int oP = x.oP + prt, oQ = x.oQ + qrt;  // of the run-time ket component, else of the shells
    const double cJ1 = 2.0 * (1 + x.f1) * (1 + x.f2);
    const double cJ2 = 2.0 * x.f3 * (1 + x.f1) * (1 + x.f2);
    // J_MN += cJ1 sum_pq D_pq I,  J_PQ += cJ2 sum_mn D_mn I
    {
        double dpq[NCr];
        static_for<0, NCr>([&](auto d_) GTF_INLINE {
            constexpr int cd = CD0 + decltype(d_)::value;
            dpq[decltype(d_)::value] = x.dk[((KRT ? crt : 0) + cd) * x.nk];
        });
        static_for<0, NAr>([&](auto c_) GTF_INLINE {
            constexpr int c = decltype(c_)::value;
            double s = 0.0;
            static_for<0, NCr>([&](auto d_) GTF_INLINE { s += dpq[decltype(d_)::value] * get(c_, d_); });
            if constexpr (JREG) jreg[c] += cJ1 * s;
            else atomicAdd(&x.jmn[RT ? crt : AB0 + c], cJ1 * s);
        });
    }
    if (x.f3) {
        double dmn[NAr];
        static_for<0, NAr>([&](auto c_) GTF_INLINE {
            constexpr int c = decltype(c_)::value;
            const int m = RT ? mrt : (AB0 + c) / NB, n = RT ? nrt : (AB0 + c) % NB;
            dmn[c] = x.Dm[(long)m * x.ld + x.oN + n];
        });
        static_for<0, NCr>([&](auto d_) GTF_INLINE {
            double s = 0.0;
            static_for<0, NAr>([&](auto c_) GTF_INLINE { s += dmn[decltype(c_)::value] * get(c_, d_); });
            const int cd = (KRT ? crt : CD0) + decltype(d_)::value;
            if (x.jpq) {
                x.jpq[cd * 64] += cJ2 * s;
                return;
            }
            // the lanes of a ket are all here (those without a component with zeros)
            for (int m = 0; m < CL; m++) s += __shfl_xor(s, x.clane << m, 64);
            if (CL > 0 && !x.lead) return;
            GTF_ATOMIC_ADD(&x.jk[cd * x.nk], cJ2 * s);
        });
    }
    // K_MP -= cMP sum_nq D_nq I,  K_MQ -= cMQ sum_np D_np I  for each m, and
    // K_NP -= cNP sum_mq D_mq I,  K_NQ -= cNQ sum_mp D_mp I  for each n
    const double c3 = -(double)(1 + x.f3);
    auto bra_side = [&](auto side_) GTF_INLINE {
        constexpr bool ROWM = decltype(side_)::value == 0;  // rows of M, sums over n
        constexpr int R0 = RT ? 0 : ROWM ? M0 : 0, R1 = RT ? 1 : ROWM ? M1 : NB;
        static_for<R0, R1>([&](auto r_) GTF_INLINE {
            constexpr int r = decltype(r_)::value;
            constexpr int O0 = RT ? 0 : ROWM ? 0 : M0, O1 = RT ? 1 : ROWM ? NB : M1;
            auto in_chunk = [](int o) {
                const int ab = ROWM ? r * NB + o : o * NB + r;
                return RT || (ab >= AB0 && ab < AB0 + NAr);
            };
            constexpr bool any = [&]() GTF_INLINE {
                for (int o = O0; o < O1; o++)
                    if (in_chunk(o)) return true;
                return false;
            }();
            if constexpr (any) {
                const int row = RT ? (ROWM ? mrt : NA + nrt) : (ROWM ? r : NA + r);
                double* out = x.strip + row * x.nbf;
                double sp[P1 - P0], sq[QN];
                static_for<0, P1 - P0>([&](auto p_) GTF_INLINE { sp[decltype(p_)::value] = 0.0; });
                static_for<0, QN>([&](auto q_) GTF_INLINE { sq[decltype(q_)::value] = 0.0; });
                static_for<O0, O1>([&](auto o_) GTF_INLINE {
                    constexpr int o = decltype(o_)::value;
                    constexpr int ab = ROWM ? r * NB + o : o * NB + r;
                    if constexpr (RT || (ab >= AB0 && ab < AB0 + NAr)) {
                        const double* dr = ROWM ? x.rn + (long)(RT ? nrt : o) * x.ld : x.rm + (long)(RT ? mrt : o) * x.ld;
                        using C = std::integral_constant<int, RT ? 0 : ab - AB0>;
                        static_for<P0, P1>([&](auto p_) GTF_INLINE {
                            constexpr int p = decltype(p_)::value;
                            const double dp = dr[oP + p];
                            static_for<0, QN>([&](auto q_) GTF_INLINE {
                                constexpr int q = decltype(q_)::value;
                                constexpr int cd = p * ND + q;
                                if constexpr (cd >= CD0 && cd < CD0 + NCr) {
                                    const double v = get(C{}, std::integral_constant<int, cd - CD0>{});
                                    sp[p - P0] += dr[oQ + q] * v;
                                    sq[q] += dp * v;
                                }
                            });
                        });
                    }
                });
                static_for<P0, P1>([&](auto p_) GTF_INLINE {
                    constexpr int p = decltype(p_)::value;
                    atomicAdd(&out[oP + p], c3 * sp[p - P0]);
                });
                if (x.f2)
                    static_for<0, QN>([&](auto q_) GTF_INLINE {
                        constexpr int q = decltype(q_)::value;
                        constexpr bool has = [&]() GTF_INLINE {
                            for (int p = P0; p < P1; p++)
                                if (p * ND + q >= CD0 && p * ND + q < CD0 + NCr) return true;
                            return false;
                        }();
                        if constexpr (has) atomicAdd(&out[oQ + q], c3 * sq[q]);
                    });
            }
        });
    };
    bra_side(std::integral_constant<int, 0>{});
    if (x.f1) bra_side(std::integral_constant<int, 1>{});
}

// Largest workgroup of a class's tile kernel (the host takes it or 256, see
// GtfSystem::tile_launch).  A kernel compiled for 512 threads has at most 256
// VGPRs; the classes of L >= 5 need more, run one wavefront per SIMD and take
// 256 threads.
template <int LA, int LB, int LC, int LD>
__host__ __device__ constexpr int tile_threads()
{
    return LA + LB + LC + LD <= 4 ? 512 : 256;
}

// Wavefronts per SIMD asked of the compiler.  Left alone it keeps addresses of
// the digestion in registers across the primitive loops.
template <int LA, int LB, int LC, int LD>
__host__ __device__ constexpr int tile_min_waves()
{
    constexpr int L = LA + LB + LC + LD;
    return L <= 1 ? 4 : L == 2 ? 3 : L <= 4 ? 2 : 1;
}

// LDS doubles of one density's work area: the strips, the J_MN copies and the
// J_PQ buffers of `bufs` wavefronts.  Without buffers (0) the wavefronts add
// J_PQ straight to the accumulators: for several densities, where the buffers
// would not fit for the d classes, and for one density of a molecule whose
// strips leave no room for them -- (dd|dd) from 1368 functions on.
__host__ __device__ constexpr int tile_work(int rows, int nbf, int nab, int ncd, int bufs)
{
    return rows * nbf + GTF_JMN_COPIES * nab + bufs * ncd * 64;
}

// One class's tile kernel.  EX = false: a thread owns NC bra components and
// every ket component of its quartet; EX = true: NC ket components and every
// bra component, the ket contracted first.
template <int LA, int LB, int LC, int LD, int NC, typename Real, bool BLDS, bool EX>
__device__ __forceinline__ void tile_kernel_body(const EriArgs& a)
{
    using S = EriShape<LA, LB, LC, LD>;
    constexpr int NA = S::NA, NB = S::NB, NCD = S::NCD, NAB = S::NAB, ND = S::ND;
    constexpr int SIDE = EX ? NCD : NAB;
    constexpr int NSPLIT = (SIDE + NC - 1) / NC;
    constexpr bool LOW = std::is_same<Real, float>::value;
    constexpr int L = S::L;
    constexpr int KREC = KetView::rec(NzTab<LC, LD>::data.nnz);
    // compile-time component chunks, or (one component of very many) run-time
    constexpr bool STATIC = tile_static(SIDE, NC);
    constexpr bool JREG_ABLE = NSPLIT == 1 && NAB <= 3;
    constexpr int CL = !STATIC && !EX ? comp_lanes<LA, LB, LC, LD>() : 0;
    extern __shared__ __attribute__((aligned(16))) double smem[];
    __shared__ int s_task, s_unit;
    const int NT = blockDim.x;
    double* work;
    const double* boys = tile_boys<L, BLDS>(a, smem, work);
    // the bra shells' density rows beside the work areas (BLDS): the digestion
    // gathers from them at the kets' columns
    const bool buffered = a.jpq_lds;
    const int wsz = tile_work(NA + NB, a.nbf, NAB, NCD, buffered ? NT / 64 : 0);
    double* drow = work + (long)a.nd * wsz;
    const long long t_begin = (long long)wall_clock64();
    const int lane = threadIdx.x & 63;
    int taken = 0;
    // the current tile, wave-uniform
    int run0, nrun, bra, oM, oN, f1, nbf, rb;
    long mat;
    double vb;
    // the full coefficients are in FP64 only
    using Coef = std::conditional_t<LOW && (STATIC || EX), float, double>;
    BraRef<Coef> br;
    br.peps = a.pv.peps;
    const Coef* lane_E = nullptr;
    // reads tile `task` (and its density rows); false when there is none
    auto open_tile = [&](int task) GTF_INLINE {
        if (task >= a.ntiles) return false;
        const_as<TileHead>& h = *as_const(a.tiles + task);
        run0 = h.run0;
        // a molecule that takes no part in this build (mol_active is written
        // between builds only)
        nrun = !a.mol_active || as_const(a.mol_active)[h.mol] ? h.nrun : 0;
        bra = h.bra;
        // strip rows are as wide as the bra's molecule (at most a.nbf)
        nbf = h.nbf;
        mat = h.mat;
        oM = h.oM;
        oN = h.oN;
        f1 = h.two;
        rb = h.rank;
        vb = as_const(a.vbra)[h.row];
        br.n = h.nprim;
        br.prim = as_const((const double*)(a.pv.prim + h.prim));
        br.q = as_const(a.pv.q + h.prim);
        if constexpr (std::is_same_v<Coef, float>) br.E = as_const(a.pv.Ezf) + h.E;
        else br.E = as_const(STATIC || EX ? a.pv.Ez : a.pv.E) + h.E;
        if constexpr (CL > 0) lane_E = a.pv.E + h.E;
        if constexpr (BLDS)
            for (int d = 0; d < a.nd; d++) {
                const double* D = a.D + d * a.dstride + mat;
                for (int r = 0; r < NA + NB; r++) {
                    const double* Dr = D + (long)(r < NA ? oM + r : oN + (r - NA)) * nbf;
                    for (int k = threadIdx.x; k < nbf; k += NT) drow[(d * (NA + NB) + r) * nbf + k] = Dr[k];
                }
            }
        return true;
    };
    if (threadIdx.x == 0) {
        s_task = atomicAdd(a.counter, 1);
        s_unit = 0;
    }
    // the work areas are zero whenever a tile starts: here, and the flush
    // clears what it read
    for (int k = threadIdx.x; k < a.nd * wsz; k += NT) work[k] = 0.0;
    __syncthreads();
    bool open = open_tile(__builtin_amdgcn_readfirstlane(s_task));
    __syncthreads();
    while (open) {
        int next = 0;  // taken now, needed at the end
        if (threadIdx.x == 0) next = atomicAdd(a.counter, 1);
        taken++;
        const int nstrip = (NA + NB) * nbf;
        double* strip = work;
        double* jmn = work + nstrip;
        double* jpq = jmn + GTF_JMN_COPIES * NAB + (threadIdx.x >> 6) * (NCD * 64);
        const bool jreg_on = JREG_ABLE && a.nd == 1;
        double jreg[JREG_ABLE ? NAB : 1];
        if constexpr (JREG_ABLE) static_for<0, NAB>([&](auto c_) { jreg[decltype(c_)::value] = 0.0; });
        // cursor: block `at` of the tile is block `blk` of run `r`
        int r = -1, left = 0, kbeg = 0, nkt = 0, lic = 0, ljc = 0, sp0 = 0, spn = 1, ic0 = 0, icn = 1;
        int blk = 0, at = -1;
        auto take = [&]() GTF_INLINE {
            int u = 0;
            if (lane == 0) u = atomicAdd(&s_unit, 1);
            return __builtin_amdgcn_readfirstlane(u);
        };
        auto seek = [&](int unit) GTF_INLINE {
            int d = unit - at;  // >= 1
            at = unit;
            while (d > left) {  // into the next run (left: blocks after the current one)
                d -= left + 1;
                if (++r >= nrun) return false;
                const_as<int>* rp = as_const((const int*)(a.runs + run0 + r));
                kbeg = rp[0];
                const int span = rp[1], chunks = rp[2];
                nkt = GTF_RUN_KETS(span), sp0 = GTF_RUN_SP0(span), spn = GTF_RUN_SPN(span);
                lic = GTF_RUN_LIC(chunks), ljc = GTF_RUN_LJC(chunks);
                ic0 = GTF_RUN_IC0(chunks), icn = GTF_RUN_ICN(chunks);
                left = (((nkt << (ljc + CL)) + 63) >> 6) - 1;
                blk = 0;
            }
            left -= d;
            blk += d;
            return true;
        };
        for (int unit = take(); seek(unit);) {
            unit = take();
            const int u = blk * 64 + lane;
            const int q = u >> (ljc + CL), cl = (u >> ljc) & ((1 << CL) - 1), jc = u & ((1 << ljc) - 1);
            const int j = kbeg + q;
            bool on = q < nkt;
            if (on) {
                const double vk = a.vket[j];
                // the Schwarz test of pfock/fock_task.c:192, the one-orientation
                // rule of a diagonal class, and the precision split on the
                // bound sqrt(v_bra v_ket) against tau
                on = vb * vk >= a.tol2 && (!a.same || a.rank_ket[j] <= rb) && (vb * vk >= a.tau2) != LOW;
            }
            if (__ballot(on) == 0) continue;
            KetRef kr{a.kv.d, a.kv.q, 0};
            int4 ki = make_int4(0, 0, 0, -1);
            int kb = 0;
            if (on) {
                kb = a.kv.base[j];
                ki = a.kv.info[j];
                kr.d = a.kv.d + (long)(kb >> 6) * (KREC * 64) + (kb & 63);
                kr.q = a.kv.q + kb;
                kr.n = a.kv.nprim[j];
            }
            const int js = 1 << (lic + ljc);
            auto finish = [&](auto a0_, auto nar_, auto c0_, auto ncr_, auto& acc, int crt) GTF_INLINE {
                constexpr int A0 = decltype(a0_)::value, NAr = decltype(nar_)::value;
                constexpr int C0 = decltype(c0_)::value, NCr = decltype(ncr_)::value;
                // acc is [NAr][NCr], or [NCr][NAr] in the exchanged form
                auto cell = [&](auto c_, auto d_) GTF_INLINE -> Real& {
                    constexpr int c = decltype(c_)::value, d = decltype(d_)::value;
                    if constexpr (EX) return acc[d][c];
                    else return acc[c][d];
                };
                for (int s = 1; s < (1 << ljc); s <<= 1)
                    static_for<0, NAr>([&](auto c_) GTF_INLINE {
                        static_for<0, NCr>([&](auto d_) GTF_INLINE { cell(c_, d_) += __shfl_xor(cell(c_, d_), s, 64); });
                    });
                if (!on || jc != 0) return;
                // (opaque, or the digestion's addresses would be formed ahead of
                // the primitive loops and held across them)
                int ox = ki.x, oy = ki.y, oj = j, onbf = nbf, orow = oM, ocol = oN;
                asm volatile("" : "+v"(ox), "+v"(oy), "+v"(oj), "+s"(onbf), "+s"(orow), "+s"(ocol));
                for (int d = 0; d < a.nd; d++) {
                    const double* D = a.D + d * a.dstride + mat;
                    DigestCtx x;
                    x.Dm = as_const(D + (long)orow * onbf);
                    x.rm = BLDS ? drow + d * (NA + NB) * onbf : D + (long)orow * onbf;
                    x.rn = BLDS ? drow + d * (NA + NB) * onbf + NA * onbf : D + (long)ocol * onbf;
                    x.ld = onbf;
                    x.oN = ocol;
                    x.oP = ox;
                    x.oQ = oy;
                    x.f1 = f1;
                    x.f2 = ki.z;
                    x.f3 = bra != ki.w;
                    x.strip = strip + d * wsz;
                    x.nbf = onbf;
                    x.jmn = jmn + d * wsz + (lane & (GTF_JMN_COPIES - 1)) * NAB;
                    x.dk = a.dk + d * NCD * a.nket + oj;
                    x.nk = a.nket;
                    x.jpq = buffered ? jpq + lane : nullptr;
                    x.clane = CL > 0 ? 1 << ljc : 0;
                    x.lead = cl == 0;
                    x.jk = a.jk + d * NCD * a.nket + oj;
                    auto get = [&](auto c_, auto d_) GTF_INLINE { return (double)cell(c_, d_); };
                    if constexpr (JREG_ABLE) {
                        if (jreg_on) {
                            digest_unit<LA, LB, LC, LD, A0, NAr, C0, NCr, true, CL>(x, crt, get, jreg);
                            continue;
                        }
                    }
                    digest_unit<LA, LB, LC, LD, A0, NAr, C0, NCr, false, CL>(x, crt, get, nullptr);
                }
            };
            for (int sp = sp0; sp < sp0 + spn; sp++)
                for (int ic = ic0; ic < ic0 + icn; ic++) {
                    const int j0 = ic + (jc << lic);
                    if constexpr (!STATIC && EX) {
                        const double* kf = on ? a.kv.f + ((long)(kb >> 6) * S::ESZ_CD + sp * S::HCD) * 64 + (kb & 63) : nullptr;
                        Real acc[1][NAB];
                        eri_lane_t<LA, LB, LC, LD, -1, 1, Real, BLDS>(br, kr, j0, js, kf, boys, acc);
                        finish(std::integral_constant<int, 0>{}, std::integral_constant<int, NAB>{},
                               std::integral_constant<int, -1>{}, std::integral_constant<int, 1>{}, acc, sp);
                    } else if constexpr (CL > 0) {
                        const int comp = (sp << CL) + cl;
                        BraRef<Coef> b1 = br;
                        b1.lane_E = lane_E + min(comp, NAB - 1) * S::HAB;
                        KetRef k1 = kr;
                        if (comp >= NAB) k1.n = 0;  // a lane without a component: zeros
                        Real acc[1][NCD];
                        eri_lane<LA, LB, LC, LD, -1, 1, Real, BLDS, true>(b1, k1, j0, js, boys, acc);
                        finish(std::integral_constant<int, -1>{}, std::integral_constant<int, 1>{},
                               std::integral_constant<int, 0>{}, std::integral_constant<int, NCD>{}, acc, min(comp, NAB - 1));
                    } else if constexpr (!STATIC) {
                        BraRef<Coef> b1 = br;
                        b1.E += sp * S::HAB;
                        Real acc[1][NCD];
                        eri_lane<LA, LB, LC, LD, -1, 1, Real, BLDS>(b1, kr, j0, js, boys, acc);
                        finish(std::integral_constant<int, -1>{}, std::integral_constant<int, 1>{},
                               std::integral_constant<int, 0>{}, std::integral_constant<int, NCD>{}, acc, sp);
                    } else {
                        split_switch<NSPLIT>(sp, [&](auto s_) GTF_INLINE {
                            constexpr int F0 = decltype(s_)::value * NC;
                            constexpr int FN = SIDE - F0 < NC ? SIDE - F0 : NC;
                            if constexpr (EX) {
                                Real acc[FN][NAB];
                                eri_lane_t<LA, LB, LC, LD, F0, FN, Real, BLDS>(br, kr, j0, js, nullptr, boys, acc);
                                finish(std::integral_constant<int, 0>{}, std::integral_constant<int, NAB>{},
                                       std::integral_constant<int, F0>{}, std::integral_constant<int, FN>{}, acc, 0);
                            } else {
                                Real acc[FN][NCD];
                                eri_lane<LA, LB, LC, LD, F0, FN, Real, BLDS>(br, kr, j0, js, boys, acc);
                                finish(std::integral_constant<int, F0>{}, std::integral_constant<int, FN>{},
                                       std::integral_constant<int, 0>{}, std::integral_constant<int, NCD>{}, acc, 0);
                            }
                        });
                    }
                }
            // the block's J_PQ
            if constexpr (CL > 0) {
                // summed over the lanes of a ket
                if (buffered)
                    for (int cd = 0; cd < NCD; cd++) {
                        double* p = jpq + cd * 64 + lane;
                        double v = *p;
                        if (v != 0.0) *p = 0.0;
                        for (int s = 0; s < CL; s++) v += __shfl_xor(v, 1 << (ljc + s), 64);
                        if (on && (jc | cl) == 0 && v != 0.0) GTF_ATOMIC_ADD(&a.jk[cd * a.nket + j], v);
                    }
            } else if (buffered && on && jc == 0)
                for (int cd = 0; cd < NCD; cd++) {
                    double* p = jpq + cd * 64 + lane;
                    const double v = *p;
                    if (v != 0.0) {
                        GTF_ATOMIC_ADD(&a.jk[cd * a.nket + j], v);
                        *p = 0.0;
                    }
                }
        }
        if constexpr (JREG_ABLE) {
            if (jreg_on)
                static_for<0, NAB>([&](auto c_) GTF_INLINE {
                    constexpr int c = decltype(c_)::value;
                    if (jreg[c] != 0.0) atomicAdd(&jmn[(lane & (GTF_JMN_COPIES - 1)) * NAB + c], jreg[c]);
                });
        }
        if (threadIdx.x == 0) s_task = next;
        __syncthreads();
        for (int d = 0; d < a.nd; d++) {
            double* sd = strip + d * wsz;
            double* jd = jmn + d * wsz;
            double* Kd = a.K + d * a.dstride + mat;
            double* Jd = a.J + d * a.dstride + mat;
            for (int o = 0; o < NA + NB; o++) {
                double* Kr = Kd + (long)(o < NA ? oM + o : oN + (o - NA)) * nbf;
                for (int k = threadIdx.x; k < nbf; k += NT) {
                    const double v = sd[o * nbf + k];
                    if (v != 0.0) {
                        GTF_ATOMIC_ADD(&Kr[k], v);
                        sd[o * nbf + k] = 0.0;
                    }
                }
            }
            for (int k = threadIdx.x; k < NAB; k += NT) {
                double v = 0.0;
                for (int c = 0; c < GTF_JMN_COPIES; c++) {
                    v += jd[c * NAB + k];
                    jd[c * NAB + k] = 0.0;
                }
                if (v != 0.0) GTF_ATOMIC_ADD(&Jd[(long)(oM + k / NB) * nbf + oN + k % NB], v);
            }
        }
        if (threadIdx.x == 0) s_unit = 0;
        open = open_tile(__builtin_amdgcn_readfirstlane(s_task));
        __syncthreads();
    }
    record_workgroup(a, t_begin, taken);
}

template <int LA, int LB, int LC, int LD, int NC, typename Real, bool BLDS>
__global__ __launch_bounds__((tile_threads<LA, LB, LC, LD>()), (tile_min_waves<LA, LB, LC, LD>())) void eri_jk_tile_kernel(EriArgs a)
{
    tile_kernel_body<LA, LB, LC, LD, NC, Real, BLDS, false>(a);
}

template <int LA, int LB, int LC, int LD, int NCT, typename Real, bool BLDS>
__global__ __launch_bounds__((tile_threads<LA, LB, LC, LD>()), (tile_min_waves<LA, LB, LC, LD>())) void eri_jk_tile_t_kernel(EriArgs a)
{
    tile_kernel_body<LA, LB, LC, LD, NCT, Real, BLDS, true>(a);
}

// launch helpers (eri_table.cpp)
typedef void (*eri_kernel_t)(EriArgs);
struct EriClassInfo {
    int la, lb, lc, ld;
    int nc;         // bra components per thread of the unit kernels (jk, diag, store)
    int nsplit;     // and threads per quartet
    int tile_threads;  // largest workgroup of the tile kernels
    int nc_tile;       // bra components per thread of the tile kernels
    int nsplit_tile;   // chunks of the bra components
    int comp_lanes;    // log2 of the lanes that share a ket, a component each, in the standard tile kernels
    bool full_E;       // the standard tile kernel reads the full coefficients
    int nints;      // integrals per quartet
    eri_kernel_t jk, diag, store;
    // tile kernels: FP64 quartets (v_bra v_ket >= tau2), [0] Boys slab read
    // from HBM, [1] staged in LDS; FP32 quartets (v_bra v_ket < tau2)
    eri_kernel_t jk_tile[2], jk_tile_lo;
    // classes that have a tile kernel with the contractions exchanged
    // (nsplit_t > 0): threads per quartet, ket components per thread
    int nsplit_t, nc_t;
    eri_kernel_t jk_tile_t[2], jk_tile_t_lo;
};
const EriClassInfo* gtf_eri_class(int cls);
