// gtf_internal.h -- shared definitions of the HIP Fock engine (host + device).
//
// Angular momentum up to d (L <= 2) per shell, spherical functions.
// Shell pairs are stored canonically with L(s1) >= L(s2); a pair type is
//   0 ss, 1 ps, 2 pp, 3 ds, 4 dp, 5 dd
// and a quartet class (bra type A >= ket type B) is A*(A+1)/2 + B (21 classes).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <type_traits>
#include <utility>

#define GTF_LMAX 2
#define GTF_NPAIRTYPES 6
#define GTF_NCLASSES 21
// ket-list block re-sorted by primitive count (one wavefront)
#define GTF_KET_BLOCK 64
// kets of a segment whose records start a block of their own (KetView)
#define GTF_KET_OWN 256

// A tile of the J/K kernels is one bra pair and several runs of its kets:
// TileHead.  A run is int4 (first ket, span word, chunk word, bra row).
// span word: kets, first component chunk and number of them
#define GTF_RUN_SPAN(kets, sp0, spn) ((kets) | (sp0) << 15 | (spn) << 20)
#define GTF_RUN_KETS(y) ((y) & 32767)
#define GTF_RUN_SP0(y) (((y) >> 15) & 31)
#define GTF_RUN_SPN(y) ((y) >> 20)
#define GTF_RUN_MAX_KETS 32767
// chunk word: log2 of the ket-primitive chunks, log2 of the lanes that share a
// ket, first ket-primitive chunk and number of them
#define GTF_RUN_CHUNKS(lic, ljc, ic0, icn) ((lic) | (ljc) << 4 | (ic0) << 8 | (icn) << 20)
#define GTF_RUN_LIC(z) ((z) & 15)
#define GTF_RUN_LJC(z) (((z) >> 4) & 15)
#define GTF_RUN_IC0(z) (((z) >> 8) & 4095)
#define GTF_RUN_ICN(z) ((z) >> 20)
#define GTF_MAX_LIC 9  // at most 512 chunks
// Everything of the bra that a workgroup needs to start a tile, read with one
// scalar load (looked up through the pair and shell arrays it was a chain of
// five dependent loads, several microseconds a tile).
struct TileHead {
    int row, run0, nrun;  // bra row, runs
    int bra;              // pair id
    int prim, nprim;      // first primitive pair, primitive pairs
    int oM, oN;           // function offsets
    int two;              // 1 if the shells differ
    int nbf, mol;         // size of the molecule's matrices, molecule
    int rank;
    long mat;             // the molecule's matrix block
    long E;               // first coefficient, in the layout that the kernel reads
};
static_assert(sizeof(TileHead) == 64, "read as 16 dwords");

// Boys-function grid: F_m(T0) for T0 = i * BOYS_DELTA, i = 0..BOYS_NGRID-1,
// m = 0..BOYS_NCOL-1; T >= BOYS_TMAX uses the asymptotic form.
#define BOYS_DELTA 0.05
#define BOYS_INV_DELTA 20.0
#define BOYS_NGRID 721
#define BOYS_NCOL 16
#define BOYS_TMAX 36.0
#define BOYS_NTAYLOR 7
// compact Taylor table of the ERI kernels: orders M = 0 .. BOYS8_NM - 1,
// T0 = i * BOYS8_DELTA for i < BOYS8_NGRID, BOYS8_NTERM coefficients per row
#define BOYS8_DELTA 0.1
#define BOYS8_INV_DELTA 10.0
#define BOYS8_NGRID 361
#define BOYS8_NTERM 8
#define BOYS8_NM 9
#define BOYS8_SLAB (BOYS8_NGRID * BOYS8_NTERM)
// the slabs, then exp(-T0) of the grid points (padded to whole double2)
#define BOYS8_EXP (BOYS8_NGRID + 1)
#define BOYS8_TOTAL (BOYS8_NM * BOYS8_SLAB + BOYS8_EXP)

#define GTF_CHECK(call)                                                                    \
    do {                                                                                   \
        hipError_t e_ = (call);                                                            \
        if (e_ != hipSuccess) {                                                            \
            fprintf(stderr, "gtfock_amd: HIP error %s at %s:%d\n", hipGetErrorString(e_), \
                    __FILE__, __LINE__);                                                   \
            return -1;                                                                     \
        }                                                                                  \
    } while (0)

__host__ __device__ constexpr int nherm(int L) { return (L + 1) * (L + 2) * (L + 3) / 6; }
__host__ __device__ constexpr int nsph(int l) { return 2 * l + 1; }
__host__ __device__ constexpr int ncart(int l) { return (l + 1) * (l + 2) / 2; }
__host__ __device__ constexpr int pair_type(int la, int lb) { return la * (la + 1) / 2 + lb; }
__host__ __device__ constexpr int class_index(int A, int B) { return A * (A + 1) / 2 + B; }

// Hermite / cartesian component index: order k = t+u+v, then t descending,
// then v ascending.  The same ordering serves cartesian components
// (lx, ly, lz) of one shell when restricted to order k.
__host__ __device__ constexpr int hidx(int t, int u, int v)
{
    return (t + u + v) * (t + u + v + 1) * (t + u + v + 2) / 6 +
           ((u + v) * (u + v + 1)) / 2 + v;
}
__host__ __device__ constexpr int horder(int h)
{
    int k = 0;
    while (nherm(k) <= h) ++k;
    return k;
}
__host__ __device__ constexpr int herm_t(int h)
{
    int k = horder(h);
    int r = h - (k == 0 ? 0 : nherm(k - 1));
    int s = 0;  // s = u + v
    while ((s + 1) * (s + 2) / 2 <= r) ++s;
    return k - s;
}
__host__ __device__ constexpr int herm_v(int h)
{
    int k = horder(h);
    int r = h - (k == 0 ? 0 : nherm(k - 1));
    int s = 0;
    while ((s + 1) * (s + 2) / 2 <= r) ++s;
    return r - s * (s + 1) / 2;
}
__host__ __device__ constexpr int herm_u(int h) { return horder(h) - herm_t(h) - herm_v(h); }

// 1/sqrt(s) from the hardware estimate refined by two Newton steps
// y <- y (3 - s y^2) / 2 (relative error ~1e-16 in FP64)
__device__ __forceinline__ double rsqrt_nr(double s)
{
    double y = __builtin_amdgcn_rsq(s);
    double h = s * y;
    y = fma(y, fma(-0.5 * h, y, 0.5), y);
    h = s * y;
    y = fma(y, fma(-0.5 * h, y, 0.5), y);
    return y;
}
__device__ __forceinline__ float rsqrt_nr(float s)
{
    float y = __builtin_amdgcn_rsqf(s);
    y = fmaf(y, fmaf(-0.5f * s * y, y, 0.5f), y);
    return y;
}

// for lambdas whose arrays must stay in registers
#define GTF_INLINE __attribute__((always_inline))

// compile-time loop: f(std::integral_constant<int, i>) for i in [B, E)
template <int B, int E, typename F>
__host__ __device__ __forceinline__ void static_for(F&& f)
{
    if constexpr (B < E) {
        f(std::integral_constant<int, B>{});
        static_for<B + 1, E>(f);
    }
}

// Device views of the engine's resident data.
struct PairView {
    const int* s1;       // canonical first shell
    const int* s2;       // canonical second shell
    const int* nprim;    // primitive pairs
    const int* poff;     // offset into prim[]
    const long* eoff;    // offset into E[]
    const double4* prim; // (p, Px, Py, Pz) per primitive pair
    const double* E;     // Hermite->spherical coefficients, scaled by c_i c_j K_ab / p
    const long* zoff;    // offset into Ez[]
    const double* Ez;    // the same, structural nonzeros only (herm_nz_pos order)
    const double* q;     // Schwarz bound per primitive pair (a pair's primitives in descending order)
    const float* Ezf;    // Ez rounded to FP32 (systems with FP32 tiles)
    double peps;         // primitive quartets with q_bra q_ket < peps are skipped (0: none)
};

// Ket side of one pair type's significant-pair list, in list order, for the
// tile kernels: 64 kets form a block whose primitive pairs are
// stored primitive by primitive, each as rec(nnz) rows of 64 double2 -- (p,
// Px), (Py, Pz) and the compact Hermite coefficients two by two -- so that the
// lanes of a wavefront, which hold consecutive kets, read whole lines.
// base[j] = 64 * (first primitive row of ket j's block) + (place in the block).
struct KetView {
    const int* base;
    const double2* d;
    const double* f;    // pair types with a chunked ket side: the full coefficients, rows of 64 doubles
    const double* q;    // Schwarz bound per primitive pair, rows of 64
    const int4* info;   // function offsets of the two shells, 1 if they differ, pair id
    const int* nprim;
    __host__ __device__ static constexpr int rec(int nnz) { return 2 + (nnz + 1) / 2; }
    // pair types whose full coefficients are stored (pp, ds, dp) in a system with
    // d functions: the exchanged kernels of a dp or dd bra take one ket component
    // at a time, known at run time.  Found among the compact ones instead, they
    // would save C54H18 33 of 327 MB and cost (dd|dp) 11 %, (dp|pp) 4 %.
    __host__ __device__ static constexpr bool full(int type) { return type >= 2 && type <= 4; }
};

// One pair type's list in the density's and J_PQ's list-ordered copies: [density]
// [component][list position].
struct JkList {
    int n;             // list length
    int nc, nd;        // functions of the two shells
    const int4* info;  // KetView::info
    double* dk;
    double* jk;
};
struct JkLists {
    JkList t[GTF_NPAIRTYPES];
    const int* s1;      // first shell of each pair
    const long* mbase;  // per shell: matrix block and leading dimension
    const int* mld;
};

struct BasisView {
    int nshells, nbf, natoms;
    const int* L;
    const int* nprim;
    const int* poff;
    const int* fstart;
    const int* atom;
    const double* alpha;
    const double* coef;
    const double* center;    // 3 per shell (bohr)
    const double* atom_xyz;  // 3 per atom
    const double* atom_Z;
};

// Spherical transform rows (m = -l..l) over cartesian components of order l
// in the hidx order (xx, xy, xz, yy, yz, zz for l = 2).
__host__ __device__ constexpr double sph_coef(int l, int m, int c)
{
    if (l == 0) return 1.0;
    if (l == 1) return m == c ? 1.0 : 0.0;
    const double r3 = 1.7320508075688772;
    switch (m) {
    case 0: return c == 1 ? r3 : 0.0;                              // xy
    case 1: return c == 4 ? r3 : 0.0;                              // yz
    case 2: return c == 5 ? 1.0 : ((c == 0 || c == 3) ? -0.5 : 0.0); // z^2 - r^2/2
    case 3: return c == 2 ? r3 : 0.0;                              // xz
    case 4: return c == 0 ? 0.5 * r3 : (c == 3 ? -0.5 * r3 : 0.0); // (x^2 - y^2)
    }
    return 0.0;
}

// Structural nonzeros of the Hermite coefficients of a spherical component
// pair (as, bs) of shells (la, lb): E^{ab}_{tuv} can be nonzero only if some
// cartesian pair (a, b) in the two spherical functions has t <= ax + bx,
// u <= ay + by, v <= az + bz.
__host__ __device__ constexpr bool herm_nz(int la, int lb, int as, int bs, int h)
{
    const int t = herm_t(h), u = herm_u(h), v = herm_v(h);
    const int ca0 = la == 0 ? 0 : nherm(la - 1), cb0 = lb == 0 ? 0 : nherm(lb - 1);
    for (int ca = 0; ca < ncart(la); ca++) {
        if (sph_coef(la, as, ca) == 0.0) continue;
        for (int cb = 0; cb < ncart(lb); cb++) {
            if (sph_coef(lb, bs, cb) == 0.0) continue;
            if (t <= herm_t(ca0 + ca) + herm_t(cb0 + cb) && u <= herm_u(ca0 + ca) + herm_u(cb0 + cb) &&
                v <= herm_v(ca0 + ca) + herm_v(cb0 + cb))
                return true;
        }
    }
    return false;
}
// The structural-nonzero table of one pair type, evaluated once at compile
// time: nz[ab][h], pos[ab][h] (position in the compact layout), nnz.
template <int LA, int LB>
struct NzTab {
    static constexpr int NAB = nsph(LA) * nsph(LB), H = nherm(LA + LB);
    struct Data {
        bool nz[NAB][H];
        int pos[NAB][H];
        int nnz;
    };
    static constexpr Data make()
    {
        Data d{};
        int n = 0;
        for (int ab = 0; ab < NAB; ab++)
            for (int h = 0; h < H; h++) {
                d.nz[ab][h] = herm_nz(LA, LB, ab / nsph(LB), ab % nsph(LB), h);
                d.pos[ab][h] = n;
                if (d.nz[ab][h]) n++;
            }
        d.nnz = n;
        return d;
    }
    static constexpr Data data = make();
};

// number of structural nonzeros of a (la, lb) pair block (runtime form), and
// the position of (component ab, hermite h) in the compact layout
__host__ __device__ constexpr int herm_nnz(int la, int lb)
{
    int n = 0;
    for (int ab = 0; ab < nsph(la) * nsph(lb); ab++)
        for (int h = 0; h < nherm(la + lb); h++)
            if (herm_nz(la, lb, ab / nsph(lb), ab % nsph(lb), h)) n++;
    return n;
}
// herm_nnz read from the compile-time tables (the runtime form takes
// thousands of steps per call; set-up code calls it once per shell pair)
inline int herm_nnz_lookup(int la, int lb)
{
    static_assert(GTF_LMAX == 2, "table below lists l = 0..2");
    static constexpr int t[3][3] = {{NzTab<0, 0>::data.nnz, NzTab<0, 1>::data.nnz, NzTab<0, 2>::data.nnz},
                                    {NzTab<1, 0>::data.nnz, NzTab<1, 1>::data.nnz, NzTab<1, 2>::data.nnz},
                                    {NzTab<2, 0>::data.nnz, NzTab<2, 1>::data.nnz, NzTab<2, 2>::data.nnz}};
    return t[la][lb];
}
__host__ __device__ constexpr int herm_nz_pos(int la, int lb, int ab, int h)
{
    int n = 0;
    for (int x = 0; x < nsph(la) * nsph(lb); x++)
        for (int y = 0; y < nherm(la + lb); y++) {
            if (x == ab && y == h) return n;
            if (herm_nz(la, lb, x / nsph(lb), x % nsph(lb), y)) n++;
        }
    return n;
}
