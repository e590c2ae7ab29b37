// batch_linalg.hip -- the dense steps of an SCF iteration (pscf/purif.c,
// pscf/scf.c:80-102) for many molecules at once.
//
// Two per-molecule layouts share one device array each:
//   packed  molecule m at off[m], row-major n_m x n_m (the Fock engine's)
//   padded  molecule m at poff[m], row-major n_m x pld[m], pld = n rounded
//           up to 64 with zero padding (the MFMA GEMM's)
// Every kernel indexes molecules by blockIdx.y (blockIdx.z for the GEMM) and
// skips a molecule whose flag in `skip` is set.  Reductions add fixed-order
// partials, so a molecule's result does not depend on which other molecules
// share the batch.
#include "batch_linalg.h"

#include "gemm_tile.h"
#include "ozaki_launch.h"

// C_m = A_m * B_m (TRANSB = 0) or A_m * B_m^T (TRANSB = 1) on padded blocks
// (gemm_tile.h).  A molecule is skipped when skip[m] != 0 or, during
// purification, when it has already converged (done[m] >= 0); fp32[m] ==
// GTF_LOW_FP32 selects the FP32 MFMA tile for it, GTF_LOW_SPLIT leaves it to
// the split-BF16 products.  above: molecules of a larger leading dimension
// only (the others are bgemm_rows_kernel's).
template <int TRANSB>
__global__ __launch_bounds__(256) void bgemm_kernel(const long* __restrict__ poff, const int* __restrict__ pld,
                                                    const int* __restrict__ skip, const int* __restrict__ done,
                                                    const int* __restrict__ fp32, int above,
                                                    const double* __restrict__ A0, const double* __restrict__ B0,
                                                    double* __restrict__ C0)
{
    const int m = blockIdx.z;
    const int ld = pld[m];
    const int row0 = blockIdx.y * GEMM_GT, col0 = blockIdx.x * GEMM_GT;
    if (row0 >= ld || col0 >= ld || ld <= above || (skip && skip[m]) || (done && done[m] >= 0)) return;
    const long o = poff[m];
    if (fp32 && fp32[m] == GTF_LOW_SPLIT) return;  // the split-BF16 products (ozaki.hip) cover it
    if (fp32 && fp32[m] == GTF_LOW_FP32) gemm_tile<TRANSB, true>(ld, A0 + o, B0 + o, C0 + o, row0, col0);
    else gemm_tile<TRANSB, false>(ld, A0 + o, B0 + o, C0 + o, row0, col0);
}

// fixed-order tree reduction of one value per thread of a block of NT threads
template <int NT = 256, typename Op>
__device__ __forceinline__ double block_reduce(double v, double* sh, Op op)
{
    sh[threadIdx.x] = v;
    __syncthreads();
    for (int s = NT / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s) sh[threadIdx.x] = op(sh[threadIdx.x], sh[threadIdx.x + s]);
        __syncthreads();
    }
    const double r = sh[0];
    __syncthreads();
    return r;
}

// C_m = A_m * B_m^T, every tile, of the molecules up to ROWS_MAX_LD
__global__ __launch_bounds__(ROWS_THREADS) void bgemm_rows_kernel(const long* __restrict__ poff, const int* __restrict__ pld,
                                                         const int* __restrict__ skip, const int* __restrict__ done,
                                                         const double* __restrict__ A0, const double* __restrict__ B0,
                                                         double* __restrict__ C0)
{
    __shared__ double red[ROWS_W][ROWS_T * ROWS_T];
    const int m = blockIdx.z, ld = pld[m], row0 = blockIdx.y * ROWS_T, col0 = blockIdx.x * ROWS_T;
    if (row0 >= ld || col0 >= ld || ld > ROWS_MAX_LD || (skip && skip[m]) || (done && done[m] >= 0)) return;
    const long o = poff[m];
    rows_tile(ld, A0 + o, B0 + o, row0, col0, red);
    for (int k = threadIdx.x; k < ROWS_T * ROWS_T; k += ROWS_THREADS) C0[o + (long)(row0 + k / ROWS_T) * ld + col0 + k % ROWS_T] = red[0][k];
}

// tiles of the lower triangle
__host__ __device__ constexpr int tri_tiles(int ld) { return (ld / ROWS_T) * (ld / ROWS_T + 1) / 2; }

// One product of the purification, C_m = D_m * B_m of symmetric commuting
// matrices (B is D, then D^2): the tiles of the lower triangle, each also
// written transposed.  The partial sums of the statistics come from the tiles:
// with B = D (CUBE false) {||D - C||_F^2, tr(D - C)}, with B = D^2 tr(B - C).
template <bool CUBE>
__global__ __launch_bounds__(ROWS_THREADS) void bpurif_product_kernel(const long* __restrict__ poff,
                                                             const int* __restrict__ pld, const int* __restrict__ skip,
                                                             const int* __restrict__ done,
                                                             const double* __restrict__ D0,
                                                             const double* __restrict__ B0, double* __restrict__ C0,
                                                             double* __restrict__ part, int mtiles)
{
    __shared__ double red[ROWS_W][ROWS_T * ROWS_T];
    const int m = blockIdx.y, t = blockIdx.x, ld = pld[m];
    if (t >= tri_tiles(ld) || (skip && skip[m]) || done[m] >= 0) return;
    int ti = (int)((sqrtf(8.0f * t + 1.0f) - 1.0f) * 0.5f);
    while ((ti + 1) * (ti + 2) / 2 <= t) ti++;
    while (ti * (ti + 1) / 2 > t) ti--;
    const int tj = t - ti * (ti + 1) / 2;
    const int row0 = ti * ROWS_T, col0 = tj * ROWS_T;
    const long o = poff[m];
    rows_tile(ld, D0 + o, B0 + o, row0, col0, red);
    double* C = C0 + o;
    const double* S = (CUBE ? B0 : D0) + o;  // what C is subtracted from
    double e = 0.0, tr = 0.0;
    for (int k = threadIdx.x; k < ROWS_T * ROWS_T; k += ROWS_THREADS) {
        const int i = k / ROWS_T, j = k % ROWS_T;
        const double low = red[0][k], up = red[0][j * ROWS_T + i];
        double v = low;
        if (ti == tj) v = 0.5 * (low + up);
        else C[(long)(col0 + i) * ld + row0 + j] = up;
        C[(long)(row0 + i) * ld + col0 + j] = v;
        if (!CUBE || (ti == tj && i == j)) {
            const double x = S[(long)(row0 + i) * ld + col0 + j] - v;
            e += x * x;
            if (ti == tj && i == j) tr += x;
        }
    }
    if (CUBE && ti != tj) return;  // tr alone
    __syncthreads();
    double* sh = red[1];
    auto add = [](double a, double b) { return a + b; };
    if (!CUBE) e = block_reduce<ROWS_THREADS>(e, sh, add);
    if (ti == tj) tr = block_reduce<ROWS_THREADS>(tr, sh, add);
    if (threadIdx.x == 0) {
        double* p = part + ((long)m * mtiles + t) * 3;
        if (CUBE) {
            p[2] = tr;
        } else {
            p[0] = ti == tj ? e : 2.0 * e;
            p[1] = ti == tj ? tr : 0.0;
            p[2] = 0.0;
        }
    }
}

// packed -> padded (zero padding) and padded -> packed
__global__ void bpad_kernel(const long* __restrict__ off, const int* __restrict__ nn, const long* __restrict__ poff,
                            const int* __restrict__ pld, const int* __restrict__ skip, const double* __restrict__ src,
                            double* __restrict__ dst)
{
    const int m = blockIdx.y;
    if (skip && skip[m]) return;
    const int n = nn[m], ld = pld[m];
    const double* s = src + off[m];
    double* d = dst + poff[m];
    for (long k = (long)blockIdx.x * blockDim.x + threadIdx.x; k < (long)ld * ld; k += (long)gridDim.x * blockDim.x) {
        const int i = (int)(k / ld), j = (int)(k - (long)i * ld);
        d[k] = (i < n && j < n) ? s[(long)i * n + j] : 0.0;
    }
}
__global__ void bunpad_kernel(const long* __restrict__ off, const int* __restrict__ nn, const long* __restrict__ poff,
                              const int* __restrict__ pld, const int* __restrict__ skip,
                              const double* __restrict__ src, double* __restrict__ dst)
{
    const int m = blockIdx.y;
    if (skip && skip[m]) return;
    const int n = nn[m], ld = pld[m];
    const double* s = src + poff[m];
    double* d = dst + off[m];
    for (long k = (long)blockIdx.x * blockDim.x + threadIdx.x; k < (long)n * n; k += (long)gridDim.x * blockDim.x) {
        const int i = (int)(k / n), j = (int)(k - (long)i * n);
        d[k] = s[(long)i * ld + j];
    }
}

// Reductions over one molecule's matrix run in BPART workgroups per molecule
// (grid BPART x nmol), each writing its partial to part[(m * BPART + p) * w
// + v]; a finishing kernel (one thread per molecule) adds the partials in
// order p = 0 .. BPART-1.  The result depends only on the molecule's data.

// Gershgorin bounds and trace of F_m (pscf/purif.c:302-358), partials
__global__ __launch_bounds__(256) void bgersh_part_kernel(const long* __restrict__ poff, const int* __restrict__ nn,
                                                          const int* __restrict__ pld, const int* __restrict__ skip,
                                                          const double* __restrict__ F0, double* __restrict__ part)
{
    __shared__ double sh[256];
    const int m = blockIdx.y, p = blockIdx.x;
    if (skip && skip[m]) return;
    const int n = nn[m], ld = pld[m];
    const double* F = F0 + poff[m];
    double mn = 1e300, mx = -1e300, tr = 0.0;
    // a wavefront per row (F is symmetric); a thread per column walked the
    // matrix with one workgroup at n = 250, 100 us
    const int lane = threadIdx.x & 63;
    for (int i = p * 4 + (threadIdx.x >> 6); i < n; i += BPART * 4) {
        double off = 0.0;
        for (int j = lane; j < n; j += 64) off += fabs(F[(long)i * ld + j]);
        for (int w = 32; w > 0; w >>= 1) off += __shfl_xor(off, w, 64);
        const double dg = F[(long)i * ld + i];
        off -= fabs(dg);
        mn = fmin(mn, dg - off);
        mx = fmax(mx, dg + off);
        if (lane == 0) tr += dg;
    }
    mn = block_reduce(mn, sh, [](double a, double b) { return fmin(a, b); });
    mx = block_reduce(mx, sh, [](double a, double b) { return fmax(a, b); });
    tr = block_reduce(tr, sh, [](double a, double b) { return a + b; });
    if (threadIdx.x == 0) {
        double* o = part + ((long)m * BPART + p) * 3;
        o[0] = mn;
        o[1] = mx;
        o[2] = tr;
    }
}

// coef[2m] = -lambda / n, coef[2m + 1] = lambda mu / n + nocc / n with
// mu = tr F / n, lambda = min(nocc / (hmax - mu), (n - nocc) / (mu - hmin))
// (pscf/purif.c:347-373)
__global__ void bgersh_fin_kernel(int nmol, const int* __restrict__ nn, const int* __restrict__ nocc,
                                  const int* __restrict__ skip, const double* __restrict__ part,
                                  double* __restrict__ coef)
{
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= nmol || (skip && skip[m])) return;
    double hmin = 1e300, hmax = -1e300, tr = 0.0;
    for (int p = 0; p < BPART; p++) {
        const double* o = part + ((long)m * BPART + p) * 3;
        hmin = fmin(hmin, o[0]);
        hmax = fmax(hmax, o[1]);
        tr += o[2];
    }
    const int n = nn[m];
    const double mu = tr / n, no = nocc[m];
    const double lambda = fmin(no / (hmax - mu), (double)(n - nocc[m]) / (mu - hmin));
    coef[2 * m] = -lambda / n;
    coef[2 * m + 1] = lambda * mu / n + no / n;
}

// D0 = coef0 (F + F^T)/2 + coef1 I on the n x n block, zero padding
__global__ void bpurif_init_kernel(const long* __restrict__ poff, const int* __restrict__ nn,
                                   const int* __restrict__ pld, const int* __restrict__ skip,
                                   const double* __restrict__ coef, const double* __restrict__ F0,
                                   double* __restrict__ D0)
{
    const int m = blockIdx.y;
    if (skip && skip[m]) return;
    const int n = nn[m], ld = pld[m];
    const double a = coef[2 * m], dshift = coef[2 * m + 1];
    const double* F = F0 + poff[m];
    double* D = D0 + poff[m];
    for (long k = (long)blockIdx.x * blockDim.x + threadIdx.x; k < (long)ld * ld; k += (long)gridDim.x * blockDim.x) {
        const int i = (int)(k / ld), j = (int)(k - (long)i * ld);
        D[k] = (i < n && j < n) ? a * (0.5 * (F[k] + F[(long)j * ld + i])) + (i == j ? dshift : 0.0) : 0.0;
    }
}

// partials of {||D - D2||_F^2, tr(D2 - D3), tr(D - D2)} of the molecules
// still iterating
__global__ __launch_bounds__(256) void bstats_part_kernel(const long* __restrict__ poff, const int* __restrict__ nn,
                                                          const int* __restrict__ pld, const int* __restrict__ skip,
                                                          const int* __restrict__ iters,
                                                          const double* __restrict__ D0,
                                                          const double* __restrict__ D20,
                                                          const double* __restrict__ D30, double* __restrict__ part)
{
    __shared__ double sh[256];
    const int m = blockIdx.y, p = blockIdx.x;
    if ((skip && skip[m]) || iters[m] >= 0) return;
    const int n = nn[m], ld = pld[m];
    const double* D = D0 + poff[m];
    const double* D2 = D20 + poff[m];
    const double* D3 = D30 + poff[m];
    double e = 0.0, t1 = 0.0, t2 = 0.0;
    for (long k = (long)p * 256 + threadIdx.x; k < (long)ld * ld; k += BPART * 256) {
        const double d = D[k] - D2[k];
        e += d * d;
    }
    for (int i = p * 256 + threadIdx.x; i < n; i += BPART * 256) {
        const long k = (long)i * ld + i;
        t1 += D2[k] - D3[k];
        t2 += D[k] - D2[k];
    }
    auto add = [](double a, double b) { return a + b; };
    e = block_reduce(e, sh, add);
    t1 = block_reduce(t1, sh, add);
    t2 = block_reduce(t2, sh, add);
    if (threadIdx.x == 0) {
        double* o = part + ((long)m * BPART + p) * 3;
        o[0] = e;
        o[1] = t1;
        o[2] = t2;
    }
}

// stats[3m..] from the partials; a molecule whose error drops below tol is
// marked done at this iteration (iters[m] = it) and still takes this
// iteration's update
__global__ void bstats_fin_kernel(int nmol, const int* __restrict__ skip, const double* __restrict__ part,
                                  int* __restrict__ iters, double* __restrict__ stats, int it, double tol,
                                  int* __restrict__ fp32, double fp32_until, int* __restrict__ low_iters)
{
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= nmol || (skip && skip[m]) || iters[m] >= 0) return;
    double e = 0.0, t1 = 0.0, t2 = 0.0;
    for (int p = 0; p < BPART; p++) {
        const double* o = part + ((long)m * BPART + p) * 3;
        e += o[0];
        t1 += o[1];
        t2 += o[2];
    }
    stats[3 * m + 0] = e;
    stats[3 * m + 1] = t1;
    stats[3 * m + 2] = t2;
    if (sqrt(e) < tol) iters[m] = it;
    // FP32 GEMMs only while the error is far above FP32 resolution
    if (fp32 && fp32[m] && sqrt(e) < fp32_until) {
        fp32[m] = 0;
        if (low_iters) low_iters[m] = it + 1;  // iterations 0..it ran in the reduced precision
    }
}

// D <- ((1-2c) D + (1+c) D2 - D3)/(1-c) if c < 1/2, else ((1+c) D2 - D3)/c
// (pscf/purif.c:432-453), for molecules iterating at `it`
__global__ void bpurif_update_kernel(const long* __restrict__ poff, const int* __restrict__ pld,
                                     const int* __restrict__ skip, const int* __restrict__ iters,
                                     const double* __restrict__ stats, double* __restrict__ D0,
                                     const double* __restrict__ D20, const double* __restrict__ D30, int it)
{
    const int m = blockIdx.y;
    if ((skip && skip[m]) || (iters[m] >= 0 && iters[m] != it)) return;
    const int ld = pld[m];
    const double c = stats[3 * m + 1] / stats[3 * m + 2];
    double* D = D0 + poff[m];
    const double* D2 = D20 + poff[m];
    const double* D3 = D30 + poff[m];
    for (long k = (long)blockIdx.x * blockDim.x + threadIdx.x; k < (long)ld * ld; k += (long)gridDim.x * blockDim.x) {
        if (c < 0.5) D[k] = ((1.0 - 2.0 * c) * D[k] + (1.0 + c) * D2[k] - D3[k]) / (1.0 - c);
        else D[k] = ((1.0 + c) * D2[k] - D3[k]) / c;
    }
}

// The same with the means of the products and their transposes: the split
// products are not symmetric, and the iterations amplify an antisymmetric part
// of D (with it C54H18's SCF with split products took 24 builds, FP64's 21;
// without it 21).  A workgroup takes a 32 x 32 tile and reads the mirrored ones
// of D2 and D3 through LDS.  A mirrored element comes out the same bit for bit,
// D being symmetric.  Bound by latency: with a tile and its mirror in one
// workgroup, half as many of them and three barriers, a split purification of
// n = 106 took 3.30 ms, now 3.15 (3.28 with the unsymmetric update).
__global__ __launch_bounds__(256) void bpurif_update_sym_kernel(const long* __restrict__ poff, const int* __restrict__ pld,
                                                            const int* __restrict__ skip, const int* __restrict__ iters,
                                                            const double* __restrict__ stats, double* __restrict__ D0,
                                                            const double* __restrict__ D20,
                                                            const double* __restrict__ D30, int it)
{
    __shared__ double s2[ROWS_T][ROWS_T + 1], s3[ROWS_T][ROWS_T + 1];
    const int m = blockIdx.z, ld = pld[m], row0 = blockIdx.y * ROWS_T, col0 = blockIdx.x * ROWS_T;
    if (row0 >= ld || col0 >= ld || (skip && skip[m]) || (iters[m] >= 0 && iters[m] != it)) return;
    constexpr int N = ROWS_T * ROWS_T / 256, STEP = 256 / ROWS_T;
    const double c = stats[3 * m + 1] / stats[3 * m + 2];
    double* D = D0 + poff[m];
    const double* D2 = D20 + poff[m];
    const double* D3 = D30 + poff[m];
    const int tx = threadIdx.x % ROWS_T, ty = threadIdx.x / ROWS_T;
    const long own = (long)(row0 + ty) * ld + col0 + tx, mirror = (long)(col0 + ty) * ld + row0 + tx;
    double d[N], d2[N], d3[N];
    for (int k = 0; k < N; k++) {
        const long o = (long)k * STEP * ld;
        d[k] = D[own + o];
        d2[k] = D2[own + o];
        d3[k] = D3[own + o];
        s2[ty + k * STEP][tx] = D2[mirror + o];
        s3[ty + k * STEP][tx] = D3[mirror + o];
    }
    __syncthreads();
    for (int k = 0; k < N; k++) {
        const int r = ty + k * STEP;
        const double x = 0.5 * (d2[k] + s2[tx][r]), y = 0.5 * (d3[k] + s3[tx][r]);
        D[own + (long)k * STEP * ld] = c < 0.5 ? ((1.0 - 2.0 * c) * d[k] + (1.0 + c) * x - y) / (1.0 - c) : ((1.0 + c) * x - y) / c;
    }
}

// The same after bpurif_product_kernel: every workgroup adds up the molecule's
// partials (in one fixed order), and the first one records the end of the
// iterations, so a purification iteration is three launches.
__global__ __launch_bounds__(256) void bpurif_step_kernel(const long* __restrict__ poff, const int* __restrict__ pld,
                                                          const int* __restrict__ skip, int* __restrict__ iters,
                                                          const double* __restrict__ part, int mtiles, double tol,
                                                          int* host_iters, double* __restrict__ D0, const double* __restrict__ D20,
                                                          const double* __restrict__ D30, int it)
{
    __shared__ double sh[256];
    const int m = blockIdx.y;
    // a molecule that ends at `it` still takes this update: its flag may be
    // set already by the time a workgroup reads it
    if ((skip && skip[m]) || (iters[m] >= 0 && iters[m] != it)) return;
    const int ld = pld[m], nt = tri_tiles(ld);
    double e = 0.0, t2 = 0.0, t1 = 0.0;
    for (int k = threadIdx.x; k < nt; k += 256) {
        const double* p = part + ((long)m * mtiles + k) * 3;
        e += p[0];
        t2 += p[1];
        t1 += p[2];
    }
    auto add = [](double a, double b) { return a + b; };
    e = block_reduce(e, sh, add);
    t2 = block_reduce(t2, sh, add);
    t1 = block_reduce(t1, sh, add);
    if (blockIdx.x == 0 && threadIdx.x == 0 && sqrt(e) < tol) {
        iters[m] = it;
        if (host_iters) __hip_atomic_store(host_iters + m, it, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    const double c = t1 / t2;
    double2* D = (double2*)(D0 + poff[m]);
    const double2* D2 = (const double2*)(D20 + poff[m]);
    const double2* D3 = (const double2*)(D30 + poff[m]);
    const double x = c < 0.5 ? (1.0 - 2.0 * c) / (1.0 - c) : 0.0, r = c < 0.5 ? 1.0 / (1.0 - c) : 1.0 / c;
    const double y = (1.0 + c) * r;
    for (long k = (long)blockIdx.x * 256 + threadIdx.x; k < (long)ld * ld / 2; k += (long)gridDim.x * 256) {
        const double2 d = D[k], d2 = D2[k], d3 = D3[k];
        D[k] = make_double2(x * d.x + y * d2.x - r * d3.x, x * d.y + y * d2.y - r * d3.y);
    }
}

// E_m = W_m - W_m^T
__global__ void bantisym_kernel(const long* __restrict__ poff, const int* __restrict__ pld,
                                const int* __restrict__ skip, const double* __restrict__ W0, double* __restrict__ E0)
{
    const int m = blockIdx.y;
    if (skip && skip[m]) return;
    const int ld = pld[m];
    const double* W = W0 + poff[m];
    double* E = E0 + poff[m];
    for (long k = (long)blockIdx.x * blockDim.x + threadIdx.x; k < (long)ld * ld; k += (long)gridDim.x * blockDim.x) {
        const int i = (int)(k / ld), j = (int)(k - (long)i * ld);
        E[k] = W[k] - W[(long)j * ld + i];
    }
}

// dots[m * BMAX_DOTS + v] = <x_m, vecs[v]_m> for v < nvec[m]; vecs[v] at
// v * stride; partials then a finishing pass
__global__ __launch_bounds__(256) void bdot_part_kernel(const long* __restrict__ poff, const int* __restrict__ pld,
                                                        const int* __restrict__ skip, const int* __restrict__ nvec,
                                                        const double* __restrict__ x0, const double* __restrict__ vecs,
                                                        long stride, double* __restrict__ part)
{
    __shared__ double sh[256];
    const int m = blockIdx.y, p = blockIdx.x;
    if (skip && skip[m]) return;
    const int ld = pld[m];
    const double* x = x0 + poff[m];
    for (int v = 0; v < nvec[m]; v++) {
        const double* y = vecs + (long)v * stride + poff[m];
        double s = 0.0;
        for (long k = (long)p * 256 + threadIdx.x; k < (long)ld * ld; k += BPART * 256) s += x[k] * y[k];
        s = block_reduce(s, sh, [](double a, double b) { return a + b; });
        if (threadIdx.x == 0) part[((long)m * BPART + p) * BMAX_DOTS + v] = s;
    }
}

__global__ void bdot_fin_kernel(int nmol, const int* __restrict__ skip, const int* __restrict__ nvec,
                                const double* __restrict__ part, double* __restrict__ dots)
{
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= nmol || (skip && skip[m])) return;
    for (int v = 0; v < nvec[m]; v++) {
        double s = 0.0;
        for (int p = 0; p < BPART; p++) s += part[((long)m * BPART + p) * BMAX_DOTS + v];
        dots[m * BMAX_DOTS + v] = s;
    }
}

// F_m = sum_v coef[m, v] vecs[v]_m   (pscf/purif.c:629-635)
__global__ void blincomb_kernel(const long* __restrict__ poff, const int* __restrict__ pld,
                                const int* __restrict__ skip, const int* __restrict__ nvec,
                                const double* __restrict__ coef, const double* __restrict__ vecs, long stride,
                                double* __restrict__ F0)
{
    const int m = blockIdx.y;
    if (skip && skip[m]) return;
    const int ld = pld[m];
    const int nv = nvec[m];
    double* F = F0 + poff[m];
    for (long k = (long)blockIdx.x * blockDim.x + threadIdx.x; k < (long)ld * ld; k += (long)gridDim.x * blockDim.x) {
        double s = 0.0;
        for (int v = 0; v < nv; v++) s += coef[m * BMAX_DOTS + v] * vecs[(long)v * stride + poff[m] + k];
        F[k] = s;
    }
}

// F = H + G and E_m = sum_ij D_ij (H_ij + F_ij) on packed blocks
// (pscf/scf.c:80-102, 339): partials, then a finishing pass
__global__ __launch_bounds__(256) void bfe_part_kernel(const long* __restrict__ off, const int* __restrict__ nn,
                                                       const double* __restrict__ H0, const double* __restrict__ G0,
                                                       const double* __restrict__ D0, double* __restrict__ F0,
                                                       double* __restrict__ part)
{
    __shared__ double sh[256];
    const int m = blockIdx.y, p = blockIdx.x;
    const long nm = (long)nn[m] * nn[m];
    const double* H = H0 + off[m];
    const double* G = G0 + off[m];
    const double* D = D0 + off[m];
    double* F = F0 + off[m];
    double e = 0.0;
    for (long k = (long)p * 256 + threadIdx.x; k < nm; k += BPART * 256) {
        const double f = H[k] + G[k];
        F[k] = f;
        e += D[k] * (H[k] + f);
    }
    e = block_reduce(e, sh, [](double a, double b) { return a + b; });
    if (threadIdx.x == 0) part[(long)m * BPART + p] = e;
}

__global__ void bfe_fin_kernel(int nmol, const double* __restrict__ part, double* __restrict__ energy)
{
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= nmol) return;
    double e = 0.0;
    for (int p = 0; p < BPART; p++) e += part[(long)m * BPART + p];
    energy[m] = e;
}

// ---- launchers ----------------------------------------------------------------

static dim3 per_mol_grid(int maxelems, int nmol)
{
    return dim3((unsigned)std::max(1, std::min((maxelems + 255) / 256, 256)), (unsigned)nmol);
}

int gtf_bgemm(hipStream_t st, const BatchLayout& L, const int* skip, const int* done, const double* A,
              const double* B, double* C, int transB, const int* fp32)
{
    if (L.nmol <= 0) return 0;
    // the two A B^T kernels add in different orders, so each molecule takes the
    // one of its own size, whatever shares the batch
    int above = 0;
    if (transB && !fp32) {
        above = ROWS_MAX_LD;
        const int t = std::min(L.maxpld, ROWS_MAX_LD) / ROWS_T;
        bgemm_rows_kernel<<<dim3(t, t, L.nmol), ROWS_THREADS, 0, st>>>(L.poff, L.pld, skip, done, A, B, C);
        GTF_CHECK(hipGetLastError());
        if (L.maxpld <= ROWS_MAX_LD) return 0;
    }
    dim3 grid(L.maxpld / GEMM_GT, L.maxpld / GEMM_GT, L.nmol);
    if (transB) bgemm_kernel<1><<<grid, 256, 0, st>>>(L.poff, L.pld, skip, done, fp32, above, A, B, C);
    else bgemm_kernel<0><<<grid, 256, 0, st>>>(L.poff, L.pld, skip, done, fp32, above, A, B, C);
    GTF_CHECK(hipGetLastError());
    return 0;
}

int gtf_bpad(hipStream_t st, const BatchLayout& L, const int* skip, const double* packed, double* padded)
{
    bpad_kernel<<<per_mol_grid(L.maxpld * L.maxpld, L.nmol), 256, 0, st>>>(L.off, L.n, L.poff, L.pld, skip, packed,
                                                                          padded);
    GTF_CHECK(hipGetLastError());
    return 0;
}

int gtf_bunpad(hipStream_t st, const BatchLayout& L, const int* skip, const double* padded, double* packed)
{
    bunpad_kernel<<<per_mol_grid(L.maxn * L.maxn, L.nmol), 256, 0, st>>>(L.off, L.n, L.poff, L.pld, skip, padded,
                                                                       packed);
    GTF_CHECK(hipGetLastError());
    return 0;
}

int gtf_bpurif_init(hipStream_t st, const BatchLayout& L, const int* nocc, const int* skip, const double* F, double* D)
{
    bgersh_part_kernel<<<dim3(BPART, L.nmol), 256, 0, st>>>(L.poff, L.n, L.pld, skip, F, L.part);
    GTF_CHECK(hipGetLastError());
    bgersh_fin_kernel<<<(L.nmol + 63) / 64, 64, 0, st>>>(L.nmol, L.n, nocc, skip, L.part, L.coef);
    GTF_CHECK(hipGetLastError());
    bpurif_init_kernel<<<per_mol_grid(L.maxpld * L.maxpld, L.nmol), 256, 0, st>>>(L.poff, L.n, L.pld, skip, L.coef,
                                                                                F, D);
    GTF_CHECK(hipGetLastError());
    return 0;
}

int gtf_bpurif_stats(hipStream_t st, const BatchLayout& L, const int* skip, const double* D, const double* D2,
                     const double* D3, int* iters, double* stats, int it, double tol, int* fp32, double fp32_until,
                     int* low_iters)
{
    bstats_part_kernel<<<dim3(BPART, L.nmol), 256, 0, st>>>(L.poff, L.n, L.pld, skip, iters, D, D2, D3, L.part);
    GTF_CHECK(hipGetLastError());
    bstats_fin_kernel<<<(L.nmol + 63) / 64, 64, 0, st>>>(L.nmol, skip, L.part, iters, stats, it, tol, fp32,
                                                          fp32_until, low_iters);
    GTF_CHECK(hipGetLastError());
    return 0;
}

int gtf_bpurif_update(hipStream_t st, const BatchLayout& L, const int* skip, const int* iters, const double* stats,
                      double* D, const double* D2, const double* D3, int it, bool sym)
{
    if (sym)
        bpurif_update_sym_kernel<<<dim3(L.maxpld / ROWS_T, L.maxpld / ROWS_T, L.nmol), 256, 0, st>>>(
            L.poff, L.pld, skip, iters, stats, D, D2, D3, it);
    else
        bpurif_update_kernel<<<per_mol_grid(L.maxpld * L.maxpld, L.nmol), 256, 0, st>>>(L.poff, L.pld, skip, iters,
                                                                                      stats, D, D2, D3, it);
    GTF_CHECK(hipGetLastError());
    return 0;
}

size_t gtf_bpurif_part(int nmol, int maxpld) { return (size_t)nmol * tri_tiles(maxpld) * 3; }

int gtf_bpurif_iterate(hipStream_t st, const BatchLayout& L, const int* skip, int* iters, double* part, double tol,
                       double* D, double* D2, double* D3, int it, int* host_iters)
{
    const int mt = tri_tiles(L.maxpld);
    const dim3 grid(mt, L.nmol);
    bpurif_product_kernel<false><<<grid, ROWS_THREADS, 0, st>>>(L.poff, L.pld, skip, iters, D, D, D2, part, mt);
    GTF_CHECK(hipGetLastError());
    bpurif_product_kernel<true><<<grid, ROWS_THREADS, 0, st>>>(L.poff, L.pld, skip, iters, D, D2, D3, part, mt);
    GTF_CHECK(hipGetLastError());
    bpurif_step_kernel<<<per_mol_grid(L.maxpld * L.maxpld / 4, L.nmol), 256, 0, st>>>(L.poff, L.pld, skip, iters, part,
                                                                                     mt, tol, host_iters, D, D2, D3, it);
    GTF_CHECK(hipGetLastError());
    return 0;
}

int gtf_bantisym(hipStream_t st, const BatchLayout& L, const int* skip, const double* W, double* E)
{
    bantisym_kernel<<<per_mol_grid(L.maxpld * L.maxpld, L.nmol), 256, 0, st>>>(L.poff, L.pld, skip, W, E);
    GTF_CHECK(hipGetLastError());
    return 0;
}

int gtf_bmultidot(hipStream_t st, const BatchLayout& L, const int* skip, const int* nvec, const double* x,
                  const double* vecs, long stride, double* dots)
{
    bdot_part_kernel<<<dim3(BPART, L.nmol), 256, 0, st>>>(L.poff, L.pld, skip, nvec, x, vecs, stride, L.part);
    GTF_CHECK(hipGetLastError());
    bdot_fin_kernel<<<(L.nmol + 63) / 64, 64, 0, st>>>(L.nmol, skip, nvec, L.part, dots);
    GTF_CHECK(hipGetLastError());
    return 0;
}

int gtf_blincomb(hipStream_t st, const BatchLayout& L, const int* skip, const int* nvec, const double* coef,
                 const double* vecs, long stride, double* F)
{
    blincomb_kernel<<<per_mol_grid(L.maxpld * L.maxpld, L.nmol), 256, 0, st>>>(L.poff, L.pld, skip, nvec, coef, vecs,
                                                                             stride, F);
    GTF_CHECK(hipGetLastError());
    return 0;
}

int gtf_bfock_energy(hipStream_t st, const BatchLayout& L, const double* H, const double* G, const double* D,
                     double* F, double* energy)
{
    bfe_part_kernel<<<dim3(BPART, L.nmol), 256, 0, st>>>(L.off, L.n, H, G, D, F, L.part);
    GTF_CHECK(hipGetLastError());
    bfe_fin_kernel<<<(L.nmol + 63) / 64, 64, 0, st>>>(L.nmol, L.part, energy);
    GTF_CHECK(hipGetLastError());
    return 0;
}
