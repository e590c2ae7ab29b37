// eri_class.hip -- instantiates part GTF_PART of the ERI kernels of quartet
// class GTF_CLASS: 0 the unit kernels, 1 the FP64 tile kernels, 2 the FP32
// tile kernels (one object each, so the heavy instantiations compile in
// parallel).
#include "eri_kernels.h"

namespace {
constexpr int CLS = GTF_CLASS;
constexpr int bra_type()
{
    int A = 0;
    while ((A + 1) * (A + 2) / 2 <= CLS) ++A;
    return A;
}
constexpr int A = bra_type(), B = CLS - A * (A + 1) / 2;
constexpr int TYPE_A[GTF_NPAIRTYPES] = {0, 1, 1, 2, 2, 2}, TYPE_B[GTF_NPAIRTYPES] = {0, 0, 1, 0, 1, 2};
constexpr int LA = TYPE_A[A], LB = TYPE_B[A], LC = TYPE_A[B], LD = TYPE_B[B];
using S = EriShape<LA, LB, LC, LD>;
constexpr int NC = default_nc<LA, LB, LC, LD>();
constexpr int NT = tile_nc<LA, LB, LC, LD>();
// the exchanged contraction, for the classes whose bra pair is large beside
// the ket pair
constexpr bool EXCHANGED = A != B && (A >= 4 || S::NAB * S::NCD >= 27);
constexpr int NCT = tile_nct<LA, LB, LC, LD>();
}  // namespace

#define GTF_CAT4(a, b, c, d) a##b##c##d
#define GTF_NAME(c, p) GTF_CAT4(gtf_eri_register_, c, _, p)
void GTF_NAME(GTF_CLASS, GTF_PART)(EriClassInfo& e)
{
#if GTF_PART == 0
    e.la = LA; e.lb = LB; e.lc = LC; e.ld = LD;
    e.nc = NC;
    e.nsplit = S::NAB / NC;
    e.nints = S::NAB * S::NCD;
    e.tile_threads = tile_threads<LA, LB, LC, LD>();
    e.nc_tile = NT;
    e.comp_lanes = tile_static(S::NAB, NT) ? 0 : comp_lanes<LA, LB, LC, LD>();
    e.nsplit_tile = (S::NAB + (NT << e.comp_lanes) - 1) / (NT << e.comp_lanes);
    e.full_E = !tile_static(S::NAB, NT);
    e.nc_t = EXCHANGED ? NCT : 0;
    e.nsplit_t = EXCHANGED ? (S::NCD + NCT - 1) / NCT : 0;
    e.jk = eri_kernel<LA, LB, LC, LD, NC, EPI_JK>;
    e.store = eri_kernel<LA, LB, LC, LD, NC, EPI_STORE>;
    if constexpr (A == B) e.diag = eri_kernel<LA, LB, LC, LD, NC, EPI_DIAG>;
#elif GTF_PART == 1
    e.jk_tile[0] = eri_jk_tile_kernel<LA, LB, LC, LD, NT, double, false>;
    e.jk_tile[1] = eri_jk_tile_kernel<LA, LB, LC, LD, NT, double, true>;
    if constexpr (EXCHANGED) {
        e.jk_tile_t[0] = eri_jk_tile_t_kernel<LA, LB, LC, LD, NCT, double, false>;
        e.jk_tile_t[1] = eri_jk_tile_t_kernel<LA, LB, LC, LD, NCT, double, true>;
    }
#else
    e.jk_tile_lo = eri_jk_tile_kernel<LA, LB, LC, LD, NT, float, false>;
    if constexpr (EXCHANGED) e.jk_tile_t_lo = eri_jk_tile_t_kernel<LA, LB, LC, LD, NCT, float, false>;
#endif
}
