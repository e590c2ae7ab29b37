// eri_table.cpp -- the class table of ERI kernels (filled once).
#include "eri_kernels.h"

#define GTF_EACH_CLASS(X) \
    X(0) X(1) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12) X(13) X(14) X(15) X(16) X(17) X(18) X(19) X(20)

#define GTF_DECLARE(c)                            \
    void gtf_eri_register_##c##_0(EriClassInfo&); \
    void gtf_eri_register_##c##_1(EriClassInfo&); \
    void gtf_eri_register_##c##_2(EriClassInfo&);
GTF_EACH_CLASS(GTF_DECLARE)

namespace {
struct EriTable {
    EriClassInfo tab[GTF_NCLASSES] = {};
    EriTable()
    {
#define GTF_FILL(c)                       \
    gtf_eri_register_##c##_0(tab[c]);     \
    gtf_eri_register_##c##_1(tab[c]);     \
    gtf_eri_register_##c##_2(tab[c]);
        GTF_EACH_CLASS(GTF_FILL)
    }
};
}  // namespace

const EriClassInfo* gtf_eri_class(int cls)
{
    // filled once, thread-safely (several batches may start at the same time)
    static const EriTable t;
    return (cls >= 0 && cls < GTF_NCLASSES) ? &t.tab[cls] : nullptr;
}
