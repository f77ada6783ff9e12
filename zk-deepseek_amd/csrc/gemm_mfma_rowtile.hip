// Instances of the kernel for many rows against the digit planes of a small B (gemm_mfma_rowtile.h).
#include "gemm_mfma_rowtile.h"

namespace zk {

RowtileForm rowtile_form(int na, int nb)
{
#define ZK_ROWTILE(NA_, NB_) \
    if (na == NA_ && nb == NB_) return RowtileForm{ gemm_mfma_rowtile_kernel<NA_, NB_>, rowtile_cols(NA_, NB_), rowtile_lds_bytes(NA_, NB_) }
    ZK_ROWTILE(3, 3);
    ZK_ROWTILE(3, 4);
    ZK_ROWTILE(4, 3);
    ZK_ROWTILE(4, 4);
    ZK_ROWTILE(3, 5);
    ZK_ROWTILE(6, 3);
    ZK_ROWTILE(5, 4);
    ZK_ROWTILE(4, 5);
    ZK_ROWTILE(5, 5);
#undef ZK_ROWTILE
    return RowtileForm{ nullptr, 0, 0 };
}

}  // namespace zk
