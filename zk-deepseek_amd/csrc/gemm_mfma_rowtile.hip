// Instances of the kernel for many rows against the digit planes of a small B (gemm_mfma_rowtile.h).
#include "gemm_mfma_rowtile.h"

namespace zk {

RowtileForm rowtile_form(int na, int nb)
{
#define ZK_ROWTILE(NA_, NB_) \
    if (na == NA_ && nb == NB_) return RowtileForm{ gemm_mfma_rowtile_kernel<NA_, NB_>, rowtile_cols(NA_, NB_), rowtile_lds_bytes(NA_, NB_) };
    ZK_PIPE_DIGITS(ZK_ROWTILE)
#undef ZK_ROWTILE
    return RowtileForm{ nullptr, 0, 0 };
}

}  // namespace zk
