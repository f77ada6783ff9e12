// Instances of the software-pipelined kernel for digit planes on both sides (gemm_mfma_pipe.h).
#include "gemm_mfma_kernels.h"
#include "gemm_mfma_pipe.h"

namespace zk {

template <int NA, int NB>
static PipeForm form()
{
    PipeForm f;
    f.fn = gemm_mfma_pipe_kernel<NA, NB>;
    if constexpr (pipe_wide(NA, NB)) f.finish = gemm_split_finish_kernel<2, 4, 2, 1>;
    else f.finish = gemm_split_finish_kernel<4, 2, 1, 1>;
    f.bn = pipe_wide(NA, NB) ? 128 : 64;
    f.lds = pipe_lds_bytes(NA, NB);
    return f;
}

PipeForm pipe_form(int na, int nb)
{
#define ZK_PIPE(NA_, NB_) if (na == NA_ && nb == NB_) return form<NA_, NB_>();
    ZK_PIPE_DIGITS(ZK_PIPE)
#undef ZK_PIPE
    return PipeForm{ nullptr, nullptr, 0, 0 };
}

}  // namespace zk
