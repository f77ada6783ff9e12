// Instances of the i8 MFMA GEMM kernels: 64x64 tiles, two workgroups to a compute unit, for a short K: (4,3) (3,4) (4,4).
#include "gemm_mfma_kernels.h"

namespace zk {

void mfma_instances_short(std::vector<Instance> &out)
{
    out.push_back(make_short_instance<4, 3, 2>());
    out.push_back(make_short_instance<3, 4, 2>());
    out.push_back(make_short_instance<4, 4, 2>());
}

}  // namespace zk
