// Instances of the i8 MFMA GEMM kernels: 32-row tiles for grouped launches on prepared four-digit planes of B (int32
// weights), two depths per step: (4,4) (5,4).
#include "gemm_mfma_kernels.h"

namespace zk {

void mfma_instances_rows32d(std::vector<Instance> &out)
{
    out.push_back(make_instance<4, 4, kTileRows32, 16, 2, kUseGroupPlanes>());
    out.push_back(make_instance<5, 4, kTileRows32, 16, 2, kUseGroupPlanes>());
}

}  // namespace zk
