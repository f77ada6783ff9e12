// Instances of the i8 MFMA GEMM kernels: (3,3) on 128x128 tiles and, for launches smaller than the device, on 128x64 ones;
// (4,3) (3,4) (4,4) (5,4) on 128x64 tiles.
#include "gemm_mfma_kernels.h"

namespace zk {

void mfma_instances_narrow(std::vector<Instance> &out)
{
    out.push_back(make_instance<3, 3>());
    out.push_back(make_instance<3, 3, kTile128x64, 16, 2>());
    out.push_back(make_instance<4, 3, kTileAuto, 16, 2>());
    out.push_back(make_instance<3, 4, kTileAuto, 16, 2>());
    out.push_back(make_instance<4, 4, kTileAuto, 16, 2>());
    out.push_back(make_instance<5, 4, kTileAuto, 16, 2>());
}

}  // namespace zk
