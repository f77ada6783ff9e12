// Instances of the i8 MFMA GEMM kernels: planes on both sides (weights prepared once), one depth per step: the digit counts of
// which the unprepared kernels have two depths per step.  (The pipelined kernel has every one of these pairs and is what runs;
// these are its dimensions and plane layouts, and the kernels that ZK_NO_PIPE puts in its place.)
#include "gemm_mfma_kernels.h"

namespace zk {

void mfma_instances_both(std::vector<Instance> &out)
{
    out.push_back(make_instance<4, 3, kTileAuto, 16, 1, kUsePlanesBoth>());
    out.push_back(make_instance<6, 3, kTileAuto, 16, 1, kUsePlanesBoth>());
    out.push_back(make_instance<3, 4, kTileAuto, 16, 1, kUsePlanesBoth>());
    out.push_back(make_instance<4, 4, kTileAuto, 16, 1, kUsePlanesBoth>());
    out.push_back(make_instance<5, 4, kTileAuto, 16, 1, kUsePlanesBoth>());
    out.push_back(make_instance<3, 5, kTileAuto, 16, 1, kUsePlanesBoth>());
    out.push_back(make_instance<4, 5, kTileAuto, 16, 1, kUsePlanesBoth>());
    out.push_back(make_instance<5, 5, kTileAuto, 16, 1, kUsePlanesBoth>());
}

}  // namespace zk
