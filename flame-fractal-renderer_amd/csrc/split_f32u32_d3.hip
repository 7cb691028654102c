// Split walker kernels for 3-D flames, float trajectories (counts: unsigned int).
#include "walk_kernel.inc"

#include "split_kernel.inc"

namespace ffr {
int launch_split_f32u32_d3(const WalkLaunch &L)
{
    return launch_split<float, unsigned int, 3>(L);
}
} // namespace ffr
