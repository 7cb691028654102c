// Split walker kernels for 2-D flames, float trajectories (counts: unsigned long long).
#include "walk_kernel.inc"

#include "split_kernel.inc"

namespace ffr {
int launch_split_f32u64_d2(const WalkLaunch &L)
{
    return launch_split<float, unsigned long long, 2>(L);
}
} // namespace ffr
