// Split walker kernels for 2-D flames, double trajectories (counts: unsigned long long).
#include "walk_kernel.inc"

#include "split_kernel.inc"

namespace ffr {
int launch_split_f64u64_d2(const WalkLaunch &L)
{
    return launch_split<double, unsigned long long, 2>(L);
}
} // namespace ffr
