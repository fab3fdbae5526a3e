// Shared launch of several models of any size, private regions in memory (row update and kinematics out of line as in
// rs_fused_gen.hip).
#define RS_LARGE_FN __attribute__((noinline)) inline
#include "rs_launch.h"

namespace rs {

void launch_fused_multi_any(dim3 grid, dim3 block, size_t lds, hipStream_t s, const FusedSegment* segs, int n_segs) {
    hipLaunchKernelGGL((k_fused_multi<false, true>), grid, block, lds, s, segs, n_segs);
}

}  // namespace rs
