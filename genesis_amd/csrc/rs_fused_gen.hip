// Fused substep kernel of models with more than 24 dofs, private regions in memory. The solver's functions stay out of
// line: inlined into the kernel they share its registers with everything else and spill (880 B of scratch per lane), box
// pile x1024, 4 steps: 10.9 ms out of line, 12.1 ms inlined.
#define RS_LARGE_FN __attribute__((noinline)) inline
#include "rs_launch.h"

namespace rs {

void launch_fused_generic(bool use_lds, dim3 grid, dim3 block, size_t lds, hipStream_t s, const DModel& m,
                          const DState& st, const FusedArgs& fa) {
    if (use_lds) launch_fused_generic_lds(grid, block, lds, s, m, st, fa);
    else hipLaunchKernelGGL((k_fused_large<false, 0>), grid, block, lds, s, FusedKernArgs{m, st, fa});
}

}  // namespace rs
