// Fused substep kernels of models with more than 24 dofs, private regions in memory. Where the Hessian is makes a kernel of
// its own, so that each holds one solver, inlined; the row update and the kinematics stay out of line. Box pile x1024, 4
// steps: 10.2 ms so, 10.9 with the solver and its line search out of line too (they then reach the Hessian in LDS by flat
// accesses), 12.1 with everything inlined, which spills 178 registers.
#define RS_LARGE_FN __attribute__((noinline)) inline
#include "rs_launch.h"

namespace rs {

void launch_fused_generic(bool use_lds, dim3 grid, dim3 block, size_t lds, hipStream_t s, const DModel& m,
                          const DState& st, const FusedArgs& fa) {
    if (use_lds) launch_fused_generic_lds(grid, block, lds, s, m, st, fa);
    else if (fa.h_off >= 0) hipLaunchKernelGGL((k_fused_large<false, 3>), grid, block, lds, s, FusedKernArgs{m, st, fa});
    else hipLaunchKernelGGL((k_fused_large<false, 0>), grid, block, lds, s, FusedKernArgs{m, st, fa});
}

}  // namespace rs
