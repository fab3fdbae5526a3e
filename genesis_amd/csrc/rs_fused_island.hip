// Fused substep kernels of models with 25 to 128 dofs and short constraint rows (island solver).
#include "rs_launch.h"

namespace rs {

void launch_fused_island(bool use_lds, dim3 grid, dim3 block, size_t lds, hipStream_t s, const DModel& m,
                         const DState& st, const FusedArgs& fa) {
    if (use_lds) hipLaunchKernelGGL((k_fused_large<true, 5>), grid, block, lds, s, FusedKernArgs{m, st, fa});
    else hipLaunchKernelGGL((k_fused_large<false, 5>), grid, block, lds, s, FusedKernArgs{m, st, fa});
}

}  // namespace rs
