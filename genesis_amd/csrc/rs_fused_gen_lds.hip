// Fused substep kernel of models with more than 24 dofs whose private regions fit in LDS (up to about 50 dofs). Everything
// is inlined: a function called out of line reaches the region by flat accesses instead of LDS ones.
#define RS_LARGE_FN __forceinline__
#include "rs_launch.h"

namespace rs {

void launch_fused_generic_lds(dim3 grid, dim3 block, size_t lds, hipStream_t s, const DModel& m, const DState& st,
                              const FusedArgs& fa) {
    hipLaunchKernelGGL((k_fused_large<true, 0>), grid, block, lds, s, FusedKernArgs{m, st, fa});
}

}  // namespace rs
