// qmm_walk_6.hip -- the kernel of qmm_walk.h for 6-bit codes.
#include "qmm_walk.h"

namespace mlxrocm {

int launch_walk_6(
    const WalkArgs& wa, const WalkPlan& pl, int gs, int dtype, int table_groups, const dim3& grid,
    hipStream_t s) {
  return launch_walk_bits<6>(wa, pl, gs, dtype, table_groups, grid, s);
}

} // namespace mlxrocm
