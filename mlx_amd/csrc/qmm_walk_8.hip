// qmm_walk_8.hip -- the kernel of qmm_walk.h for 8-bit codes.
#include "qmm_walk.h"

namespace mlxrocm {

int launch_walk_8(
    const WalkArgs& wa, const WalkPlan& pl, int gs, int dtype, int table_groups, const dim3& grid,
    hipStream_t s) {
  return launch_walk_bits<8>(wa, pl, gs, dtype, table_groups, grid, s);
}

} // namespace mlxrocm
