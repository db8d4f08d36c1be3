// qmm_walk_fp.hip -- the kernel of qmm_walk.h for the floating-point modes.
#include "qmm_walk.h"

namespace mlxrocm {

namespace {

template <typename T>
int launch_mode(
    const WalkArgs& wa, const WalkPlan& pl, int mode, int table_groups, const dim3& grid,
    hipStream_t s) {
  switch (mode) {
    case MLXROCM_MXFP4:
      return launch_walk_rows<T, 4, 32, 1>(wa, pl, table_groups, grid, s);
    case MLXROCM_MXFP8:
      return launch_walk_rows<T, 8, 32, 2>(wa, pl, table_groups, grid, s);
    default:
      return launch_walk_rows<T, 4, 16, 3>(wa, pl, table_groups, grid, s);
  }
}

} // namespace

int launch_walk_fp(
    const WalkArgs& wa, const WalkPlan& pl, int mode, int dtype, int table_groups, const dim3& grid,
    hipStream_t s) {
  return dtype == MLXROCM_BFLOAT16 ? launch_mode<bf16_t>(wa, pl, mode, table_groups, grid, s)
                                   : launch_mode<f16_t>(wa, pl, mode, table_groups, grid, s);
}

} // namespace mlxrocm
