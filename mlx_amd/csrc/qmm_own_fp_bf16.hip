// qmm_own_fp_bf16.hip -- qmm_own_tiles.h for bf16_t, floating-point codes.
#include "qmm_own_tiles.h"

namespace mlxrocm {

int launch_qmm_own_fp_bf16(const QmmArgs& a, int mode, const OwnPlan& pl, hipStream_t s) {
  return own_tiles_fp<bf16_t>(a, mode, pl, s);
}

} // namespace mlxrocm
