// qmm_own_fp_f16.hip -- qmm_own_tiles.h for f16_t, floating-point codes.
#include "qmm_own_tiles.h"

namespace mlxrocm {

int launch_qmm_own_fp_f16(const QmmArgs& a, int mode, const OwnPlan& pl, hipStream_t s) {
  return own_tiles_fp<f16_t>(a, mode, pl, s);
}

} // namespace mlxrocm
