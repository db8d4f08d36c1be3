// qmm_own_f16.hip -- qmm_own_tiles.h for f16_t, affine codes.
#include "qmm_own_tiles.h"

namespace mlxrocm {

int launch_qmm_own_f16(const QmmArgs& a, int gs, int bits, const OwnPlan& pl, hipStream_t s) {
  return own_tiles_affine<f16_t>(a, gs, bits, pl, s);
}

} // namespace mlxrocm
