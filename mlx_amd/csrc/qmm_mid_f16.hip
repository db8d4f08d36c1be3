// qmm_mid_f16.hip -- qmm_mid_kernel for float16, every width.
#include "qmm_mid.h"

namespace mlxrocm {

int launch_qmm_mid_f16(const QmmArgs& a, int gs, int bits, const MidPlan& pl, hipStream_t s) {
  return mid_launch<f16_t>(a, gs, bits, pl, s);
}

} // namespace mlxrocm
