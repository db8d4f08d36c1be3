// qmm_mid_bf16.hip -- qmm_mid_kernel for bfloat16, every width.
#include "qmm_mid.h"

namespace mlxrocm {

int launch_qmm_mid_bf16(const QmmArgs& a, int gs, int bits, const MidPlan& pl, hipStream_t s) {
  return mid_launch<bf16_t>(a, gs, bits, pl, s);
}

} // namespace mlxrocm
