// qmm_own_experts_f16.hip -- qmm_own_experts.h for f16_t.
#include "qmm_own_experts.h"

namespace mlxrocm {

int launch_qmm_own_experts_f16(
    const QmmArgs& a, int gs, int bits, bool glu, int k_splits, hipStream_t s) {
  return own_experts<f16_t>(a, gs, bits, glu, k_splits, s);
}

} // namespace mlxrocm
