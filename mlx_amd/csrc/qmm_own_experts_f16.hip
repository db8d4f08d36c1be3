// qmm_own_experts_f16.hip -- qmm_own_experts.h for f16_t.
#include "qmm_own_experts.h"

namespace mlxrocm {

int launch_qmm_own_experts_f16(const QmmArgs& a, int gs, int bits, bool glu, hipStream_t s) {
  return glu ? own_experts<f16_t, true>(a, gs, bits, s) : own_experts<f16_t, false>(a, gs, bits, s);
}

} // namespace mlxrocm
