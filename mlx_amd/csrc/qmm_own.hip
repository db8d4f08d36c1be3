// qmm_own.hip -- when qmm_own_kernel (qmm_own.h) takes a call, and its launches.
#include "qmm_own.h"

namespace mlxrocm {

namespace {

constexpr uint64_t k32Bit = uint64_t{1} << 32;

// Whole steps of K; operands within the kernel's 32-bit byte offsets.
bool own_addresses(const QmmArgs& a, int bits) {
  return a.K % kOwnBK == 0 && a.K >= kOwnBK &&
      static_cast<uint64_t>(a.N) * a.K * bits / 8 < k32Bit;
}

} // namespace

// Ahead of the tile kernel wherever it can run and tiles are many, by its unpacking and by the rows that an
// expert's last tile has not got.  us per call of the gated MLP, start -> this kernel: 2048
// tokens to 2 of 8 experts, 4096 x 14336 4-bit 1498 -> 1377 (1300 tokens 1122 -> 930, 300
// tokens 511 -> 486, 700 at 8 bits 837 -> 841); 6 of 64, 2048 x 1408 4-bit, 2048 tokens 387
// -> 310, 8-bit 438 -> 382, 800 tokens 283 -> 264.
bool qmm_own_experts_supported(const QmmArgs& a, int bits) {
  // (x: the callers check it for every grouped kernel)
  return own_addresses(a, bits) && static_cast<uint64_t>(a.L) * a.N * 2 < kNoStore;
}

int launch_qmm_own_experts(
    const QmmArgs& a, int gs, int bits, int dtype, bool glu, hipStream_t s) {
  MLXROCM_REHEARSE("qmm_own_experts%s", glu ? "_glu" : "");
  return dtype == MLXROCM_BFLOAT16 ? launch_qmm_own_experts_bf16(a, gs, bits, glu, s)
                                   : launch_qmm_own_experts_f16(a, gs, bits, glu, s);
}

} // namespace mlxrocm
