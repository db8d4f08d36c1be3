// qmm_own_experts.h -- qmm_own_kernel on tiles of rows routed to one expert: the two launches
// of an expert-routed gated MLP (switch_glu.hip), one translation unit per element type.
#pragma once

#include "qmm_own.h"

namespace mlxrocm {

namespace {

// Tiles of the worst case: the count is on the device, workgroups without one exit.
template <typename T, bool GLU>
int own_experts(const QmmArgs& a, int gs, int bits, hipStream_t s) {
  constexpr int kCols = GLU ? kOwnBN / 2 : kOwnBN;
  const long tiles = static_cast<long>((a.N + kCols - 1) / kCols) *
      gather_group_max_tiles(a.L, a.n_experts, kGroupLargeTile);
  return dispatch_bits(bits, [&](auto bval) {
    constexpr int B = decltype(bval)::value;
    return launch_own<T, T, B, 0, 0, GLU>(a, own_group_shift(gs), tiles, s);
  });
}

} // namespace

} // namespace mlxrocm
