// qmm_own_experts.h -- qmm_own_kernel on tiles of rows routed to one expert: the launches
// of an expert-routed gated MLP (switch_glu.hip), one translation unit per element type.
#pragma once

#include "qmm_own.h"

namespace mlxrocm {

namespace {

// Tiles of the worst case: the count is on the device, workgroups without one exit.
template <typename T, typename TO, bool GLU>
int own_experts(const QmmArgs& a, int gs, int bits, int k_splits, hipStream_t s) {
  constexpr int kCols = GLU ? kOwnBN / 2 : kOwnBN;
  const long tiles = static_cast<long>((a.N + kCols - 1) / kCols) *
      gather_group_max_tiles(a.L, a.n_experts, kGroupLargeTile) * k_splits;
  return dispatch_bits(bits, [&](auto bval) {
    constexpr int B = decltype(bval)::value;
    return launch_own<T, TO, B, 0, 0, GLU>(a, own_group_shift(gs), tiles, s, k_splits);
  });
}

template <typename T>
int own_experts(const QmmArgs& a, int gs, int bits, bool glu, int k_splits, hipStream_t s) {
  return glu            ? own_experts<T, T, true>(a, gs, bits, 1, s)
      : k_splits > 1 ? own_experts<T, float, false>(a, gs, bits, k_splits, s)
                     : own_experts<T, T, false>(a, gs, bits, 1, s);
}

} // namespace

} // namespace mlxrocm
