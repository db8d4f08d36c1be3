// qmm_mfma_experts.hip -- the tile kernel on tiles of rows routed to one expert,
// with the pair image of scales and biases: the two launches of an expert-routed
// gated MLP (switch_glu.hip) where qmm_own_kernel does not take them (qmm_own.hip).
#include "qmm_mfma_tile.h"

namespace mlxrocm {

// Row tiles that a routing of `pairs` rows to `experts` makes: every expert ends
// on a partial tile, half of one on average.
int expected_tiles(int pairs, int experts) {
  return (pairs + kBM - 1) / kBM + experts / 2;
}

// h = silu(x W_gate^T) * (x W_up^T): a.w / a.scales the gate weights and their pair
// images, a.w_alt / a.scales_alt the up weights.  256-column tiles, 128 of each.
int launch_qmm_mfma_experts_glu(const QmmArgs& a, int gs, int bits, int dtype, hipStream_t s) {
  if (qmm_own_experts_supported(a, bits)) { // (K a multiple of 128)
    return launch_qmm_own_experts(a, gs, bits, dtype, true, 1, s);
  }
  constexpr int kNT = 8;
  MLXROCM_REHEARSE("qmm_t_tile_experts_glu(nt=%d)", kNT);
  const int gs_shift = shift_of(gs);
  const dim3 grid(
      (a.N + 16 * kNT - 1) / (16 * kNT), gather_group_max_tiles(a.L, a.n_experts, kGroupLargeTile), 1);
  auto run = [&](auto tval) -> int {
    using T = decltype(tval);
    return dispatch_bits(bits, [&](auto bval) {
      constexpr int B = decltype(bval)::value;
      return launch_variant<T, T, T, B, kNT, true, false, true, 0, true>(a, gs_shift, grid, s);
    });
  };
  return dtype == MLXROCM_BFLOAT16 ? run(bf16_t{}) : run(f16_t{});
}

int launch_qmm_mfma_experts(
    const QmmArgs& a, int gs, int bits, int dtype, void* planes, size_t room, hipStream_t s) {
  // Tiles of 256 columns that leave half of the compute units idle over a short K are behind
  // the narrower ones here: 2400 pairs of 32 experts, 1024 x 1024, whole call 82.8 us against 81.1.
  // So they are where both kernels have one round of tiles: this one's are 192 or 224 columns and
  // meet more units.  us of the product under a trace, own / here, 8 experts, 4096 x 14336: 1300
  // pairs 4-bit 366 / 327, 8-bit 420 / 359, 2000 pairs 340 / 307 and 379 / 334; 2900 pairs, a
  // second round here 356 / 505; 32 experts, 1024 x 1024, 5800 pairs 34 / 30 and 38 / 31.
  const int row_tiles = expected_tiles(a.L, a.n_experts);
  const long own_tiles = static_cast<long>(row_tiles) * ((a.N + 255) / 256);
  // the tile count is on the device: the width that suits the expected one
  const int nt = choose_nt(row_tiles * kBM, a.N, 1);
  const bool one_round = nt > 5 &&
      static_cast<long>(row_tiles) * ((a.N + 32 * nt - 1) / (32 * nt)) <= compute_units();
  if (qmm_own_experts_supported(a, bits) && (2 * own_tiles > compute_units() || a.K > 2048)) {
    const int splits = qmm_own_experts_splits(a, bits, room);
    if (splits > 1) {
      QmmArgs part = a;
      part.out = planes;
      const int rc = launch_qmm_own_experts(part, gs, bits, dtype, false, splits, s);
      return rc != MLXROCM_OK
          ? rc
          : reduce_grouped_planes(
                a, static_cast<const float*>(planes), splits, static_cast<int64_t>(a.L) * a.N,
                dtype, s);
    }
    if (!one_round) {
      return launch_qmm_own_experts(a, gs, bits, dtype, false, 1, s);
    }
  }
  const int gs_shift = shift_of(gs);
  MLXROCM_REHEARSE("qmm_t_tile_experts(nt=%d)", nt);
  const dim3 grid(
      (a.N + 32 * nt - 1) / (32 * nt), gather_group_max_tiles(a.L, a.n_experts, kGroupLargeTile), 1);
  auto run = [&](auto tval) -> int {
    using T = decltype(tval);
    return dispatch_bits(bits, [&](auto bval) {
      constexpr int B = decltype(bval)::value;
      switch (nt) {
        case 5:
          return launch_variant<T, T, T, B, 5, true, false, true>(a, gs_shift, grid, s);
        case 6:
          return launch_variant<T, T, T, B, 6, true, false, true>(a, gs_shift, grid, s);
        default:
          return launch_variant<T, T, T, B, 7, true, false, true>(a, gs_shift, grid, s);
      }
    });
  };
  return dtype == MLXROCM_BFLOAT16 ? run(bf16_t{}) : run(f16_t{});
}

} // namespace mlxrocm
