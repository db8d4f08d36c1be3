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

// Which kernel takes the products of a routed gated MLP.  Both return the same bits at 4 and 8
// bits.  us of the whole call, both products on the tile kernel (tiles in the order of their
// experts) / here, 8 experts, 4096 x 14336: 4-bit 2048 tokens to 2 1487 / 1361, 343 tokens 548 /
// 432; 8-bit 343 tokens 569 / 501; 64 experts 2048 x 1408, 4-bit, 2000 tokens to 6 402 / 329.
//
// The last product stays on the tile kernel in one round of tiles without ranges of K: its tiles
// are 160..224 columns and meet more units.  % of the call, own against it, by rows per expert: 8
// experts 4096 x 14336, 4-bit 132 +14, 175 +6, 276 +3 (a second round from 280 on: -9), 8-bit 135
// +13, 218 +8; 16 experts 2048 x 4096 4-bit 98 +11, 8-bit 155 +13; 32 experts 1024 x 1024 4-bit
// 105 +7, 8-bit 79 +10.
//
// 8-bit codes that are put in order leave nothing to gain in the first products (-3..+3 %); over
// experts of more than 16 MB (gather_tiles_by_height) the tile kernel gains from tiles in the
// order of their experts, so it takes all three unless the last one is ahead here (up to a round
// of tiles and from nearly two on): 8 experts 4096 x 14336, 886 tokens 845 / 897 with the first
// ones here, 1868 tokens 1462 / 1563 and 2414 tokens 1833 / 2009 with all, 3482 tokens 2578 / 2472.
ExpertsPlan qmm_experts_plan(const QmmArgs& in, const QmmArgs& out, int bits, size_t room) {
  ExpertsPlan pl{qmm_own_experts_supported(in, bits), false, 1}; // (K a multiple of 128)
  const long cus = compute_units();
  const int row_tiles = expected_tiles(out.L, out.n_experts);
  const long own_tiles = static_cast<long>(row_tiles) * ((out.N + 255) / 256);
  const int nt = choose_nt(row_tiles * kBM, out.N, 1);
  const bool one_round = static_cast<long>(row_tiles) * ((out.N + 32 * nt - 1) / (32 * nt)) <= cus;
  // (half of the units idle over a short K: 2400 pairs of 32 experts, 1024 x 1024, 82.8 / 81.1)
  if (qmm_own_experts_supported(out, bits) && (2 * own_tiles > cus || out.K > 2048)) {
    pl.splits = qmm_own_experts_splits(out, bits, room);
    pl.own_second = pl.splits > 1 || !one_round;
  }
  if (bits == 8 && !gather_tiles_by_height(out.N, out.K, bits) && pl.splits <= 1 &&
      (!pl.own_second || (16 * own_tiles > 17 * cus && 4 * own_tiles < 7 * cus))) {
    pl.own_first = pl.own_second = false;
  }
  return pl;
}

// h = silu(x W_gate^T) * (x W_up^T): a.w / a.scales the gate weights and their pair
// images, a.w_alt / a.scales_alt the up weights.  256-column tiles, 128 of each.
int launch_qmm_mfma_experts_glu(
    const QmmArgs& a, int gs, int bits, int dtype, const ExpertsPlan& pl, hipStream_t s) {
  if (pl.own_first) {
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
    const QmmArgs& a, int gs, int bits, int dtype, const ExpertsPlan& pl, void* planes,
    hipStream_t s) {
  if (pl.own_second && pl.splits <= 1) {
    return launch_qmm_own_experts(a, gs, bits, dtype, false, 1, s);
  }
  if (pl.own_second) {
    QmmArgs part = a;
    part.out = planes;
    const int rc = launch_qmm_own_experts(part, gs, bits, dtype, false, pl.splits, s);
    return rc != MLXROCM_OK
        ? rc
        : reduce_grouped_planes(
              a, static_cast<const float*>(planes), pl.splits, static_cast<int64_t>(a.L) * a.N,
              dtype, s);
  }
  const int gs_shift = shift_of(gs);
  // the tile count is on the device: the width that suits the expected one
  const int nt = choose_nt(expected_tiles(a.L, a.n_experts) * kBM, a.N, 1);
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
