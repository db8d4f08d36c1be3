// qmm_mid.hip -- plan and launch of qmm_mid_kernel (qmm_mid.h).
#include "qmm_args.h"

namespace mlxrocm {

namespace {
constexpr int kStep = 128;  // codes of a K-step
constexpr int kTileN = 128; // rows of W of a tile
} // namespace

bool qmm_mid_supported(const QmmArgs& a, int gs, int bits, int dtype, bool transpose) {
  (void)gs;
  const uint64_t limit = uint64_t{1} << 32; // operands are addressed with 32-bit offsets
  return transpose && dtype != MLXROCM_FLOAT32 && a.L == 1 && a.lhs_indices == nullptr &&
      a.group_tiles == nullptr && a.w_alt == nullptr && a.K >= kStep && a.K % kStep == 0 &&
      static_cast<uint64_t>(a.M) * a.K * 2 < limit &&
      static_cast<uint64_t>(a.N) * a.K / 8 * bits < limit && a.M <= 65535 * 64;
}

// Rows of x are dealt out evenly over as few tiles as hold them.  K is cut into the
// number of ranges with the least time by this account (us): a workgroup starts and ends
// in 4 and takes 0.55 + 0.005 a row of its tile for a step; planes cost a launch, and
// are written and read once at about 3 TB/s.
MidPlan qmm_mid_plan(int M, int N, int K, int bits) {
  MidPlan pl{};
  const int most = bits == 8 ? 96 : 128; // (three stages of both operands in 160 KB)
  const int tiles = (M + most - 1) / most;
  pl.rows = ((M + tiles - 1) / tiles + 31) / 32 * 32;
  pl.rows = pl.rows < 64 ? 64 : pl.rows;
  pl.tiles = (M + pl.rows - 1) / pl.rows;
  const long cus = compute_units();
  pl.groups = static_cast<long>(pl.tiles) * ((N + kTileN - 1) / kTileN);
  const int steps = K / kStep;
  const double step = 0.55 + 0.005 * pl.rows;
  double best = 0.0;
  pl.splits = 1;
  for (int s = 1; s <= 16 && (s == 1 || s * 2 <= steps); ++s) {
    const long rounds = (pl.groups * s + cus - 1) / cus;
    double cost = rounds * (4.0 + ((steps + s - 1) / s) * step);
    if (s > 1) {
      cost += 2.5 + static_cast<double>(k_split_plane(M, N)) * s * 8.0 / 3e6;
    }
    if (s == 1 || cost < best) {
      best = cost;
      pl.splits = s;
    }
  }
  return pl;
}

int launch_qmm_mid(
    const QmmArgs& a, int gs, int bits, int dtype, const MidPlan& pl, hipStream_t s) {
  MLXROCM_REHEARSE("qmm_mid(rows=%d,tiles=%d,ksplit=%d)", pl.rows, pl.tiles, pl.splits);
  return dtype == MLXROCM_BFLOAT16 ? launch_qmm_mid_bf16(a, gs, bits, pl, s)
                                   : launch_qmm_mid_f16(a, gs, bits, pl, s);
}

} // namespace mlxrocm
