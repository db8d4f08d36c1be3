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

namespace {

// us a K-step: a tile of up to 96 rows, of 128 (8-bit codes have tiles of 64 and 96).  Odd
// widths cost more to unpack than 4 and 8 bits.
double step_us(int bits, int rows) {
  const bool tall = bits == 8 ? rows > 64 : rows > 96;
  switch (bits) {
    case 2:
      return tall ? 1.11 : 1.19;
    case 3:
      return tall ? 1.37 : 1.23;
    case 4:
      return tall ? 1.11 : 1.02;
    case 5:
      return tall ? 1.42 : 1.30;
    case 6:
      return tall ? 1.46 : 1.35;
    default:
      return tall ? 0.92 : 0.80;
  }
}

} // namespace

// Rows of x are dealt out evenly over as few tiles as hold them.  K is cut into the
// number of ranges with the least time by this account (us), fitted to 14500 calls of
// 65..2048 rows at every width and group size, each in several numbers of ranges (errors of
// 4 %): a launch and the rounds of workgroups, with 2.4 for each further filling of the
// table; then the planes and the launch that adds them up, or results stored by the
// workgroups themselves (by the element where N is no multiple of four).
MidPlan qmm_mid_plan(int M, int N, int K, int gs, int bits) {
  MidPlan pl{};
  const int most = bits == 8 ? 96 : 128; // (three stages of both operands in 160 KB)
  const int tiles = (M + most - 1) / most;
  pl.rows = ((M + tiles - 1) / tiles + 31) / 32 * 32;
  pl.rows = pl.rows < 64 ? 64 : pl.rows;
  pl.tiles = (M + pl.rows - 1) / pl.rows;
  const long cus = compute_units();
  pl.groups = static_cast<long>(pl.tiles) * ((N + kTileN - 1) / kTileN);
  const int steps = K / kStep;
  const int mf = pl.rows <= 64 ? 4 : pl.rows <= 96 ? 6 : 8; // as mid_launch() has it
  const int segment = mid_table_groups(mf, bits) * gs / kStep;
  const double step = step_us(bits, pl.rows);
  const double results = 1e-6 * static_cast<double>(k_split_plane(M, N));
  // (ranges of two steps at least; below 768 codes they gain nothing)
  const int ranges = steps < 6 ? 1 : steps < 32 ? steps / 2 : 16;
  pl.splits = 1;
  for (int s = 1; s <= ranges; ++s) {
    const long rounds = (pl.groups * s + cus - 1) / cus;
    const int each = (steps + s - 1) / s;
    const int fillings = (each + segment - 1) / segment;
    const double us = 3.5 + static_cast<double>(rounds) * (0.35 + each * step + 2.4 * (fillings - 1)) +
        (s > 1 ? 2.1 + 0.31 * s + (1.8 * s + 1.4) * results
               : 1.7 * results + (N % 4 != 0 ? 2.6 : 0.0));
    if (s == 1 || us < pl.us) {
      pl.us = us;
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
