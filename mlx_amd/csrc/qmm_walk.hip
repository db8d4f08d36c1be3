// qmm_walk.hip -- which launches of the kernel of qmm_walk.h cover a call, and the
// launch itself.
#include "qmm_walk.h"

namespace mlxrocm {

namespace {

constexpr size_t kWalkLds = 160 * 1024;

int walk_rows(int M) {
  return M <= 8 ? 8 : (M + 15) / 16 * 16;
}

int stage_codes(int config) {
  return kWalkConfigs[config].k_waves * kWkChunk;
}

int walk_table_groups(const WalkPlan& pl, int K, int gs) {
  const long in_range = static_cast<long>(pl.range) * stage_codes(pl.config) / gs;
  return in_range < K / gs ? static_cast<int>(in_range) : K / gs;
}

// (floating-point modes: scales only)
size_t walk_lds(const WalkPlan& pl, int K, int gs, bool fp) {
  const WalkConfig& c = kWalkConfigs[pl.config];
  const size_t stages = size_t(4) * c.k_waves * pl.mr * kWkChunk;
  const size_t sums = size_t(1024) * c.k_waves * c.tiles * ((pl.mr + 15) / 16);
  const size_t tables =
      static_cast<size_t>(walk_table_groups(pl, K, gs)) * c.tiles * (fp ? 64 : 128);
  return tables + (stages > sums ? stages : sums);
}

WalkPlan walk_plan(const QmmArgs& a, int gs, int bits, bool fp) {
  WalkPlan pl{};
  pl.mr = walk_rows(a.M);
  const long cus = compute_units();
  const long rows = static_cast<long>(a.N) * a.L;
  const long per_cu = (rows + cus - 1) / cus;
  const bool wide = bits == 8; // registers: half as many stages ahead
  if (pl.mr == 8) {
    pl.config = per_cu <= 16 ? 0 : per_cu <= 32 ? 2 : 3;
  } else if (pl.mr == 16) {
    pl.config = per_cu <= 16 ? 0 : per_cu <= 32 || wide ? 2 : 1;
  } else if (pl.mr == 32) {
    pl.config = per_cu <= 16 && a.K < 8192 ? 0 : 1;
  } else {
    pl.config = 1;
  }
  // many rows of x against few of W per unit: K in ranges, so that a unit multiplies
  // a range of x by up to 64 rows of W instead of the whole of x by a few
  int splits = 1;
  if (pl.mr >= 32 && pl.config == 1 && per_cu <= 32) {
    const long blocks = (rows + 63) / 64;
    splits = static_cast<int>(cus / blocks < 4 ? cus / blocks : 4);
  }
  const int tiles = kWalkConfigs[pl.config].tiles;
  const int stages = (a.K + stage_codes(pl.config) - 1) / stage_codes(pl.config);
  for (;; ++splits) {
    const long most = 16 * tiles;
    const long units = (cus + splits - 1) / splits;
    const long rounds = (rows + units * most - 1) / (units * most);
    pl.tile_rows = static_cast<int>((rows + units * rounds * tiles - 1) / (units * rounds * tiles));
    pl.range = (stages + splits - 1) / splits;
    pl.splits = (stages + pl.range - 1) / pl.range;
    if (splits >= stages || walk_lds(pl, a.K, gs, fp) <= kWalkLds) {
      return pl;
    }
  }
}

} // namespace

namespace {

bool walk_fits(const QmmArgs& a, int gs, int bits, int dtype, bool transpose, bool fp) {
  const uint64_t limit = uint64_t{1} << 32; // operands are addressed by 32-bit byte offsets
  if (!transpose || dtype == MLXROCM_FLOAT32 || a.M < 1 || a.M > 64 || a.K % 32 != 0 || a.K < 128 ||
      a.group_tiles != nullptr || a.L > 65535 ||
      static_cast<uint64_t>(a.N) * a.K / 8 * bits >= limit ||
      static_cast<uint64_t>(a.M) * a.K * 2 >= limit) {
    return false;
  }
  const WalkPlan pl = walk_plan(a, gs, bits, fp);
  return walk_lds(pl, a.K, gs, fp) <= kWalkLds &&
      (pl.splits == 1 || (static_cast<int64_t>(a.L) * a.M * a.N) % 4 == 0);
}

size_t walk_planes(const QmmArgs& a, const WalkPlan& pl) {
  return pl.splits > 1 ? static_cast<size_t>(pl.splits) * a.L * a.M * a.N * sizeof(float) : 0;
}

constexpr int kFpGroup = 32; // codes per entry of the scale table
int fp_bits(int mode) {
  return mode == MLXROCM_MXFP8 ? 8 : 4;
}

} // namespace

bool qmm_walk_supported(const QmmArgs& a, int gs, int bits, int dtype, bool transpose) {
  return walk_fits(a, gs, bits, dtype, transpose, false);
}

size_t qmm_walk_plane_bytes(const QmmArgs& a, int gs, int bits) {
  return walk_planes(a, walk_plan(a, gs, bits, false));
}

bool qmm_walk_fp_supported(const QmmArgs& a, int mode, int dtype) {
  return a.K % kWkChunk == 0 && walk_fits(a, kFpGroup, fp_bits(mode), dtype, true, true);
}

size_t qmm_walk_fp_plane_bytes(const QmmArgs& a, int mode) {
  return walk_planes(a, walk_plan(a, kFpGroup, fp_bits(mode), true));
}

namespace {

int walk_launch(
    const QmmArgs& a, const WalkPlan& pl, WalkLauncher* launcher, int gs, int dtype, int groups,
    bool glu, void* planes, hipStream_t s) {
  WalkArgs wa{};
  wa.a = a;
  wa.tile_rows = pl.tile_rows;
  wa.range = pl.range;
  wa.glu = glu;
  wa.planes = static_cast<float*>(planes);
  const int rows = kWalkConfigs[pl.config].tiles * pl.tile_rows / (glu ? 2 : 1);
  const dim3 grid(static_cast<unsigned>((a.N + rows - 1) / rows), pl.splits, a.L);
  const int rc = launcher(wa, pl, gs, dtype, groups, grid, s);
  if (rc != MLXROCM_OK || pl.splits == 1) {
    return rc;
  }
  return reduce_planes(
      static_cast<const float*>(planes), a.out, static_cast<size_t>(a.L) * a.M * a.N, pl.splits,
      dtype, s);
}

WalkLauncher* walk_launcher(int bits) {
  switch (bits) {
    case 2:
      return launch_walk_2;
    case 3:
      return launch_walk_3;
    case 4:
      return launch_walk_4;
    case 5:
      return launch_walk_5;
    case 6:
      return launch_walk_6;
    default:
      return launch_walk_8;
  }
}

} // namespace

int launch_qmm_walk(const QmmArgs& a, int gs, int bits, int dtype, void* planes, hipStream_t s) {
  const WalkPlan pl = walk_plan(a, gs, bits, false);
  MLXROCM_REHEARSE(
      "qmm_walk(config=%d,rows=%d,tile=%d,splits=%d)", pl.config, pl.mr, pl.tile_rows, pl.splits);
  return walk_launch(
      a, pl, walk_launcher(bits), gs, dtype, walk_table_groups(pl, a.K, gs), false, planes, s);
}

int launch_qmm_walk_fp(const QmmArgs& a, int mode, int dtype, void* planes, hipStream_t s) {
  const WalkPlan pl = walk_plan(a, kFpGroup, fp_bits(mode), true);
  MLXROCM_REHEARSE(
      "qmm_walk_fp(config=%d,rows=%d,tile=%d,splits=%d)", pl.config, pl.mr, pl.tile_rows,
      pl.splits);
  return walk_launch(
      a, pl, launch_walk_fp, mode, dtype, walk_table_groups(pl, a.K, kFpGroup), false, planes,
      s);
}

// `a`: one problem (L = 1) with w_alt, scales_alt, biases_alt
bool qmm_walk_glu_supported(const QmmArgs& a, int gs, int bits, int dtype) {
  QmmArgs both = a;
  both.L = 2;
  const WalkPlan pl = walk_plan(both, gs, bits, false);
  return qmm_walk_supported(both, gs, bits, dtype, true) && pl.config != 0 && pl.splits == 1;
}

int launch_qmm_walk_glu(const QmmArgs& a, int gs, int bits, int dtype, hipStream_t s) {
  QmmArgs both = a;
  both.L = 2;
  const WalkPlan pl = walk_plan(both, gs, bits, false);
  MLXROCM_REHEARSE("qmm_walk_glu(config=%d,rows=%d,tile=%d)", pl.config, pl.mr, pl.tile_rows);
  return walk_launch(
      a, pl, walk_launcher(bits), gs, dtype, walk_table_groups(pl, a.K, gs), true, nullptr, s);
}

} // namespace mlxrocm
