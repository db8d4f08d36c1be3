// qmm_own.hip -- when qmm_own_kernel (qmm_own.h) takes a call, and its launches.
#include "qmm_own.h"

namespace mlxrocm {

namespace {

constexpr uint64_t k32Bit = uint64_t{1} << 32;

// Whole steps of K; operands within the kernel's 32-bit byte offsets.
bool own_addresses(int N, int K, int bits) {
  return K % kOwnBK == 0 && K >= kOwnBK && static_cast<uint64_t>(N) * K * bits / 8 < k32Bit;
}

// us of a step of 128 codes: fixed + 16-row blocks of the tile * (each + busy * share of the
// compute units at work, by which the clock gives way).
struct Step {
  double fixed, each, busy;
};
constexpr Step kSteps[] = {
    {0.73, 0.0845, 0.0263}, // 2-bit
    {0.77, 0.0876, 0.0326}, // 3-bit
    {0.62, 0.0817, 0.0398}, // 4-bit
    {1.13, 0.0851, 0.0215}, // 5-bit
    {1.16, 0.0830, 0.0229}, // 6-bit
    {1.11, 0.0652, 0.0287}, // 8-bit
    {0.59, 0.0720, 0.0337}, // mxfp4
    {1.14, 0.0574, 0.0184}, // mxfp8
    {0.64, 0.0794, 0.0388}, // nvfp4
};
const Step& step_of(int codes) {
  return kSteps[codes >= kOwnFpCodes ? 6 + codes - kOwnFpCodes : codes == 8 ? 5 : codes - 2];
}

// Scratch of ranges of K that a plan may ask for.
constexpr size_t kOwnMostPlanes = size_t(128) << 20;

} // namespace

// (which products it takes: qmm_experts_plan)
bool qmm_own_experts_supported(const QmmArgs& a, int bits) {
  // (x: the callers check it for every grouped kernel)
  return own_addresses(a.N, a.K, bits) && static_cast<uint64_t>(a.L) * a.N * 2 < kNoStore;
}

bool qmm_own_supported(int M, int N, int K, int L, int bits, int dtype) {
  return M > 64 && L == 1 && dtype != MLXROCM_FLOAT32 && own_addresses(N, K, bits) &&
      static_cast<uint64_t>(M) * K * 2 < k32Bit &&
      static_cast<uint64_t>(kOwnBM) * (N + 3) * 4 < kNoStore;
}

// The height of the tiles and the number of K ranges with the least time by this account,
// fitted to 27000 calls of 65..8192 rows on 14 shapes, every width and mode, each in every
// height and several numbers of ranges (errors of 5 %; the choice takes 1.2 % longer than the
// best one on average): the launches and the image of scales, rounds of tiles, planes written
// and added up.  Ranges are cut only while one round of workgroups holds their tiles.  Rows of y
// of an odd number of elements are stored element by element: 17 us a tile of 256 rows (planes
// have whole pieces).  Heights of 96, 160 and 224 rows make the 41 % of 2500 calls that take them 6 %
// shorter than 64, 128, 192 and 256 alone.
OwnPlan qmm_own_plan(int M, int N, int K, int codes) {
  const Step& step = step_of(codes);
  const int cus = static_cast<int>(compute_units());
  const int nx = (N + kOwnBN - 1) / kOwnBN;
  const int steps = K / kOwnBK;
  const size_t plane_size = k_split_plane(M, N) * sizeof(float);
  const double plane = 1e-6 / sizeof(float) * static_cast<double>(plane_size);
  // (4-bit codes in one range are put in order: kInOrder)
  const double in_order = codes == 4 ? 0.12 : 0.0;
  size_t most = kOwnMostPlanes / plane_size;
  most = most > 16 ? 16 : most;
  const int ranges = static_cast<int>(most) * 2 > steps ? steps / 2 : static_cast<int>(most);
  OwnPlan pl{};
  for (int mt = 4; mt <= 16; mt += 2) {
    if (mt > 4 && 16 * mt > (M + 31) / 32 * 32) {
      break;
    }
    const long tiles = static_cast<long>(nx) * ((M + 16 * mt - 1) / (16 * mt));
    const double tile = 0.36 * mt - 1.1;
    const long rounds = (tiles + cus - 1) / cus;
    const double busy = static_cast<double>(tiles) / static_cast<double>(rounds * cus);
    const double us = 5.9 + 0.34 * plane +
        rounds * (tile + steps * (step.fixed + in_order + mt * (step.each + busy * step.busy)) +
                  (N % 2 != 0 ? 1.05 * mt : 0.0));
    if (pl.mt == 0 || us < pl.us) {
      pl = {mt, 1, us};
    }
    for (int s = 2; s <= ranges && tiles * s <= cus; ++s) { // (one round)
      const double share = static_cast<double>(tiles * s) / cus;
      const double each =
          (steps + s - 1) / s * (step.fixed + mt * (step.each + share * step.busy));
      const double cut = 5.9 + tile + each + 6.6 + (0.89 * s + 0.15) * plane;
      if (cut < pl.us) {
        pl = {mt, s, cut};
      }
    }
  }
  return pl;
}

// With the accounts of both sides, which err by 5 and 7..15 %, these margins leave 1.0 % of the
// 4000 calls taken behind by more than 3 %, the worst by 15 %; the mean takes 0.85 of the time.  us against the tile kernel, bf16 g64 4-bit: 2048 x 4096 x 14336 198 / 243,
// 2048 x 8192 x 8192 198 / 275, 2048 x 4096 x 4096 66 / 78, 320 x 14336 x 4096 51 / 60, 320 x 8192 x
// 8192 54 / 80; the tile kernel stays ahead where its widths make whole rounds: 1024 x 14336 x
// 4096 8-bit 102 / 99, 512 x 18944 x 3584 8-bit 77 / 72.  Less is to be gained where its
// unpacking is one convert for two codes (mxfp8: 512 x 18944 x 3584 75 / 66; mxfp4 in one tile of
// rows, 103 x 18944 x 3584 42 / 38), its steps are cheap (8-bit, one range: 1921 x 5120 x 13824 313
// / 280) or this kernel has to put the codes in order (4-bit, one range: 5291 x 6853 x 8192 557 /
// 553).
bool qmm_own_pays(const OwnPlan& pl, int M, int codes, double other) {
  const bool one = pl.splits == 1;
  const double margin = codes == kOwnFpCodes + MLXROCM_MXFP8      ? 0.82
      : one && codes == 4                                         ? 0.82
      : one && codes == 8                                         ? 0.84
      : one && codes == kOwnFpCodes + MLXROCM_MXFP4 && M <= 256 ? 0.82
                                                                  : 0.88;
  return pl.us < margin * other;
}

int launch_qmm_own(
    const QmmArgs& a, int gs, int codes, int dtype, const OwnPlan& pl, hipStream_t s) {
  if (a.out_scale != nullptr) {
    return fail(MLXROCM_UNSUPPORTED, "[qmm_own] a scale of the results"); // (mlxrocm_fp_qmm takes it)
  }
  MLXROCM_REHEARSE("qmm_own(rows=%d,ksplit=%d)", 16 * pl.mt, pl.splits);
  if (codes >= kOwnFpCodes) {
    const int mode = codes - kOwnFpCodes;
    return dtype == MLXROCM_BFLOAT16 ? launch_qmm_own_fp_bf16(a, mode, pl, s)
                                     : launch_qmm_own_fp_f16(a, mode, pl, s);
  }
  return dtype == MLXROCM_BFLOAT16 ? launch_qmm_own_bf16(a, gs, codes, pl, s)
                                   : launch_qmm_own_f16(a, gs, codes, pl, s);
}

// Tiles that leave units idle over a long K: ranges of 1024 codes or more, up to four, with the
// least time by qmm_own_plan's account of a step, of planes and their sum.  8 experts, 4096 x
// 14336 4-bit, 300 tokens to 2 experts each: the product 231 us without ranges, the whole call
// 486 / 407 (600 tokens, by scratch without: 643 against 692 of the tile kernel).  From a round
// of tiles on the order of the list evens the workgroups' shares out, and ranges gain nothing
// (2048 tokens, two ranges: 1.07 of the tile kernel, 1.07..1.12 without).  One expert more with a
// second tile may start a second round of ranges, which codes that are dear to unpack feel: 8-bit,
// 493 tokens, 9 tiles of rows instead of 8, 595 us on the tile kernel, 717 in two ranges (4-bit,
// 489 tokens: 614 / 523).  So more than half a tile is counted there beyond the full ones.
int qmm_own_experts_splits(const QmmArgs& a, int bits, size_t room) {
  const size_t plane = static_cast<size_t>(a.L) * a.N * sizeof(float);
  if (a.N % 4 != 0 || plane >= kNoStore) {
    return 1;
  }
  const long cus = compute_units();
  const long expected =
      bits == 4 ? expected_tiles(a.L, a.n_experts) : (5L * a.L / 256 + 3L * a.n_experts + 4) / 5;
  const long least = a.n_experts < a.L ? a.n_experts : a.L;
  const long high = expected > least ? expected : least;
  const long tiles = high * ((a.N + kOwnBN - 1) / kOwnBN);
  if (tiles >= cus) {
    return 1;
  }
  const int mt = static_cast<int>((a.L / high + 31) / 32 * 2);
  const Step& step = step_of(bits);
  const double each =
      a.K / kOwnBK * (step.fixed + (mt < 4 ? 4 : mt > 16 ? 16 : mt) * (step.each + step.busy));
  int best = 1;
  double best_us = 0.0;
  for (int s = 1; s <= 4 && (s == 1 || (s * 1024 <= a.K && s * plane <= room)); ++s) {
    const double us = each / s * static_cast<double>((tiles * s + cus - 1) / cus) +
        (s > 1 ? 6.6 + (0.89 * s + 0.15) * 1e-6 / sizeof(float) * static_cast<double>(plane) : 0.0);
    if (s == 1 || us < 0.95 * best_us) {
      best = s;
      best_us = us;
    }
  }
  return best;
}

int launch_qmm_own_experts(
    const QmmArgs& a, int gs, int bits, int dtype, bool glu, int k_splits, hipStream_t s) {
  MLXROCM_REHEARSE("qmm_own_experts%s(ksplit=%d)", glu ? "_glu" : "", k_splits);
  return dtype == MLXROCM_BFLOAT16 ? launch_qmm_own_experts_bf16(a, gs, bits, glu, k_splits, s)
                                   : launch_qmm_own_experts_f16(a, gs, bits, glu, k_splits, s);
}

} // namespace mlxrocm
