// qmm_own_tiles.h -- qmm_own_kernel on one product, one translation unit per element type and
// kind of codes.
#pragma once

#include "qmm_own.h"

namespace mlxrocm {

namespace {

// pl.splits > 1: a.out points at that many planes.
template <typename T, int BITS, int FP = 0>
int own_tiles(const QmmArgs& a, int gs, const OwnPlan& pl, hipStream_t s) {
  const long tiles = static_cast<long>((a.N + kOwnBN - 1) / kOwnBN) *
      ((a.M + 16 * pl.mt - 1) / (16 * pl.mt)) * pl.splits;
  const int shift = FP != 0 ? 5 : own_group_shift(gs);
  auto run = [&](auto mtval) {
    constexpr int MT = decltype(mtval)::value;
    return pl.splits > 1 ? launch_own<T, float, BITS, MT, FP>(a, shift, tiles, s, pl.splits)
                         : launch_own<T, T, BITS, MT, FP>(a, shift, tiles, s);
  };
  switch (pl.mt) {
    case 4:
      return run(IntC<4>{});
    case 6:
      return run(IntC<6>{});
    case 8:
      return run(IntC<8>{});
    case 10:
      return run(IntC<10>{});
    case 12:
      return run(IntC<12>{});
    case 14:
      return run(IntC<14>{});
    default:
      return run(IntC<16>{});
  }
}

template <typename T>
int own_tiles_affine(const QmmArgs& a, int gs, int bits, const OwnPlan& pl, hipStream_t s) {
  return dispatch_bits(bits, [&](auto bval) {
    return own_tiles<T, decltype(bval)::value>(a, gs, pl, s);
  });
}

template <typename T>
int own_tiles_fp(const QmmArgs& a, int mode, const OwnPlan& pl, hipStream_t s) {
  switch (mode) {
    case MLXROCM_MXFP4:
      return own_tiles<T, 4, 1>(a, 32, pl, s);
    case MLXROCM_MXFP8:
      return own_tiles<T, 8, 2>(a, 32, pl, s);
    default:
      return own_tiles<T, 4, 3>(a, 32, pl, s);
  }
}

} // namespace

} // namespace mlxrocm
