// qmm_own.h -- tiles of up to 256 rows of x by 256 rows of W whose wavefronts own their
// rows of W (transpose=true, 16-bit types, every width and mode, pair images of scales).
//
// What bounds it: the matrix units at the clock that the card's power leaves them.  8192 x
// 14336 x 4096 4-bit g64 bf16 takes 680 us (1415 TFLOP/s) on ordinary values and 517 (1861)
// where x and W are zero, the same instructions; the tile kernel (qmm_mfma_tile.h) takes 757
// and 579, a library product of the dequantized weights 1426 TFLOP/s.  Hence the split: each
// of the eight wavefronts unpacks 32 rows of W and no other does, straight from global memory
// into the registers that the matrix instructions read, so that the unpacked weights neither
// pass through LDS nor are unpacked twice, and a step has one barrier.  x is the operand that
// all share: 128 columns at a time go to LDS by direct loads, two stages, and every fragment
// of 16 rows that a wavefront reads meets two 16-row tiles of W.  Every instruction has its
// slot between two matrix instructions: loads of the next step in the first of them, the 64
// pairs of codes spread over all, four fragments of x read ahead.
//
// Workgroups are persistent, one on a compute unit (128 KB of LDS, 256 registers): the last
// step of a tile loads the first of the next, so that only the first tile of a launch waits
// for memory.  A tile's height is its own in steps of 32 rows where rows are routed to experts:
// the rows of an expert's last tile that are none cost at most 31 rows' instructions.
#pragma once

#include "mfma_dequant.h"
#include "mfma_loads.h"
#include "qmm_args.h"

namespace mlxrocm {

namespace {

constexpr int kOwnBM = 256;
constexpr int kOwnBN = 256;
constexpr int kOwnBK = 128;
constexpr int kOwnThreads = 512;
// bytes of an x stage of tiles of 16 mt rows (0: up to kOwnBM)
constexpr int own_stage_bytes(int mt) {
  return (mt == 0 ? kOwnBM : 16 * mt) * kOwnBK * 2;
}
inline int own_group_shift(int gs) {
  return gs == 32 ? 5 : (gs == 64 ? 6 : 7);
}
constexpr int kOwnRing = 4; // fragments of x in registers
// Offset of a result that is not stored: it lies past the bound of the buffer, and so do the
// 32 bytes behind it.  The outputs are shorter (qmm_own.hip).
constexpr uint32_t kNoStore = 0xffffffe0u;

// f(0), f(1), .. f(N - 1) with the numbers as constants
template <int... I, typename F>
__device__ __forceinline__ void own_unroll_impl(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void own_unroll(F&& f) {
  own_unroll_impl(f, std::make_integer_sequence<int, N>{});
}

#define OWN_INLINE __attribute__((always_inline))

// Lanes 16 g + i, g = 0..3, as a 4 x 4 matrix of registers v[0..3]: transposed, so that
// lanes of g hold in v[j] what lanes of j held in v[g].
__device__ __forceinline__ void transpose_rows(uint32_t& v0, uint32_t& v1, uint32_t& v2, uint32_t& v3) {
  auto swap32 = [](uint32_t& a, uint32_t& b) { // a's lanes 32.. for b's lanes 0..31
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0];
    b = r[1];
  };
  auto swap16 = [](uint32_t& a, uint32_t& b) { // a's odd 16s of lanes for b's even ones
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0];
    b = r[1];
  };
  swap32(v0, v2);
  swap32(v1, v3);
  swap16(v0, v1);
  swap16(v2, v3);
}

// out = x W^T.  MT: tiles have 16 MT rows of x (4..16, even; grouped: 0, as many as the tile list says, in
// steps of 32).  TO float with k_splits > 1: planes (k_split_plane(); grouped: of a.L rows in
// the order of a.group_perm, N % 4 == 0) of K ranges.  FP: the
// modes of FpPairDequant.  GLU: gated pairs of columns of W and a.w_alt, 128 to a tile.
template <typename T, typename TO, int BITS, int MT_, int FP = 0, bool GLU = false>
__global__ __launch_bounds__(kOwnThreads) void qmm_own_kernel(
    const QmmArgs a, const int gs_shift, const int k_splits) {
  constexpr bool GROUPED = MT_ == 0;
  using DQ = std::conditional_t<FP != 0, FpPairDequant<T, (FP != 0 ? FP : 1)>, PairDequant<T, BITS>>;
  constexpr int kStage = own_stage_bytes(MT_);
  constexpr int kTileRows = GROUPED ? kOwnBM : 16 * MT_;
  // Without ranges of K the matrix instructions of a step take its 4-bit codes 32 by 32 in their
  // order, and those of routed rows at 8 bits too: a result has the bits that the tile kernel
  // gives in one range, so that which of the two runs does not show.  A lane loads 32 codes in a
  // row and gives 24 of them to the three lanes that hold the same row of W (swaps of registers
  // between lanes, with scales and biases 24 vector instructions a step, 32 at 8 bits: 8192 x
  // 14336 x 4096 685 -> 712 us; routed, 2048 tokens to 2 of 8 experts, 4096 x 14336, the call 1401
  // -> 1454.  Loads of a lane's own 8 codes instead, four for one: 1791).  Everywhere else the
  // codes stay where they were loaded.
  constexpr bool kInOrder = (BITS == 4 || (BITS == 8 && GROUPED)) && FP == 0 && sizeof(TO) == 2;
  constexpr int kCols = GLU ? kOwnBN / 2 : kOwnBN; // columns of y of a tile
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int N = a.N;
  const int K = a.K;
  const int pad = sizeof(TO) == 4 && k_splits > 1 ? 3 : 0;
  const int ldy = (N + pad) & ~pad;

  // ---- the tiles of this workgroup ----
  const int nx = (N + kCols - 1) / kCols;
  const int ny = __builtin_amdgcn_readfirstlane(
      GROUPED ? *a.group_ntiles : (a.M + kTileRows - 1) / kTileRows);
  const int plane = nx * ny;
  const int tiles = plane * k_splits;
  // Rounds of gridDim.x tiles.  Workgroups b, b + 8, .. share an XCD: they take neighbouring
  // tiles, and what is left for the last round is dealt out evenly to the XCDs.
  const int stride = gridDim.x;
  int base = 0; // first tile of the round
  auto tile_of_round = [&]() OWN_INLINE {
    const int left = tiles - base < stride ? tiles - base : stride;
    if constexpr (GROUPED) {
      // (the list is sorted by height: every other round runs backwards)
      const int b = blockIdx.x;
      const int in = base / stride % 2 == 0 ? b : stride - 1 - b;
      return in < left ? base + in : tiles;
    }
    if (stride % 8 != 0) {
      return static_cast<int>(blockIdx.x) < left ? base + static_cast<int>(blockIdx.x) : tiles;
    }
    const int xcd = blockIdx.x % 8, in = blockIdx.x / 8;
    const int each = left / 8, more = left % 8;
    return in < each + (xcd < more ? 1 : 0)
        ? base + xcd * each + (xcd < more ? xcd : more) + in
        : tiles;
  };
  int tile = tile_of_round();
  if (tile >= tiles) {
    return;
  }

  // what the loads of a tile need
  const uint8_t* px;
  const uint8_t* pw[2];
  const uint8_t* ps[2];
  constexpr int kLoads = kTileRows / 32; // direct-to-LDS loads of a wavefront for a stage
  uint32_t w_voff[2], sb_voff[2], xoff[kLoads];
  int kbeg = 0, ksteps = K / kOwnBK;
  // what its results need
  int rows = 0, m0 = 0, n0 = 0, row0 = 0, z = 0;

  // The lane as a number that is new wherever it is asked for: what is formed from it stays
  // where it is needed and takes no register in the K loops.
  auto lane_here = [&]() OWN_INLINE {
    int v = lane;
    asm volatile("" : "+v"(v));
    return v;
  };

  auto enter = [&](int id) OWN_INLINE {
    // (the quotients are formed in vector registers)
    auto uniform = [](int v) OWN_INLINE { return __builtin_amdgcn_readfirstlane(v); };
    z = uniform(id / plane);
    const int in = id - z * plane;
    // four row tiles by all columns at a time
    const int band = uniform(in / (4 * nx));
    const int in_band = in - band * 4 * nx;
    const int high = ny - 4 * band < 4 ? ny - 4 * band : 4;
    const int col = uniform(in_band / high);
    const int ty = 4 * band + in_band - col * high;
    n0 = col * kCols + wave * (kCols / 8);
    int64_t wb = 0;
    if constexpr (GROUPED) {
      wb = uniform(a.group_tiles[3 * ty]);
      row0 = uniform(a.group_tiles[3 * ty + 1]);
      rows = uniform(a.group_tiles[3 * ty + 2]);
    } else {
      m0 = ty * kTileRows;
      rows = a.M - m0 < kTileRows ? a.M - m0 : kTileRows;
    }
    px = static_cast<const uint8_t*>(a.x);
    const int64_t wo = wb * a.w_batch_stride * 4;
    const int64_t so = wb * a.sb_batch_stride * 2;
    pw[0] = reinterpret_cast<const uint8_t*>(a.w) + wo;
    ps[0] = static_cast<const uint8_t*>(a.scales) + so;
    pw[1] = GLU ? reinterpret_cast<const uint8_t*>(a.w_alt) + wo : pw[0];
    ps[1] = GLU ? static_cast<const uint8_t*>(a.scales_alt) + so : ps[0];
    const uint32_t row_words = static_cast<uint32_t>(K / 32 * BITS);
    const int at = lane_here();
    const int wi = at & 15, wk = at >> 4;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int n = GLU ? n0 + wi : n0 + 2 * wi + j;
      const int nc = n < N ? n : N - 1; // loads stay in bounds
      w_voff[j] = (static_cast<uint32_t>(nc) * row_words + wk * BITS) * 4u;
      sb_voff[j] = (static_cast<uint32_t>((32 * wk) >> gs_shift) * N + nc) * 4u;
    }
    // x: load i of wavefront w moves rows 32 i + 4 w .. + 3, the 16 pieces of a row in 16
    // lanes.  Piece p of row r (eight columns) is read in slice s by the lanes of k, p = 4 s + k
    // in order and 4 k + s otherwise.  It sits at 8 (k % 2) + (q ^ (r % 8)), q being what
    // else there is of p: the 64 lanes of a fragment read, 16 rows by four k, then hit every
    // bank of LDS once in each quarter.
    const int xr0 = 4 * wave + (at >> 4);
    const uint32_t xlow = static_cast<uint32_t>((at ^ xr0) & 7);
    const uint32_t odd = (at >> 3) & 1;
    const uint32_t xpiece =
        kInOrder ? 2 * xlow + odd : ((xlow >> 2) * 2 + odd) * 4 + (xlow & 3);
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int r = 32 * i + xr0;
      const int rc = r < rows ? r : rows - 1; // rows past M are never stored
      if constexpr (GROUPED) {
        const uint32_t pair = static_cast<uint32_t>(a.group_perm[row0 + rc]);
        xoff[i] = (a.lhs_indices[pair] * static_cast<uint32_t>(a.x_batch_stride) + xpiece * 8) * 2u;
      } else {
        xoff[i] = (static_cast<uint32_t>(m0 + rc) * static_cast<uint32_t>(K) + xpiece * 8) * 2u;
      }
    }
    if (k_splits > 1) {
      const int steps = K / kOwnBK;
      const int begin = uniform(steps * z / k_splits);
      ksteps = uniform(steps * (z + 1) / k_splits) - begin;
      kbeg = begin * kOwnBK;
    }
  };

  uint32_t wreg[2][BITS];
  constexpr int kScales = kInOrder ? 4 : 1; // of a row in a step: of each 32 codes
  uint32_t sb[2][kScales]; // pairs of scale and bias
  float sf[2], bf[2];      // those of the codes being unpacked
  RawWords<BITS> wnext[2];
  RawTuple<1> snext[2];
  uint32_t rd[4]; // byte offset of this lane's piece of slice s in a row block
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const int fi = lane & 15, fk = lane >> 4;
    const int of_half = kInOrder ? 2 * s + (fk >> 1) : 4 * (fk >> 1) + s;
    rd[s] = fi * 256 + (8 * (fk & 1) + (of_half ^ (fi & 7))) * 16;
  }

  auto load_w = [&](int k) OWN_INLINE {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      wnext[j].load(w_voff[j], pw[j] + static_cast<size_t>(k / 32 * BITS) * 4);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      snext[j].template load<0>(sb_voff[j], ps[j] + static_cast<size_t>(k >> gs_shift) * N * 4);
    }
  };
  // behind the wait that covers the loads of load_w()
  auto take_w = [&](auto jval) OWN_INLINE {
    constexpr int j = decltype(jval)::value;
    wnext[j].pin();
    snext[j].pin();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < BITS; ++i) {
      wreg[j][i] = wnext[j].get(i);
    }
    sb[j][0] = snext[j].get(0);
    if constexpr (kInOrder) {
      constexpr int each = BITS / 4; // dwords of eight codes
#pragma unroll
      for (int i = 0; i < each; ++i) {
        transpose_rows(
            wreg[j][i], wreg[j][each + i], wreg[j][2 * each + i], wreg[j][3 * each + i]);
      }
      sb[j][1] = sb[j][2] = sb[j][3] = sb[j][0];
      transpose_rows(sb[j][0], sb[j][1], sb[j][2], sb[j][3]);
    }
  };
  auto dma_x = [&](int stage, int k, auto i) OWN_INLINE {
    dma16(lds_address(smem + stage + (32 * i + 4 * wave) * 256), xoff[decltype(i)::value],
          px + static_cast<size_t>(k) * 2);
  };
  int cur = 0; // stage of the step being multiplied

  // K loop and results of a tile of at most 16 MT rows; the loads of its last step are
  // those of the next tile's first.
  auto run_tile = [&](auto mtval) OWN_INLINE {
    constexpr int MT = decltype(mtval)::value;
    constexpr int kNS = 8 * MT;  // matrix instructions of a wavefront and step
    constexpr int kF = 4 * MT;   // fragments of x of a step
    constexpr int kDma = MT / 2; // direct-to-LDS loads of a wavefront and step
    constexpr int kBarrier = kNS - 6;
    constexpr int kP1 = kBarrier * 2 / 5, kP2 = kBarrier * 7 / 10, kP3 = kBarrier * 19 / 20;
    uint4 xr[kOwnRing];
    auto read_x = [&](int stage, auto F, int e) OWN_INLINE {
      constexpr int s = decltype(F)::value / MT;
      constexpr int f = decltype(F)::value % MT;
      xr[e] = *reinterpret_cast<const uint4*>(smem + stage + rd[s] + f * 4096);
    };
    uint32_t wf[2][2][4]; // [slice % 2][16-row tile of W]: operands of a slice
    DQ dq[2];
    // pair q (0..7) of slice s: four dwords of each of the two rows
    auto pair = [&](auto s, auto q) OWN_INLINE {
      constexpr int j = decltype(q)::value / 4;
      constexpr int i = decltype(q)::value % 4;
      if constexpr (i == 0 && (kInOrder || decltype(s)::value == 0)) {
        constexpr int g = kInOrder ? decltype(s)::value : 0;
        sf[j] = raw_value<T>(sb[j][g]) * DQ::kCodeScale;
        bf[j] = raw_value<T>(sb[j][g] >> 16);
      }
      wf[s % 2][j][i] = dq[j].template pair<4 * decltype(s)::value + i>(wreg[j], sf[j], bf[j]);
    };
    own_unroll<8>([&](auto q) OWN_INLINE { pair(std::integral_constant<int, 0>{}, q); });
    own_unroll<kOwnRing>([&](auto f) OWN_INLINE { read_x(cur, f, f); });
    floatx4 acc[2][MT];
    own_unroll<MT>([&](auto f) OWN_INLINE {
      acc[0][f] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
      acc[1][f] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    });
    const int my_rows = rows, my_m0 = m0, my_n0 = n0, my_row0 = row0, my_z = z;
    int k2 = kbeg;
    int left = ksteps - 1; // steps before the last
    bool last = false;
#pragma nounroll
    for (;;) {
#pragma nounroll
    for (; left > 0; --left) {
      k2 += kOwnBK;
      const int nxt = kStage - cur;
      __builtin_amdgcn_sched_barrier(0);
      own_unroll<kNS>([&](auto mi) OWN_INLINE {
        constexpr int m = decltype(mi)::value;
        constexpr int s = m / (2 * MT);
        constexpr int f = m % (2 * MT) / 2;
        constexpr int n = m % 2;
        constexpr int F = m / 2;
        constexpr int e = F % kOwnRing;
        constexpr int in_slice = m % (2 * MT);
        if constexpr (m == 6 * MT) {
          // the packed W asked for in slot 0 is older than the loads of x
          asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kDma) : "memory");
          take_w(std::integral_constant<int, 0>{});
        }
        if constexpr (m == 7 * MT - 1) { // before the first pair of the second row
          take_w(std::integral_constant<int, 1>{});
        }
        if constexpr (m == kBarrier) {
          asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
          __syncthreads();
          read_x(nxt, std::integral_constant<int, 0>{}, 0);
        }
        // the wavefront that is behind goes first: its partner on the same unit waits at the
        // barrier for it
        if constexpr (m == kP1 || m == kP2 || m == kP3 || m == kBarrier) {
          __builtin_amdgcn_s_setprio(m == kP1 ? 2 : m == kP2 ? 1 : m == kP3 ? 0 : 3);
        }
        acc[n][f] = mfma16<T>(
            make_uint4(wf[s % 2][n][0], wf[s % 2][n][1], wf[s % 2][n][2], wf[s % 2][n][3]), xr[e],
            acc[n][f]);
        if constexpr (n == 1) {
          constexpr int G = F + kOwnRing; // the fragment that takes this one's registers
          if constexpr (G < kF) {
            read_x(cur, std::integral_constant<int, G>{}, e);
          } else if constexpr (m > kBarrier) {
            read_x(nxt, std::integral_constant<int, G - kF>{}, e);
          }
        }
        if constexpr (m == 0) {
          load_w(k2);
        }
        if constexpr (m % 8 == 5 && m / 8 < kDma) {
          dma_x(nxt, k2, std::integral_constant<int, m / 8>{});
        }
        constexpr int q = in_slice * 8 / (2 * MT);
        if constexpr (in_slice == (q * 2 * MT + 7) / 8) {
          pair(std::integral_constant<int, (s + 1) % 4>{}, std::integral_constant<int, q>{});
        }
        __builtin_amdgcn_sched_barrier(0);
      });
      cur = nxt;
    }
      if (last) {
        break;
      }
      last = true;
      left = 1;
      base += stride;
      tile = base < tiles ? tile_of_round() : tiles;
      if (tile < tiles) {
        enter(tile);
      }
      k2 = kbeg - kOwnBK;
    }

    // lane (fi, fk) holds row fi of x and rows 4 fk + r of both tiles of W
    const int at = lane_here();
    const int fi = at & 15, fk = at >> 4;
    TO* out = static_cast<TO*>(a.out);
    uint32_t bytes; // behind `out`: what lies past it is not stored
    if constexpr (GROUPED) {
      out += static_cast<int64_t>(my_z) * a.L * ldy; // (of a plane)
      bytes = static_cast<uint32_t>(a.L) * static_cast<uint32_t>(ldy) * sizeof(TO);
    } else {
      out += (static_cast<int64_t>(my_z) * a.M + my_m0) * ldy;
      bytes = static_cast<uint32_t>(my_rows) * static_cast<uint32_t>(ldy) * sizeof(TO);
    }
    // (stores without a branch that differs between lanes: such a branch here makes the
    // compiler lay out the choice of the tile's height as one, with every register of every
    // height alive)
    auto rsrc = __builtin_amdgcn_make_buffer_rsrc(out, 0, static_cast<int>(bytes), 0x00020000);
    // results of a lane in a row: of its four rows of one 16-row tile of W, or of both
    constexpr int kRun = GLU ? 4 : 8;
    const int n = my_n0 + kRun * fk;
    const int bound = sizeof(TO) == 4 ? ldy : N; // rows of planes are whole 16-byte pieces
    const bool whole = my_n0 + kCols / 8 <= bound && (sizeof(TO) == 4 || N % 2 == 0);
    uint32_t off[MT];
    own_unroll<MT>([&](auto f) OWN_INLINE {
      const int mr = 16 * f + fi;
      if constexpr (GROUPED) {
        // (planes: rows in their sorted order)
        const int pos = my_row0 + (mr < my_rows ? mr : my_rows - 1);
        const uint32_t row = sizeof(TO) == 4 ? pos : a.group_perm[pos];
        off[f] = mr < my_rows ? (row * static_cast<uint32_t>(ldy) + n) * sizeof(TO) : kNoStore;
      } else {
        off[f] = (static_cast<uint32_t>(mr) * static_cast<uint32_t>(ldy) + n) * sizeof(TO);
      }
    });
    auto store = [&](auto f, auto by_piece) OWN_INLINE {
      float v[kRun];
#pragma unroll
      for (int e = 0; e < kRun; ++e) {
        if constexpr (GLU) {
          v[e] = gated<TO>(round_to<TO>(acc[0][f][e]), round_to<TO>(acc[1][f][e]));
        } else {
          v[e] = acc[e % 2][f][e / 2];
        }
      }
      typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
      typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
      if constexpr (sizeof(TO) == 4) {
        const u32x4 lo = {__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]),
                          __float_as_uint(v[3])};
        const u32x4 hi = {__float_as_uint(v[4]), __float_as_uint(v[5]), __float_as_uint(v[6]),
                          __float_as_uint(v[7])};
        const uint32_t at_lo = n + 4 <= bound ? off[f] : kNoStore;
        const uint32_t at_hi = n + 8 <= bound ? off[f] + 16 : kNoStore;
        __builtin_amdgcn_raw_buffer_store_b128(lo, rsrc, at_lo, 0, 0);
        __builtin_amdgcn_raw_buffer_store_b128(hi, rsrc, at_hi, 0, 0);
      } else if constexpr (decltype(by_piece)::value) {
        uint32_t d[kRun / 2];
#pragma unroll
        for (int e = 0; e < kRun; e += 2) {
          d[e / 2] = pack2<TO>(v[e], v[e + 1]);
        }
        if constexpr (GLU) {
          __builtin_amdgcn_raw_buffer_store_b64(u32x2{d[0], d[1]}, rsrc, off[f], 0, 0);
        } else {
          __builtin_amdgcn_raw_buffer_store_b128(
              u32x4{d[0], d[1], d[2], d[3]}, rsrc, off[f], 0, 0);
        }
      } else {
#pragma unroll
        for (int e = 0; e < kRun; ++e) {
          const uint32_t at_e = n + e < bound ? off[f] + e * sizeof(TO) : kNoStore;
          __builtin_amdgcn_raw_buffer_store_b16(
              __builtin_bit_cast(uint16_t, static_cast<TO>(v[e])), rsrc, at_e, 0, 0);
        }
      }
    };
    if (whole) {
      own_unroll<MT>([&](auto f) OWN_INLINE { store(f, std::true_type{}); });
    } else {
      own_unroll<MT>([&](auto f) OWN_INLINE { store(f, std::false_type{}); });
    }
  };

  // first tile: its first stage and weights
  enter(tile);
  own_unroll<kLoads>([&](auto i) OWN_INLINE { dma_x(0, kbeg, i); });
  load_w(kbeg);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  take_w(std::integral_constant<int, 0>{});
  take_w(std::integral_constant<int, 1>{});
  __syncthreads();
  __builtin_amdgcn_s_setprio(3);
  if constexpr (!GROUPED) {
    while (tile < tiles) {
      run_tile(std::integral_constant<int, MT_>{});
    }
  } else {
    int have = 16; // 16-row blocks of the current tile that its first stage holds
    while (tile < tiles) {
      const int need = __builtin_amdgcn_readfirstlane((rows + 15) >> 4);
      if (need > have) {
        // the tile before was lower: its last step fetched too few rows
        own_unroll<kLoads>([&](auto i) OWN_INLINE { dma_x(cur, kbeg, i); });
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
      }
      if (need > 14) {
        run_tile(std::integral_constant<int, 16>{});
        have = 16;
      } else if (need > 12) {
        run_tile(std::integral_constant<int, 14>{});
        have = 14;
      } else if (need > 10) {
        run_tile(std::integral_constant<int, 12>{});
        have = 12;
      } else if (need > 8) {
        run_tile(std::integral_constant<int, 10>{});
        have = 10;
      } else if (need > 6) {
        run_tile(std::integral_constant<int, 8>{});
        have = 8;
      } else if (need > 4) {
        run_tile(std::integral_constant<int, 6>{});
        have = 6;
      } else {
        run_tile(std::integral_constant<int, 4>{});
        have = 4;
      }
    }
  }
}

template <typename T, typename TO, int BITS, int MT, int FP = 0, bool GLU = false>
int launch_own(
    const QmmArgs& a, int gs_shift, long tiles, hipStream_t s, int k_splits = 1) {
  auto kern = qmm_own_kernel<T, TO, BITS, MT, FP, GLU>;
  constexpr int smem = 2 * own_stage_bytes(MT);
  static bool configured = false; // per instantiation
  if (!configured) {
    MLXROCM_HIP_TRY(hipFuncSetAttribute(
        reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, smem));
    configured = true;
  }
  const long room = compute_units(); // one workgroup each
  const unsigned grid = static_cast<unsigned>(tiles < room ? tiles : room);
  kern<<<grid, kOwnThreads, smem, s>>>(a, gs_shift, k_splits);
  MLXROCM_HIP_TRY(hipGetLastError());
  return static_cast<int>(MLXROCM_OK);
}

} // namespace

} // namespace mlxrocm
