// qmm_walk.h -- transpose=true products with a few rows of x (2..64), 16-bit
// element types: the kernel template; the .hip files beside it instantiate it per
// code width.
//
//   y[M, N] = x[M, K] * dequant(W)[N, K]^T
//
// The bound is the stream of packed weights: at 48 rows a weight of 14336 x 4096
// at 4 bits is 33 MB (6.5 us at the rate of a large copy) against 4 us of matrix
// instructions.  What it takes to come near that with x of up to 64 rows:
//   * every compute unit owns an equal number of rows of W (R = 4..64, chosen by
//     the host as N / units, so that the last round of workgroups is full) and
//     the whole of K: y is finished where it is computed.  Only where 17 rows of x or
//     more meet few rows of W per unit, or the tables of the whole of K do not fit LDS,
//     is K cut into ranges with fp32 planes (walk_plan);
//   * W goes from memory to registers, asked for four stages ahead of its use (two
//     where registers are short: kAhead).  Loads arrive in order, so the wait for x
//     (below) is one for the W asked for before it, too: across it only the newest
//     stage of W is in flight where x has one set of registers (48 and 64 rows; 16 and
//     32 rows with one tile of W), two where it has two.  A lane
//     (r = lane % 16, q = lane / 16) holds 32 consecutive codes of row r, the
//     quads side by side: 16 rows x 128 codes per wavefront and stage.  The matrix
//     instruction sums over the four quads, and a sum may not leave a quantization
//     group, so for groups of 32 or 64 the quads first exchange registers
//     (v_permlane32_swap / v_permlane16_swap, one instruction per two dwords);
//   * x walks through LDS in stages of KW x 128 codes, double-buffered, one
//     barrier per stage, fetched through registers and asked for XD stages (one or
//     two) before it is stored for the next.  KW wavefronts
//     (times NW that share them) split the 128-code chunks of a stage, and add
//     their sums up through LDS at the end;
//   * codes are multiplied as they are (widened exactly into the 16-bit type, with
//     an offset where that saves instructions), one chain of v_mfma_f32_16x16x32
//     per quantization group starting from zero, then acc += scale * chain in
//     fp32.  What offset and biases add, sum_g X[m][g] * (bias[n][g] - offset *
//     scale[n][g]), is one v_mfma_f32_16x16x4_f32 per tile and four groups; X, the
//     sums of x over a group, come from a chain with a matrix of ones.  Nothing is
//     rounded before the final conversion, but the offset is taken back in fp32, so
//     its size against the codes matters (walk_offset);
//   * scales and biases of the workgroup's rows go to LDS once, as [group][row]
//     pairs.
#pragma once

#include <type_traits>

#include "mfma_dequant.h"
#include "qmm_args.h"

namespace mlxrocm {

// Shape of one launch, chosen by walk_plan() (qmm_walk.hip).
struct WalkPlan {
  int config;    // an entry of kWalkConfigs
  int mr;        // rows of x staged: 8, 16, 32, 48, 64
  int tile_rows; // rows of W per tile, at most 16
  int splits;    // K ranges over blockIdx.y (fp32 planes), 1 = none
  int range;     // stages per K range
};

struct WalkConfig {
  int tiles;   // 16-row tiles of W per workgroup
  int k_waves; // wavefronts that share K
};
// One tile and K over 8 wavefronts (few rows of W per compute unit); four tiles
// and K over 4; two tiles and K over 4 with room for two workgroups per unit; the
// same of four tiles (8 rows of x).
constexpr WalkConfig kWalkConfigs[] = {{1, 8}, {4, 4}, {2, 4}, {4, 4}};

struct WalkArgs {
  QmmArgs a;
  int tile_rows;
  int range;     // stages of a K range
  int glu;       // silu(w . x) * (w_alt . x): half the tiles are rows of each
  float* planes; // splits > 1: fp32 [splits][L][M][N]
};

namespace {

constexpr int kWkChunk = 128; // codes of a row per wavefront and stage
constexpr int kWkUnroll = 4;  // stages per turn of the loop: four groups or more

template <typename T>
struct WalkMagic;
template <>
struct WalkMagic<bf16_t> {
  static constexpr int kMantissa = 7; // bits: a code and an offset above it
  static constexpr uint32_t kOnes = 0x3F803F80u; // 1.0 twice
  static constexpr uint32_t kBits4 = 0x43004300u; // 128.0 twice: 4-bit codes fit below
  static constexpr int kShift4 = 0;
  static constexpr float kOffset4 = 128.0f;
};
template <>
struct WalkMagic<f16_t> {
  static constexpr int kMantissa = 10;
  static constexpr uint32_t kOnes = 0x3C003C00u;
  static constexpr uint32_t kBits4 = 0x54005400u; // 64.0 twice: 1 is bit 4
  static constexpr int kShift4 = 4;
  static constexpr float kOffset4 = 64.0f;
  static constexpr uint32_t kBits8 = 0x64006400u; // 1024.0 twice: 1 is bit 0
};

// A widened code is (code + offset) / unit.  The offset costs the fp32 sums what it is
// above the codes, so it is kept as small as the instructions allow.  2, 3, 5 and 6
// bits, whose pairs are put together code by code: at the top of the mantissa, offset
// 2^bits (1024 + c, in the same time, loses more than a float16 result hides: x of one
// sign, K = 4096, error of the result 5.9e-4 / 3.6e-4 at 2 / 3 bits in groups of 64
// against 2.1e-4, which is what rounding the exact result loses).  4 bits: where one of
// the four shifts of a dword falls away (float16: 1024 + c loses 3.4e-4 in groups of
// 128; at the top of the mantissa, one shift more, 16 rows of 14336 x 4096 take 13.9 us
// instead of 13.3).  8 bits: a byte, against codes that reach 255.
template <int BITS>
constexpr bool walk_at_top() {
  return BITS < 8 && BITS != 4;
}
template <int BITS>
constexpr float walk_unit() {
  return walk_at_top<BITS>() ? static_cast<float>(1 << BITS) : 1.0f;
}
template <typename T, int BITS>
constexpr float walk_offset() {
  if (BITS == 4) {
    return WalkMagic<T>::kOffset4;
  }
  if (BITS == 8) { // (bfloat16: no room, converted)
    return WalkMagic<T>::kMantissa < 8 ? 0.0f : 1024.0f;
  }
  return static_cast<float>(1 << BITS);
}
template <typename T, int BITS>
constexpr uint32_t walk_offset_bits() {
  if constexpr (BITS == 8) {
    return WalkMagic<f16_t>::kBits8;
  }
  return BITS == 4 ? WalkMagic<T>::kBits4 : WalkMagic<T>::kOnes;
}

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x3_t __attribute__((ext_vector_type(3)));

// As loads of packed codes see memory: 4-byte aligned whatever their width (rows
// of 3, 5 and 6 bits start where they start).
typedef u32x2_t u32x2_a4 __attribute__((aligned(4)));
typedef u32x3_t u32x3_a4 __attribute__((aligned(4)));
typedef u32x4_t u32x4_a4 __attribute__((aligned(4)));

// The packed dwords of a lane, in the tuples that its loads fill: whole vectors,
// because values that cross the loop's back edge while their load is in flight
// must not be taken apart there (that would be a wait).
template <int BITS>
struct WalkRegs {
  static constexpr int kB = BITS > 4 ? BITS - 4 : 0;
  std::conditional_t<BITS == 2, u32x2_t, std::conditional_t<BITS == 3, u32x3_t, u32x4_t>> a;
  std::conditional_t<kB == 4, u32x4_t, std::conditional_t<kB == 2, u32x2_t, uint32_t>> b;

  // off2: the second piece (8 bits: 64 codes on; 5 and 6 bits: 16 bytes on)
  __device__ __forceinline__ void load(const uint8_t* p, uint32_t off, uint32_t off2) {
    if constexpr (BITS == 2) {
      a = *reinterpret_cast<const u32x2_a4*>(p + off);
    } else if constexpr (BITS == 3) {
      a = *reinterpret_cast<const u32x3_a4*>(p + off);
    } else if constexpr (BITS == 4 || BITS == 8) {
      a = *reinterpret_cast<const u32x4_t*>(p + off);
    } else {
      a = *reinterpret_cast<const u32x4_a4*>(p + off);
    }
    if constexpr (BITS == 8) {
      b = *reinterpret_cast<const u32x4_t*>(p + off2);
    } else if constexpr (BITS == 6) {
      b = *reinterpret_cast<const u32x2_a4*>(p + off + 16);
    } else if constexpr (BITS == 5) {
      b = *reinterpret_cast<const uint32_t*>(p + off + 16);
    }
  }
  __device__ __forceinline__ void get(uint32_t (&w)[BITS]) const {
#pragma unroll
    for (int i = 0; i < (BITS < 4 ? BITS : 4); ++i) {
      w[i] = a[i];
    }
    if constexpr (BITS == 5) {
      w[4] = b;
    } else if constexpr (BITS > 5) {
#pragma unroll
      for (int i = 4; i < BITS; ++i) {
        w[i] = b[i - 4];
      }
    }
  }
};

// a's upper 32 lanes and b's lower 32 change places
__device__ __forceinline__ void swap_halves(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}
// a's odd runs of 16 lanes and b's even ones change places
__device__ __forceinline__ void swap_quads(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}

// Four operands (one per run of 32 summed codes) from the packed dwords of a
// lane.  Before: quad q holds codes 32 q .. of the chunk (8 bits: 16 q .. and
// 64 + 16 q ..).  After: operand i holds, over its four quads, codes of group
// i * 32 / GS only; k_of() says which.
template <typename T, int BITS, int GS>
struct WalkCodes {
  static constexpr bool kMagic = BITS <= WalkMagic<T>::kMantissa;
  static constexpr uint32_t kOffsetBits = walk_offset_bits<T, BITS>();
  static constexpr int kShift = // of a code
      BITS == 4 ? WalkMagic<T>::kShift4 : (BITS == 8 ? 0 : WalkMagic<T>::kMantissa - BITS);
  static constexpr uint32_t kMask = // of a code in the low half (4 bits: in both)
      (BITS == 4 ? 0x000f000fu : (1u << BITS) - 1u) << kShift;

  // first code (within the chunk) of the eight that quad q holds in operand i
  static __device__ __forceinline__ int k_of(int i, int q) {
    if constexpr (BITS == 8) {
      const int j = i / 2;
      const int h = i % 2;
      if constexpr (GS == 32) {
        return 64 * j + (h == 0 ? (q < 2 ? 16 * q : 16 * (q - 2) + 8)
                                : (q < 2 ? 16 * (q + 2) : 16 * q + 8));
      }
      return 64 * j + 16 * q + 8 * h;
    } else if constexpr (GS == 32) {
      return 32 * i + 8 * q;
    } else if constexpr (GS == 64) {
      const int h = i % 2;
      return i < 2 ? (q < 2 ? 32 * q + 8 * h : 32 * (q - 2) + 16 + 8 * h)
                   : (q < 2 ? 32 * (q + 2) + 8 * h : 32 * q + 16 + 8 * h);
    } else {
      return 32 * q + 8 * i;
    }
  }

  static __device__ __forceinline__ uint32_t pair(uint32_t c0, uint32_t c1) {
    return pack2<T>(static_cast<float>(c0), static_cast<float>(c1));
  }

  // (codes that straddle dwords) code i of w with its lowest bit at bit `at`
  static __device__ __forceinline__ uint32_t
  placed(const uint32_t (&w)[BITS], int i, int at) {
    const int d = i * BITS / 32;
    const int b = i * BITS % 32;
    if (b + BITS > 32) {
      return __builtin_amdgcn_alignbit(w[d + 1 < BITS ? d + 1 : d], w[d], b - at);
    }
    return b >= at ? w[d] >> (b - at) : w[d] << (at - b);
  }

  // The registers the operands of a stage are made from: the packed dwords with
  // every quad's share in place, or, for the widths whose codes straddle dwords,
  // the operands themselves.
  static constexpr bool kWhole = BITS == 4 || BITS == 8;
  static constexpr int kKept = kWhole ? BITS : 16;

  static __device__ __forceinline__ void
  regroup(const uint32_t (&w)[BITS], uint32_t (&d)[kKept], uint32_t mask, uint32_t magic) {
    if constexpr (BITS == 4) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        d[i] = w[i];
      }
      if constexpr (GS <= 64) {
        swap_halves(d[0], d[2]);
        swap_halves(d[1], d[3]);
      }
      if constexpr (GS == 32) {
        swap_quads(d[0], d[1]);
        swap_quads(d[2], d[3]);
      }
    } else if constexpr (BITS == 8) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        d[i] = w[i];
      }
      if constexpr (GS == 32) {
        swap_halves(d[0], d[2]);
        swap_halves(d[1], d[3]);
        swap_halves(d[4], d[6]);
        swap_halves(d[5], d[7]);
      }
    } else {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        d[i] = (placed(w, 2 * i, kShift) & mask) | magic;
        asm("" : "+v"(d[i])); // (two v_and_or_b32, not regrouped into three instructions)
        d[i] = (placed(w, 2 * i + 1, kShift + 16) & (mask << 16)) | d[i];
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) { // d[4 i + j]: dword j of operand i
        if constexpr (GS <= 64) {
          swap_halves(d[j], d[8 + j]);
          swap_halves(d[4 + j], d[12 + j]);
        }
        if constexpr (GS == 32) {
          swap_quads(d[j], d[4 + j]);
          swap_quads(d[8 + j], d[12 + j]);
        }
      }
    }
    // (opaque: the packed registers are free from here on, and the load that
    // fills them again is not held up by later uses)
#pragma unroll
    for (int i = 0; i < kKept; ++i) {
      asm volatile("" : "+v"(d[i]));
    }
  }

  // mask and magic come in registers: one v_and_or_b32 per pair
  static __device__ __forceinline__ uint4
  operand(const uint32_t (&d)[kKept], int i, uint32_t mask, uint32_t magic) {
    uint4 o;
    if constexpr (BITS == 4) {
      // codes 0,4 1,5 2,6 3,7: x is staged in that order
      const auto at = [&](int bit) { // the codes at `bit` and 16 on, in their place
        return bit >= kShift ? d[i] >> (bit - kShift) : d[i] << (kShift - bit);
      };
      o.x = (at(0) & mask) | magic;
      o.y = (at(4) & mask) | magic;
      o.z = (at(8) & mask) | magic;
      o.w = (at(12) & mask) | magic;
    } else if constexpr (BITS == 8 && kMagic) {
      // byte, 0x64, byte, 0x64
      o.x = __builtin_amdgcn_perm(magic, d[2 * i], 0x07010700u);
      o.y = __builtin_amdgcn_perm(magic, d[2 * i], 0x07030702u);
      o.z = __builtin_amdgcn_perm(magic, d[2 * i + 1], 0x07010700u);
      o.w = __builtin_amdgcn_perm(magic, d[2 * i + 1], 0x07030702u);
    } else if constexpr (BITS == 8) {
      const uint32_t v = d[2 * i];
      const uint32_t u = d[2 * i + 1];
      o.x = pair(v & 0xffu, (v >> 8) & 0xffu);
      o.y = pair((v >> 16) & 0xffu, v >> 24);
      o.z = pair(u & 0xffu, (u >> 8) & 0xffu);
      o.w = pair((u >> 16) & 0xffu, u >> 24);
    } else {
      o = make_uint4(d[4 * i], d[4 * i + 1], d[4 * i + 2], d[4 * i + 3]);
    }
    return o;
  }
};

// The floating-point modes (FP = 1 mxfp4, 2 mxfp8, 3 nvfp4): the scales go into
// the operands, which are exact in bf16 (and in f16 while they are in its range),
// so that one chain runs over the whole of K.
__device__ __forceinline__ float walk_e8m0(uint32_t s) {
  return __uint_as_float((s == 0 ? 0x40u : (s << 7)) << 16);
}
// sign, bias 7, subnormals, no special codes
__device__ __forceinline__ float walk_e4m3(uint32_t x) {
  const uint32_t e = (x >> 3) & 0xFu;
  const uint32_t m = x & 7u;
  const float mag = e == 0 ? static_cast<float>(m) * 0.001953125f
                           : __uint_as_float(((e + 120u) << 23) | (m << 20));
  return (x & 0x80u) ? -mag : mag;
}

template <typename T, int FP, int Q>
__device__ __forceinline__ uint32_t
walk_fp_pair(const uint32_t (&w)[FP == 2 ? 8 : 4], float s0, float s1) {
  FpPairDequant<T, FP> dq;
  if constexpr (FP == 2) { // dwords 4..7 are the second piece, of another group
    return dq.template pair<Q>(w, Q < 8 ? s0 : s1, 0.0f);
  } else {
    return dq.template pair<Q>(w, s0, s1);
  }
}
template <typename T, int FP, int... Q>
__device__ __forceinline__ void walk_fp_widen(
    const uint32_t (&w)[FP == 2 ? 8 : 4], float s0, float s1, uint32_t (&d)[16],
    std::integer_sequence<int, Q...>) {
  ((d[Q] = walk_fp_pair<T, FP, Q>(w, s0, s1)), ...);
}

// The 16 dwords of a lane's four operands.  s0, s1: the scales of the lane's two
// pieces (mxfp8), of its two runs of 16 codes (nvfp4), of all its codes (mxfp4: s0).
template <typename T, int FP>
__device__ __forceinline__ void walk_fp_operands(
    const uint32_t (&w)[FP == 2 ? 8 : 4], float s0, float s1, uint32_t (&d)[16]) {
  if constexpr (FP == 2) {
    // the bytes 0x7f and 0xff are NaN to the convert and +-480 to the format (no
    // quantizer writes them)
    uint32_t special = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      special |= (w[i] & 0x7f7f7f7fu) + 0x01010101u;
    }
    if (__builtin_expect(__any((special & 0x80808080u) != 0), 0)) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const uint32_t h = w[i / 2] >> (16 * (i % 2));
        const float s = i < 8 ? s0 : s1;
        d[i] = pack2<T>(walk_e4m3(h & 0xffu) * s, walk_e4m3((h >> 8) & 0xffu) * s);
        __builtin_amdgcn_sched_barrier(0); // (one at a time: no registers for this path)
      }
      return;
    }
  }
  walk_fp_widen<T, FP>(w, s0, s1, d, std::make_integer_sequence<int, 16>{});
}

template <typename T>
__device__ __forceinline__ float half_value(uint32_t v) {
  if constexpr (std::is_same<T, bf16_t>::value) {
    return __uint_as_float(v << 16);
  } else {
    return static_cast<float>(__builtin_bit_cast(f16_t, static_cast<uint16_t>(v)));
  }
}
// x . w over codes [k0, k1) of a row, term by term with the weights as dequantize gives
// them.  Only for sums that did not come out finite: an infinite x, or one whose
// products with the offset codes leave fp32, would otherwise turn every result of its
// row into inf - inf.  One thread per result, some hundred microseconds (a NaN in x ends
// it at once).
template <typename T, int BITS, int GS>
__device__ __forceinline__ float walk_terms(
    const T* x, const uint32_t* w, const T* scales, const T* biases, int k0, int k1) {
  float v = 0.0f;
#pragma unroll 1
  for (int k = k0; k < k1 && v == v; k += 32) {
    const uint32_t* p = w + static_cast<size_t>(k / 32) * BITS;
    const float s = to_f32(scales[k / GS]);
    const float b = to_f32(biases[k / GS]);
#pragma unroll 1
    for (int i = 0; i < 32; ++i) {
      const int d = i * BITS / 32;
      const int at = i * BITS % 32;
      const uint64_t high = at + BITS > 32 ? p[d + 1] : 0u; // the code goes on there
      const uint32_t c = static_cast<uint32_t>((high << 32 | p[d]) >> at) & ((1u << BITS) - 1u);
      v = fmaf(to_f32(x[k + i]), round_to<T>(fmaf(s, static_cast<float>(c), b)), v);
    }
  }
  return v;
}

// LDS: the [group][row] tables, then two x stages, which the final sums reuse.
template <int MR, int NW, int KW, int NPW>
constexpr size_t walk_x_bytes() {
  constexpr int mt = (MR + 15) / 16;
  constexpr size_t stages = 2u * KW * MR * 2 * kWkChunk;
  constexpr size_t sums = static_cast<size_t>(KW) * NW * NPW * mt * 1024;
  return stages > sums ? stages : sums;
}

template <typename T, int BITS, int GS, int FP, int MR, int NW, int KW, int NPW, int OCC>
__global__ __launch_bounds__(64 * NW * KW) __attribute__((amdgpu_waves_per_eu(OCC, OCC)))
void qmm_walk_kernel(WalkArgs wa) {
  constexpr int MT = (MR + 15) / 16;
  constexpr int NT = NW * NPW;             // 16-row tiles of W per workgroup
  constexpr int GT = FP != 0 ? 32 : GS;    // codes per table entry
  constexpr int NG = kWkChunk / GT;        // groups per chunk
  constexpr int OPG = FP != 0 ? 4 : GS / 32; // operands per group (affine)
  constexpr int kThreads = 64 * NW * KW;
  constexpr int kPieces = KW * MR * 16 / kThreads; // 16-byte pieces of x per thread and stage
  constexpr int kRowBytes = 2 * kWkChunk;
  constexpr int kStageBytes = KW * MR * kRowBytes;
  // how far ahead W and x are fetched: what the registers hold
  constexpr int kAhead = BITS >= 6 && (OCC == 4 || MR == 64) ? 2 : 4; // stages of W
  constexpr int XD = kPieces <= (OCC == 4 ? 2 : 4) ? 2 : 1; // sets of registers for x
  static_assert(KW * MR * 16 % kThreads == 0, "whole pieces per thread");
  using Codes = WalkCodes<T, BITS, FP != 0 ? 128 : GS>;
  constexpr float kOff = walk_offset<T, BITS>();

  extern __shared__ __align__(16) uint8_t smem[];
  const QmmArgs& a = wa.a;
  const int M = a.M, N = a.N, K = a.K;
  const int G = K / GT;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kw = wave % KW;
  const int nw = wave / KW;
  const int r = lane & 15;
  const int q = lane >> 4;
  const QmmProblem<T> p = resolve_problem<T>(a, blockIdx.z);
  const int tile_rows = wa.tile_rows;
  // gated form: the tiles of the second half are the same rows of the other matrix
  const bool glu = NW == 2 && wa.glu != 0;
  const int tiles_n = glu ? NPW : NT;
  const int n0 = blockIdx.x * (tiles_n * tile_rows);
  const uint8_t* w_base = p.w;
  if (glu && nw == 1) {
    w_base = reinterpret_cast<const uint8_t*>(a.w_alt);
  }
  // row of W (of its matrix) that row rr of a tile stands for
  const auto row_of = [&](int tile, int rr) {
    const int n = n0 + (tile < tiles_n ? tile : tile - tiles_n) * tile_rows +
        (rr < tile_rows ? rr : tile_rows - 1);
    return n < N ? n : N - 1;
  };
  const int stages_all = (K + KW * kWkChunk - 1) / (KW * kWkChunk);
  const int s0 = blockIdx.y * wa.range;
  const int s1 = s0 + wa.range < stages_all ? s0 + wa.range : stages_all;

  const int g0 = s0 * KW * NG;
  const int g_count = (s1 * KW * NG < G ? s1 * KW * NG : G) - g0;
  const int table_groups = wa.range * KW * NG < G ? wa.range * KW * NG : G;
  // [group of the range][NT * 16]: scales, and (affine) biases less offset * scale;
  // nvfp4: the two scales of 32 codes as a pair of bf16
  float* stab = reinterpret_cast<float*>(smem);
  float* btab = stab + table_groups * (NT * 16);
  uint8_t* xs = smem + static_cast<size_t>(table_groups) * NT * 16 * (FP != 0 ? 4 : 8);

  // ---- W: where this lane reads (32-bit offsets from a uniform base) ---------
  const uint32_t row_bytes = static_cast<uint32_t>(K) / 8 * BITS;
  constexpr uint32_t kLaneBytes = BITS == 8 ? 16 : 4 * BITS;  // one piece of a lane
  constexpr uint32_t kStageW = KW * kWkChunk / 8 * BITS;
  uint32_t wrow[NPW]; // start of the row
#pragma unroll
  for (int t = 0; t < NPW; ++t) {
    wrow[t] = static_cast<uint32_t>(row_of(nw * NPW + t, r)) * row_bytes;
  }
  WalkRegs<BITS> w[kAhead][NPW];
  const uint32_t w_lane = kw * (kWkChunk / 8 * BITS) + kLaneBytes * q;
  const auto fetch_w = [&](int s, WalkRegs<BITS> (&dst)[NPW]) {
    // (past the end of a row its last piece again: finite codes, and either x is
    // zero there or nothing is multiplied)
    const uint32_t at = s * kStageW + w_lane;
    const uint32_t last = row_bytes - kLaneBytes;
    const uint32_t off = at < last ? at : last;
    const uint32_t off2 = at + 64 < last ? at + 64 : last; // (8 bits)
#pragma unroll
    for (int t = 0; t < NPW; ++t) {
      dst[t].load(w_base, wrow[t] + off, wrow[t] + off2);
    }
  };
  // ---- x: pieces of 16 bytes, 16 of them a row of a chunk --------------------
  u32x4_t xr[XD][kPieces];
  uint32_t x_at[kPieces];   // byte offset of the piece in stage 0
  uint32_t x_last[kPieces]; // the last piece of that row of x
#pragma unroll
  for (int j = 0; j < kPieces; ++j) {
    const int piece = j * kThreads + tid;
    const int row = piece / (16 * KW); // KW chunks of a row are contiguous
    const int m = row < M ? row : M - 1;
    x_at[j] = static_cast<uint32_t>(m) * K * 2 + piece % (16 * KW) * 16;
    x_last[j] = static_cast<uint32_t>(m + 1) * K * 2 - 16;
  }
  const uint8_t* x_bytes = reinterpret_cast<const uint8_t*>(p.x);
  const auto fetch_x = [&](int s, u32x4_t (&dst)[kPieces]) {
#pragma unroll
    for (int j = 0; j < kPieces; ++j) {
      const uint32_t at = x_at[j] + s * (KW * kRowBytes);
      dst[j] = *reinterpret_cast<const u32x4_t*>(x_bytes + (at < x_last[j] ? at : x_last[j]));
    }
  };
  const int tail = K % kWkChunk != 0 ? K / (KW * kWkChunk) : -1; // stage where a chunk ends early
  const auto put_x = [&](int s, u32x4_t (&src)[kPieces]) {
    uint8_t* base = xs + (s & 1) * kStageBytes;
#pragma unroll
    for (int j = 0; j < kPieces; ++j) {
      const int piece = j * kThreads + tid;
      const int row = piece / (16 * KW);
      const int within = piece % (16 * KW);
      const int chunk = within / 16;
      const int slot = (within % 16) ^ (row & 15);
      u32x4_t v = src[j];
      if (BITS == 4 && FP == 0) { // elements 0,4 1,5 2,6 3,7
        v = u32x4_t{
            __builtin_amdgcn_perm(v.z, v.x, 0x05040100u), __builtin_amdgcn_perm(v.z, v.x, 0x07060302u),
            __builtin_amdgcn_perm(v.w, v.y, 0x05040100u), __builtin_amdgcn_perm(v.w, v.y, 0x07060302u)};
      }
      if (s == tail) {
        if (s * KW * kWkChunk + within * 8 >= K) {
          v = u32x4_t{0, 0, 0, 0};
        }
      }
      *reinterpret_cast<u32x4_t*>(base + (chunk * MR + row) * kRowBytes + slot * 16) = v;
    }
  };

  // ---- scales and biases -> LDS ----------------------------------------------
  // (lanes along the rows, so that the writes run over the banks; a row's groups
  // eight at a time where they start at 16 bytes, else one by one.  The first
  // eight are asked for before W, since loads complete in order.)
  constexpr int kRows = NT * 16;
  constexpr int kRuns = kThreads / kRows; // runs of groups in flight
  const int trow = tid % kRows;
  const int trun = tid / kRows;
  const T* srow = p.scales;
  const T* brow = p.biases;
  if constexpr (FP == 0) {
    const int tile = trow >> 4;
    if (glu && tile >= tiles_n) {
      srow = static_cast<const T*>(a.scales_alt);
      brow = static_cast<const T*>(a.biases_alt);
    }
    const size_t at = static_cast<size_t>(row_of(tile, trow & 15)) * G + g0;
    srow += at;
    brow += at;
  }
  // (the problem's own base counts: a stack's stride is the caller's)
  const bool eights = FP == 0 && ((G | g0 | g_count) & 7) == 0 &&
      ((reinterpret_cast<uintptr_t>(p.scales) | reinterpret_cast<uintptr_t>(p.biases)) & 15) == 0;
  const auto put_group = [&](int g, uint32_t s, uint32_t b) { // 16 bits each
    const float sv = half_value<T>(s);
    stab[g * kRows + trow] = sv * walk_unit<BITS>();
    btab[g * kRows + trow] = fmaf(-kOff, sv, half_value<T>(b));
  };
  const auto put_eight = [&](int g, const uint4& s, const uint4& b) {
    const uint32_t sd[4] = {s.x, s.y, s.z, s.w};
    const uint32_t bd[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      put_group(g + 2 * i, sd[i] & 0xffffu, bd[i] & 0xffffu);
      put_group(g + 2 * i + 1, sd[i] >> 16, bd[i] >> 16);
    }
  };
  uint4 s8 = make_uint4(0, 0, 0, 0);
  uint4 b8 = s8;
  if (eights) {
    const int g = trun * 8 < g_count ? trun * 8 : 0;
    s8 = *reinterpret_cast<const uint4*>(srow + g);
    b8 = *reinterpret_cast<const uint4*>(brow + g);
  }
  if constexpr (FP != 0) { // four scale bytes at a time (K is whole chunks), four loads at once
    // (as dwords where they start at one: scales may be a view at any byte)
    const uint8_t* s_base = static_cast<const uint8_t*>(a.scales) +
        static_cast<int64_t>(blockIdx.z) * a.sb_batch_stride;
    constexpr int kBytes = 32 / GS; // per entry
    const uint32_t first =
        static_cast<uint32_t>(row_of(trow >> 4, trow & 15)) * (K / GS) + g0 * kBytes;
    const int bytes = g_count * kBytes;
    const bool dwords = (reinterpret_cast<uintptr_t>(s_base) & 3) == 0;
    for (int g = trun * 4; g < bytes; g += 4 * 4 * kRuns) {
      uint32_t v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int at = g + j * 4 * kRuns;
        const uint8_t* four = s_base + first + (at < bytes ? at : 0);
        if (dwords) { // uniform
          v[j] = *reinterpret_cast<const uint32_t*>(four);
        } else {
          v[j] = four[0] | four[1] << 8 | four[2] << 16 | static_cast<uint32_t>(four[3]) << 24;
        }
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int at = g + j * 4 * kRuns;
        if (at < bytes) {
          if constexpr (FP == 3) {
            float f[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              f[i] = walk_e4m3((v[j] >> (8 * i)) & 0xffu);
            }
#pragma unroll
            for (int i = 0; i < 2; ++i) {
              stab[(at / 2 + i) * kRows + trow] =
                  __uint_as_float(pack2<bf16_t>(f[2 * i], f[2 * i + 1]));
            }
          } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              stab[(at + i) * kRows + trow] = walk_e8m0((v[j] >> (8 * i)) & 0xffu);
            }
          }
        }
      }
    }
  }
  fetch_x(s0, xr[0]);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int u = 0; u < kAhead; ++u) { // as in the loop: stage j asks for W (j + kAhead), x (j + 1 + XD)
    fetch_w(s0 + u, w[u]);
    if (u == 0) {
      __builtin_amdgcn_sched_barrier(0);
      put_x(s0, xr[0]);
    }
    if (u >= kAhead - XD) {
      fetch_x(s0 + 1 + u - (kAhead - XD), xr[(1 + u - (kAhead - XD)) % XD]);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  if (eights) {
    if (trun * 8 < g_count) {
      put_eight(trun * 8, s8, b8);
    }
    for (int g = (trun + kRuns) * 8; g < g_count; g += kRuns * 8) {
      put_eight(
          g, *reinterpret_cast<const uint4*>(srow + g), *reinterpret_cast<const uint4*>(brow + g));
    }
  } else if (FP == 0) {
    for (int g = trun; g < g_count; g += kRuns) {
      put_group(g, __builtin_bit_cast(uint16_t, srow[g]), __builtin_bit_cast(uint16_t, brow[g]));
    }
  }
  __syncthreads();

  floatx4 acc[NPW][MT];
#pragma unroll
  for (int t = 0; t < NPW; ++t) {
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      acc[t][m] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    }
  }
  float xsum[MT]; // quad q: the sum of x over the q-th of four groups
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    xsum[m] = 0.0f;
  }
  const uint32_t one2 = pack2<T>(1.0f, 1.0f);
  const uint4 ones = make_uint4(one2, one2, one2, one2);

  uint32_t mask = Codes::kMask;
  uint32_t magic = Codes::kOffsetBits;
  asm("" : "+v"(mask));
  asm("" : "+v"(magic));

  // byte offset of this lane's pieces within a row of x, per operand
  int xoff[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    xoff[i] = ((Codes::k_of(i, q) / 8) ^ ((r % MR) & 15)) * 16;
  }

  // What the biases add for the (up to) four groups collected in xsum; `first` is
  // the stage the first of them belongs to.
  const auto add_biases = [&](int first) {
    const int g = ((first + q / NG) * KW + kw) * NG + q % NG - g0;
    const int gi = g < g_count ? g : 0; // (xsum is zero there)
#pragma unroll
    for (int t = 0; t < NPW; ++t) {
      const float b = btab[gi * (NT * 16) + (nw * NPW + t) * 16 + r];
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        acc[t][m] = __builtin_amdgcn_mfma_f32_16x16x4f32(b, xsum[m], acc[t][m], 0, 0, 0);
      }
    }
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      xsum[m] = 0.0f;
    }
  };

  for (int sb = s0; sb < s1; sb += kWkUnroll) {
#pragma unroll
    for (int u = 0; u < kWkUnroll; ++u) {
      const int s = sb + u; // (stages past the range: x is zero, nothing is multiplied)
      const int c = s * KW + kw; // this wavefront's chunk
      const uint8_t* xbase = xs + (s & 1) * kStageBytes + (kw * MR + r % MR) * kRowBytes;
      // x of the first half of the chunk: on its way while W is waited for
      uint4 xf[2][MT];
      const auto read_x = [&](int half) {
#pragma unroll
        for (int o = 0; o < 2; ++o) {
#pragma unroll
          for (int m = 0; m < MT; ++m) {
            xf[o][m] = *reinterpret_cast<const uint4*>(
                xbase + m * 16 * kRowBytes + xoff[2 * half + o]);
          }
        }
      };
      read_x(0);
      float fs[NPW][2]; // scales of the floating-point modes
      if constexpr (FP != 0) {
        const int gc = c * NG - g0 < g_count ? c * NG - g0 : 0;
#pragma unroll
        for (int t = 0; t < NPW; ++t) {
          const float* at = stab +
              (gc + (FP == 2 ? q / 2 : q)) * kRows + (nw * NPW + t) * 16 + r;
          fs[t][0] = at[0];
          fs[t][1] = 0.0f;
          if constexpr (FP == 2) {
            fs[t][1] = at[2 * kRows];
          } else if constexpr (FP == 3) {
            const uint32_t pair = __float_as_uint(fs[t][0]);
            fs[t][0] = __uint_as_float(pair << 16);
            fs[t][1] = __uint_as_float(pair & 0xffff0000u);
          }
        }
      }
      uint32_t kept[NPW][FP != 0 ? 16 : Codes::kKept];
#pragma unroll
      for (int t = 0; t < NPW; ++t) {
        uint32_t d[BITS];
        w[u % kAhead][t].get(d);
        if constexpr (FP != 0) {
          walk_fp_operands<T, FP>(d, fs[t][0], fs[t][1], kept[t]);
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            asm volatile("" : "+v"(kept[t][i]));
          }
        } else {
          Codes::regroup(d, kept[t], mask, magic);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      fetch_w(s + kAhead, w[u % kAhead]);
      if (s < s1 && c * kWkChunk < K) {
        floatx4 ch[NPW][MT];
        floatx4 cx[MT];
#pragma unroll
        for (int half = 0; half < 2; ++half) {
          if (half == 1) {
            read_x(1);
          }
#pragma unroll
          for (int o = 0; o < 2; ++o) {
            const int i = 2 * half + o;   // operand of the chunk
            if constexpr (FP != 0) {
#pragma unroll
              for (int t = 0; t < NPW; ++t) {
                const uint4 op = make_uint4(
                    kept[t][4 * i], kept[t][4 * i + 1], kept[t][4 * i + 2], kept[t][4 * i + 3]);
#pragma unroll
                for (int m = 0; m < MT; ++m) {
                  acc[t][m] = mfma16<T>(op, xf[o][m], acc[t][m]);
                }
              }
              continue;
            }
            const int g = i / OPG;        // its group
            if (i % OPG == 0) {
#pragma unroll
              for (int m = 0; m < MT; ++m) {
                cx[m] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int t = 0; t < NPW; ++t) {
                  ch[t][m] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
                }
              }
            }
#pragma unroll
            for (int m = 0; m < MT; ++m) {
              cx[m] = mfma16<T>(ones, xf[o][m], cx[m]);
            }
#pragma unroll
            for (int t = 0; t < NPW; ++t) {
              uint4 op;
              if constexpr (FP == 0) {
                op = Codes::operand(kept[t], i, mask, magic);
              }
#pragma unroll
              for (int m = 0; m < MT; ++m) {
                ch[t][m] = mfma16<T>(op, xf[o][m], ch[t][m]);
              }
            }
            if (i % OPG == OPG - 1) {
              const int gi = c * NG + g - g0;
              const int gt = gi < g_count ? gi : 0; // (a group past K: x is zero)
#pragma unroll
              for (int m = 0; m < MT; ++m) {
                xsum[m] = q == (u * NG + g) % 4 ? cx[m][0] : xsum[m];
              }
#pragma unroll
              for (int t = 0; t < NPW; ++t) {
                const floatx4 sc = *reinterpret_cast<const floatx4*>(
                    &stab[gt * (NT * 16) + (nw * NPW + t) * 16 + 4 * q]);
#pragma unroll
                for (int m = 0; m < MT; ++m) {
#pragma unroll
                  for (int j = 0; j < 4; ++j) {
                    acc[t][m][j] = fmaf(sc[j], ch[t][m][j], acc[t][m][j]);
                  }
                }
              }
            }
          }
        }
      }
      if (FP == 0 && (u + 1) * NG % 4 == 0) {
        add_biases(s + 1 - 4 / NG);
      }
      // x of the next stage, late: it has had XD stages to arrive
      put_x(s + 1, xr[(u + 1) % XD]);
      __builtin_amdgcn_sched_barrier(0);
      fetch_x(s + 1 + XD, xr[(u + 1) % XD]);
      __syncthreads();
    }
  }

  // ---- the KW partial sums meet ----------------------------------------------
  float* sums = reinterpret_cast<float*>(xs); // [kw][tile][m tile][lane][4]
#pragma unroll
  for (int t = 0; t < NPW; ++t) {
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      *reinterpret_cast<floatx4*>(
          sums + (((kw * NT + nw * NPW + t) * MT + m) * 64 + lane) * 4) = acc[t][m];
    }
  }
  __syncthreads();
  const bool planes = gridDim.y > 1;
  float* plane = planes ? wa.planes +
          (static_cast<size_t>(blockIdx.y) * gridDim.z + blockIdx.z) * static_cast<size_t>(M) * N
                        : nullptr;
  float factor = 1.0f; // weights quantized with a tensor-wide scale
  if (FP == 3 && a.out_scale != nullptr) {
    factor = *a.out_scale / (448.0f * 6.0f);
  }
  // lanes along the rows of W
  constexpr int kSumRows = NT * 16;
  constexpr int kSumM = kThreads / kSumRows;
  const int row = tid % kSumRows;
  const int t = row / 16;
  const int rr = row % 16;
  const int n = n0 + t * tile_rows + rr;
  if (t < tiles_n && rr < tile_rows && n < N) {
    const auto sum_of = [&](int tile, int m) {
      float v = 0.0f;
#pragma unroll
      for (int k = 0; k < KW; ++k) {
        v += sums[(((k * NT + tile) * MT + m / 16) * 64 + (rr / 4) * 16 + m % 16) * 4 + rr % 4];
      }
      return v * factor;
    };
    const auto finish = [&](int m, auto&& sum) {
      const float v = sum(t, m);
      const size_t at = static_cast<size_t>(m) * N + n;
      if (glu) {
        // the roundings of the unfused chain: both products, the sigmoid, gate *
        // sigmoid and the result
        const float g = round_to<T>(v);
        const float up = round_to<T>(sum(t + NT / 2, m));
        const float sg = round_to<T>(1.0f / (1.0f + __expf(-g)));
        p.out[at] = from_f32<T>(round_to<T>(g * sg) * up);
      } else if (planes) {
        plane[at] = v;
      } else {
        p.out[at] = from_f32<T>(p.valid ? v : 0.0f);
      }
    };
    bool finite = true;
    for (int m = tid / kSumRows; m < M; m += kSumM) {
      finish(m, [&](int tile, int row_of_x) {
        const float v = sum_of(tile, row_of_x);
        finite = finite && __builtin_isfinite(v);
        return v;
      });
    }
    if constexpr (FP == 0) {
      if (!finite) { // (this thread's results alone)
        const int k1 = s1 * KW * kWkChunk < K ? s1 * KW * kWkChunk : K;
        for (int m = tid / kSumRows; m < M; m += kSumM) {
          finish(m, [&](int tile, int row_of_x) {
            const float v = sum_of(tile, row_of_x);
            if (__builtin_isfinite(v)) {
              return v;
            }
            const bool alt = tile >= tiles_n;
            const size_t at = static_cast<size_t>(n);
            return walk_terms<T, BITS, GS>(
                p.x + static_cast<size_t>(row_of_x) * K,
                (alt ? a.w_alt : reinterpret_cast<const uint32_t*>(p.w)) + at * (K / 32) * BITS,
                (alt ? static_cast<const T*>(a.scales_alt) : p.scales) + at * G,
                (alt ? static_cast<const T*>(a.biases_alt) : p.biases) + at * G,
                s0 * KW * kWkChunk, k1);
          });
        }
      }
    }
  }
}

template <typename T, int BITS, int GS, int FP, int MR, int NW, int KW, int NPW, int OCC>
int launch_walk_shape(const WalkArgs& wa, int table_groups, const dim3& grid, hipStream_t s) {
  const auto kernel = &qmm_walk_kernel<T, BITS, GS, FP, MR, NW, KW, NPW, OCC>;
  const size_t lds = static_cast<size_t>(table_groups) * NW * NPW * 16 * (FP != 0 ? 4 : 8) +
      walk_x_bytes<MR, NW, KW, NPW>();
  if (lds > 64 * 1024) {
    static const hipError_t attr = hipFuncSetAttribute(
        reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
        160 * 1024);
    MLXROCM_HIP_TRY(attr);
  }
  kernel<<<grid, 64 * NW * KW, lds, s>>>(wa);
  MLXROCM_HIP_TRY(hipGetLastError());
  return MLXROCM_OK;
}

template <typename T, int BITS, int GS, int FP>
int launch_walk_rows(
    const WalkArgs& wa, const WalkPlan& pl, int table_groups, const dim3& grid, hipStream_t s) {
#define WALK_CASE(C, R, ...)                                                                  \
  if (pl.config == C && pl.mr == R) {                                                         \
    return launch_walk_shape<T, BITS, GS, FP, R, __VA_ARGS__>(wa, table_groups, grid, s);     \
  }
  WALK_CASE(0, 8, 1, 8, 1, 4)
  WALK_CASE(0, 16, 1, 8, 1, 4)
  WALK_CASE(0, 32, 1, 8, 1, 2)
  WALK_CASE(1, 16, 2, 4, 2, 2)
  WALK_CASE(1, 32, 2, 4, 2, 2)
  WALK_CASE(1, 48, 2, 4, 2, 2)
  WALK_CASE(1, 64, 2, 4, 2, 2)
  WALK_CASE(2, 8, 2, 4, 1, 4)
  WALK_CASE(2, 16, 2, 4, 1, 4)
  WALK_CASE(3, 8, 2, 4, 2, 4)
#undef WALK_CASE
  return fail(MLXROCM_UNSUPPORTED, "[qmm_walk] no shape for %d rows", pl.mr);
}

template <int BITS>
int launch_walk_bits(
    const WalkArgs& wa, const WalkPlan& pl, int gs, int dtype, int table_groups, const dim3& grid,
    hipStream_t s) {
  return dispatch_group(gs, [&](auto g) {
    constexpr int GS = decltype(g)::value;
    return dtype == MLXROCM_BFLOAT16
        ? launch_walk_rows<bf16_t, BITS, GS, 0>(wa, pl, table_groups, grid, s)
        : launch_walk_rows<f16_t, BITS, GS, 0>(wa, pl, table_groups, grid, s);
  });
}

} // namespace

// per width, in the .hip file of that width
using WalkLauncher = int(
    const WalkArgs&, const WalkPlan&, int gs, int dtype, int table_groups, const dim3&,
    hipStream_t);
WalkLauncher launch_walk_2, launch_walk_3, launch_walk_4, launch_walk_5, launch_walk_6,
    launch_walk_8;
// the floating-point modes: gs holds the mlxrocm_fp_mode
WalkLauncher launch_walk_fp;

} // namespace mlxrocm
