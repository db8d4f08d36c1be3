// qmm_mid.h -- x @ dequantize(w)^T for some tens to some hundreds of rows of x:
// tiles of up to 128 rows of x by 128 rows of W, packed W and x both walking
// through LDS several K-steps ahead.
//
// What bounds this regime: 128 x 2876 x 9152 at 4 bits reads 13 MB (3 us) and does
// 6.7 GFLOP (4 us at the rate of a large product), so neither: a workgroup's steps follow
// one another, and there are few.  The 256-row tile kernel (qmm_mfma_tile.h) asks for W one
// K-step of 64 ahead and dequantizes it through LDS: 1.5 us a step however few rows it has.
// Here a step of 128 takes 1.0 us with 66 rows and 1.15 with 128 (32000 x 4096 and 8192, one
// workgroup per compute unit): 0.07 for the matrix instructions of every 16 rows and 0.6
// for the vector instructions that dequantize, which add up; without any loads it is 1.1.
// us per call, 4-bit g64 bf16, tile kernel -> this: 4096 x 14336, 96 rows 37.2 -> 26.6;
// 4096 x 4096, 256 rows 29.5 -> 22.3; 1024 x 1024, 512 rows 23.8 -> 13.5.
// (Dequantizing at the head of the step that uses it: 52 us instead of 44 at 32000 x 4096,
// 128 rows.  The loads of a step spread between its matrix instructions: no gain.)
//  * a K-step is 128 codes.  Direct-to-LDS loads bring the packed rows of W (16 bytes
//    a lane: 128 codes are whole 16-byte pieces at every width) and the rows of x; three
//    to five stages fit 160 KB, so two to four steps are in flight.  One barrier a step.
//    Scales and biases go to a table in LDS ahead of the steps that read them.
//  * a wavefront owns 32 rows of W and 64 of the 128 codes of a step, and dequantizes
//    them in registers straight into the operands of its matrix instructions: no
//    dequantized W in LDS, each code once per workgroup.  (Eight wavefronts along N
//    alone would read x from LDS twice as often, which then takes longer than the
//    matrix instructions; the halves of K meet once, at the end.)
//  * the order of k within a step is the same permutation for both operands: lane
//    quarter q holds codes 16 q .. 16 q + 15 of its wavefront's 64, eight for each of
//    two matrix instructions, so a lane's codes lie side by side at every width and
//    belong to one group.
#pragma once

#include "mfma_dequant.h"
#include "mfma_loads.h"
#include "qmm_args.h"

namespace mlxrocm {

namespace {

constexpr int kMidThreads = 512;
constexpr int kMidBN = 128; // rows of W of a tile
constexpr int kMidBK = 128; // codes of a K-step
constexpr size_t kMidLds = 163840;

// LDS bytes of a stage: x, packed W
constexpr int mid_x_bytes(int mf) {
  return mf * 16 * kMidBK * 2;
}
constexpr int mid_w_bytes(int bits) {
  return kMidBN * kMidBK * bits / 8;
}
// (the table of (scale, bias) pairs in front of the stages: mid_table_groups())
constexpr int mid_table_bytes(int mf, int bits) {
  return mid_table_groups(mf, bits) * kMidBN * 4;
}
// stages of x; W has one more, since its codes are widened a step before they are used
constexpr int mid_stages(int mf, int bits) {
  const int fit = (static_cast<int>(kMidLds) - mid_table_bytes(mf, bits) - mid_w_bytes(bits)) /
      (mid_x_bytes(mf) + mid_w_bytes(bits));
  return fit > 5 ? 5 : fit;
}
constexpr size_t mid_stage_bytes(int mf, int bits) {
  return static_cast<size_t>(mid_stages(mf, bits)) * mid_x_bytes(mf) +
      static_cast<size_t>(mid_stages(mf, bits) + 1) * mid_w_bytes(bits);
}

// Lets all but the `LEFT` newest loads of this wavefront land and its LDS reads end (the
// stage they read is filled again behind the barrier), then meets the others.
template <int LEFT>
__device__ __forceinline__ void wait_and_meet() {
  static_assert(LEFT < 64, "vmcnt counts to 63");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(LEFT) : "memory");
}

// The 2 x 16 codes of a lane's two rows for one step, dequantized a pair at a time.
template <typename T, int BITS>
struct MidCodes {
  uint32_t w[2][BITS];
  float s[2], b[2];
  PairDequant<T, BITS> dq[2];

  // pair P (0..15): rows take turns, so that two chains run side by side
  template <int P>
  __device__ __forceinline__ void pair(uint4 (&out)[2][2]) {
    constexpr int f = P % 2;
    constexpr int q = P / 2; // codes 2 q, 2 q + 1 of 16
    const uint32_t v = dq[f].template pair<q>(w[f], s[f], b[f]);
    if constexpr (q % 4 == 0) {
      out[f][q / 4].x = v;
    } else if constexpr (q % 4 == 1) {
      out[f][q / 4].y = v;
    } else if constexpr (q % 4 == 2) {
      out[f][q / 4].z = v;
    } else {
      out[f][q / 4].w = v;
    }
  }
  template <int FROM, int... I>
  __device__ __forceinline__ void pairs(uint4 (&out)[2][2], std::integer_sequence<int, I...>) {
    (pair<FROM + I>(out), ...);
  }
};

template <int M, int MF, typename F>
__device__ __forceinline__ void for_tiles(F&& fn) {
  if constexpr (M < MF) {
    fn(std::integral_constant<int, M>{});
    for_tiles<M + 1, MF>(fn);
  }
}

// MF: tiles of 16 rows of x (a workgroup has up to 16 MF of them).  splits > 1: `a.out`
// is that many fp32 planes, blockIdx.z the range of K.  K % 128 == 0; operands below 4 GiB.
template <typename T, int BITS, int MF>
__global__ __launch_bounds__(kMidThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void qmm_mid_kernel(
    QmmArgs a, int gs_shift, int rows_per_tile, int splits) {
  extern __shared__ __align__(16) uint8_t smem_all[];
  constexpr int kTable = mid_table_bytes(MF, BITS);
  uint32_t* table = reinterpret_cast<uint32_t*>(smem_all); // [group][row]: scale low, bias high
  uint8_t* xs_lds = smem_all + kTable;
  constexpr int kX = mid_x_bytes(MF);
  constexpr int kW = mid_w_bytes(BITS);
  constexpr int kStages = mid_stages(MF, BITS);
  static_assert(kStages >= 3, "two steps in flight");
  uint8_t* ws_lds = xs_lds + kStages * kX;
  constexpr int kXLoads = kX / 1024 / 8;          // per wavefront and step
  constexpr int kWUnits = kW / 1024;              // of the workgroup
  constexpr int kWLoads = (kWUnits + 7) / 8;      // per wavefront: surplus ones repeat the last
  constexpr int kLoads = kXLoads + kWLoads;
  static_assert(MF % 2 == 0 && kX % 8192 == 0, "x loads are dealt out evenly");

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave & 3;  // rows 32 wn .. 32 wn + 31 of the tile
  const int wk = wave >> 2; // codes 64 wk .. 64 wk + 63 of a step
  const int l16 = lane & 15;
  const int q = lane >> 4;

  const int N = a.N;
  const int K = a.K;
  const int n0 = blockIdx.x * kMidBN;
  const int m0 = blockIdx.y * rows_per_tile;
  const int rows = a.M - m0 < rows_per_tile ? a.M - m0 : rows_per_tile;
  const int G = K >> gs_shift;

  // this range's steps: the first (steps % splits) ranges have one more
  const int all_steps = K / kMidBK;
  const int z = blockIdx.z;
  const int each = all_steps / splits;
  const int extra = all_steps - each * splits;
  const int first = z * each + (z < extra ? z : extra);
  const int steps = each + (z < extra ? 1 : 0);

  // ---- byte offsets of this lane's loads from the bases of a step ----
  // x: an instruction covers four rows of 256 bytes; piece p of row r is kept at
  // p ^ (r % 16), so that the 16 rows of a fragment read lie in different banks
  uint32_t x_off[kXLoads];
#pragma unroll
  for (int j = 0; j < kXLoads; ++j) {
    const int r = (wave * kXLoads + j) * 4 + q;
    const int m = m0 + (r < rows ? r : rows - 1);
    x_off[j] = static_cast<uint32_t>(m) * (static_cast<uint32_t>(K) * 2u) +
        static_cast<uint32_t>(l16 ^ (r & 15)) * 16u;
  }
  uint32_t w_off[kWLoads];
  int w_unit[kWLoads];
#pragma unroll
  for (int j = 0; j < kWLoads; ++j) {
    const int unit = wave + 8 * j < kWUnits ? wave + 8 * j : kWUnits - 1;
    w_unit[j] = unit;
    const int piece = unit * 64 + lane;
    const int r = piece / BITS;
    const int n = n0 + r < N ? n0 + r : N - 1;
    w_off[j] = static_cast<uint32_t>(n) * (static_cast<uint32_t>(K) / 8u * BITS) +
        static_cast<uint32_t>(piece - r * BITS) * 16u;
  }
  const char* x_base = static_cast<const char*>(a.x);
  const char* w_base = reinterpret_cast<const char*>(a.w);

  const uint32_t lds_x = __builtin_amdgcn_readfirstlane(lds_address(xs_lds));
  const uint32_t lds_w = __builtin_amdgcn_readfirstlane(lds_address(ws_lds));
  auto fetch_w = [&](int step, int stage) {
    const char* ws = w_base + static_cast<size_t>(step) * (kMidBK / 8 * BITS);
#pragma unroll
    for (int j = 0; j < kWLoads; ++j) {
      dma16(lds_w + stage * kW + w_unit[j] * 1024, w_off[j], ws);
    }
  };
  auto fetch_x = [&](int step, int stage) {
    const char* xs = x_base + static_cast<size_t>(step) * (kMidBK * 2);
#pragma unroll
    for (int j = 0; j < kXLoads; ++j) {
      dma16(lds_x + stage * kX + (wave * kXLoads + j) * 1024, x_off[j], xs);
    }
  };

  floatx4 acc[2][MF];
#pragma unroll
  for (int f = 0; f < 2; ++f) {
#pragma unroll
    for (int m = 0; m < MF; ++m) {
      acc[f][m] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    }
  }

  // ---- where this lane reads ----
  constexpr int kCodeBytes = 2 * BITS;                   // of 16 codes
  constexpr int kCodeWords = (kCodeBytes + 3) / 4;       // dwords that hold them, aligned
  constexpr bool kHalf = kCodeBytes % 4 != 0;            // odd widths: may start mid-dword
  const int code_byte = (4 * wk + q) * kCodeBytes;       // in a row of a stage
  const bool mid_dword = kHalf && (q & 1) != 0;
  const int w_read = (wn * 32 + l16) * (kMidBK / 8 * BITS) + (code_byte & ~3);
  const int group = (64 * wk + 16 * q) >> gs_shift;      // of the step
  const uint32_t* sb_read = table + group * kMidBN + wn * 32 + l16;
  const int x_row = l16 * (kMidBK * 2);
  const int x_piece0 = ((wk * 8 + 2 * q) ^ l16) * 16;
  const int x_piece1 = ((wk * 8 + 2 * q + 1) ^ l16) * 16;

  using Codes = MidCodes<T, BITS>;
  auto read_codes = [&](Codes& c, int stage, int step_in_table) {
#pragma unroll
    for (int f = 0; f < 2; ++f) {
      const uint32_t* wp = reinterpret_cast<const uint32_t*>(
          ws_lds + stage * kW + w_read + f * 16 * (kMidBK / 8 * BITS));
      if constexpr (kHalf) {
        uint32_t raw[kCodeWords];
#pragma unroll
        for (int i = 0; i < kCodeWords; ++i) {
          raw[i] = wp[i];
        }
#pragma unroll
        for (int i = 0; i < kCodeWords; ++i) {
          const uint32_t next = i + 1 < kCodeWords ? raw[i + 1] : 0u;
          c.w[f][i] = mid_dword ? (raw[i] >> 16) | (next << 16) : raw[i];
        }
      } else {
#pragma unroll
        for (int i = 0; i < kCodeWords; ++i) {
          c.w[f][i] = wp[i];
        }
      }
#pragma unroll
      for (int i = kCodeWords; i < BITS; ++i) {
        c.w[f][i] = 0u;
      }
      const uint32_t pair = sb_read[((step_in_table * kMidBK) >> gs_shift) * kMidBN + f * 16];
      c.s[f] = half_of<T>(pair, 0) * PairDequant<T, BITS>::kCodeScale;
      c.b[f] = half_of<T>(pair, 1);
    }
  };

  // One step: the matrix instructions of this step's operands, the dequantization of the
  // next step's between them.
  uint4 wf[2][2];
  auto compute = [&](int stage, Codes& c) {
    const uint8_t* xp = xs_lds + stage * kX + x_row;
    uint4 next[2][2];
    for_tiles<0, MF / 2>([&](auto mval) {
      constexpr int m = 2 * decltype(mval)::value;
      uint4 x[2][2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        x[i][0] = *reinterpret_cast<const uint4*>(xp + (m + i) * 16 * (kMidBK * 2) + x_piece0);
        x[i][1] = *reinterpret_cast<const uint4*>(xp + (m + i) * 16 * (kMidBK * 2) + x_piece1);
      }
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          acc[0][m + i] = mfma16<T>(wf[0][h], x[i][h], acc[0][m + i]);
          acc[1][m + i] = mfma16<T>(wf[1][h], x[i][h], acc[1][m + i]);
        }
      }
      constexpr int from = 16 * m / MF;
      constexpr int to = 16 * (m + 2) / MF;
      c.template pairs<from>(next, std::make_integer_sequence<int, to - from>{});
    });
    wf[0][0] = next[0][0];
    wf[0][1] = next[0][1];
    wf[1][0] = next[1][0];
    wf[1][1] = next[1][1];
  };

  // ---- K loop, in segments whose scales and biases fit the table.  x of step t and W of
  // step t + 1 are asked for together and waited for while the kStages - 2 pairs behind
  // them are in flight; the stages that were read last before the barrier of step t are
  // filled again behind it ----
  const int segment = mid_table_groups(MF, BITS) * (1 << gs_shift) / kMidBK; // steps
  const T* scales = static_cast<const T*>(a.scales);
  const T* biases = static_cast<const T*>(a.biases);
  for (int done = 0; done < steps; done += segment) {
    const int here = steps - done < segment ? steps - done : segment;
    const int from = first + done;
    __syncthreads(); // the stages and the table of the segment before have been read
    fetch_w(from, 0);
#pragma unroll
    for (int t = 0; t < kStages - 1; ++t) {
      if (t + 1 < here) {
        fetch_w(from + t + 1, t + 1);
      }
      if (t < here) {
        fetch_x(from + t, t);
      }
    }
    // a quarter of the threads' lanes along a row's groups: whole lines of the caller's arrays
    {
      const int g0 = (from * kMidBK) >> gs_shift;
      const int groups = (here * kMidBK) >> gs_shift;
      const int r = tid >> 2;
      const int n = n0 + r < N ? n0 + r : N - 1;
      const size_t row = static_cast<size_t>(n) * G + g0;
      for (int g = tid & 3; g < groups; g += 16) {
        uint16_t v[4][2];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int gi = g + 4 * i < groups ? g + 4 * i : g;
          v[i][0] = __builtin_bit_cast(uint16_t, scales[row + gi]);
          v[i][1] = __builtin_bit_cast(uint16_t, biases[row + gi]);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (g + 4 * i < groups) {
            table[(g + 4 * i) * kMidBN + r] = v[i][0] | static_cast<uint32_t>(v[i][1]) << 16;
          }
        }
      }
    }
    int x_stage = 0, x_spare = kStages - 1; // of step t; where step t + kStages - 1 goes
    int w_next = 1, w_spare = kStages;      // of step t + 1; where step t + kStages goes
    for (int t = 0; t < here; ++t) {
      const int left = here - 1 - t; // steps behind this one
      if (left >= kStages - 1) {
        wait_and_meet<(kStages - 2) * kLoads>();
      } else if (kStages > 4 && left == 3) {
        wait_and_meet<2 * kLoads + kXLoads>();
      } else if (kStages > 3 && left == 2) {
        wait_and_meet<kLoads + kXLoads>();
      } else if (left == 1) {
        wait_and_meet<kXLoads>();
      } else {
        wait_and_meet<0>();
      }
      if (left >= kStages) {
        fetch_w(from + t + kStages, w_spare);
      }
      if (left >= kStages - 1) {
        fetch_x(from + t + kStages - 1, x_spare);
      }
      Codes c;
      if (t == 0) {
        read_codes(c, 0, 0);
        c.template pairs<0>(wf, std::make_integer_sequence<int, 16>{});
      }
      // (behind the last step: the codes of the stage before, for nothing)
      read_codes(c, left > 0 ? w_next : 0, left > 0 ? t + 1 : t);
      compute(x_stage, c);
      x_spare = x_stage;
      x_stage = x_stage + 1 == kStages ? 0 : x_stage + 1;
      w_spare = w_spare == kStages ? 0 : w_spare + 1;
      w_next = w_next == kStages ? 0 : w_next + 1;
    }
  }

  // ---- the halves of K meet: each wavefront gives the other of its pair half of the
  // tiles of x and finishes the rest ----
  __syncthreads(); // (no load is in flight: the last step waited for all)
  float4* swap = reinterpret_cast<float4*>(xs_lds);
  constexpr int kHalfTiles = MF / 2;
#pragma unroll
  for (int f = 0; f < 2; ++f) {
#pragma unroll
    for (int i = 0; i < kHalfTiles; ++i) {
      const floatx4 v = wk == 0 ? acc[f][kHalfTiles + i] : acc[f][i];
      swap[((wave * 2 + f) * kHalfTiles + i) * 64 + lane] = make_float4(v[0], v[1], v[2], v[3]);
    }
  }
  __syncthreads();
  const int other = wave ^ 4;
#pragma unroll
  for (int f = 0; f < 2; ++f) {
#pragma unroll
    for (int i = 0; i < kHalfTiles; ++i) {
      const float4 o = swap[((other * 2 + f) * kHalfTiles + i) * 64 + lane];
      const floatx4 v = wk == 0 ? acc[f][i] : acc[f][kHalfTiles + i];
      const float y[4] = {v[0] + o.x, v[1] + o.y, v[2] + o.z, v[3] + o.w};
      const int mr = (wk * kHalfTiles + i) * 16 + l16;
      const int n = n0 + wn * 32 + f * 16 + q * 4;
      if (mr >= rows || n >= N) {
        continue;
      }
      const size_t m = static_cast<size_t>(m0 + mr);
      if (splits > 1) {
        // (rows of a plane are whole 16-byte pieces)
        float* plane = static_cast<float*>(a.out) + static_cast<size_t>(z) * k_split_plane(a.M, N);
        *reinterpret_cast<float4*>(plane + m * k_split_row(N) + n) =
            make_float4(y[0], y[1], y[2], y[3]);
      } else {
        T* out = static_cast<T*>(a.out) + m * N + n;
        if ((N & 3) == 0) {
          *reinterpret_cast<uint2*>(out) = make_uint2(pack2<T>(y[0], y[1]), pack2<T>(y[2], y[3]));
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            if (n + j < N) {
              out[j] = static_cast<T>(y[j]);
            }
          }
        }
      }
    }
  }
}

template <typename T, int BITS, int MF>
int mid_variant(const QmmArgs& a, int gs_shift, const MidPlan& pl, hipStream_t s) {
  constexpr size_t stages = mid_stage_bytes(MF, BITS);
  constexpr size_t smem = mid_table_bytes(MF, BITS) + stages;
  static_assert(stages >= static_cast<size_t>(8) * MF * 64 * 16, "the halves of K meet in the stages");
  auto kern = qmm_mid_kernel<T, BITS, MF>;
  static const hipError_t attr = hipFuncSetAttribute(
      reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
      static_cast<int>(smem));
  MLXROCM_HIP_TRY(attr);
  const dim3 grid((a.N + kMidBN - 1) / kMidBN, pl.tiles, pl.splits);
  kern<<<grid, kMidThreads, smem, s>>>(a, gs_shift, pl.rows, pl.splits);
  MLXROCM_HIP_TRY(hipGetLastError());
  return static_cast<int>(MLXROCM_OK);
}

template <typename T>
int mid_launch(const QmmArgs& a, int gs, int bits, const MidPlan& pl, hipStream_t s) {
  const int gs_shift = gs == 32 ? 5 : (gs == 64 ? 6 : 7);
  return dispatch_bits(bits, [&](auto bval) -> int {
    constexpr int B = decltype(bval)::value;
    if (pl.rows <= 64) {
      return mid_variant<T, B, 4>(a, gs_shift, pl, s);
    }
    if (pl.rows <= 96) {
      return mid_variant<T, B, 6>(a, gs_shift, pl, s);
    }
    if constexpr (B == 8) {
      return fail(MLXROCM_UNSUPPORTED, "[qmm] %d rows of x in a tile of 8-bit codes", pl.rows);
    } else {
      return mid_variant<T, B, 8>(a, gs_shift, pl, s);
    }
  });
}

} // namespace

} // namespace mlxrocm
