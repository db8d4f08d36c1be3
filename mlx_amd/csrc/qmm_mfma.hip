// qmm_mfma.hip -- launchers of the prefill tile kernel (qmm_mfma_tile.h):
// transpose=true with the caller's scale layout or the two transposed images,
// split K, float32 through split bf16 operands, [K, N] weights, grouped gathers.
// The launches that read the (scale, bias) pair image are in qmm_mfma_pairs.hip.
#include "qmm_mfma_tile.h"

namespace mlxrocm {

bool qmm_mfma_supported(const QmmArgs& a, int gs, int bits, int dtype, bool transpose) {
  (void)gs;
  if (dtype == MLXROCM_FLOAT32) {
    return false;
  }
  if (!transpose && !(bits == 4 || bits == 8)) {
    return false; // [K, N] weights: the column loader reads whole words per 8 codes
  }
  return a.K % kBK == 0 && a.K >= kBK;
}

namespace {

// [K, N] weights (transpose=false), 4- or 8-bit; TO = float when K is split.
template <typename T, typename TO, int NT>
int launch_wn(const QmmArgs& a, int gs_shift, int bits, dim3 grid, hipStream_t s, int k_splits) {
  if (bits == 4) {
    return launch_variant<T, T, TO, 4, NT, false, true>(a, gs_shift, grid, s, k_splits);
  }
  return launch_variant<T, T, TO, 8, NT, false, true>(a, gs_shift, grid, s, k_splits);
}

} // namespace

namespace {

// [K][G] -> [G][K] for scales and biases (blockIdx.z: which of the two, then
// which batch entry), 32 x 32 tiles through LDS.
template <typename T>
__global__ __launch_bounds__(256) void transpose_sb_kernel(
    const T* scales,
    const T* biases,
    T* out,
    int K,
    int G,
    int64_t src_stride) {
  __shared__ T tile[32][33];
  const int which = blockIdx.z & 1;
  const int l = blockIdx.z >> 1;
  const T* src = (which == 0 ? scales : biases) + l * src_stride;
  T* dst = out + (static_cast<size_t>(l) * 2 + which) * K * G;
  const int tx = threadIdx.x & 31;
  const int ty = threadIdx.x >> 5; // 0..7
  const int g0 = blockIdx.x * 32;
  const int k0 = blockIdx.y * 32;
#pragma unroll
  for (int r = ty; r < 32; r += 8) {
    const int k = k0 + r;
    const int g = g0 + tx;
    if (k < K && g < G) {
      tile[r][tx] = src[static_cast<size_t>(k) * G + g];
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = ty; r < 32; r += 8) {
    const int g = g0 + r;
    const int k = k0 + tx;
    if (k < K && g < G) {
      dst[static_cast<size_t>(g) * K + k] = tile[tx][r];
    }
  }
}

} // namespace

// Scratch bytes of the transposed scale / bias image of `batches` weight matrices.
size_t qmm_n_sb_bytes(int K, int G, int batches, int dtype) {
  return static_cast<size_t>(2) * batches * K * G * dtype_size(dtype);
}

// out: per batch entry the [G][K] scales followed by the [G][K] biases.
int transpose_sb_for_qmm_n(
    const void* scales,
    const void* biases,
    void* out,
    int K,
    int G,
    int batches,
    int64_t src_stride,
    int dtype,
    hipStream_t s) {
  const dim3 grid((G + 31) / 32, (K + 31) / 32, 2 * batches);
  if (grid.y > 65535u || grid.z > 65535u) {
    return fail(MLXROCM_UNSUPPORTED, "[qmm] K=%d or batch=%d exceed the grid", K, batches);
  }
  MLXROCM_REHEARSE("transpose_sb");
  if (dtype == MLXROCM_FLOAT32) {
    transpose_sb_kernel<float><<<grid, 256, 0, s>>>(
        static_cast<const float*>(scales), static_cast<const float*>(biases),
        static_cast<float*>(out), K, G, src_stride);
  } else if (dtype == MLXROCM_BFLOAT16) {
    transpose_sb_kernel<bf16_t><<<grid, 256, 0, s>>>(
        static_cast<const bf16_t*>(scales), static_cast<const bf16_t*>(biases),
        static_cast<bf16_t*>(out), K, G, src_stride);
  } else {
    transpose_sb_kernel<f16_t><<<grid, 256, 0, s>>>(
        static_cast<const f16_t*>(scales), static_cast<const f16_t*>(biases),
        static_cast<f16_t*>(out), K, G, src_stride);
  }
  MLXROCM_HIP_TRY(hipGetLastError());
  return MLXROCM_OK;
}

// [K, N] weights: the width of the tiles and the number of K ranges that finish
// first.  What a launch costs, in nanoseconds, from timing every width and number of
// ranges on eight shapes (errors up to 15 %): a K-step takes longer the wider its
// tile, and the more compute units work beside it (the clock gives way: 224 columns
// 1.46 us with 76 of 256 units at work, 1.78 with 228); a tile costs some
// microseconds before and after its steps; ranges cost the fp32 planes, written and
// read again.
TilePlan qmm_n_plan(int M, int N, int K, int L) {
  const long cus = compute_units();
  const long mt = (M + kBM - 1) / kBM;
  const long steps = K / kBK;
  auto cost = [&](int nt, int splits) -> double {
    const long wgs = mt * ((N + 32 * nt - 1) / (32 * nt)) * (splits > 1 ? splits : L);
    const double rounds = static_cast<double>((wgs + cus - 1) / cus);
    const double busy = static_cast<double>(wgs) / (rounds * cus);
    const double step = (400.0 + 110.0 * nt) * (1.0 + 0.3 * busy);
    double ns = rounds * (static_cast<double>((steps + splits - 1) / splits) * step + 4000.0);
    if (splits > 1) {
      ns += 3000.0 + static_cast<double>(splits) * M * N * 4.0 / 5000.0; // 5 TB/s
    }
    return ns;
  };
  TilePlan best = {choose_nt(M, N, L), 1};
  if (L != 1 || (static_cast<int64_t>(M) * N) % 4 != 0) {
    return best;
  }
  // a margin of 8 % for the plain launch: it needs no planes
  double best_ns = cost(best.nt, 1) / 1.08;
  for (int nt = 6; nt <= 7; ++nt) { // the widths built with fp32 planes
    const long tiles = mt * ((N + 32 * nt - 1) / (32 * nt));
    for (int splits = 2; splits <= 16 && splits * 8 <= steps && splits * tiles <= 2 * cus;
         ++splits) {
      const double ns = cost(nt, splits);
      if (ns < best_ns) {
        best = {nt, splits};
        best_ns = ns;
      }
    }
  }
  return best;
}

// transpose=false on the matrix cores: same tiles, column loader for W.  a.scales
// / a.biases point at the transposed images made by transpose_sb_for_qmm_n.
// Tiles of 224 columns as for transpose=true (245 registers; 256 columns spill):
// dy [1024, 14336] x W [14336, 4096] at 4 bits takes 133 us in three K ranges of
// them (228 workgroups), against 206 in three of 192 columns (264: a second round
// for eight workgroups) and 157 in two.
int launch_qmm_mfma_n(
    const QmmArgs& a, int gs, int bits, int dtype, const TilePlan& pl, hipStream_t s) {
  const int gs_shift = shift_of(gs);
  const int nt = pl.nt;
  MLXROCM_REHEARSE("qmm_n_tile(ksplit=%d)", pl.splits);
  const dim3 grid(
      (a.N + 32 * nt - 1) / (32 * nt), (a.M + kBM - 1) / kBM, pl.splits > 1 ? pl.splits : a.L);
  auto run = [&](auto tval) -> int {
    using T = decltype(tval);
    if (pl.splits > 1) {
      return nt == 6 ? launch_wn<T, float, 6>(a, gs_shift, bits, grid, s, pl.splits)
                     : launch_wn<T, float, 7>(a, gs_shift, bits, grid, s, pl.splits);
    }
    switch (nt) {
      case 5:
        return launch_wn<T, T, 5>(a, gs_shift, bits, grid, s, 1);
      case 6:
        return launch_wn<T, T, 6>(a, gs_shift, bits, grid, s, 1);
      default:
        return launch_wn<T, T, 7>(a, gs_shift, bits, grid, s, 1);
    }
  };
  return dtype == MLXROCM_BFLOAT16 ? run(bf16_t{}) : run(f16_t{});
}

int launch_qmm_mfma(const QmmArgs& a, int gs, int bits, int dtype, hipStream_t s) {
  const int gs_shift = shift_of(gs);
  // (128-wide tiles, which would make x [2048, .] x W [4096, .] exactly one round
  // of 256 workgroups, were measured and are not offered: a K-step costs nearly
  // the same whatever the tile's width -- the x tile, the barrier and the
  // dequantization work per thread do not shrink with it -- so 4096 x 4096 went
  // from 83 to 82 us at 2048 rows and from 292 to 338 us at 8192)
  const int nt = choose_nt(a.M, a.N, a.L);
  MLXROCM_REHEARSE("qmm_t_tile(nt=%d)", nt);
  const dim3 grid((a.N + 32 * nt - 1) / (32 * nt), (a.M + kBM - 1) / kBM, a.L);
  auto run = [&](auto tval) -> int {
    using T = decltype(tval);
    return dispatch_bits(bits, [&](auto bval) {
      constexpr int B = decltype(bval)::value;
      switch (nt) {
        case 5:
          return launch_variant<T, T, T, B, 5, false>(a, gs_shift, grid, s);
        case 6:
          return launch_variant<T, T, T, B, 6, false>(a, gs_shift, grid, s);
        default:
          return launch_variant<T, T, T, B, 7, false>(a, gs_shift, grid, s);
      }
    });
  };
  return dtype == MLXROCM_BFLOAT16 ? run(bf16_t{}) : run(f16_t{});
}

// How many ranges to cut K into so that a launch with few tiles still fills the
// compute units (1 = no split): only for a single problem, and every range
// keeps at least eight steps.  nt: the width of the launcher's tiles.
int qmm_mfma_k_splits(int M, int N, int K, int L, int nt) {
  if (L != 1) {
    return 1;
  }
  const long cus = compute_units();
  const long tiles = static_cast<long>((M + kBM - 1) / kBM) * ((N + 32 * nt - 1) / (32 * nt));
  const long steps = K / kBK;
  long s = cus / tiles;
  if (s > steps / 8) {
    s = steps / 8;
  }
  // (up to 16 ranges: a narrow N over a long K -- 3584 x 18944, 128 rows: 45.6 us
  // against 57.5 with at most 8, 2048 x 8192: 26.7 against 32.7)
  if (s > 16) {
    s = 16;
  }
  if (s < 2) {
    return 1;
  }
  // Results stored by the element (N no multiple of four), 16-bit tiles: ranges where the
  // steps they save, some 0.4 us each beside narrower tiles without ranges, are worth more
  // than the planes, written and read at about 10 GB/ms.  us without / with two ranges,
  // bf16: 1495 x 4099 x 1024 38 / 44, 6334 x 1001 x 1344 (mxfp4) 41 / 46; 990 x 3001 x 1344
  // (nvfp4) 42 / 37, 319 x 10762 x 2048 53 / 43.
  if (nt != kSplitFp32Width && N % 4 != 0) {
    const double saved = 0.4 * static_cast<double>(steps - (steps + s - 1) / s);
    if (saved < 1.0 + static_cast<double>(k_split_plane(M, N)) * s * 4e-7) {
      return 1;
    }
  }
  return static_cast<int>(s);
}

// Fitted to 14500 calls of 65..2048 rows at every width (errors of 7 %): a step of 64 codes
// costs by the rows of x in a tile and by the share of the compute units at work; from 512
// rows on scales and biases are transposed first.
double qmm_mfma_us(int M, int N, int K, int bits) {
  const int splits = qmm_mfma_k_splits(M, N, K, 1);
  const int nt = splits > 1 ? 7 : choose_nt(M, N, 1);
  const long cus = compute_units();
  const long wgs = static_cast<long>((M + kBM - 1) / kBM) * ((N + 32 * nt - 1) / (32 * nt)) * splits;
  const double rounds = static_cast<double>((wgs + cus - 1) / cus);
  const double steps = rounds * ((K / kBK + splits - 1) / splits);
  const double width = bits == 3 ? 0.06 : bits == 5 ? 0.17 : bits == 6 ? 0.13 : bits == 8 ? 0.06 : 0.0;
  double us = 11.1 + steps * (width + 0.68 * (M < kBM ? M : kBM) / kBM +
                              0.71 * static_cast<double>(wgs) / (rounds * cus));
  if (splits > 1) {
    us += 5.2 + 0.9e-6 * static_cast<double>(k_split_plane(M, N)) * splits;
  }
  return M >= 512 ? us + 1.8 : us;
}

// 16-bit operands with K cut into k_splits ranges: `a.out` points at k_splits
// fp32 planes (k_split_plane(); reduce_k_splits adds them up into y).
int launch_qmm_mfma_ksplit(
    const QmmArgs& a,
    int gs,
    int bits,
    int dtype,
    int k_splits,
    hipStream_t s) {
  constexpr int kNT = 7;
  const int gs_shift = shift_of(gs);
  const dim3 grid((a.N + 32 * kNT - 1) / (32 * kNT), (a.M + kBM - 1) / kBM, k_splits);
  MLXROCM_REHEARSE("qmm_t_tile(ksplit=%d)", k_splits);
  auto run = [&](auto tval) -> int {
    using T = decltype(tval);
    return dispatch_bits(bits, [&](auto bval) {
      constexpr int B = decltype(bval)::value;
      return launch_variant<T, T, float, B, kNT, false>(a, gs_shift, grid, s, k_splits);
    });
  };
  return dtype == MLXROCM_BFLOAT16 ? run(bf16_t{}) : run(f16_t{});
}

namespace {

// Four consecutive elements of a row of the planes per thread, with 16-byte loads: rows of
// the planes are whole 16-byte pieces, also where rows of y (N) are not.  There the row is
// found by one 32-bit division and the store starts at any element.  With four elements of
// y per thread, each with a 64-bit division and loads of its own, whole calls took 2 to 10 %
// longer: 1660 x 803 x 5888 mxfp4 48.5 us against 42.9, 1285 x 4099 x 8192 4-bit 122 against 116.
template <typename TO>
__global__ __launch_bounds__(256) void reduce_k_splits_kernel(
    const float* partial,
    TO* out,
    size_t pieces, // of a plane
    int N,
    int k_splits) {
  const size_t piece = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (piece >= pieces) {
    return;
  }
  const float4* p = reinterpret_cast<const float4*>(partial) + piece;
  float4 acc = *p;
  for (int z = 1; z < k_splits; ++z) {
    const float4 v = p[z * pieces];
    acc.x += v.x;
    acc.y += v.y;
    acc.z += v.z;
    acc.w += v.w;
  }
  // (one store, wherever an element may start)
  auto store = [&](TO* y) {
    if constexpr (sizeof(TO) == 4) {
      typedef float __attribute__((ext_vector_type(4), aligned(4))) four;
      *reinterpret_cast<four*>(y) = four{acc.x, acc.y, acc.z, acc.w};
    } else {
      typedef uint32_t __attribute__((ext_vector_type(2), aligned(2))) four;
      *reinterpret_cast<four*>(y) = four{pack2<TO>(acc.x, acc.y), pack2<TO>(acc.z, acc.w)};
    }
  };
  if ((N & 3) == 0) {
    store(out + piece * 4);
    return;
  }
  const uint32_t row_pieces = static_cast<uint32_t>(k_split_row(N)) / 4;
  const uint32_t m = static_cast<uint32_t>(piece) / row_pieces; // (the launcher checks the size)
  const int n = static_cast<int>(static_cast<uint32_t>(piece) - m * row_pieces) * 4;
  TO* y = out + static_cast<size_t>(m) * N + n;
  if (n + 4 <= N) {
    store(y);
    return;
  }
  const float v[3] = {acc.x, acc.y, acc.z};
#pragma unroll
  for (int e = 0; e < 3; ++e) {
    if (n + e < N) {
      y[e] = static_cast<TO>(v[e]);
    }
  }
}

} // namespace

// y[M, N] = sum of the k_splits fp32 planes (k_split_plane(M, N) elements apart);
// y must be 16-byte aligned.
int reduce_k_splits(
    const void* partial, void* out, int M, int N, int k_splits, int dtype, hipStream_t s) {
  const size_t pieces = k_split_plane(M, N) / 4;
  const size_t blocks = (pieces + 255) / 256;
  if (blocks > 0x7fffffffull || (N % 4 != 0 && pieces > 0xffffffffull)) {
    return fail(MLXROCM_UNSUPPORTED, "[qmm] output too large for the split-K reduction");
  }
  MLXROCM_REHEARSE("reduce_k_splits(%d)", k_splits);
  const float* p = static_cast<const float*>(partial);
  const unsigned g = static_cast<unsigned>(blocks);
  return dispatch_dtype(dtype, [&](auto tval) {
    using T = decltype(tval);
    reduce_k_splits_kernel<T><<<g, 256, 0, s>>>(
        p, static_cast<T*>(out), pieces, N, k_splits);
    MLXROCM_HIP_TRY(hipGetLastError());
    return static_cast<int>(MLXROCM_OK);
  });
}

// fp32 operands: `a.x` already points at the [hi | lo | hi] bf16 image of x
// (split_x_for_mfma) and a.x_batch_stride counts its elements (M * 3 K).
int launch_qmm_mfma_split(const QmmArgs& a, int gs, int bits, hipStream_t s, int k_splits) {
  // six column blocks: with fp32 scales and the weight split, seven spill
  // registers to scratch memory (measured 620 against 415 us at 1024 x 11008 x 4096)
  constexpr int kNT = kSplitFp32Width;
  const int gs_shift = shift_of(gs);
  const dim3 grid(
      (a.N + 32 * kNT - 1) / (32 * kNT), (a.M + kBM - 1) / kBM, k_splits > 1 ? k_splits : a.L);
  MLXROCM_REHEARSE("qmm_t_tile_split_fp32(ksplit=%d)", k_splits);
  return dispatch_bits(bits, [&](auto bval) {
    constexpr int B = decltype(bval)::value;
    return launch_variant<bf16_t, float, float, B, kNT, false>(a, gs_shift, grid, s, k_splits);
  });
}

namespace {

// 8 consecutive fp32 of x -> 8 bf16 high parts and 8 bf16 low parts, written to
// blocks 0/2 and 1 of the element's group of three 64-wide blocks.
__global__ __launch_bounds__(256) void split_x_kernel(
    const float* x,
    bf16_t* xs,
    size_t rows,
    int K) {
  const size_t unit = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const size_t units_per_row = static_cast<size_t>(K) / 8;
  if (unit >= rows * units_per_row) {
    return;
  }
  const size_t row = unit / units_per_row;
  const int k = static_cast<int>(unit - row * units_per_row) * 8;
  const float4 v0 = *reinterpret_cast<const float4*>(x + row * K + k);
  const float4 v1 = *reinterpret_cast<const float4*>(x + row * K + k + 4);
  const float v[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
  uint32_t hi[4], lo[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float h0 = static_cast<float>(static_cast<bf16_t>(v[2 * i]));
    const float h1 = static_cast<float>(static_cast<bf16_t>(v[2 * i + 1]));
    hi[i] = pack2<bf16_t>(v[2 * i], v[2 * i + 1]);
    lo[i] = pack2<bf16_t>(v[2 * i] - h0, v[2 * i + 1] - h1);
  }
  bf16_t* dst = xs + row * (3 * static_cast<size_t>(K)) + static_cast<size_t>(k / 64) * 192 + k % 64;
  const uint4 h = make_uint4(hi[0], hi[1], hi[2], hi[3]);
  *reinterpret_cast<uint4*>(dst) = h;
  *reinterpret_cast<uint4*>(dst + 64) = make_uint4(lo[0], lo[1], lo[2], lo[3]);
  *reinterpret_cast<uint4*>(dst + 128) = h;
}

} // namespace

size_t split_x_bytes(size_t rows, int K) {
  return rows * 3 * static_cast<size_t>(K) * sizeof(bf16_t);
}

int split_x_for_mfma(const void* x, void* xs, size_t rows, int K, hipStream_t s) {
  const size_t units = rows * (static_cast<size_t>(K) / 8);
  const size_t blocks = (units + 255) / 256;
  if (blocks > 0x7fffffffull) {
    return fail(MLXROCM_UNSUPPORTED, "[qmm] x is too large to split");
  }
  MLXROCM_REHEARSE("split_x");
  split_x_kernel<<<static_cast<unsigned>(blocks), 256, 0, s>>>(
      static_cast<const float*>(x), static_cast<bf16_t*>(xs), rows, K);
  MLXROCM_HIP_TRY(hipGetLastError());
  return MLXROCM_OK;
}

// Gather grouped by expert: `a` carries the tile list; one grid row per
// possible tile, rows past the device-side tile count exit at once.
int launch_qmm_mfma_grouped(const QmmArgs& a, int gs, int bits, int dtype, hipStream_t s) {
  MLXROCM_REHEARSE("qmm_t_tile_grouped");
  constexpr int kNT = 7;
  const int gs_shift = shift_of(gs);
  const dim3 grid(
      (a.N + 32 * kNT - 1) / (32 * kNT), gather_group_max_tiles(a.L, a.n_experts, kGroupLargeTile), 1);
  auto run = [&](auto tval) -> int {
    using T = decltype(tval);
    return dispatch_bits(bits, [&](auto bval) {
      constexpr int B = decltype(bval)::value;
      return launch_variant<T, T, T, B, kNT, true>(a, gs_shift, grid, s);
    });
  };
  return dtype == MLXROCM_BFLOAT16 ? run(bf16_t{}) : run(f16_t{});
}

// The same for [K, N] weights (transpose=false): a.scales / a.biases point at
// the transposed images of all experts (transpose_sb_for_qmm_n), a.sb_batch_stride
// is the distance between two experts' images.
int launch_qmm_mfma_grouped_n(const QmmArgs& a, int gs, int bits, int dtype, hipStream_t s) {
  MLXROCM_REHEARSE("qmm_n_tile_grouped");
  constexpr int kNT = 6;
  const int gs_shift = shift_of(gs);
  const dim3 grid(
      (a.N + 32 * kNT - 1) / (32 * kNT), gather_group_max_tiles(a.L, a.n_experts, kGroupLargeTile), 1);
  auto run = [&](auto tval) -> int {
    using T = decltype(tval);
    if (bits == 4) {
      return launch_variant<T, T, T, 4, kNT, true, true>(a, gs_shift, grid, s);
    }
    return launch_variant<T, T, T, 8, kNT, true, true>(a, gs_shift, grid, s);
  };
  return dtype == MLXROCM_BFLOAT16 ? run(bf16_t{}) : run(f16_t{});
}

} // namespace mlxrocm
