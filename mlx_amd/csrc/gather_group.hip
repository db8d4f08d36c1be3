// gather_group.hip -- groups the index pairs of a GatherQMM call by expert so
// that the matrix-core GEMM reads every expert's weights once for all the rows
// routed to it (the reference loops over the pairs one GEMV at a time,
// mlx/backend/cpu/quantized.cpp:700-747; the Metal backend groups sorted runs,
// mlx/backend/metal/quantized.cpp:1905-1923).
//
// Three small kernels fill a caller-provided workspace (one workgroup does all
// three steps in a single launch when there are at most 16384 pairs):
//   count    a histogram per workgroup in LDS, then one global atomic per
//            workgroup and expert into counts[expert] (one global atomic per
//            pair serializes on the few counters, worst for sorted indices);
//            pairs with an index out of range are left out and their output
//            rows are zero-filled here;
//   plan     one workgroup: exclusive scan of the counts -> first sorted
//            position of every expert, and the list of tiles {expert, first
//            position, rows} of up to tile_rows rows (256 for the tile GEMMs, 32
//            for the few-row kernel when the groups are small); the tile count
//            stays on the device;
//   scatter  perm[position] = pair: rank inside the workgroup from an LDS
//            counter, the workgroup's base from one atomic on a per-expert cursor.
// The order inside an expert's run is arbitrary; every output row depends on
// its own x row only, so the result does not depend on it.
#include "qmm_args.h"

namespace mlxrocm {

namespace {

constexpr int kMaxExperts = 4096; // plan kernel keeps the counts in LDS

template <typename T>
__global__ __launch_bounds__(256) void group_count_kernel(
    const uint32_t* lhs,
    const uint32_t* rhs,
    int n_indices,
    int x_batches,
    int n_experts,
    int32_t* counts,
    T* out,
    int N) {
  __shared__ int32_t hist[kMaxExperts];
  for (int e = threadIdx.x; e < n_experts; e += blockDim.x) {
    hist[e] = 0;
  }
  __syncthreads();
  const int l = blockIdx.x * blockDim.x + threadIdx.x;
  if (l < n_indices) {
    const uint32_t xi = lhs[l];
    const uint32_t wi = rhs[l];
    if (xi < static_cast<uint32_t>(x_batches) && wi < static_cast<uint32_t>(n_experts)) {
      atomicAdd(&hist[wi], 1);
    } else {
      T* row = out + static_cast<size_t>(l) * N;
      for (int n = 0; n < N; ++n) {
        row[n] = static_cast<T>(0.0f);
      }
    }
  }
  __syncthreads();
  for (int e = threadIdx.x; e < n_experts; e += blockDim.x) {
    if (hist[e] != 0) {
      atomicAdd(&counts[e], hist[e]);
    }
  }
}

// First sorted position of every expert and the list of tiles from the counts in LDS, by all
// threads of the workgroup: in the order of their experts, or (by_height) those that are full
// first and the others behind them by eighths of their height, highest first.
constexpr int kHeights = 8;
__device__ __forceinline__ void plan_tiles(
    int n_experts,
    int tile_rows, // a power of two
    bool by_height,
    const int32_t* cnt,
    int32_t* first_pos,
    int32_t* first_tile,
    int32_t* offsets,
    int32_t* tiles,
    int32_t* n_tiles) {
  __shared__ int32_t next[kHeights]; // of the tiles of a height: how many, then the next one
  const int shift = __ffs(tile_rows) - 1;
  auto height = [&](int rows) { return ((rows * kHeights - 1) >> shift); };
  if (threadIdx.x < kHeights) {
    next[threadIdx.x] = 0;
  }
  __syncthreads();
  for (int e = threadIdx.x; by_height && e < n_experts; e += blockDim.x) {
    const int rest = cnt[e] & (tile_rows - 1);
    if (rest != 0) {
      atomicAdd(&next[height(rest)], 1);
    }
  }
  __syncthreads();
  // sums over the experts before each, 64 experts at a time by the first wavefront (one thread
  // after the other: a round trip to LDS per expert)
  if (threadIdx.x < 64) {
    const int lane = threadIdx.x;
    int pos = 0;
    int tile = 0;
    for (int first = 0; first < n_experts; first += 64) {
      const int e = first + lane;
      const int c = e < n_experts ? cnt[e] : 0;
      const int t = (c + (by_height ? 0 : tile_rows - 1)) >> shift;
      int c_sum = c;
      int t_sum = t;
      for (int d = 1; d < 64; d *= 2) {
        const int c_below = __shfl_up(c_sum, d, 64);
        const int t_below = __shfl_up(t_sum, d, 64);
        c_sum += lane >= d ? c_below : 0;
        t_sum += lane >= d ? t_below : 0;
      }
      if (e < n_experts) {
        first_pos[e] = pos + c_sum - c;
        first_tile[e] = tile + t_sum - t;
      }
      pos += __shfl(c_sum, 63, 64);
      tile += __shfl(t_sum, 63, 64);
    }
    if (lane == 0) {
      for (int h = kHeights - 1; h >= 0; --h) {
        const int n = next[h];
        next[h] = tile;
        tile += n;
      }
      n_tiles[0] = tile;
      n_tiles[1] = pos; // pairs with both indices in range
    }
  }
  __syncthreads();
  for (int e = threadIdx.x; e < n_experts; e += blockDim.x) {
    offsets[e] = first_pos[e];
    const int c = cnt[e];
    int t = first_tile[e];
    for (int r = 0; r < c; r += tile_rows, ++t) {
      const int rows = c - r < tile_rows ? c - r : tile_rows;
      if (by_height && rows < tile_rows) {
        t = atomicAdd(&next[height(rows)], 1); // (the expert's last)
      }
      tiles[3 * t + 0] = e;
      tiles[3 * t + 1] = first_pos[e] + r;
      tiles[3 * t + 2] = rows;
    }
  }
}

__global__ __launch_bounds__(256) void group_plan_kernel(
    int n_experts,
    int tile_rows,
    bool by_height,
    const int32_t* counts,
    int32_t* offsets,
    int32_t* tiles,
    int32_t* n_tiles) {
  __shared__ int32_t cnt[kMaxExperts];
  __shared__ int32_t first_pos[kMaxExperts];
  __shared__ int32_t first_tile[kMaxExperts];
  for (int e = threadIdx.x; e < n_experts; e += blockDim.x) {
    cnt[e] = counts[e];
  }
  __syncthreads();
  plan_tiles(n_experts, tile_rows, by_height, cnt, first_pos, first_tile, offsets, tiles, n_tiles);
}

__global__ __launch_bounds__(256) void group_scatter_kernel(
    const uint32_t* lhs,
    const uint32_t* rhs,
    int n_indices,
    int x_batches,
    int n_experts,
    const int32_t* offsets,
    int32_t* cursor,
    int32_t* perm) {
  __shared__ int32_t hist[kMaxExperts]; // pairs of this workgroup per expert, then its base
  for (int e = threadIdx.x; e < n_experts; e += blockDim.x) {
    hist[e] = 0;
  }
  __syncthreads();
  const int l = blockIdx.x * blockDim.x + threadIdx.x;
  bool live = false;
  uint32_t wi = 0;
  int rank = 0;
  if (l < n_indices) {
    const uint32_t xi = lhs[l];
    wi = rhs[l];
    live = xi < static_cast<uint32_t>(x_batches) && wi < static_cast<uint32_t>(n_experts);
    if (live) {
      rank = atomicAdd(&hist[wi], 1);
    }
  }
  __syncthreads();
  for (int e = threadIdx.x; e < n_experts; e += blockDim.x) {
    const int c = hist[e];
    if (c != 0) {
      hist[e] = atomicAdd(&cursor[e], c);
    }
  }
  __syncthreads();
  if (live) {
    perm[offsets[wi] + hist[wi] + rank] = l;
  }
}

// All three steps in one workgroup, for calls with so few pairs that four
// launches cost more than the work: counts, scan and cursors stay in LDS, no
// global atomics, nothing to clear beforehand.
constexpr int kFusedThreads = 1024;
constexpr int kFusedMaxPairs = 16384;

// counter[key] += 1 for every lane with `live`; returns the lane's old value.  The
// lanes of a wavefront that share a key find each other by ballots over the key's
// bits and go together: one atomic instruction per wavefront, an address per key.
// (One per lane serializes on the counters of a few experts.)
__device__ __forceinline__ int wave_counter_add(
    int32_t* counter, uint32_t key, bool live, int key_bits) {
  const int lane = threadIdx.x & 63;
  uint64_t same = __ballot(live);
  for (int b = 0; b < key_bits; ++b) {
    const uint64_t ones = __ballot((key >> b) & 1u);
    same &= (key >> b) & 1u ? ones : ~ones;
  }
  const int leader = __ffsll(static_cast<unsigned long long>(same)) - 1;
  int base = 0;
  if (live && lane == leader) {
    base = atomicAdd(&counter[key], __popcll(same));
  }
  base = __shfl(base, leader < 0 ? 0 : leader, 64);
  return base + __popcll(same & ((uint64_t{1} << lane) - 1));
}

// What bounds it: the vector instructions of one compute unit, about 70 per wavefront and call of
// wave_counter_add.  A pair's expert, and its rank among that expert's, which the count gives by the
// way, stay in registers: the scatter adds them to the expert's first position and counts nothing
// again.  us of a routed MLP whose pairs it groups, counting twice -> once: 64 experts 2048 x
// 1408, 2048 tokens to 6 265 -> 260 (this kernel under a trace 23.0 -> 19.4), 32 experts 1024 x
// 1024, 900 tokens to 4 69.2 -> 67.3; 8 experts 4096 x 14336, 600 tokens 552 -> 553.
template <typename T>
__global__ __launch_bounds__(kFusedThreads) void group_fused_kernel(
    const uint32_t* lhs,
    const uint32_t* rhs,
    int n_indices,
    int x_batches,
    int n_experts,
    int key_bits,
    int tile_rows,
    bool by_height,
    int32_t* offsets,
    int32_t* tiles,
    int32_t* n_tiles,
    int32_t* perm,
    T* out,
    int N) {
  constexpr int kPer = kFusedMaxPairs / kFusedThreads;
  constexpr uint32_t kNone = 0xffffffffu;
  __shared__ int32_t cnt[kMaxExperts];
  __shared__ int32_t first_pos[kMaxExperts];
  __shared__ int32_t first_tile[kMaxExperts];
  uint32_t key[kPer];
  int rank[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int l = i * kFusedThreads + threadIdx.x;
    key[i] = kNone;
    if (l < n_indices) {
      const uint32_t xi = lhs[l];
      const uint32_t wi = rhs[l];
      key[i] = xi < static_cast<uint32_t>(x_batches) && wi < static_cast<uint32_t>(n_experts)
          ? wi : kNone - 1;
    }
  }
  for (int e = threadIdx.x; e < n_experts; e += kFusedThreads) {
    cnt[e] = 0;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    if (i * kFusedThreads < n_indices) { // (uniform: whole wavefronts stay together)
      rank[i] =
          wave_counter_add(cnt, key[i], key[i] < static_cast<uint32_t>(n_experts), key_bits);
      if (key[i] == kNone - 1) {
        T* row = out + static_cast<size_t>(i * kFusedThreads + threadIdx.x) * N;
        for (int n = 0; n < N; ++n) {
          row[n] = static_cast<T>(0.0f);
        }
      }
    }
  }
  __syncthreads();
  plan_tiles(n_experts, tile_rows, by_height, cnt, first_pos, first_tile, offsets, tiles, n_tiles);
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    if (i * kFusedThreads < n_indices && key[i] < static_cast<uint32_t>(n_experts)) {
      perm[first_pos[key[i]] + rank[i]] = i * kFusedThreads + threadIdx.x;
    }
  }
}

__global__ __launch_bounds__(256) void fill_i32_kernel(int32_t* p, int n, int32_t v) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    p[i] = v;
  }
}

size_t align_up(size_t v, size_t a) {
  return (v + a - 1) / a * a;
}

} // namespace

int gather_group_max_tiles(int n_indices, int n_experts, int tile_rows) {
  // every expert may end on a partial tile
  return (n_indices + tile_rows - 1) / tile_rows + n_experts;
}

size_t gather_group_workspace_bytes(int n_indices, int n_experts) {
  if (n_indices <= 0 || n_experts <= 0 || n_experts > kMaxExperts) {
    return 0;
  }
  const size_t ints = static_cast<size_t>(3) * n_experts + 4 +
      static_cast<size_t>(3) * gather_group_max_tiles(n_indices, n_experts, kGroupSmallTile) +
      n_indices; // sized for the smaller tile
  return align_up(ints * sizeof(int32_t), 256);
}

void bind_gather_group(QmmArgs& a, int tile_rows, void* workspace) {
  const int E = a.n_experts;
  int32_t* ws = static_cast<int32_t*>(workspace);
  int32_t* n_tiles = ws + 3 * E;
  int32_t* tiles = n_tiles + 4;
  a.group_tiles = tiles;
  a.group_perm = tiles + 3 * gather_group_max_tiles(a.L, E, tile_rows);
  a.group_ntiles = n_tiles;
  a.group_tile_rows = tile_rows;
}

// Fills the workspace and points the grouped-mode fields of `a` into it.
int launch_gather_group(
    QmmArgs& a, int dtype, int tile_rows, bool by_height, void* workspace, hipStream_t s) {
  const int E = a.n_experts;
  const int n = a.L;
  int32_t* ws = static_cast<int32_t*>(workspace);
  int32_t* counts = ws;
  int32_t* cursor = counts + E;
  int32_t* offsets = cursor + E;
  int32_t* n_tiles = offsets + E;
  int32_t* tiles = n_tiles + 4;
  int32_t* perm = tiles + 3 * gather_group_max_tiles(n, E, tile_rows);

  a.group_tiles = tiles;
  a.group_perm = perm;
  a.group_ntiles = n_tiles;
  MLXROCM_REHEARSE(n <= kFusedMaxPairs ? "gather_group(fused)" : "gather_group(3 kernels)");
  a.group_tile_rows = tile_rows;
  if (n <= kFusedMaxPairs) {
    int key_bits = 1;
    while ((1 << key_bits) < E) {
      ++key_bits;
    }
    if (dtype == MLXROCM_BFLOAT16) {
      group_fused_kernel<bf16_t><<<1, kFusedThreads, 0, s>>>(
          a.lhs_indices, a.rhs_indices, n, a.x_batches, E, key_bits, tile_rows, by_height, offsets, tiles,
          n_tiles, perm, static_cast<bf16_t*>(a.out), a.N);
    } else {
      group_fused_kernel<f16_t><<<1, kFusedThreads, 0, s>>>(
          a.lhs_indices, a.rhs_indices, n, a.x_batches, E, key_bits, tile_rows, by_height, offsets, tiles,
          n_tiles, perm, static_cast<f16_t*>(a.out), a.N);
    }
    MLXROCM_HIP_TRY(hipGetLastError());
    return MLXROCM_OK;
  }

  // counts and cursors start at zero (a fill kernel, so that the sequence can be
  // captured into a graph)
  fill_i32_kernel<<<(2 * E + 255) / 256, 256, 0, s>>>(counts, 2 * E, 0);
  MLXROCM_HIP_TRY(hipGetLastError());
  const int blocks = (n + 255) / 256;
  if (dtype == MLXROCM_BFLOAT16) {
    group_count_kernel<bf16_t><<<blocks, 256, 0, s>>>(
        a.lhs_indices, a.rhs_indices, n, a.x_batches, E, counts,
        static_cast<bf16_t*>(a.out), a.N);
  } else {
    group_count_kernel<f16_t><<<blocks, 256, 0, s>>>(
        a.lhs_indices, a.rhs_indices, n, a.x_batches, E, counts,
        static_cast<f16_t*>(a.out), a.N);
  }
  MLXROCM_HIP_TRY(hipGetLastError());
  group_plan_kernel<<<1, 256, 0, s>>>(E, tile_rows, by_height, counts, offsets, tiles, n_tiles);
  MLXROCM_HIP_TRY(hipGetLastError());
  group_scatter_kernel<<<blocks, 256, 0, s>>>(
      a.lhs_indices, a.rhs_indices, n, a.x_batches, E, offsets, cursor, perm);
  MLXROCM_HIP_TRY(hipGetLastError());
  return MLXROCM_OK;
}

} // namespace mlxrocm
