// switch_glu.hip -- the expert-routed gated MLP in one call:
//   out[t, j] = (silu(x[t] W_gate[e]^T) * (x[t] W_up[e]^T)) W_down[e]^T,  e = indices[t, j]
// (three gathers and the arithmetic between them, as a model's mixture-of-experts
// block issues them).  What the call saves over those: the pairs are grouped by
// expert once instead of three times (and instead of being sorted beforehand), the
// indices are read as they come, the gate is applied where its operands are, and
// from 64 pairs per expert on (fewer: least_pairs) the two first products run as one launch
// of a tile kernel whose epilogue writes the gated result -- 8 experts of [14336, 4096], 4096
// pairs: 2 x 117 MB written and read again are left out, and one pass over x.
#include "qmm_args.h"

#include "mfma_dequant.h"

namespace mlxrocm {

namespace {

// pair p: expert indices[p], row p / top of x; and the pair itself, as the row of h
template <typename I>
__global__ __launch_bounds__(256) void expert_pairs_kernel(
    const I* indices, int pairs, int top, uint32_t* expert, uint32_t* row, uint32_t* self) {
  const int p = blockIdx.x * 256 + threadIdx.x;
  if (p < pairs) {
    expert[p] = static_cast<uint32_t>(indices[p]); // as astype(indices, uint32)
    row[p] = static_cast<uint32_t>(p) / static_cast<uint32_t>(top);
    self[p] = p;
  }
}

// h[i] = silu(gate[i]) * up[i], eight values per thread
template <typename T>
__global__ __launch_bounds__(256) void gate_kernel(const T* gate, const T* up, T* h, size_t n) {
  const size_t i = (static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x) * 8;
  if (i + 8 <= n) {
    const uint4 g = *reinterpret_cast<const uint4*>(gate + i);
    const uint4 u = *reinterpret_cast<const uint4*>(up + i);
    const uint32_t gd[4] = {g.x, g.y, g.z, g.w};
    const uint32_t ud[4] = {u.x, u.y, u.z, u.w};
    uint32_t hd[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      hd[e] = pack2<T>(
          gated<T>(half_of<T>(gd[e], 0), half_of<T>(ud[e], 0)),
          gated<T>(half_of<T>(gd[e], 1), half_of<T>(ud[e], 1)));
    }
    *reinterpret_cast<uint4*>(h + i) = make_uint4(hd[0], hd[1], hd[2], hd[3]);
  } else {
    for (size_t e = i; e < n; ++e) {
      h[e] = from_f32<T>(gated<T>(to_f32(gate[e]), to_f32(up[e])));
    }
  }
}

size_t round256(size_t n) {
  return (n + 255) / 256 * 256;
}

// The first products and the last, as plans look at them.
struct Shapes {
  QmmArgs in, out;
};
Shapes shapes_of(int pairs, int D, int F, int E) {
  Shapes s{};
  s.in.N = F;
  s.in.K = D;
  s.in.L = pairs;
  s.in.n_experts = E;
  s.out = s.in;
  s.out.N = D;
  s.out.K = F;
  return s;
}

// Pairs per expert from which the tiles are ahead: as many as mlxrocm_gather_qmm asks for of
// the tile kernel, fewer where qmm_own_kernel takes both products and the products one by one
// would run on the staged kernel of 32 rows (4-bit codes have one that rounds no weight, and
// keep it).  us per call, products / tiles, 8-bit, by pairs per expert: 4096 x 14336, 8
// experts 24 525 / 529, 32 546 / 532, 44 707 / 554, 64 876 / 580; 2048 x 1408, 64 experts 12
// 189 / 194, 17 193 / 204, 22 217 / 209, 32 246 / 201, 64 375 / 248; 1024 x 1024, 32 experts 16 75
// / 64, 64 109 / 82 (3-bit: 28 458 / 469, 28 238 / 185, 28 70 / 57; 2048 x 1408 16 173 / 140).
int least_pairs(const Shapes& s, int bits) {
  if (bits == 4 || !qmm_own_experts_supported(s.in, bits) ||
      !qmm_own_experts_supported(s.out, bits)) {
    return 64;
  }
  const int widest = s.in.N > s.in.K ? s.in.N : s.in.K;
  return widest > 2048 ? 32 : widest > 1024 && bits == 8 ? 20 : 16;
}

// The tile kernels' grouped form: operands within 32-bit byte offsets.
bool tiled(int tokens, int top, int D, int F, int E, int least) {
  const int64_t pairs = static_cast<int64_t>(tokens) * top;
  const int64_t limit = int64_t{1} << 32;
  return pairs > least * static_cast<int64_t>(E) && D % 64 == 0 &&
      F % 64 == 0 && static_cast<int64_t>(tokens) * D * 2 < limit && pairs * F * 2 < limit &&
      gather_group_max_tiles(static_cast<int>(pairs), E, kGroupLargeTile) <= 65535 &&
      gather_group_workspace_bytes(static_cast<int>(pairs), E) > 0;
}

struct Layout {
  size_t expert, row, self; // u32 [pairs] each
  size_t h;                 // [pairs, F]
  size_t up;                // [pairs, F] (products one by one)
  bool gated;               // not tiled: the first two products meet in h (gather_gated)
  size_t rest;              // workspace of the products (tables and images: tiled)
  size_t gate_image, up_image, down_image;
  size_t total;
};

// room: what the caller has.  One with too little for tiles of few pairs, or for the planes of
// two products, has the products one by one.
Layout layout_of(
    int tokens, int top, int D, int F, int E, int gs, int bits, int dtype, bool* tiles,
    size_t room = SIZE_MAX, int least = 0) {
  const size_t pairs = static_cast<size_t>(tokens) * top;
  Layout l{};
  size_t at = 0;
  const auto take = [&](size_t bytes) {
    const size_t here = at;
    at += round256(bytes);
    return here;
  };
  l.expert = take(pairs * 4);
  l.row = take(pairs * 4);
  l.self = take(pairs * 4);
  l.h = take(pairs * F * dtype_size(dtype));
  const int fewest = least_pairs(shapes_of(static_cast<int>(pairs), D, F, E), bits);
  *tiles = tiled(tokens, top, D, F, E, least > fewest ? least : fewest);
  if (*tiles) {
    l.rest = take(gather_group_workspace_bytes(static_cast<int>(pairs), E));
    l.gate_image = take(qmm_n_sb_bytes(F, D / gs, E, dtype));
    l.up_image = take(qmm_n_sb_bytes(F, D / gs, E, dtype));
    l.down_image = take(qmm_n_sb_bytes(D, F / gs, E, dtype));
  } else {
    const size_t in = mlxrocm_gather_qmm_workspace_size(
        1, F, D, static_cast<int>(pairs), E, gs, bits, dtype, 1, 0);
    const size_t out = mlxrocm_gather_qmm_workspace_size(
        1, D, F, static_cast<int>(pairs), E, gs, bits, dtype, 1, 0);
    const size_t both = gather_gated_bytes(
        F, D, static_cast<int>(pairs), E, tokens, D, gs, bits, dtype);
    l.gated = both != 0 && at + round256(both > out ? both : out) <= room;
    l.up = l.gated ? 0 : take(pairs * F * dtype_size(dtype));
    const size_t first = l.gated ? both : in;
    l.rest = take(first > out ? first : out);
  }
  l.total = at;
  return l.total > room && *tiles && least == 0
      ? layout_of(tokens, top, D, F, E, gs, bits, dtype, tiles, room, 64)
      : l;
}

bool good_shape(int tokens, int top, int D, int F, int E, int gs, int bits, int dtype) {
  return tokens > 0 && top > 0 && D > 0 && F > 0 && E > 0 && valid_group(gs) && valid_bits(bits) &&
      dtype != MLXROCM_FLOAT32 && valid_dtype(dtype) && D % gs == 0 && F % gs == 0 &&
      static_cast<int64_t>(tokens) * top < (int64_t{1} << 31) &&
      static_cast<int64_t>(D) * bits % 128 == 0 && static_cast<int64_t>(F) * bits % 128 == 0;
}

} // namespace

} // namespace mlxrocm

using namespace mlxrocm;

extern "C" size_t mlxrocm_switch_glu_workspace_size(
    int tokens, int top, int D, int F, int n_experts, int group_size, int bits, int dtype) {
  if (!good_shape(tokens, top, D, F, n_experts, group_size, bits, dtype)) {
    return 0;
  }
  bool tiles;
  return layout_of(tokens, top, D, F, n_experts, group_size, bits, dtype, &tiles).total;
}

extern "C" int mlxrocm_switch_glu(
    const void* x,
    const void* indices,
    int index_bytes,
    const uint32_t* gate_w,
    const void* gate_scales,
    const void* gate_biases,
    const uint32_t* up_w,
    const void* up_scales,
    const void* up_biases,
    const uint32_t* down_w,
    const void* down_scales,
    const void* down_biases,
    void* out,
    int tokens,
    int top,
    int D,
    int F,
    int n_experts,
    int group_size,
    int bits,
    int dtype,
    void* workspace,
    size_t workspace_bytes,
    mlxrocm_stream_t stream) {
  mlxrocm::ApiRange api_range("mlxrocm_switch_glu");
  const int E = n_experts;
  if (!good_shape(tokens, top, D, F, E, group_size, bits, dtype) ||
      (index_bytes != 4 && index_bytes != 8)) {
    return fail(
        MLXROCM_INVALID_ARGUMENT,
        "[switch_glu] tokens=%d top=%d D=%d F=%d experts=%d group_size=%d bits=%d dtype=%d "
        "index_bytes=%d: not a shape of this call",
        tokens, top, D, F, E, group_size, bits, dtype, index_bytes);
  }
  for (const void* p : {x, indices, static_cast<const void*>(gate_w), gate_scales, gate_biases,
                        static_cast<const void*>(up_w), up_scales, up_biases,
                        static_cast<const void*>(down_w), down_scales, down_biases,
                        static_cast<const void*>(out), static_cast<const void*>(workspace)}) {
    if (p == nullptr) {
      return fail(MLXROCM_INVALID_ARGUMENT, "[switch_glu] null device pointer");
    }
    if (p != indices && (reinterpret_cast<uintptr_t>(p) & 15u) != 0) {
      return fail(MLXROCM_UNSUPPORTED, "[switch_glu] operands must be 16-byte aligned");
    }
  }
  bool tiles;
  const Layout l =
      layout_of(tokens, top, D, F, E, group_size, bits, dtype, &tiles, workspace_bytes);
  if (workspace_bytes < l.total) {
    return fail(
        MLXROCM_INVALID_ARGUMENT,
        "[switch_glu] this shape needs a workspace of %zu bytes (mlxrocm_switch_glu_workspace_size); "
        "got %zu",
        l.total, workspace_bytes);
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  char* ws = static_cast<char*>(workspace);
  const int pairs = tokens * top;
  uint32_t* expert = reinterpret_cast<uint32_t*>(ws + l.expert);
  uint32_t* row = reinterpret_cast<uint32_t*>(ws + l.row);
  uint32_t* self = reinterpret_cast<uint32_t*>(ws + l.self);
  const unsigned blocks = (pairs + 255) / 256;
  if (index_bytes == 8) {
    expert_pairs_kernel<int64_t><<<blocks, 256, 0, s>>>(
        static_cast<const int64_t*>(indices), pairs, top, expert, row, self);
  } else {
    expert_pairs_kernel<uint32_t><<<blocks, 256, 0, s>>>(
        static_cast<const uint32_t*>(indices), pairs, top, expert, row, self);
  }
  MLXROCM_HIP_TRY(hipGetLastError());
  const int64_t w_in = static_cast<int64_t>(F) * (static_cast<int64_t>(D) * bits / 32);
  const int64_t w_out = static_cast<int64_t>(D) * (static_cast<int64_t>(F) * bits / 32);
  const int64_t sb_in = static_cast<int64_t>(F) * (D / group_size);
  const int64_t sb_out = static_cast<int64_t>(D) * (F / group_size);
  void* h = ws + l.h;

  if (!tiles) {
    void* up = ws + l.up;
    void* rest = ws + l.rest;
    const size_t rest_bytes = workspace_bytes - l.rest;
    int rc;
    if (l.gated) {
      // two launches less: 8 tokens to 2 of 8 experts, 4096 x 14336, 190.3 -> 185.3 us
      // (64 tokens 236 -> 231, 256 tokens 555 -> 549; 64 experts 2048 x 1408, 32 tokens to 6
      // 114 -> 109)
      QmmArgs gate{};
      gate.x = x;
      gate.w = gate_w;
      gate.scales = gate_scales;
      gate.biases = gate_biases;
      gate.out = h;
      gate.M = 1;
      gate.N = F;
      gate.K = D;
      gate.L = pairs;
      gate.x_batch_stride = D;
      gate.w_batch_stride = w_in;
      gate.sb_batch_stride = sb_in;
      gate.lhs_indices = row;
      gate.rhs_indices = expert;
      gate.x_batches = tokens;
      gate.n_experts = E;
      QmmArgs other = gate;
      other.w = up_w;
      other.scales = up_scales;
      other.biases = up_biases;
      rc = gather_gated(gate, other, group_size, bits, dtype, rest, s);
      return rc != MLXROCM_OK
          ? rc
          : mlxrocm_gather_qmm(
                h, down_w, down_scales, down_biases, self, expert, out, 1, D, F, pairs, pairs, E, F,
                w_out, sb_out, group_size, bits, dtype, 1, 0, rest, rest_bytes, stream);
    }
    rc = mlxrocm_gather_qmm(
        x, gate_w, gate_scales, gate_biases, row, expert, h, 1, F, D, pairs, tokens, E, D, w_in,
        sb_in, group_size, bits, dtype, 1, 0, rest, rest_bytes, stream);
    if (rc == MLXROCM_OK) {
      rc = mlxrocm_gather_qmm(
          x, up_w, up_scales, up_biases, row, expert, up, 1, F, D, pairs, tokens, E, D, w_in, sb_in,
          group_size, bits, dtype, 1, 0, rest, rest_bytes, stream);
    }
    if (rc != MLXROCM_OK) {
      return rc;
    }
    const size_t n = static_cast<size_t>(pairs) * F;
    const unsigned gate_blocks = static_cast<unsigned>((n / 8 + 256) / 256);
    if (dtype == MLXROCM_BFLOAT16) {
      gate_kernel<bf16_t><<<gate_blocks, 256, 0, s>>>(
          static_cast<const bf16_t*>(h), static_cast<const bf16_t*>(up), static_cast<bf16_t*>(h), n);
    } else {
      gate_kernel<f16_t><<<gate_blocks, 256, 0, s>>>(
          static_cast<const f16_t*>(h), static_cast<const f16_t*>(up), static_cast<f16_t*>(h), n);
    }
    MLXROCM_HIP_TRY(hipGetLastError());
    return mlxrocm_gather_qmm(
        h, down_w, down_scales, down_biases, self, expert, out, 1, D, F, pairs, pairs, E, F, w_out,
        sb_out, group_size, bits, dtype, 1, 0, rest, rest_bytes, stream);
  }

  // one grouping for all three products (rows of out whose expert is out of range
  // are cleared by it; no product touches them)
  QmmArgs a{};
  a.lhs_indices = row;
  a.rhs_indices = expert;
  a.x_batches = tokens;
  a.n_experts = E;
  a.L = pairs;
  a.M = 1;
  a.out = out;
  a.N = D;
  // (planes of K ranges where the images of the first two products were: side by side, done with)
  const Shapes shapes = shapes_of(pairs, D, F, E);
  const ExpertsPlan pl =
      qmm_experts_plan(shapes.in, shapes.out, bits, l.down_image - l.gate_image);
  int rc = launch_gather_group(
      a, dtype, kGroupLargeTile,
      pl.own_first || pl.own_second || gather_tiles_by_height(D, F, bits), ws + l.rest, s);
  const struct {
    const void *scales, *biases;
    size_t image;
    int rows, groups;
    int64_t stride;
  } images[3] = {{gate_scales, gate_biases, l.gate_image, F, D / group_size, sb_in},
                 {up_scales, up_biases, l.up_image, F, D / group_size, sb_in},
                 {down_scales, down_biases, l.down_image, D, F / group_size, sb_out}};
  for (int i = 0; i < 3 && rc == MLXROCM_OK; ++i) {
    rc = interleave_sb_for_qmm_t(
        images[i].scales, images[i].biases, ws + images[i].image, images[i].rows, images[i].groups,
        E, images[i].stride, s);
  }
  if (rc != MLXROCM_OK) {
    return rc;
  }
  QmmArgs in = a;
  in.x = x;
  in.w = gate_w;
  in.scales = ws + l.gate_image;
  in.biases = in.scales;
  in.w_alt = up_w;
  in.scales_alt = ws + l.up_image;
  in.biases_alt = in.scales_alt;
  in.out = h;
  in.N = F;
  in.K = D;
  in.x_batch_stride = D;
  in.w_batch_stride = w_in;
  in.sb_batch_stride = 2 * sb_in; // pairs
  in.sb_transposed = 2;
  rc = launch_qmm_mfma_experts_glu(in, group_size, bits, dtype, pl, s);
  if (rc != MLXROCM_OK) {
    return rc;
  }
  QmmArgs o = a;
  o.x = h;
  o.w = down_w;
  o.scales = ws + l.down_image;
  o.biases = o.scales;
  o.out = out;
  o.N = D;
  o.K = F;
  o.lhs_indices = self;
  o.x_batches = pairs;
  o.x_batch_stride = F;
  o.w_batch_stride = w_out;
  o.sb_batch_stride = 2 * sb_out;
  o.sb_transposed = 2;
  return launch_qmm_mfma_experts(o, group_size, bits, dtype, pl, ws + l.gate_image, s);
}
