// fast_ops.cpp -- the host path of the operators in ops.py for the calls that
// need none of their conversions, as a CPython extension.
//
// What bounds it: nothing on the GPU.  A decode step is a chain of kernels of
// 3..13 us each, and the Python body of one operator call (argument rules,
// shape arithmetic, two allocations, twenty ctypes conversions) took 13..16 us,
// so the GPU waited for the host between any two of them: the projections of
// four layers with 4096 x 14336 MLPs at 4 bits took 420 us where their kernels
// take 161.  Each function here takes the operator's arguments, looks at the
// tensors through libtorch, allocates the output (and the workspace, which
// torch's caching allocator hands out per stream) and calls the C ABI.
//
// A function returns None -- and ops.py goes on with its own body -- for
// everything that is not the plain case: another device than the current one,
// operands to be converted, expanded or made contiguous, a gradient to be
// recorded, a shape or an option that ops.py refuses, and any status other than
// MLXROCM_OK (ops.py then makes the same call and turns it into an exception).
// So the rules and messages stay in one place; here are only the conditions
// under which nothing of them applies.
#include <ATen/ATen.h>
#include <ATen/core/grad_mode.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>
#include <cstring>

#include "mlx_rocm_qmm.h"

namespace {

// Entry points of the library that ops.py has loaded (bind()): the extension
// does not link it, so that both always use the same one.
struct Abi {
  decltype(&mlxrocm_qmm_workspace_size) qmm_workspace_size;
  decltype(&mlxrocm_qmm_prepacked) qmm_prepacked;
  decltype(&mlxrocm_qmm_sb_image_size) qmm_sb_image_size;
  decltype(&mlxrocm_qmm_rows_supported) rows_supported;
  decltype(&mlxrocm_qmm_rows_workspace_size) rows_workspace_size;
  decltype(&mlxrocm_qmm_rows_prepacked) rows_prepacked;
  decltype(&mlxrocm_fp_qmm_workspace_size) fp_qmm_workspace_size;
  decltype(&mlxrocm_fp_qmm) fp_qmm;
  decltype(&mlxrocm_fp_qmm_rows_supported) fp_rows_supported;
  decltype(&mlxrocm_fp_qmm_rows_workspace_size) fp_rows_workspace_size;
  decltype(&mlxrocm_fp_qmm_rows) fp_rows;
  decltype(&mlxrocm_qmm_swiglu_workspace_size) swiglu_workspace_size;
  decltype(&mlxrocm_qmm_swiglu) swiglu;
  decltype(&mlxrocm_fp_qqmm_workspace_size) fp_qqmm_workspace_size;
  decltype(&mlxrocm_fp_qqmm) fp_qqmm;
  decltype(&mlxrocm_switch_glu_workspace_size) switch_glu_workspace_size;
  decltype(&mlxrocm_switch_glu) switch_glu;
  decltype(&mlxrocm_affine_quantize) affine_quantize;
  decltype(&mlxrocm_affine_dequantize) affine_dequantize;
  decltype(&mlxrocm_fp_quantize) fp_quantize;
  decltype(&mlxrocm_fp_dequantize) fp_dequantize;
};
Abi abi{};
bool bound = false;

constexpr int kAffine = -1;
constexpr int kNoMode = -2;

// "affine" -> kAffine, a floating-point mode -> its mlxrocm_fp_mode
int mode_of(PyObject* o) {
  if (!PyUnicode_CheckExact(o)) {
    return kNoMode;
  }
  Py_ssize_t n = 0;
  const char* s = PyUnicode_AsUTF8AndSize(o, &n);
  if (s == nullptr) {
    PyErr_Clear();
    return kNoMode;
  }
  const auto is = [&](const char* name) {
    return static_cast<size_t>(n) == std::strlen(name) && std::memcmp(s, name, n) == 0;
  };
  return is("affine") ? kAffine
      : is("mxfp4")   ? static_cast<int>(MLXROCM_MXFP4)
      : is("mxfp8")   ? static_cast<int>(MLXROCM_MXFP8)
      : is("nvfp4")   ? static_cast<int>(MLXROCM_NVFP4)
                      : kNoMode;
}

// group_size or bits: an exact int, or None for the mode's default; -1 otherwise
int int_or(PyObject* o, int fallback) {
  if (o == Py_None) {
    return fallback;
  }
  if (!PyLong_CheckExact(o)) {
    return -1;
  }
  int overflow = 0;
  const long v = PyLong_AsLongAndOverflow(o, &overflow);
  return overflow == 0 && v > 0 && v < 1024 ? static_cast<int>(v) : -1;
}

// The parameters of a call; false where ops.py would complain.
bool params_of(int mode, PyObject* group, PyObject* bits_obj, int* gs, int* bits) {
  if (mode == kAffine) {
    *gs = int_or(group, 64);
    *bits = int_or(bits_obj, 4);
    return (*gs == 32 || *gs == 64 || *gs == 128) && *bits >= 2 && *bits <= 8 && *bits != 7;
  }
  const int want_gs = mode == MLXROCM_NVFP4 ? 16 : 32;
  const int want_bits = mode == MLXROCM_MXFP8 ? 8 : 4;
  *gs = int_or(group, want_gs);
  *bits = int_or(bits_obj, want_bits);
  return *gs == want_gs && *bits == want_bits;
}

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kFloat:
      return MLXROCM_FLOAT32;
    case at::kHalf:
      return MLXROCM_FLOAT16;
    case at::kBFloat16:
      return MLXROCM_BFLOAT16;
    default:
      return -1;
  }
}

// The device of the first operand; -1 unless that is the current GPU.
c10::DeviceIndex device_of(PyObject* o) {
  if (!THPVariable_CheckExact(o)) {
    return -1;
  }
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda()) {
    return -1;
  }
  const c10::DeviceIndex device = t.device().index();
  return device == c10::hip::current_device() ? device : -1;
}

// A plain contiguous tensor on `device` with something in it.
const at::Tensor* tensor_of(PyObject* o, c10::DeviceIndex device) {
  if (!THPVariable_CheckExact(o)) {
    return nullptr;
  }
  const at::Tensor& t = THPVariable_Unpack(o);
  return t.defined() && t.is_cuda() && t.device().index() == device && t.is_contiguous() &&
          t.numel() > 0 && !t.is_conj() && !t.is_neg()
      ? &t
      : nullptr;
}

// The same of two dimensions and the given type.
const at::Tensor* matrix_of(PyObject* o, c10::DeviceIndex device, at::ScalarType type) {
  const at::Tensor* t = tensor_of(o, device);
  return t != nullptr && t->dim() == 2 && t->scalar_type() == type ? t : nullptr;
}

bool fits_int(int64_t v) {
  return v > 0 && v < (int64_t{1} << 31);
}

at::Tensor new_tensor(at::IntArrayRef sizes, at::ScalarType type, c10::DeviceIndex device) {
  return at::Tensor(at::detail::empty_cuda(
      sizes, type, c10::Device(c10::DeviceType::CUDA, device), std::nullopt));
}

void* stream_of(c10::DeviceIndex device) {
  return c10::hip::getCurrentHIPStream(device).stream();
}

// A workspace: gone to the allocator again when the call returns, which hands
// it to later work of the same stream only.
struct Workspace {
  at::Tensor t;
  size_t bytes = 0;
  Workspace(size_t n, c10::DeviceIndex device) : bytes(n) {
    if (n != 0) {
      t = new_tensor({static_cast<int64_t>(n)}, at::kByte, device);
    }
  }
  void* ptr() const {
    return bytes != 0 ? t.data_ptr() : nullptr;
  }
};

// shape of x with its last dimension replaced
c10::SmallVector<int64_t, 6> with_last(const at::Tensor& x, int64_t last) {
  c10::SmallVector<int64_t, 6> s(x.sizes().begin(), x.sizes().end());
  s.back() = last;
  return s;
}

bool records_grad(const at::Tensor& t) {
  return t.requires_grad() && at::GradMode::is_enabled();
}

PyObject* wrap(at::Tensor&& t) {
  return THPVariable_Wrap(std::move(t));
}

#define NOT_PLAIN Py_RETURN_NONE
#define FAST_TRY try {
#define FAST_CATCH                                      \
  }                                                     \
  catch (const c10::OutOfMemoryError&) {                \
    Py_RETURN_NONE; /* ops.py allocates and raises */   \
  }                                                     \
  catch (const std::exception& e) {                     \
    PyErr_SetString(PyExc_RuntimeError, e.what());      \
    return nullptr;                                     \
  }

// quantized_matmul(x, w, scales, biases, transpose, group_size, bits, mode, sb_image)
PyObject* quantized_matmul(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (!bound || n != 9) {
    NOT_PLAIN;
  }
  FAST_TRY
  const c10::DeviceIndex device = device_of(args[0]);
  if (device < 0) {
    NOT_PLAIN;
  }
  const at::Tensor* x = tensor_of(args[0], device);
  const at::Tensor* w = matrix_of(args[1], device, at::kUInt32);
  const int mode = mode_of(args[7]);
  int gs = 0;
  int bits = 0;
  if (x == nullptr || w == nullptr || x->dim() < 1 || mode == kNoMode ||
      !params_of(mode, args[5], args[6], &gs, &bits)) {
    NOT_PLAIN;
  }
  const int code = dtype_code(x->scalar_type());
  if (code < 0 || records_grad(*x)) {
    NOT_PLAIN;
  }
  const at::Tensor* scales =
      matrix_of(args[2], device, mode == kAffine ? x->scalar_type() : at::kByte);
  const at::Tensor* biases = nullptr;
  if (scales == nullptr || records_grad(*scales)) {
    NOT_PLAIN;
  }
  if (mode == kAffine) {
    biases = matrix_of(args[3], device, x->scalar_type());
    if (biases == nullptr || records_grad(*biases) || biases->sizes() != scales->sizes()) {
      NOT_PLAIN;
    }
  } else if (args[3] != Py_None || args[8] != Py_None) {
    NOT_PLAIN;
  }
  const int transpose = PyObject_IsTrue(args[4]);
  if (transpose < 0) {
    return nullptr;
  }
  const int64_t rows_w = w->size(0);
  const int64_t codes_w = w->size(1) * 32 / bits;
  const int64_t K = transpose ? codes_w : rows_w;
  const int64_t N = transpose ? rows_w : codes_w;
  if (x->size(-1) != K || scales->size(0) != rows_w || scales->size(1) * gs != codes_w ||
      w->size(1) * 32 != codes_w * bits) {
    NOT_PLAIN;
  }
  const int64_t M = x->numel() / K;
  if (!fits_int(M) || !fits_int(N) || !fits_int(K)) {
    NOT_PLAIN;
  }
  const void* image = nullptr;
  if (args[8] != Py_None) {
    const at::Tensor* t = tensor_of(args[8], device);
    if (t == nullptr || !transpose || t->scalar_type() != x->scalar_type() ||
        t->nbytes() != abi.qmm_sb_image_size(N, K, 1, gs, code)) {
      NOT_PLAIN;
    }
    image = t->data_ptr();
  }
  at::Tensor out = new_tensor(with_last(*x, N), x->scalar_type(), device);
  void* stream = stream_of(device);
  int rc = 0;
  if (mode == kAffine) {
    const bool rows = transpose && abi.rows_supported(M, N, K, 1, gs, bits, code);
    const Workspace ws(
        rows ? abi.rows_workspace_size(M, N, K, 1, gs, bits, code)
             : abi.qmm_workspace_size(M, N, K, 1, 0, gs, bits, code, transpose),
        device);
    Py_BEGIN_ALLOW_THREADS;
    if (rows) {
      rc = abi.rows_prepacked(
          x->data_ptr(), static_cast<const uint32_t*>(w->data_ptr()), scales->data_ptr(),
          biases->data_ptr(), image, out.data_ptr(), M, N, K, 1, M * K, 0, 0, gs, bits, code,
          ws.ptr(), ws.bytes, stream);
    } else {
      rc = abi.qmm_prepacked(
          x->data_ptr(), static_cast<const uint32_t*>(w->data_ptr()), scales->data_ptr(),
          biases->data_ptr(), image, out.data_ptr(), M, N, K, 1, M * K, 0, 0, gs, bits, code,
          transpose, ws.ptr(), ws.bytes, stream);
    }
    Py_END_ALLOW_THREADS;
  } else if (transpose && abi.fp_rows_supported(M, N, K, 1, mode, code)) {
    const Workspace ws(abi.fp_rows_workspace_size(M, N, K, 1, mode, code), device);
    Py_BEGIN_ALLOW_THREADS;
    rc = abi.fp_rows(
        x->data_ptr(), static_cast<const uint32_t*>(w->data_ptr()),
        static_cast<const uint8_t*>(scales->data_ptr()), out.data_ptr(), M, N, K, 1, M * K, 0, 0,
        mode, code, ws.ptr(), ws.bytes, stream);
    Py_END_ALLOW_THREADS;
  } else {
    const Workspace ws(abi.fp_qmm_workspace_size(M, N, K, 1, 0, mode, code, transpose), device);
    Py_BEGIN_ALLOW_THREADS;
    rc = abi.fp_qmm(
        x->data_ptr(), static_cast<const uint32_t*>(w->data_ptr()),
        static_cast<const uint8_t*>(scales->data_ptr()), out.data_ptr(), M, N, K, 1, M * K, 0, 0,
        mode, code, transpose, ws.ptr(), ws.bytes, stream);
    Py_END_ALLOW_THREADS;
  }
  if (rc != MLXROCM_OK) {
    NOT_PLAIN;
  }
  return wrap(std::move(out));
  FAST_CATCH
}

// quantized_swiglu(x, gate, up, group_size, bits); gate and up are triplets
PyObject* quantized_swiglu(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (!bound || n != 5) {
    NOT_PLAIN;
  }
  FAST_TRY
  const c10::DeviceIndex device = device_of(args[0]);
  if (device < 0) {
    NOT_PLAIN;
  }
  const at::Tensor* x = tensor_of(args[0], device);
  int gs = 0;
  int bits = 0;
  if (x == nullptr || x->dim() < 1 || !params_of(kAffine, args[3], args[4], &gs, &bits) ||
      !PyTuple_CheckExact(args[1]) || PyTuple_GET_SIZE(args[1]) != 3 ||
      !PyTuple_CheckExact(args[2]) || PyTuple_GET_SIZE(args[2]) != 3) {
    NOT_PLAIN;
  }
  const int code = dtype_code(x->scalar_type());
  const at::Tensor* t[2][3];
  for (int i = 0; i < 2; ++i) {
    for (int j = 0; j < 3; ++j) {
      t[i][j] = matrix_of(
          PyTuple_GET_ITEM(args[1 + i], j), device, j == 0 ? at::kUInt32 : x->scalar_type());
      if (t[i][j] == nullptr || t[i][j]->sizes() != t[0][j]->sizes()) {
        NOT_PLAIN;
      }
    }
  }
  const int64_t N = t[0][0]->size(0);
  const int64_t K = t[0][0]->size(1) * 32 / bits;
  const at::Tensor& scales = *t[0][1];
  if (code < 0 || x->size(-1) != K || t[0][2]->sizes() != scales.sizes() || scales.size(0) != N ||
      scales.size(1) * gs != K || t[0][0]->size(1) * 32 != K * bits) {
    NOT_PLAIN;
  }
  const int64_t M = x->numel() / K;
  if (M > 8 || !fits_int(N) || !fits_int(K)) {
    NOT_PLAIN;
  }
  at::Tensor out = new_tensor(with_last(*x, N), x->scalar_type(), device);
  const size_t need = abi.swiglu_workspace_size(M, N, code);
  const Workspace ws(need < 16 ? 16 : need, device);
  void* stream = stream_of(device);
  int rc = 0;
  Py_BEGIN_ALLOW_THREADS;
  rc = abi.swiglu(
      x->data_ptr(), static_cast<const uint32_t*>(t[0][0]->data_ptr()), t[0][1]->data_ptr(),
      t[0][2]->data_ptr(), static_cast<const uint32_t*>(t[1][0]->data_ptr()),
      t[1][1]->data_ptr(), t[1][2]->data_ptr(), out.data_ptr(), ws.ptr(), M, N, K, gs, bits, code,
      stream);
  Py_END_ALLOW_THREADS;
  if (rc != MLXROCM_OK) {
    NOT_PLAIN;
  }
  return wrap(std::move(out));
  FAST_CATCH
}

// switch_glu(x, indices, gate, up, down, group_size, bits): the expert-routed gated
// MLP of nn.SwitchGLU over three (weight, scales, biases) stacks
PyObject* switch_glu(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (!bound || n != 7) {
    NOT_PLAIN;
  }
  FAST_TRY
  const c10::DeviceIndex device = device_of(args[0]);
  if (device < 0) {
    NOT_PLAIN;
  }
  const at::Tensor* x = tensor_of(args[0], device);
  const at::Tensor* indices = tensor_of(args[1], device);
  int gs = 0;
  int bits = 0;
  if (x == nullptr || indices == nullptr || x->dim() < 1 || indices->dim() != x->dim() ||
      !params_of(kAffine, args[5], args[6], &gs, &bits)) {
    NOT_PLAIN;
  }
  const at::ScalarType it = indices->scalar_type();
  const int index_bytes = it == at::kLong ? 8 : it == at::kInt || it == at::kUInt32 ? 4 : 0;
  const int code = dtype_code(x->scalar_type());
  const auto lead = [](const at::Tensor& t) { return t.sizes().slice(0, t.dim() - 1); };
  if (index_bytes == 0 || code < 0 || code == MLXROCM_FLOAT32 || lead(*x) != lead(*indices)) {
    NOT_PLAIN;
  }
  const int64_t D = x->size(-1);
  const at::Tensor* t[3][3];
  for (int i = 0; i < 3; ++i) {
    PyObject* triplet = args[2 + i];
    if (!PyTuple_CheckExact(triplet) || PyTuple_GET_SIZE(triplet) != 3) {
      NOT_PLAIN;
    }
    for (int j = 0; j < 3; ++j) {
      t[i][j] = tensor_of(PyTuple_GET_ITEM(triplet, j), device);
      if (t[i][j] == nullptr || t[i][j]->dim() != 3 ||
          t[i][j]->scalar_type() != (j == 0 ? at::kUInt32 : x->scalar_type())) {
        NOT_PLAIN;
      }
    }
  }
  const int64_t E = t[0][0]->size(0);
  const int64_t F = t[0][0]->size(1);
  for (int i = 0; i < 3; ++i) {
    const int64_t rows = i < 2 ? F : D;
    const int64_t inner = i < 2 ? D : F;
    const at::Tensor& w = *t[i][0];
    if (w.size(0) != E || w.size(1) != rows || w.size(2) * 32 != inner * bits) {
      NOT_PLAIN;
    }
    for (int j = 1; j < 3; ++j) {
      const at::Tensor& s = *t[i][j];
      if (s.size(0) != E || s.size(1) != rows || s.size(2) * gs != inner) {
        NOT_PLAIN;
      }
    }
  }
  const int64_t top = indices->size(-1);
  const int64_t tokens = indices->numel() / top;
  if (!fits_int(tokens * top) || !fits_int(D) || !fits_int(F) || !fits_int(E)) {
    NOT_PLAIN;
  }
  const size_t need = abi.switch_glu_workspace_size(tokens, top, D, F, E, gs, bits, code);
  if (need == 0) {
    NOT_PLAIN;
  }
  c10::SmallVector<int64_t, 6> shape(indices->sizes().begin(), indices->sizes().end());
  shape.push_back(D);
  at::Tensor out = new_tensor(shape, x->scalar_type(), device);
  const Workspace ws(need, device);
  void* stream = stream_of(device);
  int rc = 0;
  Py_BEGIN_ALLOW_THREADS;
  rc = abi.switch_glu(
      x->data_ptr(), indices->data_ptr(), index_bytes,
      static_cast<const uint32_t*>(t[0][0]->data_ptr()), t[0][1]->data_ptr(), t[0][2]->data_ptr(),
      static_cast<const uint32_t*>(t[1][0]->data_ptr()), t[1][1]->data_ptr(), t[1][2]->data_ptr(),
      static_cast<const uint32_t*>(t[2][0]->data_ptr()), t[2][1]->data_ptr(), t[2][2]->data_ptr(),
      out.data_ptr(), tokens, top, D, F, E, gs, bits, code, ws.ptr(), ws.bytes, stream);
  Py_END_ALLOW_THREADS;
  if (rc != MLXROCM_OK) {
    NOT_PLAIN;
  }
  return wrap(std::move(out));
  FAST_CATCH
}

// qqmm(x, w, scales, group_size, bits, mode) with a quantized w
PyObject* qqmm(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (!bound || n != 6) {
    NOT_PLAIN;
  }
  FAST_TRY
  const c10::DeviceIndex device = device_of(args[0]);
  if (device < 0) {
    NOT_PLAIN;
  }
  const at::Tensor* x = tensor_of(args[0], device);
  const at::Tensor* w = matrix_of(args[1], device, at::kUInt32);
  const at::Tensor* scales = matrix_of(args[2], device, at::kByte);
  const int mode = mode_of(args[5]);
  int gs = 0;
  int bits = 0;
  if (x == nullptr || w == nullptr || scales == nullptr || x->dim() < 1 || mode < 0 ||
      !params_of(mode, args[3], args[4], &gs, &bits)) {
    NOT_PLAIN;
  }
  const int code = dtype_code(x->scalar_type());
  const int64_t N = w->size(0);
  const int64_t K = w->size(1) * 32 / bits;
  if (code < 0 || x->size(-1) != K || scales->size(0) != N || scales->size(1) * gs != K) {
    NOT_PLAIN;
  }
  const int64_t M = x->numel() / K;
  if (!fits_int(M) || !fits_int(N) || !fits_int(K)) {
    NOT_PLAIN;
  }
  at::Tensor out = new_tensor(with_last(*x, N), x->scalar_type(), device);
  const size_t need = abi.fp_qqmm_workspace_size(M, N, K, mode, code);
  const Workspace ws(need < 256 ? 256 : need, device);
  void* stream = stream_of(device);
  int rc = 0;
  Py_BEGIN_ALLOW_THREADS;
  rc = abi.fp_qqmm(
      x->data_ptr(), static_cast<const uint32_t*>(w->data_ptr()),
      static_cast<const uint8_t*>(scales->data_ptr()), out.data_ptr(), M, N, K, mode, code,
      ws.ptr(), need, stream);
  Py_END_ALLOW_THREADS;
  if (rc != MLXROCM_OK) {
    NOT_PLAIN;
  }
  return wrap(std::move(out));
  FAST_CATCH
}

// quantize(w, group_size, bits, mode)
PyObject* quantize(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (!bound || n != 4) {
    NOT_PLAIN;
  }
  FAST_TRY
  const c10::DeviceIndex device = device_of(args[0]);
  if (device < 0) {
    NOT_PLAIN;
  }
  const at::Tensor* w = tensor_of(args[0], device);
  const int mode = mode_of(args[3]);
  int gs = 0;
  int bits = 0;
  if (w == nullptr || w->dim() < 2 || mode == kNoMode ||
      !params_of(mode, args[1], args[2], &gs, &bits)) {
    NOT_PLAIN;
  }
  const int code = dtype_code(w->scalar_type());
  const int64_t K = w->size(-1);
  if (code < 0 || K % gs != 0) {
    NOT_PLAIN;
  }
  at::Tensor wq = new_tensor(with_last(*w, K * bits / 32), at::kUInt32, device);
  at::Tensor scales = new_tensor(
      with_last(*w, K / gs), mode == kAffine ? w->scalar_type() : at::kByte, device);
  at::Tensor biases;
  if (mode == kAffine) {
    biases = new_tensor(scales.sizes(), w->scalar_type(), device);
  }
  void* stream = stream_of(device);
  const size_t elements = static_cast<size_t>(w->numel());
  int rc = 0;
  Py_BEGIN_ALLOW_THREADS;
  if (mode == kAffine) {
    rc = abi.affine_quantize(
        w->data_ptr(), static_cast<uint32_t*>(wq.data_ptr()), scales.data_ptr(),
        biases.data_ptr(), elements, gs, bits, code, stream);
  } else {
    rc = abi.fp_quantize(
        w->data_ptr(), static_cast<uint32_t*>(wq.data_ptr()),
        static_cast<uint8_t*>(scales.data_ptr()), elements, mode, code, stream);
  }
  Py_END_ALLOW_THREADS;
  if (rc != MLXROCM_OK) {
    NOT_PLAIN;
  }
  PyObject* out = PyTuple_New(mode == kAffine ? 3 : 2);
  if (out == nullptr) {
    return nullptr;
  }
  PyTuple_SET_ITEM(out, 0, wrap(std::move(wq)));
  PyTuple_SET_ITEM(out, 1, wrap(std::move(scales)));
  if (mode == kAffine) {
    PyTuple_SET_ITEM(out, 2, wrap(std::move(biases)));
  }
  return out;
  FAST_CATCH
}

// dequantize(w, scales, biases, group_size, bits, mode, dtype); dtype None or the
// type the result has anyway (bfloat16 where None in a floating-point mode)
PyObject* dequantize(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (!bound || n != 7) {
    NOT_PLAIN;
  }
  FAST_TRY
  const c10::DeviceIndex device = device_of(args[0]);
  if (device < 0) {
    NOT_PLAIN;
  }
  const at::Tensor* w = tensor_of(args[0], device);
  const at::Tensor* scales = tensor_of(args[1], device);
  const int mode = mode_of(args[5]);
  int gs = 0;
  int bits = 0;
  if (w == nullptr || scales == nullptr || w->dim() < 2 || w->dim() != scales->dim() ||
      w->scalar_type() != at::kUInt32 || mode == kNoMode ||
      !params_of(mode, args[3], args[4], &gs, &bits)) {
    NOT_PLAIN;
  }
  at::ScalarType type = mode == kAffine ? scales->scalar_type() : at::kBFloat16;
  if (args[6] != Py_None) {
    if (!THPDtype_Check(args[6])) {
      NOT_PLAIN;
    }
    const at::ScalarType asked = reinterpret_cast<THPDtype*>(args[6])->scalar_type;
    if (mode == kAffine && asked != type) {
      NOT_PLAIN;
    }
    type = asked;
  }
  const int code = dtype_code(type);
  const int64_t K = w->size(-1) * 32 / bits;
  const auto lead = [](const at::Tensor& t) { return t.sizes().slice(0, t.dim() - 1); };
  if (code < 0 || scales->size(-1) * gs != K || w->size(-1) * 32 != K * bits ||
      lead(*w) != lead(*scales)) {
    NOT_PLAIN;
  }
  const at::Tensor* biases = nullptr;
  if (mode == kAffine) {
    biases = tensor_of(args[2], device);
    if (biases == nullptr || biases->scalar_type() != scales->scalar_type() ||
        biases->sizes() != scales->sizes()) {
      NOT_PLAIN;
    }
  } else if (args[2] != Py_None || scales->scalar_type() != at::kByte) {
    NOT_PLAIN;
  }
  at::Tensor out = new_tensor(with_last(*w, K), type, device);
  void* stream = stream_of(device);
  const size_t elements = static_cast<size_t>(out.numel());
  int rc = 0;
  Py_BEGIN_ALLOW_THREADS;
  if (mode == kAffine) {
    rc = abi.affine_dequantize(
        static_cast<const uint32_t*>(w->data_ptr()), scales->data_ptr(), biases->data_ptr(),
        out.data_ptr(), elements, gs, bits, code, stream);
  } else {
    rc = abi.fp_dequantize(
        static_cast<const uint32_t*>(w->data_ptr()),
        static_cast<const uint8_t*>(scales->data_ptr()), out.data_ptr(), elements, mode, code,
        stream);
  }
  Py_END_ALLOW_THREADS;
  if (rc != MLXROCM_OK) {
    NOT_PLAIN;
  }
  return wrap(std::move(out));
  FAST_CATCH
}

// bind({entry point: address}): the library whose entry points are to be called
PyObject* bind(PyObject*, PyObject* table) {
  if (!PyDict_Check(table)) {
    PyErr_SetString(PyExc_TypeError, "bind() takes a dict of addresses");
    return nullptr;
  }
  const auto take = [&](const char* name, auto& slot) {
    PyObject* v = PyDict_GetItemString(table, name); // borrowed
    if (v == nullptr) {
      PyErr_Format(PyExc_KeyError, "no address for %s", name);
      return false;
    }
    void* p = PyLong_AsVoidPtr(v);
    if (p == nullptr) {
      if (!PyErr_Occurred()) {
        PyErr_Format(PyExc_ValueError, "null address for %s", name);
      }
      return false;
    }
    slot = reinterpret_cast<std::remove_reference_t<decltype(slot)>>(p);
    return true;
  };
  bound = take("mlxrocm_qmm_workspace_size", abi.qmm_workspace_size) &&
      take("mlxrocm_qmm_prepacked", abi.qmm_prepacked) &&
      take("mlxrocm_qmm_sb_image_size", abi.qmm_sb_image_size) &&
      take("mlxrocm_qmm_rows_supported", abi.rows_supported) &&
      take("mlxrocm_qmm_rows_workspace_size", abi.rows_workspace_size) &&
      take("mlxrocm_qmm_rows_prepacked", abi.rows_prepacked) &&
      take("mlxrocm_fp_qmm_workspace_size", abi.fp_qmm_workspace_size) &&
      take("mlxrocm_fp_qmm", abi.fp_qmm) &&
      take("mlxrocm_fp_qmm_rows_supported", abi.fp_rows_supported) &&
      take("mlxrocm_fp_qmm_rows_workspace_size", abi.fp_rows_workspace_size) &&
      take("mlxrocm_fp_qmm_rows", abi.fp_rows) &&
      take("mlxrocm_qmm_swiglu_workspace_size", abi.swiglu_workspace_size) &&
      take("mlxrocm_qmm_swiglu", abi.swiglu) &&
      take("mlxrocm_fp_qqmm_workspace_size", abi.fp_qqmm_workspace_size) &&
      take("mlxrocm_fp_qqmm", abi.fp_qqmm) &&
      take("mlxrocm_switch_glu_workspace_size", abi.switch_glu_workspace_size) &&
      take("mlxrocm_switch_glu", abi.switch_glu) &&
      take("mlxrocm_affine_quantize", abi.affine_quantize) &&
      take("mlxrocm_affine_dequantize", abi.affine_dequantize) &&
      take("mlxrocm_fp_quantize", abi.fp_quantize) &&
      take("mlxrocm_fp_dequantize", abi.fp_dequantize);
  if (!bound) {
    return nullptr;
  }
  Py_RETURN_NONE;
}

#define FASTCALL(f) \
  {#f, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    FASTCALL(quantized_matmul),
    FASTCALL(quantized_swiglu),
    FASTCALL(switch_glu),
    FASTCALL(qqmm),
    FASTCALL(quantize),
    FASTCALL(dequantize),
    {"bind", bind, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {
    PyModuleDef_HEAD_INIT, "fast_ops", "The operators' host path for plain calls.", -1, methods,
    nullptr, nullptr, nullptr, nullptr};

} // namespace

PyMODINIT_FUNC PyInit_fast_ops(void) {
  return PyModule_Create(&module);
}
