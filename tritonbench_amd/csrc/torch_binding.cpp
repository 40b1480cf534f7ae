// The short way from a PyTorch call to the C ABI: checks the operands, allocates the results, looks up the current
// stream and calls the library, all without going back to the interpreter.
//
// Every function returns None for whatever is not an everyday call (an operand of another kind, shape, type or
// stride, a tensor subclass, a device that is not set up yet, a status other than OK). ops.py then takes the call
// through its own checks, which say what is wrong with it or handle it; nothing is decided differently here.
//
// What it is for: launches of a few microseconds. A product of one row against a 2304 x 2048 weight takes 3.3 us on the
// GPU and took 12.2 us a call, the rest of it attribute look-ups, conversions of 18 arguments and wrapper objects.
#include <Python.h>
#include <ATen/Context.h>
#include <ATen/core/Tensor.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/ops/empty.h>
#include <ATen/record_function.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <atomic>

#include "../../include/mi355x_fp8_rowwise.h"

namespace {

constexpr int kMaxDevices = 64;
std::atomic<bool> g_ready[kMaxDevices];

constexpr at::ScalarType kCodes = at::ScalarType::Float8_e4m3fn;

// An operand: a plain tensor with memory on a device that has been set up.
const at::Tensor* operand(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || !t.unsafeGetTensorImpl()->has_storage()) return nullptr;
  const auto index = t.get_device();
  if (index < 0 || index >= kMaxDevices || !g_ready[index].load(std::memory_order_acquire)) return nullptr;
  return &t;
}

bool matrix(const at::Tensor* t, at::ScalarType type) { return t && t->scalar_type() == type && t->dim() == 2 && t->stride(1) == 1; }
bool factors(const at::Tensor* t, int64_t count) {
  return t && t->scalar_type() == at::kFloat && t->numel() == count && t->is_contiguous();
}
bool result(const at::Tensor* t, at::ScalarType type, int64_t m, int64_t n) {
  return matrix(t, type) && t->size(0) == m && t->size(1) == n;
}
// Straight from the device's allocator, without the dispatcher, which is half of what a tensor of a few kilobytes costs (a quantiser and a product of
// 5 x 512 x 2560, three tensors and two launches: 9.8 -> 9.1 us a call) - where nothing would see the difference: no dispatch mode, tracer,
// transform, inference mode or autocast in this thread, nobody who records operators, and no filling of new memory, which the operator does
// under deterministic algorithms.
bool dispatch_is_plain() {
  const auto keys = c10::impl::tls_local_dispatch_key_set();
  return keys.included_ == c10::default_included_set && keys.excluded_ == c10::default_excluded_set && !at::hasCallbacks() &&
         !(at::globalContext().deterministicAlgorithms() && at::globalContext().deterministicFillUninitializedMemory());
}
at::Tensor fresh(at::IntArrayRef shape, at::ScalarType type, const at::Tensor& like) {
  if (!dispatch_is_plain()) return at::empty(shape, at::TensorOptions().dtype(type).device(like.device()));
  return at::detail::empty_cuda(shape, type, like.device(), std::nullopt);
}
void* current_stream() { return (void*)c10::hip::getCurrentHIPStream().stream(); }
float* f32(const at::Tensor& t) { return (float*)t.data_ptr(); }

// One call of the library, with the interpreter's lock released (the arguments are taken before).
template <typename Entry, typename... Args>
bool enqueue(Entry entry, Args... args) {
  int st;
  Py_BEGIN_ALLOW_THREADS
  st = entry(args...);
  Py_END_ALLOW_THREADS
  return st == MI355X_FP8_OK;
}
PyObject* one(const at::Tensor& t) { return THPVariable_Wrap(t); }
PyObject* two(const at::Tensor& a, const at::Tensor& b) {
  PyObject* pa = THPVariable_Wrap(a);
  PyObject* pb = pa ? THPVariable_Wrap(b) : nullptr;
  PyObject* r = pb ? PyTuple_Pack(2, pa, pb) : nullptr;
  Py_XDECREF(pa);
  Py_XDECREF(pb);
  return r;
}

// (no C++ exception and no half-way error reaches the interpreter: such a call goes the long way, which raises it properly)
template <PyObject* (*Body)(PyObject* const*, Py_ssize_t)>
PyObject* guarded(PyObject*, PyObject* const* args, Py_ssize_t count) {
  try {
    if (PyObject* r = Body(args, count)) return r;
  } catch (...) {
  }
  PyErr_Clear();
  Py_RETURN_NONE;
}

// (device index) after the library has set the device up
PyObject* mark_ready(PyObject* const* args, Py_ssize_t count) {
  if (count != 1) return nullptr;
  const long index = PyLong_AsLong(args[0]);
  if (index >= 0 && index < kMaxDevices) g_ready[index].store(true, std::memory_order_release);
  return nullptr;
}

// (xq, wq, x_scale, w_scale, bias, out, variant, workspace, float16 result)
PyObject* gemm_rowwise(PyObject* const* a, Py_ssize_t count) {
  if (count != 9) return nullptr;
  const at::Tensor *xq = operand(a[0]), *wq = operand(a[1]), *xs = operand(a[2]), *ws = operand(a[3]);
  if (!matrix(xq, kCodes) || !matrix(wq, kCodes) || xq->size(1) != wq->size(1)) return nullptr;
  const int64_t m = xq->size(0), n = wq->size(0), k = xq->size(1);
  if (!factors(xs, m) || !factors(ws, n)) return nullptr;
  const void* bias = nullptr;
  if (a[4] != Py_None) {
    const at::Tensor* b = operand(a[4]);
    if (!b || b->scalar_type() != at::kBFloat16 || b->numel() != n || !b->is_contiguous()) return nullptr;
    bias = b->data_ptr();
  }
  const long variant = PyLong_AsLong(a[6]);
  if (variant < 0 || variant > INT32_MAX) return nullptr;
  const bool f16 = a[8] == Py_True;
  const at::ScalarType type = f16 ? at::kHalf : at::kBFloat16;
  at::Tensor made;
  const at::Tensor* out = &made;
  if (a[5] != Py_None) {
    out = operand(a[5]);
    if (!result(out, type, m, n)) return nullptr;
  } else {
    made = fresh({m, n}, type, *xq);
  }
  void* space = nullptr;
  size_t space_bytes = 0;
  at::Tensor made_space;
  if (a[7] != Py_None) {
    const at::Tensor* w = operand(a[7]);
    if (!w || !w->is_contiguous()) return nullptr;
    space = w->data_ptr();
    space_bytes = w->nbytes();
  } else if ((space_bytes = mi355x_fp8_rowwise_workspace_bytes(m, n, k, (int)variant))) {
    made_space = fresh({(int64_t)space_bytes}, at::kByte, *xq);
    space = made_space.data_ptr();
  }
  void* stream = current_stream();
  const bool ok = enqueue(mi355x_fp8_rowwise_gemm_ex, xq->data_ptr(), wq->data_ptr(), f32(*xs), f32(*ws), bias, out->data_ptr(),
                                      f16 ? MI355X_FP8_OUT_F16 : MI355X_FP8_OUT_BF16, m, n, k, xq->stride(0), wq->stride(0),
                                      out->stride(0), space, space_bytes, (int)variant, stream);
  if (!ok) return nullptr;
  if (a[5] == Py_None) return one(made);
  Py_INCREF(a[5]);
  return a[5];
}

// (group_a, group_b, m_sizes, a_scale, b_scale, out, tile configuration)
PyObject* gemm_grouped(PyObject* const* a, Py_ssize_t count) {
  if (count != 7) return nullptr;
  const at::Tensor *xq = operand(a[0]), *wq = operand(a[1]), *sizes = operand(a[2]), *xs = operand(a[3]), *ws = operand(a[4]);
  if (!matrix(xq, kCodes) || !matrix(wq, kCodes) || xq->size(1) != wq->size(1)) return nullptr;
  if (!sizes || sizes->scalar_type() != at::kInt || sizes->dim() != 1 || !sizes->is_contiguous() || sizes->numel() < 1) return nullptr;
  const int64_t m = xq->size(0), k = xq->size(1), groups = sizes->numel();
  if (wq->size(0) % groups) return nullptr;
  const int64_t n = wq->size(0) / groups;
  if (!factors(xs, m) || !factors(ws, groups * n)) return nullptr;
  const long config = PyLong_AsLong(a[6]);
  if (config < -1 || config > 255 || PyErr_Occurred()) return nullptr;
  at::Tensor made;
  const at::Tensor* out = &made;
  if (a[5] != Py_None) {
    out = operand(a[5]);
    if (!result(out, at::kBFloat16, m, n)) return nullptr;
  } else {
    made = fresh({m, n}, at::kBFloat16, *xq);
  }
  void* stream = current_stream();
  const bool ok = enqueue(mi355x_fp8_rowwise_grouped_gemm_ex, xq->data_ptr(), wq->data_ptr(), f32(*xs), f32(*ws), (const int32_t*)sizes->data_ptr(),
                                           out->data_ptr(), groups, m, n, k, xq->stride(0), wq->stride(0), out->stride(0),
                                           (int)config, a[5] == Py_None, stream);
  if (!ok) return nullptr;
  if (a[5] == Py_None) return one(made);
  Py_INCREF(a[5]);
  return a[5];
}

int64_t blocks(int64_t v) { return (v + 127) / 128; }

// (xq, wq, x_scale, w_scale, out)
PyObject* gemm_blockwise(PyObject* const* a, Py_ssize_t count) {
  if (count != 5) return nullptr;
  const at::Tensor *xq = operand(a[0]), *wq = operand(a[1]), *xs = operand(a[2]), *ws = operand(a[3]);
  if (!matrix(xq, kCodes) || !matrix(wq, kCodes) || xq->size(1) != wq->size(1)) return nullptr;
  const int64_t m = xq->size(0), n = wq->size(0), k = xq->size(1);
  if (!factors(xs, blocks(m) * blocks(k)) || xs->dim() != 2 || xs->size(0) != blocks(m) || xs->size(1) != blocks(k)) return nullptr;
  if (!factors(ws, blocks(n) * blocks(k)) || ws->dim() != 2 || ws->size(0) != blocks(n) || ws->size(1) != blocks(k)) return nullptr;
  at::Tensor made;
  const at::Tensor* out = &made;
  if (a[4] != Py_None) {
    out = operand(a[4]);
    if (!result(out, at::kBFloat16, m, n)) return nullptr;
  } else {
    made = fresh({m, n}, at::kBFloat16, *xq);
  }
  void* stream = current_stream();
  void* space = nullptr;
  at::Tensor made_space;
  const size_t space_bytes = mi355x_fp8_blockwise_workspace_bytes(m, n, k);
  if (space_bytes) {
    made_space = fresh({(int64_t)space_bytes}, at::kByte, *xq);
    space = made_space.data_ptr();
  }
  const bool ok = enqueue(mi355x_fp8_blockwise_gemm_ws, xq->data_ptr(), wq->data_ptr(), f32(*xs), f32(*ws), out->data_ptr(), m, n, k,
                          xq->stride(0), wq->stride(0), out->stride(0), space, space_bytes, -1, stream);
  if (!ok) return nullptr;
  if (a[4] == Py_None) return one(made);
  Py_INCREF(a[4]);
  return a[4];
}

// (x), block-wise or row-wise
template <bool BLOCKWISE>
PyObject* quantize(PyObject* const* a, Py_ssize_t count) {
  if (count != 1) return nullptr;
  const at::Tensor* x = operand(a[0]);
  const bool wide = x && x->scalar_type() == at::kFloat;
  if (!matrix(x, wide ? at::kFloat : at::kBFloat16)) return nullptr;
  const int64_t r = x->size(0), k = x->size(1);
  const int src = wide ? MI355X_FP8_SRC_F32 : MI355X_FP8_SRC_BF16;
  const at::Tensor q = fresh({r, k}, kCodes, *x);
  const at::Tensor inv = BLOCKWISE ? fresh({blocks(r), blocks(k)}, at::kFloat, *x) : fresh({r}, at::kFloat, *x);
  void* stream = current_stream();
  const bool ok = enqueue(BLOCKWISE ? mi355x_fp8_blockwise_quantize : mi355x_fp8_rowwise_quantize, x->data_ptr(), src, q.data_ptr(),
                          f32(inv), r, k, x->stride(0), q.stride(0), stream);
  return ok ? two(q, inv) : nullptr;
}

// (x, weight, eps)
PyObject* rms_norm_quantize(PyObject* const* a, Py_ssize_t count) {
  if (count != 3) return nullptr;
  const at::Tensor *x = operand(a[0]), *w = operand(a[1]);
  if (!matrix(x, at::kBFloat16) || !w || w->scalar_type() != at::kBFloat16 || w->dim() != 1 || w->size(0) != x->size(1) ||
      w->stride(0) != 1 || !PyFloat_CheckExact(a[2]))
    return nullptr;
  const int64_t r = x->size(0), k = x->size(1);
  const float eps = (float)PyFloat_AS_DOUBLE(a[2]);
  const at::Tensor q = fresh({r, k}, kCodes, *x), inv = fresh({r}, at::kFloat, *x);
  void* stream = current_stream();
  const bool ok = enqueue(mi355x_fp8_rmsnorm_rowwise_quantize, x->data_ptr(), w->data_ptr(), eps, q.data_ptr(), f32(inv), r, k, x->stride(0),
                                               q.stride(0), stream);
  return ok ? two(q, inv) : nullptr;
}

// (x1, x2)
PyObject* silu_mul_quantize(PyObject* const* a, Py_ssize_t count) {
  if (count != 2) return nullptr;
  const at::Tensor *x1 = operand(a[0]), *x2 = operand(a[1]);
  if (!matrix(x1, at::kBFloat16) || !matrix(x2, at::kBFloat16) || x1->sizes() != x2->sizes()) return nullptr;
  const int64_t r = x1->size(0), k = x1->size(1);
  const at::Tensor q = fresh({r, k}, kCodes, *x1), inv = fresh({r}, at::kFloat, *x1);
  void* stream = current_stream();
  const bool ok = enqueue(mi355x_fp8_silu_mul_rowwise_quantize, x1->data_ptr(), x2->data_ptr(), q.data_ptr(), f32(inv), r, k, x1->stride(0),
                                                x2->stride(0), q.stride(0), stream);
  return ok ? two(q, inv) : nullptr;
}

#define ENTRY(name, ...) {name, (PyCFunction)(void (*)(void))guarded<__VA_ARGS__>, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    ENTRY("mark_ready", mark_ready),
    ENTRY("gemm_rowwise", gemm_rowwise),
    ENTRY("gemm_grouped", gemm_grouped),
    ENTRY("gemm_blockwise", gemm_blockwise),
    ENTRY("row_quantize", quantize<false>),
    ENTRY("block_quantize", quantize<true>),
    ENTRY("rms_norm_quantize", rms_norm_quantize),
    ENTRY("silu_mul_quantize", silu_mul_quantize),
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "mi355x_torch_binding", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_mi355x_torch_binding() { return PyModule_Create(&module); }
