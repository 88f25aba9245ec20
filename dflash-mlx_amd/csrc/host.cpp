// Host side of the launches, native: the checks, allocations and argument lists of the calls a decoding step is made of.
//
// A 16-row projection takes 6 to 20 us of device time, and issued from Python its launch took 12 us around the 3.5 us of
// the HIP runtime: extents and types compared one attribute at a time, results allocated through the argument parser, every
// pointer and number converted for ctypes.  Here the same is done on the tensors themselves.  One verify_matmul of
// 1024 x 512 13.9 -> 6.9 us (its device time: 6.0), a GatedDeltaNet layer's verify block with its rollback 106 -> 51 us (49),
// the attention layer of one over 4096 keys 81 -> 54 us, one token through the projections of a 9B-shaped layer 61 -> 44 us.
// Results that skip the dispatcher and a block's operands read from the joint product: the call 5.6 -> 4.8 us, the recurrent
// layer's block of a 1024-wide model, which waits for its host, 43.6 -> 33.7, one token 34.9 -> 27.6.
//
// Each function serves the ordinary form of a call - strided device tensors of the exact extents, in one piece - and
// returns None for every other form and for whatever it would have to refuse: the Python function that asked then goes on
// as if it had not, copying, falling back to the array operators, or raising.  So nothing is decided here about what a
// call means, only how fast the common form of it gets to the device.  What Python holds (workspaces, options in the
// environment) is passed in, never kept; tensors are only held while a function runs.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/Context.h>
#include <ATen/EmptyTensor.h>
#include <ATen/record_function.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/Device.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>
#include <torch/csrc/utils/pybind.h>

#include <initializer_list>

#include "dflash_mi355.h"

namespace {

PyObject* g_error = nullptr;  // _native.NativeLibraryError

using at::Tensor;

constexpr int kNoCode = -1;

int dtype_code(at::ScalarType t) {
  return t == at::kBFloat16 ? DFLASH_BF16 : t == at::kHalf ? DFLASH_FP16 : t == at::kFloat ? DFLASH_FP32 : kNoCode;
}
int half_code(at::ScalarType t) { return t == at::kFloat ? kNoCode : dtype_code(t); }

// A tensor that is memory on the device and nothing else: no subclass, no wrapper of a transform, no lazy conjugate.
const Tensor* device_tensor(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const Tensor& t = THPVariable_Unpack(o);
  static const c10::DispatchKeySet ordinary =
      c10::DispatchKeySet({c10::DispatchKey::Dense, c10::DispatchKey::ADInplaceOrView, c10::DispatchKey::AutogradFunctionality,
                           c10::DispatchKey::AutocastCUDA}) | c10::DispatchKeySet(c10::BackendComponent::CUDABit);
  if (!t.defined() || (t.key_set().raw_repr() & ~ordinary.raw_repr()) != 0 || !t.is_cuda() || !t.has_storage()) return nullptr;
  return &t;
}
bool is_matrix(const Tensor& t, int64_t a, int64_t b) { return t.dim() == 2 && t.size(0) == a && t.size(1) == b && t.is_contiguous(); }
bool has_shape(const Tensor& t, std::initializer_list<int64_t> shape) { return t.sizes() == at::IntArrayRef(shape); }
bool aligned(const void* p, uintptr_t n) { return (reinterpret_cast<uintptr_t>(p) & (n - 1)) == 0; }
const void* at_of(const Tensor& t) { return t.const_data_ptr(); }

void* stream_of(const Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

bool integer(PyObject* o, long* out) {
  if (!PyLong_CheckExact(o)) return false;
  int overflow = 0;
  *out = PyLong_AsLongAndOverflow(o, &overflow);
  return overflow == 0 && *out >= 0 && *out < (1l << 31);
}
bool integer(PyObject* o, int* out) {
  long v = 0;
  if (!integer(o, &v)) return false;
  *out = (int)v;
  return true;
}

// The scratch that Python keeps for a key in one of its dictionaries, if there is enough of it; undefined if not.
Tensor kept_workspace(PyObject* held, PyObject* key, size_t need) {
  Tensor ws;
  if (key != nullptr && PyDict_CheckExact(held)) {
    PyObject* entry = PyDict_GetItemWithError(held, key);
    const Tensor* t = entry == nullptr ? nullptr : device_tensor(entry);
    if (t != nullptr && (size_t)t->nbytes() >= need && t->is_contiguous()) ws = *t;
  }
  Py_XDECREF(key);
  if (PyErr_Occurred()) PyErr_Clear();
  return ws;
}
PyObject* by_index(const Tensor& x, void* stream) {
  return Py_BuildValue("(iK)", (int)x.device().index(), (unsigned long long)(uintptr_t)stream);
}

PyObject* fail(int rc, const char* what) {
  PyErr_Format(g_error == nullptr ? PyExc_RuntimeError : g_error, "%s failed (code %d): %s", what, rc, dflash_last_error());
  return nullptr;
}

// Runs `work` (allocations and launches) without the interpreter lock, as the calls did that this replaces.
template <class F>
int released(F&& work) {
  pybind11::gil_scoped_release release;
  return work();
}

// Somebody looks at what goes through the dispatcher - a dispatch mode, a transform, a trace, the profiler - or wants new memory filled.
bool watched() {
  return !(c10::impl::tls_local_dispatch_key_set().included_ - c10::default_included_set).empty() || at::hasCallbacks() ||
         (at::globalContext().deterministicAlgorithms() && at::globalContext().deterministicFillUninitializedMemory());
}

// A new tensor beside `like`: at::empty without the way through the dispatcher, half of its 0.5 us, where nobody is there to see it.  A verify
// block of a recurrent layer with its rollback makes ten.
Tensor fresh(at::IntArrayRef shape, const Tensor& like, at::ScalarType type) {
  c10::Allocator* const allocator = like.storage().allocator();
  if (allocator == nullptr || c10::hip::current_device() != like.device().index() || watched())
    return at::empty(shape, like.options().dtype(type));
  return Tensor(at::detail::empty_generic(shape, allocator, c10::DispatchKeySet(c10::DispatchKey::CUDA), type, std::nullopt));
}
Tensor fresh(at::IntArrayRef shape, const Tensor& like) { return fresh(shape, like, like.scalar_type()); }

std::vector<int64_t> rows_by(const Tensor& x, int64_t n) {
  std::vector<int64_t> shape(x.sizes().begin(), x.sizes().end());
  shape.back() = n;
  return shape;
}

// ---- 4-bit products -------------------------------------------------------------------------------------------------
struct Product {
  const Tensor *x, *w, *s, *b;
  int64_t rows;
  int K, N, group, act, sb;
};

// x [.., K], w [N, K/8] of 32-bit words, scales and biases [N, K/group], all in one piece on one device.
bool product_of(PyObject* const* a, Product* p) {
  p->x = device_tensor(a[0]), p->w = device_tensor(a[1]), p->s = device_tensor(a[2]), p->b = device_tensor(a[3]);
  if (!p->x || !p->w || !p->s || !p->b || !integer(a[4], &p->group)) return false;
  const Tensor &x = *p->x, &w = *p->w, &s = *p->s, &b = *p->b;
  if (p->group != 32 && p->group != 64 && p->group != 128) return false;
  if (x.dim() < 1 || w.dim() != 2 || w.element_size() != 4) return false;
  const int64_t K = x.size(-1), N = w.size(0);
  if (K < p->group || K >= (1 << 30) || N < 1 || N >= (1 << 30) || K % p->group != 0 || N % 16 != 0) return false;
  p->K = (int)K, p->N = (int)N, p->rows = x.numel() / K;
  p->act = half_code(x.scalar_type()), p->sb = half_code(s.scalar_type());
  return p->rows >= 1 && p->rows < (1 << 30) && p->act != kNoCode && p->sb != kNoCode && b.scalar_type() == s.scalar_type() &&
         x.is_contiguous() && is_matrix(w, N, K / 8) && is_matrix(s, N, K / p->group) && is_matrix(b, N, K / p->group) &&
         w.device() == x.device() && s.device() == x.device() && b.device() == x.device();
}

// qmm_m16(x, w, scales, biases, group_size, kernel, workspaces): the verify product of 16 rows, variant chosen as "auto" does.
PyObject* qmm_m16(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Product p;
  int kernel;
  if (n != 7 || !product_of(a, &p) || p.rows != 16 || !integer(a[5], &kernel)) Py_RETURN_NONE;
  const bool pipe = p.K >= 8192 || p.N <= 8192;
  const int variant = pipe ? DFLASH_QMM_MMA2BIG_PIPE : DFLASH_QMM_MMA2BIG, parts = pipe ? 8 : 1;
  if (p.N % 32 != 0 || p.K % (32 * parts) != 0) Py_RETURN_NONE;
  void* stream = stream_of(*p.x);
  const size_t need = dflash_qmm_m16_workspace_bytes(p.K, p.N, p.group, variant, parts, kernel);
  Tensor ws, y;
  if (need != 0 && !(ws = kept_workspace(a[6], by_index(*p.x, stream), need)).defined()) Py_RETURN_NONE;
  const int rc = released([&] {
    y = fresh(rows_by(*p.x, p.N), *p.x);
    return dflash_qmm_m16(at_of(*p.x), (const uint32_t*)at_of(*p.w), at_of(*p.s), at_of(*p.b), y.mutable_data_ptr(),
                          need ? ws.mutable_data_ptr() : nullptr, need ? ws.nbytes() : 0, p.K, p.N, p.group, p.act, p.sb,
                          variant, parts, kernel, stream);
  });
  return rc != 0 ? fail(rc, "dflash_qmm_m16") : THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

// qmm_packed(x, codes, scales, biases, K, N, group_size, kernel, workspaces): the same on images of pack_weights.
PyObject* qmm_packed(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 9) Py_RETURN_NONE;
  const Tensor *x = device_tensor(a[0]), *w = device_tensor(a[1]), *s = device_tensor(a[2]), *b = device_tensor(a[3]);
  int K, N, group, kernel;
  if (!x || !w || !s || !b || !integer(a[4], &K) || !integer(a[5], &N) || !integer(a[6], &group) || !integer(a[7], &kernel)) Py_RETURN_NONE;
  const int act = half_code(x->scalar_type()), sb = half_code(s->scalar_type());
  if (act == kNoCode || sb == kNoCode || x->dim() < 1 || x->size(-1) != K || x->numel() != 16 * (int64_t)K ||
      !x->is_contiguous() || w->device() != x->device())
    Py_RETURN_NONE;
  void* stream = stream_of(*x);
  const size_t need = dflash_qmm_m16_workspace_bytes(K, N, group, DFLASH_QMM_MMA2BIG, 1, DFLASH_QMM_KERNEL_STREAM);
  Tensor y, ws = kept_workspace(a[8], by_index(*x, stream), need);
  if (!ws.defined()) Py_RETURN_NONE;
  const int rc = released([&] {
    y = fresh(rows_by(*x, N), *x);
    return dflash_qmm_m16_packed_by(at_of(*x), at_of(*w), at_of(*s), at_of(*b), y.mutable_data_ptr(), ws.mutable_data_ptr(),
                                    ws.nbytes(), K, N, group, act, sb, kernel, stream);
  });
  return rc != 0 ? fail(rc, "dflash_qmm_m16_packed") : THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

// qmm_few(x, w, scales, biases, group_size, kernel, workspaces): 1 to 16 rows outside the verify switch.
PyObject* qmm_few(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Product p;
  int kernel;
  if (n != 7 || !product_of(a, &p) || p.rows > 16 || !integer(a[5], &kernel)) Py_RETURN_NONE;
  if (p.rows < 16 && !aligned(at_of(*p.x), 16)) Py_RETURN_NONE;
  void* stream = stream_of(*p.x);
  const size_t need = dflash_qmm_m16_workspace_bytes(p.K, p.N, p.group, DFLASH_QMM_MMA2BIG, 1, kernel);
  Tensor ws, y;
  if (need != 0 && !(ws = kept_workspace(a[6], by_index(*p.x, stream), need)).defined()) Py_RETURN_NONE;
  const int rc = released([&] {
    y = fresh(rows_by(*p.x, p.N), *p.x);
    return dflash_qmm_few(at_of(*p.x), (const uint32_t*)at_of(*p.w), at_of(*p.s), at_of(*p.b), y.mutable_data_ptr(),
                          need ? ws.mutable_data_ptr() : nullptr, need ? ws.nbytes() : 0, (int)p.rows, p.K, p.N, p.group,
                          p.act, p.sb, kernel, stream);
  });
  return rc != 0 ? fail(rc, "dflash_qmm_few") : THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

// qmm_few_silu_mul(x, w, scales, biases, group_size, kernel, workspaces): the gated activation of 1 to 16 rows.
PyObject* qmm_few_silu_mul(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Product p;
  int kernel;
  if (n != 7 || !product_of(a, &p) || p.rows > 16 || p.act != p.sb || !integer(a[5], &kernel)) Py_RETURN_NONE;
  if (!aligned(at_of(*p.x), 16) || !aligned(at_of(*p.w), 16) || !aligned(at_of(*p.s), 4) || !aligned(at_of(*p.b), 4)) Py_RETURN_NONE;
  const size_t need = dflash_qmm_few_silu_mul_workspace_bytes(p.K, p.N, p.group);
  if (need == 0) Py_RETURN_NONE;
  void* stream = stream_of(*p.x);
  Tensor y, ws = kept_workspace(a[6], by_index(*p.x, stream), need);
  if (!ws.defined()) Py_RETURN_NONE;
  const int rc = released([&] {
    y = fresh(rows_by(*p.x, p.N / 2), *p.x);
    return dflash_qmm_few_silu_mul_by(at_of(*p.x), (const uint32_t*)at_of(*p.w), at_of(*p.s), at_of(*p.b), y.mutable_data_ptr(),
                                   ws.mutable_data_ptr(), ws.nbytes(), (int)p.rows, p.K, p.N, p.group, p.act, kernel, stream);
  });
  return rc != 0 ? fail(rc, "dflash_qmm_few_silu_mul") : THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

// qmm_rows(x, w, scales, biases, group_size, epilogue, workspaces): any number of rows.  Not on a stream that records: the
// scratch of a recorded launch is its own, which Python sees to.
PyObject* qmm_rows(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Product p;
  int epilogue;
  if (n != 7 || !product_of(a, &p) || !integer(a[5], &epilogue)) Py_RETURN_NONE;
  const bool silu = epilogue == DFLASH_QMM_EPILOGUE_SILU_MUL;
  if ((silu && (p.N % 32 != 0 || p.act != p.sb)) || !aligned(at_of(*p.x), 16) || !aligned(at_of(*p.w), 16)) Py_RETURN_NONE;
  void* stream = stream_of(*p.x);
  const size_t need = dflash_qmm_rows_workspace_bytes((int)p.rows, p.K, p.N, p.group, p.act, p.sb, epilogue);
  Tensor y, ws;
  if (need != 0) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing((hipStream_t)stream, &status) != hipSuccess || status != hipStreamCaptureStatusNone) Py_RETURN_NONE;
    if (!(ws = kept_workspace(a[6], by_index(*p.x, stream), need)).defined()) Py_RETURN_NONE;
  }
  const int rc = released([&] {
    y = fresh(rows_by(*p.x, silu ? p.N / 2 : p.N), *p.x);
    return dflash_qmm_rows(at_of(*p.x), (const uint32_t*)at_of(*p.w), at_of(*p.s), at_of(*p.b), y.mutable_data_ptr(),
                           need ? ws.mutable_data_ptr() : nullptr, need ? ws.nbytes() : 0, (int)p.rows, p.K, p.N, p.group,
                           p.act, p.sb, epilogue, stream);
  });
  return rc != 0 ? fail(rc, "dflash_qmm_rows") : THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

// gather(x, w, scales, biases, ids, group_size, kernel, workspaces): a row of x with the expert ids names, w [E, N, K/8].
PyObject* gather(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 8) Py_RETURN_NONE;
  const Tensor *x = device_tensor(a[0]), *w = device_tensor(a[1]), *s = device_tensor(a[2]), *b = device_tensor(a[3]),
               *ids = device_tensor(a[4]);
  int group, kernel;
  if (!x || !w || !s || !b || !ids || !integer(a[5], &group) || !integer(a[6], &kernel) || group < 1 || x->dim() < 1 || w->dim() != 3)
    Py_RETURN_NONE;
  const int64_t K = x->size(-1), E = w->size(0), N = w->size(1);
  if (K < group || K >= (1 << 30) || E < 1 || E >= (1 << 30) || N < 1 || N >= (1 << 30)) Py_RETURN_NONE;
  const int64_t P = x->numel() / K;
  const int act = half_code(x->scalar_type()), sb = half_code(s->scalar_type());
  if (P < 1 || P >= (1 << 30) || act == kNoCode || sb == kNoCode || b->scalar_type() != s->scalar_type() || w->element_size() != 4 ||
      ids->scalar_type() != at::kInt || ids->numel() != P || !has_shape(*w, {E, N, K / 8}) ||
      !has_shape(*s, {E, N, K / group}) || !has_shape(*b, {E, N, K / group}))
    Py_RETURN_NONE;
  for (const Tensor* t : {x, w, s, b, ids})
    if (!t->is_contiguous() || t->device() != x->device()) Py_RETURN_NONE;
  void* stream = stream_of(*x);
  const size_t need =
      kernel != DFLASH_QMM_KERNEL_TILE ? dflash_qmm_m16_gather_workspace_bytes((int)P, (int)K, (int)N, (int)E, group) : 0;
  Tensor ws, y;
  if (need != 0 && !(ws = kept_workspace(a[7], by_index(*x, stream), need)).defined()) Py_RETURN_NONE;
  const int rc = released([&] {
    y = fresh(rows_by(*x, N), *x);
    return dflash_qmm_m16_gather_by(at_of(*x), (const int32_t*)at_of(*ids), (const uint32_t*)at_of(*w), at_of(*s), at_of(*b),
                                    y.mutable_data_ptr(), need ? ws.mutable_data_ptr() : nullptr, need ? ws.nbytes() : 0, (int)P,
                                    (int)K, (int)N, (int)E, group, act, sb, kernel, stream);
  });
  return rc != 0 ? fail(rc, "dflash_qmm_m16_gather") : THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

// chain_bind(problem, x, x_before, columns): points a planned one-problem launch at other rows and at a result of their
// shape, which it returns.  problem: address of the caller's dflash_qmm_problem; x_before: rows of the type it was planned for.
PyObject* chain_bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 4 || !PyLong_CheckExact(a[0])) Py_RETURN_NONE;
  const Tensor *x = device_tensor(a[1]), *before = device_tensor(a[2]);
  int cols;
  if (!x || !before || !integer(a[3], &cols)) Py_RETURN_NONE;
  auto* problem = (dflash_qmm_problem*)PyLong_AsVoidPtr(a[0]);
  if (problem == nullptr || problem->wait_for >= 0 || x->dim() < 1 || x->size(-1) != problem->K || x->numel() != 16 * (int64_t)problem->K ||
      !x->is_contiguous() || x->scalar_type() != before->scalar_type() || x->device() != before->device())
    Py_RETURN_NONE;
  Tensor out = fresh(rows_by(*x, cols), *x);
  problem->x = at_of(*x);
  problem->y = out.mutable_data_ptr();
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// chain_launch(problems, count, need, group_size, act, scales, spin_limit, flags, x, workspaces): the workspace it used.
PyObject* chain_launch(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 10 || !PyLong_CheckExact(a[0])) Py_RETURN_NONE;
  int count, group, act, sb, spin, flags;
  long need;
  const Tensor* x = device_tensor(a[8]);
  if (!x || !integer(a[1], &count) || !integer(a[2], &need) || !integer(a[3], &group) || !integer(a[4], &act) ||
      !integer(a[5], &sb) || !integer(a[6], &spin) || !integer(a[7], &flags))
    Py_RETURN_NONE;
  const auto* problems = (const dflash_qmm_problem*)PyLong_AsVoidPtr(a[0]);
  void* stream = stream_of(*x);
  Tensor ws = kept_workspace(a[9], by_index(*x, stream), (size_t)need);
  if (problems == nullptr || !ws.defined()) Py_RETURN_NONE;
  const int rc = released([&] {
    return dflash_qmm_m16_chain(problems, count, ws.mutable_data_ptr(), ws.nbytes(), group, act, sb, spin, flags, stream);
  });
  return rc != 0 ? fail(rc, "dflash_qmm_m16_chain") : THPVariable_Wrap(std::move(ws));
  END_HANDLE_TH_ERRORS
}

// columns(product, bounds): product[..., lo:hi] for every pair of bounds.
PyObject* columns(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const Tensor* t = n == 2 ? device_tensor(a[0]) : nullptr;
  if (t == nullptr || t->dim() < 1 || !PyList_CheckExact(a[1])) Py_RETURN_NONE;
  const Py_ssize_t count = PyList_GET_SIZE(a[1]);
  const int64_t width = t->size(-1);
  THPObjectPtr out(PyTuple_New(count));
  if (!out) return nullptr;
  for (Py_ssize_t i = 0; i < count; ++i) {
    PyObject* pair = PyList_GET_ITEM(a[1], i);
    long lo, hi;
    if (!PyTuple_CheckExact(pair) || PyTuple_GET_SIZE(pair) != 2 || !integer(PyTuple_GET_ITEM(pair, 0), &lo) ||
        !integer(PyTuple_GET_ITEM(pair, 1), &hi) || lo > hi || hi > width)
      Py_RETURN_NONE;
    PyObject* part = THPVariable_Wrap(t->narrow(-1, lo, hi - lo));
    if (part == nullptr) return nullptr;
    PyTuple_SET_ITEM(out.get(), i, part);
  }
  return out.release();
  END_HANDLE_TH_ERRORS
}

// ---- GatedDeltaNet ----------------------------------------------------------------------------------------------------
// gdn_prepare(qkv, conv_state, conv_w, a, b, A_log, dt_bias, qkv_out, Hk, Hv, Dk, Dv, eps): without a mask;
// (conv_next, q, k, v, g, beta).
PyObject* gdn_prepare(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 13) Py_RETURN_NONE;
  const Tensor *qkv = device_tensor(a[0]), *cs = nullptr, *w = device_tensor(a[2]), *ga = device_tensor(a[3]),
               *gb = device_tensor(a[4]), *A = device_tensor(a[5]), *dt = device_tensor(a[6]), *out = nullptr;
  if (!qkv || !w || !ga || !gb || !A || !dt || qkv->dim() != 3) Py_RETURN_NONE;
  if (a[1] != Py_None && !(cs = device_tensor(a[1]))) Py_RETURN_NONE;
  if (a[7] != Py_None && !(out = device_tensor(a[7]))) Py_RETURN_NONE;
  int Hk, Hv, Dk, Dv;
  if (!integer(a[8], &Hk) || !integer(a[9], &Hv) || !integer(a[10], &Dk) || !integer(a[11], &Dv) || !PyFloat_CheckExact(a[12]))
    Py_RETURN_NONE;
  const auto covers = [](int d) { return d > 0 && d <= 256 && d % 64 == 0; };
  const int code = dtype_code(qkv->scalar_type()), param = dtype_code(A->scalar_type());
  const int64_t B = qkv->size(0), S = qkv->size(1), C = qkv->size(2);
  if (code == kNoCode || param == kNoCode || !covers(Dk) || !covers(Dv) || B < 1 || S < 1 || B * S >= (1 << 30) ||
      Hk > (1 << 15) || Hv > (1 << 15) || C != 2 * (int64_t)Hk * Dk + (int64_t)Hv * Dv)
    Py_RETURN_NONE;
  if (w->dim() < 2 || w->dim() > 3 || w->size(0) != C || (w->dim() == 3 && w->size(2) != 1) || !w->is_contiguous()) Py_RETURN_NONE;
  const int64_t K = w->size(1);
  const auto type = qkv->scalar_type();
  const auto device = qkv->device();
  if (K < 2 || K > 4 || w->scalar_type() != type || ga->scalar_type() != type || gb->scalar_type() != type ||
      dt->scalar_type() != A->scalar_type() || !has_shape(*ga, {B, S, Hv}) || !has_shape(*gb, {B, S, Hv}) ||
      !has_shape(*A, {Hv}) || !has_shape(*dt, {Hv}) || !A->is_contiguous() || !dt->is_contiguous() || w->device() != device ||
      ga->device() != device || gb->device() != device || A->device() != device || dt->device() != device)
    Py_RETURN_NONE;
  if (cs && (cs->scalar_type() != type || !has_shape(*cs, {B, K - 1, C}) || cs->device() != device || !cs->is_contiguous()))
    Py_RETURN_NONE;
  if (out && (out->scalar_type() != type || !has_shape(*out, {B, S, C}) || out->device() != device || !out->is_contiguous()))
    Py_RETURN_NONE;
  const int64_t step = qkv->element_size();
  if (qkv->stride(2) != 1 || ((int64_t)(uintptr_t)at_of(*qkv) | qkv->stride(0) * step | qkv->stride(1) * step) % 8 != 0 ||
      ga->stride(2) != 1 || gb->stride(2) != 1)
    Py_RETURN_NONE;
  const long long strides[6] = {qkv->stride(0), qkv->stride(1), ga->stride(0), ga->stride(1), gb->stride(0), gb->stride(1)};
  void* stream = stream_of(*qkv);
  const float eps = (float)PyFloat_AS_DOUBLE(a[12]);
  Tensor next, q, k, v, g, beta;
  const int rc = released([&] {
    next = fresh({B, K - 1, C}, *qkv);
    q = fresh({B, S, Hk, Dk}, *qkv);
    k = fresh({B, S, Hk, Dk}, *qkv);
    v = fresh({B, S, Hv, Dv}, *qkv);
    g = fresh({B, S, Hv}, *qkv, at::kFloat);
    beta = fresh({B, S, Hv}, *qkv);
    return dflash_gdn_prepare_rows(at_of(*qkv), cs ? at_of(*cs) : nullptr, at_of(*w), at_of(*ga), at_of(*gb), at_of(*A), at_of(*dt),
                                   nullptr, next.mutable_data_ptr(), q.mutable_data_ptr(), k.mutable_data_ptr(),
                                   v.mutable_data_ptr(), (float*)g.mutable_data_ptr(), beta.mutable_data_ptr(),
                                   out ? out->mutable_data_ptr() : nullptr, strides, (int)B, (int)S, Hk, Hv, Dk, Dv, (int)K, code,
                                   param, eps, stream);
  });
  if (rc != 0) return fail(rc, "dflash_gdn_prepare");
  return Py_BuildValue("(NNNNNN)", THPVariable_Wrap(std::move(next)), THPVariable_Wrap(std::move(q)), THPVariable_Wrap(std::move(k)),
                       THPVariable_Wrap(std::move(v)), THPVariable_Wrap(std::move(g)), THPVariable_Wrap(std::move(beta)));
  END_HANDLE_TH_ERRORS
}

// gdn_forward(q, k, v, g, beta, state, z, weight, eps, with_tape): without a mask, gates per head; z and weight None, or the
// gate and the weight of the output norm.  state None: zeros of q's type, for prompts that a kernel starts with them.
// (y, state, tape or None).
PyObject* gdn_forward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 10) Py_RETURN_NONE;
  const Tensor *q = device_tensor(a[0]), *k = device_tensor(a[1]), *v = device_tensor(a[2]), *g = device_tensor(a[3]),
               *beta = device_tensor(a[4]), *state = nullptr, *z = nullptr, *w = nullptr;
  if (a[5] != Py_None && !(state = device_tensor(a[5]))) Py_RETURN_NONE;
  if (!q || !k || !v || !g || !beta || k->dim() != 4 || v->dim() != 4 || !PyFloat_CheckExact(a[8])) Py_RETURN_NONE;
  if (a[6] != Py_None && (!(z = device_tensor(a[6])) || !(w = device_tensor(a[7])))) Py_RETURN_NONE;
  const int64_t B = k->size(0), T = k->size(1), hk = k->size(2), dk = k->size(3), hv = v->size(2), dv = v->size(3);
  const int code = dtype_code(q->scalar_type()), g_code = dtype_code(g->scalar_type()), b_code = dtype_code(beta->scalar_type()),
            s_code = state ? dtype_code(state->scalar_type()) : code;
  if (B < 1 || T < 1 || hk < 1 || hv < 1 || dv < 1 || hv % hk != 0 || dk < 32 || dk % 32 != 0 || B * T * hv >= (1 << 30) ||
      code == kNoCode || g_code == kNoCode || b_code == kNoCode || s_code == kNoCode || k->scalar_type() != q->scalar_type() ||
      v->scalar_type() != q->scalar_type())
    Py_RETURN_NONE;
  if (!has_shape(*q, {B, T, hk, dk}) || !has_shape(*v, {B, T, hv, dv}) || !has_shape(*g, {B, T, hv}) ||
      !has_shape(*beta, {B, T, hv}))
    Py_RETURN_NONE;
  if (state && (!has_shape(*state, {B, hv, dv, dk}) || !state->is_contiguous() || state->device() != q->device())) Py_RETURN_NONE;
  for (const Tensor* t : {q, k, v, g, beta})
    if (!t->is_contiguous() || t->device() != q->device()) Py_RETURN_NONE;
  int w_code = code;
  if (z != nullptr) {
    w_code = dtype_code(w->scalar_type());
    const int64_t step = z->element_size();
    if (w_code == kNoCode || z->scalar_type() != q->scalar_type() || !has_shape(*z, {B, T, hv, dv}) ||
        z->device() != q->device() || w->device() != q->device() || w->numel() != dv || !w->is_contiguous() || !aligned(at_of(*w), 16) ||
        dv % 64 != 0 || dv > 256)
      Py_RETURN_NONE;
    if (z->stride(3) != 1 || z->stride(2) != dv || z->stride(1) == 0 || !aligned(at_of(*z), 16) ||
        (z->stride(0) | z->stride(1)) * step % 16 != 0)
      Py_RETURN_NONE;
  }
  size_t need = T > 16 ? dflash_gdn_forward_workspace_bytes((int)B, (int)T, (int)hk, (int)hv, (int)dk, (int)dv, code, 0) : 0;
  for (const Tensor* t : {q, k, v, state})
    if (t != nullptr && !aligned(at_of(*t), 16)) need = 0;
  if (state == nullptr && (need == 0 || dflash_get_option(DFLASH_OPT_GDN_STEP_BY_STEP) != 0)) Py_RETURN_NONE;
  const bool with_tape = a[9] == Py_True || need == 0 || dflash_get_option(DFLASH_OPT_GDN_STEP_BY_STEP) != 0;
  void* stream = stream_of(*q);
  const float eps = (float)PyFloat_AS_DOUBLE(a[8]);
  Tensor y, next, tape, ws;
  const int rc = released([&] {
    y = fresh({B, T, hv, dv}, *q);
    if (need != 0) ws = fresh({(int64_t)need}, *q, at::kByte);
    if (with_tape) tape = fresh({B, T, hv, dv}, *q, at::kFloat);
    next = fresh({B, hv, dv, dk}, state ? *state : *q);
    return dflash_gdn_forward(at_of(*q), at_of(*k), at_of(*v), at_of(*g), at_of(*beta), state ? at_of(*state) : nullptr, next.mutable_data_ptr(),
                              z ? at_of(*z) : nullptr, z ? at_of(*w) : nullptr, y.mutable_data_ptr(),
                              with_tape ? (float*)tape.mutable_data_ptr() : nullptr, nullptr,
                              need ? ws.mutable_data_ptr() : nullptr, need, z ? z->stride(0) : 0, z ? z->stride(1) : 0, (int)B,
                              (int)T, (int)hk, (int)hv, (int)dk, (int)dv, code, g_code, b_code, s_code, w_code, 0, eps, stream);
  });
  if (rc != 0) return fail(rc, "dflash_gdn_forward");
  PyObject* tape_out = with_tape ? THPVariable_Wrap(std::move(tape)) : (Py_INCREF(Py_None), Py_None);
  return Py_BuildValue("(NNN)", THPVariable_Wrap(std::move(y)), THPVariable_Wrap(std::move(next)), tape_out);
  END_HANDLE_TH_ERRORS
}

// [B, S, width] of a product of three extents: all of it, or some of its columns.
struct Columns {
  const Tensor* of = nullptr;
  int64_t first = 0, width = 0;
  const void* at() const { return static_cast<const char*>(at_of(*of)) + first * of->element_size(); }
  int64_t slot() const { return of->stride(0); }
  int64_t row() const { return of->stride(1); }
  bool whole() const { return width == of->size(2) && of->is_contiguous(); }
  bool is(int64_t B, int64_t S, int64_t n, at::ScalarType type, c10::Device device) const {
    return of->dim() == 3 && of->size(0) == B && of->size(1) == S && width == n && of->scalar_type() == type && of->device() == device &&
           of->stride(2) == 1;
  }
};
bool columns_of(PyObject* o, Columns* c) {
  c->of = device_tensor(o);
  if (c->of == nullptr || c->of->dim() != 3) return false;
  c->width = c->of->size(2);
  return true;
}
bool columns_of(const Tensor& product, PyObject* pair, Columns* c) {
  long lo, hi;
  if (!PyTuple_CheckExact(pair) || PyTuple_GET_SIZE(pair) != 2 || !integer(PyTuple_GET_ITEM(pair, 0), &lo) ||
      !integer(PyTuple_GET_ITEM(pair, 1), &hi) || lo > hi || hi > product.size(2))
    return false;
  c->of = &product, c->first = lo, c->width = hi - lo;
  return true;
}

// The launch behind gdn_block and gdn_block_of: a block of up to 16 tokens without a mask, where that has a form for it; rest: conv_state, conv_w,
// A_log, dt_bias, weight, state, Hk, Hv, Dk, Dv, eps, norm_eps, record.  z.of null: no output norm.
PyObject* block_of(const Columns& qkv, const Columns& z, const Columns& b, const Columns& a, PyObject* const (&rest)[13]) {
  const Tensor *cs = nullptr, *w = device_tensor(rest[1]), *A = device_tensor(rest[2]), *dt = device_tensor(rest[3]), *weight = nullptr,
               *state = nullptr;
  if (!w || !A || !dt) Py_RETURN_NONE;
  if (rest[0] != Py_None && !(cs = device_tensor(rest[0]))) Py_RETURN_NONE;
  if (z.of && !(weight = device_tensor(rest[4]))) Py_RETURN_NONE;
  if (rest[5] != Py_None && !(state = device_tensor(rest[5]))) Py_RETURN_NONE;
  int Hk, Hv, D, Dv;
  if (!integer(rest[6], &Hk) || !integer(rest[7], &Hv) || !integer(rest[8], &D) || !integer(rest[9], &Dv) || !PyFloat_CheckExact(rest[10]) ||
      !PyFloat_CheckExact(rest[11]))
    Py_RETURN_NONE;
  const bool record = rest[12] == Py_True;
  const Tensor& first = *qkv.of;
  const int64_t B = first.size(0), S = first.size(1), C = qkv.width;
  const auto type = at::kBFloat16;
  const auto device = first.device();
  const int param = dtype_code(A->scalar_type()), s_code = state ? dtype_code(state->scalar_type()) : DFLASH_BF16;
  if (param == kNoCode || s_code == kNoCode || D != Dv || (D != 64 && D != 128) || B < 1 || S < 1 ||
      S > 16 || Hk < 1 || Hv < 1 || Hk > (1 << 15) || Hv > (1 << 15) || Hv % Hk != 0 ||
      !qkv.is(B, S, 2 * (int64_t)Hk * D + (int64_t)Hv * D, type, device) ||
      B * S * (2 * Hk + Hv) * D >= (1ll << 31) || dflash_get_option(DFLASH_OPT_GDN_STEP_BY_STEP) != 0)
    Py_RETURN_NONE;
  if (w->dim() < 2 || w->dim() > 3 || w->size(0) != C || w->size(1) != 4 || (w->dim() == 3 && w->size(2) != 1) ||
      !w->is_contiguous() || w->scalar_type() != type || !a.is(B, S, Hv, type, device) || !b.is(B, S, Hv, type, device) ||
      dt->scalar_type() != A->scalar_type() || !has_shape(*A, {Hv}) || !has_shape(*dt, {Hv}) || !A->is_contiguous() || !dt->is_contiguous())
    Py_RETURN_NONE;
  for (const Tensor* t : {w, A, dt})
    if (t->device() != device) Py_RETURN_NONE;
  if (state && (!has_shape(*state, {B, Hv, D, D}) || !state->is_contiguous() || !aligned(at_of(*state), 16) || state->device() != device))
    Py_RETURN_NONE;
  if (cs && (cs->scalar_type() != type || !has_shape(*cs, {B, 3, C}) || cs->device() != device || !cs->is_contiguous() ||
             !aligned(at_of(*cs), 8)))
    Py_RETURN_NONE;
  if (!aligned(qkv.at(), 8) || (qkv.slot() | qkv.row()) % 4 != 0 || qkv.row() >= (1 << 26) || !aligned(at_of(*w), 8)) Py_RETURN_NONE;
  if (z.of && (!z.is(B, S, (int64_t)Hv * D, type, device) || (z.slot() | z.row()) % 8 != 0 || !aligned(z.at(), 16) ||
               dtype_code(weight->scalar_type()) == kNoCode || weight->numel() != D || !weight->is_contiguous() ||
               weight->device() != device || !aligned(at_of(*weight), 16)))
    Py_RETURN_NONE;
  dflash_gdn_block_args p = {};
  p.qkv = qkv.at(), p.conv_state = cs ? at_of(*cs) : nullptr, p.conv_w = at_of(*w), p.a = a.at(), p.b = b.at();
  p.A_log = at_of(*A), p.dt_bias = at_of(*dt);
  p.qkv_slot = qkv.slot(), p.qkv_row = qkv.row(), p.a_slot = a.slot(), p.a_row = a.row();
  p.b_slot = b.slot(), p.b_row = b.row();
  if (z.of) p.z = z.at(), p.norm_weight = at_of(*weight), p.z_slot = z.slot(), p.z_row = z.row();
  p.slots = (int)B, p.T = (int)S, p.Hk = Hk, p.Hv = Hv, p.D = D, p.param_dtype = param, p.state_dtype = s_code;
  p.weight_dtype = z.of ? dtype_code(weight->scalar_type()) : DFLASH_BF16;
  p.eps = (float)PyFloat_AS_DOUBLE(rest[10]), p.norm_eps = (float)PyFloat_AS_DOUBLE(rest[11]);
  void* stream = stream_of(first);
  Tensor y, next, conv, tape, k, g, one, zeros;
  const int rc = released([&] {
    if (!state) zeros = at::zeros({B, Hv, D, D}, first.options()), state = &zeros;
    p.state_in = at_of(*state);
    y = fresh({B, S, (int64_t)Hv * D}, first);
    next = fresh({B, Hv, D, D}, *state);
    conv = fresh({B, 3, C}, first);
    tape = fresh({B, S, Hv, D}, first, at::kFloat);
    p.y = y.mutable_data_ptr(), p.state_out = next.mutable_data_ptr(), p.conv_next = conv.mutable_data_ptr();
    p.tape = (float*)tape.mutable_data_ptr();
    if (record) {
      k = fresh({B, S, Hk, D}, first);
      g = fresh({B, S, Hv}, first, at::kFloat);
      p.k = k.mutable_data_ptr(), p.g = (float*)g.mutable_data_ptr();
      if (!qkv.whole()) {
        one = fresh({B, S, C}, first);
        p.qkv_out = one.mutable_data_ptr();
      }
    }
    return dflash_gdn_block(&p, stream);
  });
  if (rc != 0) return fail(rc, "dflash_gdn_block");
  const auto wrapped = [](Tensor&& t) -> PyObject* {
    if (!t.defined()) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(t));
  };
  return Py_BuildValue("(NNNNNNN)", wrapped(std::move(y)), wrapped(std::move(next)), wrapped(std::move(conv)), wrapped(std::move(tape)),
                       wrapped(std::move(k)), wrapped(std::move(g)), wrapped(std::move(one)));
}

// gdn_block(qkv, conv_state, conv_w, a, b, A_log, dt_bias, z, weight, state, Hk, Hv, Dk, Dv, eps, norm_eps, record): z [B, S, Hv Dv] and the norm's
// weight None, or what the output norm takes; state None: zeros of qkv's type, filled once the call is known to be served.
// (y [B, S, Hv Dv], state, conv_next, tape, k, g, qkv in one piece); the last three None unless recorded, the last one also where
// qkv is in one piece already.
PyObject* gdn_block(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Columns qkv, z, gb, ga;
  if (n != 17 || !columns_of(a[0], &qkv) || !columns_of(a[3], &ga) || !columns_of(a[4], &gb) || (a[7] != Py_None && !columns_of(a[7], &z)))
    Py_RETURN_NONE;
  return block_of(qkv, z, gb, ga, {a[1], a[2], a[5], a[6], a[8], a[9], a[10], a[11], a[12], a[13], a[14], a[15], a[16]});
  END_HANDLE_TH_ERRORS
}

// gdn_block_of(product, bounds, conv_state, conv_w, A_log, dt_bias, weight, state, Hk, Hv, Dk, Dv, eps, norm_eps, record): the same from the joint
// product of the layer's input projections; bounds: the columns of qkv, z, b and a.  weight None: no output norm.
PyObject* gdn_block_of(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const Tensor* product = n == 15 ? device_tensor(a[0]) : nullptr;
  Columns part[4];
  if (product == nullptr || product->dim() != 3 || !PyList_CheckExact(a[1]) || PyList_GET_SIZE(a[1]) != 4) Py_RETURN_NONE;
  for (int i = 0; i < 4; ++i)
    if (!columns_of(*product, PyList_GET_ITEM(a[1], i), &part[i])) Py_RETURN_NONE;
  if (a[6] == Py_None) part[1].of = nullptr;
  return block_of(part[0], part[1], part[2], part[3], {a[2], a[3], a[4], a[5], a[6], a[7], a[8], a[9], a[10], a[11], a[12], a[13], a[14]});
  END_HANDLE_TH_ERRORS
}

// What a rollback of one cache takes: device tensors as record_tape() keeps them, of extents that the kernel can index.
struct Rollback {
  const Tensor *tape, *k, *g, *qkv, *state, *prev;
  int64_t B, T, hv, dv, hk, dk, C;
  int t_code, k_code, g_code, s_code;
};
bool rollback_of(PyObject* const (&a)[6], int steps, int keep, Rollback* r) {
  r->tape = device_tensor(a[0]), r->k = device_tensor(a[1]), r->g = device_tensor(a[2]), r->qkv = device_tensor(a[3]);
  r->state = device_tensor(a[4]), r->prev = nullptr;
  if (!r->tape || !r->k || !r->g || !r->qkv || !r->state) return false;
  const Tensor &tape = *r->tape, &k = *r->k, &g = *r->g, &qkv = *r->qkv, &state = *r->state;
  if (tape.dim() != 4 || k.dim() != 4 || g.dim() != 3 || qkv.dim() != 3 || keep < 1) return false;
  if (a[5] != Py_None && !(r->prev = device_tensor(a[5]))) return false;
  const int64_t B = r->B = tape.size(0), T = r->T = tape.size(1), hv = r->hv = tape.size(2), dv = r->dv = tape.size(3);
  const int64_t hk = r->hk = k.size(2), dk = r->dk = k.size(3), C = r->C = qkv.size(2);
  if (hk < 1 || steps > T || !has_shape(k, {B, T, hk, dk}) || !has_shape(g, {B, T, hv}) || !has_shape(qkv, {B, T, C}) ||
      !has_shape(state, {B, hv, dv, dk}) || dk < 32 || dk % 32 != 0 || hv % hk != 0 ||
      T * (dv + 2 * dk + 1) * 4 + dk * 4 > 64 * 1024)
    return false;
  for (const Tensor* t : {&tape, &k, &g, &qkv, &state})
    if (!t->is_contiguous() || t->device() != state.device()) return false;
  if (r->prev && (r->prev->device() != qkv.device() || !r->prev->is_contiguous() || r->prev->scalar_type() != qkv.scalar_type() ||
                  !has_shape(*r->prev, {B, keep, C})))
    return false;
  r->t_code = dtype_code(tape.scalar_type()), r->k_code = dtype_code(k.scalar_type()), r->g_code = dtype_code(g.scalar_type());
  r->s_code = dtype_code(state.scalar_type());
  return r->t_code != kNoCode && r->k_code != kNoCode && r->g_code != kNoCode && r->s_code != kNoCode;
}

// rollback_layer(tape, k, g, qkv, state, conv_prev, steps, keep, exact): replay and conv window of one cache's tape;
// (state, conv window).
PyObject* rollback_layer(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 9) Py_RETURN_NONE;
  Rollback r = {};
  int steps, keep, exact;
  if (!integer(a[6], &steps) || !integer(a[7], &keep) || !integer(a[8], &exact) ||
      !rollback_of({a[0], a[1], a[2], a[3], a[4], a[5]}, steps, keep, &r))
    Py_RETURN_NONE;
  void* stream = stream_of(*r.state);
  Tensor next, conv;
  const int rc = released([&] {
    next = fresh({r.B, r.hv, r.dv, r.dk}, *r.state);
    conv = fresh({r.B, keep, r.C}, *r.qkv);
    return dflash_rollback_layer(at_of(*r.tape), at_of(*r.k), at_of(*r.g), at_of(*r.state), next.mutable_data_ptr(),
                                 r.prev ? at_of(*r.prev) : nullptr, at_of(*r.qkv), conv.mutable_data_ptr(), nullptr, steps, (int)r.B,
                                 (int)r.T, (int)r.hk, (int)r.hv, (int)r.dk, (int)r.dv, r.s_code, r.t_code, r.k_code, r.g_code, 0,
                                 exact, keep, (int)r.C, (int)r.qkv->element_size(), stream);
  });
  if (rc != 0) return fail(rc, "dflash_rollback_layer");
  return Py_BuildValue("(NN)", THPVariable_Wrap(std::move(next)), THPVariable_Wrap(std::move(conv)));
  END_HANDLE_TH_ERRORS
}

// rollback_layers(operands, steps, keep, exact): the same for several caches whose operands have the same extents, types and
// device.  operands: a list of the tuples (tape, k, g, qkv, state, conv_prev).  A list of (conv window, state): a cache's entries.
PyObject* rollback_layers(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  int steps, keep, exact;
  if (n != 4 || !PyList_CheckExact(a[0]) || !integer(a[1], &steps) || !integer(a[2], &keep) || !integer(a[3], &exact)) Py_RETURN_NONE;
  const Py_ssize_t count = PyList_GET_SIZE(a[0]);
  if (count < 2 || count >= (1 << 20)) Py_RETURN_NONE;
  std::vector<dflash_rollback_operands> at(count);
  Rollback r = {};
  for (Py_ssize_t i = 0; i < count; ++i) {
    PyObject* one = PyList_GET_ITEM(a[0], i);
    if (!PyTuple_CheckExact(one) || PyTuple_GET_SIZE(one) != 6) Py_RETURN_NONE;
    Rollback o = {};
    PyObject* const parts[6] = {PyTuple_GET_ITEM(one, 0), PyTuple_GET_ITEM(one, 1), PyTuple_GET_ITEM(one, 2),
                                PyTuple_GET_ITEM(one, 3), PyTuple_GET_ITEM(one, 4), PyTuple_GET_ITEM(one, 5)};
    if (!rollback_of(parts, steps, keep, &o)) Py_RETURN_NONE;
    if (i == 0) r = o;
    if (o.B != r.B || o.T != r.T || o.hv != r.hv || o.dv != r.dv || o.hk != r.hk || o.dk != r.dk || o.C != r.C || o.t_code != r.t_code ||
        o.k_code != r.k_code || o.g_code != r.g_code || o.s_code != r.s_code || o.qkv->scalar_type() != r.qkv->scalar_type() ||
        o.state->device() != r.state->device())
      Py_RETURN_NONE;
    at[i] = {at_of(*o.tape), at_of(*o.k), at_of(*o.g), at_of(*o.state), nullptr, o.prev ? at_of(*o.prev) : nullptr, at_of(*o.qkv), nullptr};
  }
  void* stream = stream_of(*r.state);
  std::vector<Tensor> made(2 * count);
  const int rc = released([&] {
    for (Py_ssize_t i = 0; i < count; ++i) {
      made[2 * i] = fresh({r.B, keep, r.C}, *r.qkv);
      made[2 * i + 1] = fresh({r.B, r.hv, r.dv, r.dk}, *r.state);
      at[i].conv_out = made[2 * i].mutable_data_ptr(), at[i].state_out = made[2 * i + 1].mutable_data_ptr();
    }
    return dflash_rollback_layers(at.data(), (int)count, steps, (int)r.B, (int)r.T, (int)r.hk, (int)r.hv, (int)r.dk, (int)r.dv, r.s_code,
                                  r.t_code, r.k_code, r.g_code, exact, keep, (int)r.C, (int)r.qkv->element_size(), stream);
  });
  if (rc != 0) return fail(rc, "dflash_rollback_layers");
  THPObjectPtr out(PyList_New(count));
  if (!out) return nullptr;
  for (Py_ssize_t i = 0; i < count; ++i) {
    PyObject* pair = PyList_New(2);
    if (pair == nullptr) return nullptr;
    PyList_SET_ITEM(out.get(), i, pair);
    for (int j = 0; j < 2; ++j) {
      PyObject* t = THPVariable_Wrap(std::move(made[2 * i + j]));
      if (t == nullptr) return nullptr;
      PyList_SET_ITEM(pair, j, t);
    }
  }
  return out.release();
  END_HANDLE_TH_ERRORS
}

// ---- attention --------------------------------------------------------------------------------------------------------
// attn_prepare(q_proj_output, keys, values, q_weight, k_weight, cache_keys, cache_values, Hq, Hk, rope_dims, offset): what a
// launch of dflash_attn_prepare into a cache with room for the block takes: (queries, the cache's keys and values up to the block's
// end, the arguments from q to offset, the strides, the three dtype codes).  The caller launches.
PyObject* attn_prepare(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 11) Py_RETURN_NONE;
  const Tensor* t[7];
  for (int i = 0; i < 7; ++i)
    if (!(t[i] = device_tensor(a[i]))) Py_RETURN_NONE;
  const Tensor &q = *t[0], &k = *t[1], &v = *t[2], &qw = *t[3], &kw = *t[4], &ck = *t[5], &cv = *t[6];
  int Hq, Hk, rope, offset;
  if (!integer(a[7], &Hq) || !integer(a[8], &Hk) || !integer(a[9], &rope) || !integer(a[10], &offset) || Hq < 1 || Hk < 1 ||
      q.dim() != 3 || ck.dim() != 4 || cv.dim() != 4)
    Py_RETURN_NONE;
  const int64_t B = q.size(0), L = q.size(1), D = q.size(2) / (2 * (int64_t)Hq), per = D / 64, capacity = ck.size(2);
  const int code = half_code(q.scalar_type()), q_code = dtype_code(qw.scalar_type()), k_code = dtype_code(kw.scalar_type());
  if (code == kNoCode || q_code == kNoCode || k_code == kNoCode || (D != 64 && D != 128 && D != 192 && D != 256) ||
      q.size(2) != 2 * (int64_t)Hq * D || rope < 1 || rope > D || rope % (2 * per) != 0 || B < 1 || L < 1 || B * L >= (1 << 30) ||
      offset + L > capacity || !has_shape(k, {B, L, Hk * D}) || !has_shape(v, {B, L, Hk * D}) || !has_shape(qw, {D}) ||
      !has_shape(kw, {D}) || !qw.is_contiguous() || !kw.is_contiguous() || !aligned(at_of(qw), 8) || !aligned(at_of(kw), 8) ||
      !has_shape(ck, {B, Hk, capacity, D}) || !has_shape(cv, {B, Hk, capacity, D}))
    Py_RETURN_NONE;
  for (const Tensor* x : {&k, &v, &ck, &cv})
    if (x->scalar_type() != q.scalar_type() || x->device() != q.device()) Py_RETURN_NONE;
  if (qw.device() != q.device() || kw.device() != q.device()) Py_RETURN_NONE;
  for (const Tensor* x : {&q, &k, &v})
    if (x->stride(2) != 1 || (x->stride(0) | x->stride(1)) % 4 != 0 || !aligned(at_of(*x), 8)) Py_RETURN_NONE;
  for (const Tensor* x : {&ck, &cv})
    if (x->stride(3) != 1 || (x->stride(0) | x->stride(1) | x->stride(2)) % 4 != 0 || !aligned(at_of(*x), 8)) Py_RETURN_NONE;
  Tensor queries = fresh({B, Hq, L, D}, q);
  const auto address = [](const void* p, int64_t elements) { return (unsigned long long)(uintptr_t)p + 2 * (unsigned long long)elements; };
  PyObject* args = Py_BuildValue("(KKKKKKKKiiiiiii)", address(at_of(q), 0), address(at_of(k), 0), address(at_of(v), 0), address(at_of(qw), 0),
                                 address(at_of(kw), 0), address(queries.mutable_data_ptr(), 0),
                                 address(ck.mutable_data_ptr(), offset * ck.stride(2)), address(cv.mutable_data_ptr(), offset * cv.stride(2)),
                                 (int)B, (int)L, Hq, Hk, (int)D, rope, offset);
  PyObject* strides = Py_BuildValue("(LLLLLLLLLLLL)", (long long)q.stride(0), (long long)q.stride(1), (long long)k.stride(0),
                                    (long long)k.stride(1), (long long)v.stride(0), (long long)v.stride(1), (long long)ck.stride(0),
                                    (long long)ck.stride(1), (long long)ck.stride(2), (long long)cv.stride(0), (long long)cv.stride(1),
                                    (long long)cv.stride(2));
  return Py_BuildValue("(NNNNN(iii))", THPVariable_Wrap(std::move(queries)), THPVariable_Wrap(ck.narrow(2, 0, offset + L)),
                       THPVariable_Wrap(cv.narrow(2, 0, offset + L)), args, strides, code, q_code, k_code);
  END_HANDLE_TH_ERRORS
}

// sdpa_q16(queries, keys, values, scale, gate, workspaces): a block of 16 queries without a mask; gate None, or the output
// of the projection that carries it.
PyObject* sdpa_q16(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 6) Py_RETURN_NONE;
  const Tensor *q = device_tensor(a[0]), *k = device_tensor(a[1]), *v = device_tensor(a[2]), *gate = nullptr;
  if (!q || !k || !v || q->dim() != 4 || k->dim() != 4 || v->dim() != 4 || !PyFloat_CheckExact(a[3])) Py_RETURN_NONE;
  if (a[4] != Py_None && !(gate = device_tensor(a[4]))) Py_RETURN_NONE;
  const int64_t B = q->size(0), hq = q->size(1), d = q->size(3), hk = k->size(1), N = k->size(2);
  const int code = half_code(q->scalar_type());
  if (code == kNoCode || q->size(2) != 16 || (d != 128 && d != 256) || hk < 1 || hq % hk != 0 || hq / hk > 8 || N < 16 ||
      N >= (1 << 30) || k->scalar_type() != q->scalar_type() || v->scalar_type() != q->scalar_type() ||
      !has_shape(*k, {B, hk, N, d}) || !has_shape(*v, {B, hk, N, d}) || k->device() != q->device() || v->device() != q->device() ||
      !q->is_contiguous())
    Py_RETURN_NONE;
  for (const Tensor* t : {k, v})
    if (t->stride(3) != 1 || (t->stride(0) | t->stride(1) | t->stride(2)) % 8 != 0 || !aligned(at_of(*t), 16)) Py_RETURN_NONE;
  const size_t need = dflash_sdpa_q16_workspace_bytes((int)B, (int)hq, (int)hk, (int)N, (int)d);
  void* stream = stream_of(*q);
  Tensor out, ws;
  if (need != 0) {
    PyObject* key = Py_BuildValue("(NK)", THPDevice_New(q->device()), (unsigned long long)(uintptr_t)stream);
    if (!(ws = kept_workspace(a[5], key, need)).defined()) Py_RETURN_NONE;
  }
  const bool gated = gate != nullptr && need != 0 && has_shape(*gate, {B, 16, hq * 2 * d}) &&
                     gate->scalar_type() == q->scalar_type() && gate->device() == q->device() && gate->stride(2) == 1 &&
                     (gate->stride(0) | gate->stride(1)) % 4 == 0 && aligned(at_of(*gate), 8);
  const float scale = (float)PyFloat_AS_DOUBLE(a[3]);
  const int rc = released([&] {
    void* scratch = need ? ws.mutable_data_ptr() : nullptr;
    const size_t bytes = need ? ws.nbytes() : 0;
    if (gated) {
      out = fresh({B, 16, hq * d}, *q);
      return dflash_sdpa_q16_gated(at_of(*q), at_of(*k), at_of(*v), nullptr, at_of(*gate), out.mutable_data_ptr(), scratch, bytes,
                                   (int)B, (int)hq, (int)hk, (int)N, (int)d, k->stride(0), k->stride(1), k->stride(2),
                                   v->stride(0), v->stride(1), v->stride(2), gate->stride(0), gate->stride(1), scale, code, stream);
    }
    out = fresh({B, hq, 16, d}, *q);
    return dflash_sdpa_q16(at_of(*q), at_of(*k), at_of(*v), nullptr, out.mutable_data_ptr(), scratch, bytes, (int)B, (int)hq,
                           (int)hk, (int)N, (int)d, k->stride(0), k->stride(1), k->stride(2), v->stride(0), v->stride(1),
                           v->stride(2), scale, code, stream);
  });
  return rc != 0 ? fail(rc, gated ? "dflash_sdpa_q16_gated" : "dflash_sdpa_q16") : THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// first_rows(keys, values, rows): a cache's buffers [B, H, capacity, D] up to a row.
PyObject* first_rows(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 3) Py_RETURN_NONE;
  const Tensor *k = device_tensor(a[0]), *v = device_tensor(a[1]);
  int rows;
  if (!k || !v || !integer(a[2], &rows) || k->dim() != 4 || v->dim() != 4 || rows > k->size(2) || rows > v->size(2)) Py_RETURN_NONE;
  return Py_BuildValue("(NN)", THPVariable_Wrap(k->narrow(2, 0, rows)), THPVariable_Wrap(v->narrow(2, 0, rows)));
  END_HANDLE_TH_ERRORS
}

// attn_block(q_proj_output, keys, values, q_weight, k_weight, cache_keys, cache_values, rope_dims, q_eps, k_eps, base, scale, workspaces):
// a block of 16 tokens from its projections to its gated attention; cache_keys and cache_values [B, Hk, N, D] hold the block's rows
// last, which are written here.
PyObject* attn_block(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 13) Py_RETURN_NONE;
  const Tensor* t[7];
  for (int i = 0; i < 7; ++i)
    if (!(t[i] = device_tensor(a[i]))) Py_RETURN_NONE;
  const Tensor &q = *t[0], &k = *t[1], &v = *t[2], &qw = *t[3], &kw = *t[4], &ck = *t[5], &cv = *t[6];
  int rope;
  if (!integer(a[7], &rope) || q.dim() != 3 || ck.dim() != 4) Py_RETURN_NONE;
  for (int i = 8; i < 12; ++i)
    if (!PyFloat_CheckExact(a[i])) Py_RETURN_NONE;
  const int64_t B = q.size(0), Hk = ck.size(1), N = ck.size(2), D = ck.size(3);
  const int code = half_code(q.scalar_type());
  if (code == kNoCode || B < 1 || Hk < 1 || (D != 128 && D != 256) || N <= 16 || N >= (1 << 30) || q.size(1) != 16 ||
      q.size(2) % (2 * D) != 0 || (rope != 64 && rope != 128 && (rope != 256 || D != 256)))
    Py_RETURN_NONE;
  const int64_t Hq = q.size(2) / (2 * D);
  if (Hq < 1 || Hq % Hk != 0 || Hq / Hk > 8 || B * Hq >= (1 << 26) || !has_shape(k, {B, 16, Hk * D}) || !has_shape(v, {B, 16, Hk * D}) ||
      !has_shape(qw, {D}) || !has_shape(kw, {D}) || !qw.is_contiguous() || !kw.is_contiguous() || !has_shape(ck, {B, Hk, N, D}) ||
      !has_shape(cv, {B, Hk, N, D}))
    Py_RETURN_NONE;
  for (const Tensor* x : t)
    if (x->scalar_type() != q.scalar_type() || x->device() != q.device() || !aligned(at_of(*x), 16)) Py_RETURN_NONE;
  for (const Tensor* x : {&q, &k, &v})
    if (x->stride(2) != 1 || (x->stride(0) | x->stride(1)) % 8 != 0) Py_RETURN_NONE;
  for (const Tensor* x : {&ck, &cv})
    if (x->stride(3) != 1 || (x->stride(0) | x->stride(1) | x->stride(2)) % 8 != 0 || x->stride(2) < D) Py_RETURN_NONE;
  const size_t need = dflash_attn_block_workspace_bytes((int)B, (int)Hq, (int)Hk, (int)N, (int)D);
  if (need == 0) Py_RETURN_NONE;
  void* stream = stream_of(q);
  Tensor out, ws = kept_workspace(a[12], Py_BuildValue("(NK)", THPDevice_New(q.device()), (unsigned long long)(uintptr_t)stream), need);
  if (!ws.defined()) Py_RETURN_NONE;
  dflash_attn_block_args p = {};
  p.q = at_of(q), p.k = at_of(k), p.v = at_of(v), p.q_weight = at_of(qw), p.k_weight = at_of(kw);
  p.k_cache = ck.mutable_data_ptr(), p.v_cache = cv.mutable_data_ptr(), p.workspace = ws.mutable_data_ptr(), p.workspace_bytes = ws.nbytes();
  p.q_batch = q.stride(0), p.q_row = q.stride(1), p.k_batch = k.stride(0), p.k_row = k.stride(1);
  p.v_batch = v.stride(0), p.v_row = v.stride(1);
  p.k_cache_batch = ck.stride(0), p.k_cache_head = ck.stride(1), p.k_cache_row = ck.stride(2);
  p.v_cache_batch = cv.stride(0), p.v_cache_head = cv.stride(1), p.v_cache_row = cv.stride(2);
  p.B = (int)B, p.Hq = (int)Hq, p.Hk = (int)Hk, p.N = (int)N, p.D = (int)D, p.rope_dims = rope, p.dtype = code;
  p.q_eps = (float)PyFloat_AS_DOUBLE(a[8]), p.k_eps = (float)PyFloat_AS_DOUBLE(a[9]);
  p.rope_base = (float)PyFloat_AS_DOUBLE(a[10]), p.scale = (float)PyFloat_AS_DOUBLE(a[11]);
  const int rc = released([&] {
    out = fresh({B, 16, Hq * D}, q);
    p.out = out.mutable_data_ptr();
    return dflash_attn_block(&p, stream);
  });
  return rc != 0 ? fail(rc, "dflash_attn_block") : THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// ---- module -----------------------------------------------------------------------------------------------------------
PyObject* bind(PyObject*, PyObject* error) {  // the class that failed launches raise
  Py_INCREF(error);
  Py_XDECREF(g_error);
  g_error = error;
  Py_RETURN_NONE;
}

#define DFLASH_HOST(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {DFLASH_HOST(qmm_m16), DFLASH_HOST(qmm_packed), DFLASH_HOST(qmm_few), DFLASH_HOST(qmm_few_silu_mul),
                          DFLASH_HOST(qmm_rows), DFLASH_HOST(columns), DFLASH_HOST(gather), DFLASH_HOST(chain_bind), DFLASH_HOST(chain_launch), DFLASH_HOST(gdn_prepare), DFLASH_HOST(gdn_forward), DFLASH_HOST(gdn_block), DFLASH_HOST(gdn_block_of),
                          DFLASH_HOST(rollback_layer), DFLASH_HOST(rollback_layers), DFLASH_HOST(attn_prepare), DFLASH_HOST(sdpa_q16), DFLASH_HOST(first_rows), DFLASH_HOST(attn_block), {"bind", bind, METH_O, nullptr},
                          {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_dflash_host", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__dflash_host() { return PyModule_Create(&kModule); }
