// The package's call path from torch tensors to the kernels, as one CPython extension (daisy_amd/_native.so).
//
// A decode step of one sequence, or a prompt of a few hundred tokens, keeps the GPU busy for 20 to 60 us per layer;
// walking the same step through Python wrappers, ctypes and tensor views took the host 55 to 120 us.  The functions
// here take the tensors as they are, check shapes, types and strides in C++, allocate the outputs and launch.  Each
// returns None for anything out of the ordinary (other dtypes, layouts, devices, autograd, a kernel that refused its
// arguments): the Python function in front of it then runs its own path, which serves the case or raises.  What has been
// written by then it writes again, the same values to the same places; only the KDA layer's states would not bear that.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/autocast_mode.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <algorithm>
#include <array>
#include <cmath>

#include "internal.h"

namespace {

using at::Tensor;
using daisy::GateSource;

// ---- arguments ----------------------------------------------------------------------------------------------------
// A tensor whose operations nothing intercepts: no Python subclass, and none of the dispatch keys of vmap, function
// transforms, fake or lazily conjugated or negated tensors, no tangent of forward-mode differentiation.
bool is_tensor(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return false;
  constexpr c10::DispatchKeySet plain = c10::DispatchKeySet({c10::DispatchKey::CUDA, c10::DispatchKey::AutogradCUDA, c10::DispatchKey::AutocastCUDA,
                                                             c10::DispatchKey::ADInplaceOrView});
  const Tensor& t = THPVariable_Unpack(o);
  return t.defined() && (t.key_set().raw_repr() & ~plain.raw_repr()) == 0 && !t._fw_grad(0).defined();
}
bool tensor_or_none(PyObject* o) { return o == Py_None || is_tensor(o); }
const Tensor* opt_tensor(PyObject* o) { return o == Py_None ? nullptr : &THPVariable_Unpack(o); }
// Whether someone watches or redirects the calls of this thread: those have to reach the library's operators one by one.
bool intercepted() {
  return c10::impl::TorchDispatchModeTLS::any_modes_set() || at::impl::torch_function_mode_enabled() || torch::jit::tracer::isTracing() ||
         at::autocast::is_autocast_enabled(at::kCUDA);
}

// The current device when the tensor lives there, else -1 (asked of CPU tensors' processes too, which may have no device).
int gpu_of(const Tensor& t) {
  if (!t.is_cuda()) return -1;
  const int dev = c10::hip::current_device();
  return t.device().index() == dev ? dev : -1;
}
bool on_gpu(const Tensor& t, int dev) { return t.is_cuda() && t.device().index() == dev; }
bool bf16(const Tensor& t) { return t.scalar_type() == at::kBFloat16; }
bool f32(const Tensor& t) { return t.scalar_type() == at::kFloat; }
// bf16, `dims` dimensions, the last one contiguous
bool rows_bf16(const Tensor& t, int64_t dims, int dev) {
  return on_gpu(t, dev) && bf16(t) && t.dim() == dims && (t.size(-1) == 1 || t.stride(-1) == 1);
}
bool rotary_table(const Tensor& t, int64_t rows, int64_t half, int dev) {
  return on_gpu(t, dev) && f32(t) && t.dim() == 2 && t.size(1) == half && t.size(0) >= rows && t.is_contiguous();
}
bool int32_vector(const Tensor& t, int64_t n, int dev) {
  return on_gpu(t, dev) && t.scalar_type() == at::kInt && t.numel() == n && t.is_contiguous();
}
bool needs_autograd(std::initializer_list<const Tensor*> ts) {
  if (!c10::GradMode::is_enabled()) return false;
  for (const Tensor* t : ts)
    if (t && t->requires_grad()) return true;
  return false;
}

struct Strides3 {
  int64_t s[3];
  Strides3() : s{0, 0, 0} {}
  explicit Strides3(const Tensor& t) : s{t.stride(0), t.stride(1), t.stride(2)} {}
};
struct Strides2 {
  int64_t s[2];
  Strides2() : s{0, 0} {}
  explicit Strides2(const Tensor& t) : s{t.stride(0), t.stride(1)} {}
};

Tensor empty(at::IntArrayRef sizes, at::ScalarType type, const Tensor& like) {
  return Tensor(at::detail::empty_cuda(sizes, type, like.device(), std::nullopt));
}
void* ptr(const Tensor& t) { return t.data_ptr(); }
void* ptr(const Tensor* t) { return t ? t->data_ptr() : nullptr; }
hipStream_t stream_of(int dev) { return c10::hip::getCurrentHIPStream(dev).stream(); }

// "Not here": borrowed, also without the interpreter lock (the method table's wrapper adds the reference).
PyObject* none() { return Py_None; }
PyObject* new_none() { Py_RETURN_NONE; }

// The interpreter lock is given up while memory is allocated and kernels are launched, as the library's operators do.
class Unlocked {
 public:
  Unlocked() : state_(PyEval_SaveThread()) {}
  ~Unlocked() { end(); }
  void end() {
    if (state_) PyEval_RestoreThread(state_);
    state_ = nullptr;
  }

 private:
  PyThreadState* state_;
};

PyObject* wrap(const Tensor& t) { return THPVariable_Wrap(t); }

// For a kernel behind which a call cannot be given back to the Python function in front of it.
void must(int rc) { TORCH_CHECK(rc == DAISY_OK, "daisy_amd: a kernel refused its arguments (code ", rc, "): ", daisy_last_error()); }

// The gate logit of a layer with value embeddings; false when it is not a lone fp32 or bf16 number on the GPU.
bool gate_source(const Tensor& g, int dev, GateSource& out) {
  if (!on_gpu(g, dev) || g.numel() != 1 || !(f32(g) || bf16(g))) return false;
  out = GateSource{g.data_ptr(), f32(g) ? GateSource::kLogitF32 : GateSource::kLogitBf16};
  return true;
}

// ---- projections --------------------------------------------------------------------------------------------------
// Activations [..., K] as M rows at one stride.
struct Rows { const uint16_t* p; int64_t stride; int M, K; };
bool as_rows(const Tensor& x, int dev, Rows& r) {
  if (!on_gpu(x, dev) || !bf16(x) || x.dim() < 1 || x.numel() == 0) return false;
  const int64_t K = x.size(-1), M = x.numel() / K;
  if (M > (1 << 30) || K > (1 << 22)) return false;
  int64_t stride = K;
  if (!x.is_contiguous()) {
    if (x.stride(-1) != 1 || x.dim() < 2) return false;
    stride = x.stride(-2);
    for (int64_t d = x.dim() - 3; d >= 0; --d)
      if (x.size(d) != 1 && x.stride(d) != x.stride(d + 1) * x.size(d + 1)) return false;
  }
  r = Rows{(const uint16_t*)x.data_ptr(), stride, (int)M, (int)K};
  return stride % 8 == 0 && (reinterpret_cast<uintptr_t>(r.p) & 15) == 0;
}

// y = x w^T for one of this library's kernels: up to max_rows rows through the weight-streaming kernel, larger
// products through the tiled one where the sizes favour it.  False: the library GEMM is the better choice.
bool own_linear(const Rows& x, const uint16_t* w, int64_t w_sn, int N, const uint16_t* bias, uint16_t* y, int64_t y_sm,
                int max_rows, hipStream_t s) {
  if (max_rows <= 0) return false;
  if (x.M <= max_rows && !bias) return daisy_linear_rows_fwd(x.p, x.stride, w, w_sn, y, y_sm, x.M, N, x.K, s) == DAISY_OK;
  if (!daisy::proj_wanted(x.M, N, x.K)) return false;
  return daisy::proj_linear(x.p, x.stride, w, w_sn, bias, y, y_sm, x.M, N, x.K, s) == DAISY_OK;
}

// linear(x, w, bias, max_rows, tile): x w^T (+ bias) through an own kernel, or None.  tile != 0 forces the tiled kernel
// with that tile (tests and sweeps).
PyObject* py_linear(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (intercepted() || n != 5 || !is_tensor(a[0]) || !is_tensor(a[1]) || !tensor_or_none(a[2])) return none();
  const Tensor &x = THPVariable_Unpack(a[0]), &w = THPVariable_Unpack(a[1]);
  const Tensor* bias = opt_tensor(a[2]);
  const int max_rows = (int)PyLong_AsLong(a[3]), tile = (int)PyLong_AsLong(a[4]);
  const int dev = gpu_of(x);
  if (dev < 0) return none();
  Rows r;
  if (!as_rows(x, dev, r) || !rows_bf16(w, 2, dev) || w.size(1) != r.K || needs_autograd({&x, &w, bias})) return none();
  if (w.stride(0) % 8 != 0 || w.stride(0) < r.K || (reinterpret_cast<uintptr_t>(ptr(w)) & 15) != 0) return none();
  if (bias && (!on_gpu(*bias, dev) || !bf16(*bias) || bias->numel() != w.size(0) || !bias->is_contiguous())) return none();
  const int N = (int)w.size(0);
  if (!tile && !(r.M <= max_rows && !bias) && !(max_rows > 0 && daisy::proj_wanted(r.M, N, r.K))) return none();
  c10::SmallVector<int64_t, 5> sizes(x.sizes().begin(), x.sizes().end());
  sizes.back() = N;
  Unlocked unlocked;
  Tensor y = empty(sizes, at::kBFloat16, x);
  const uint16_t* wp = (const uint16_t*)ptr(w);
  const hipStream_t s = stream_of(dev);
  const bool ok = tile ? daisy::proj_linear(r.p, r.stride, wp, w.stride(0), (const uint16_t*)ptr(bias), (uint16_t*)ptr(y), N, r.M, N, r.K, s, tile) == DAISY_OK
                       : own_linear(r, wp, w.stride(0), N, (const uint16_t*)ptr(bias), (uint16_t*)ptr(y), N, max_rows, s);
  unlocked.end();
  return ok ? wrap(y) : none();
  END_HANDLE_TH_ERRORS
}

// norm(x, eps): the weightless RMS norm over the last dim of contiguous bf16 rows, one token per sequence ([.., 1, C]), or None.
PyObject* py_norm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 2 || intercepted() || !is_tensor(a[0])) return none();
  const Tensor& x = THPVariable_Unpack(a[0]);
  const float eps = (float)PyFloat_AsDouble(a[1]);
  if (PyErr_Occurred()) { PyErr_Clear(); return none(); }
  const int dev = gpu_of(x);
  if (dev < 0 || !bf16(x) || x.dim() < 2 || x.size(-2) != 1 || !x.is_contiguous() || x.numel() == 0 || needs_autograd({&x})) return none();
  const int64_t C = x.size(-1), rows = x.numel() / C;
  if (!daisy::rms_rows_serves(rows, C) || (reinterpret_cast<uintptr_t>(x.data_ptr()) & 15) != 0) return none();
  Unlocked unlocked;
  Tensor y = empty(x.sizes(), at::kBFloat16, x);
  const bool ok = daisy::rms_rows((const uint16_t*)ptr(x), (uint16_t*)ptr(y), (int)rows, (int)C, eps, stream_of(dev)) == DAISY_OK;
  unlocked.end();
  return ok ? wrap(y) : none();
  END_HANDLE_TH_ERRORS
}

// linears(x, weights, biases, max_rows, tile): the products of x with several matrices in one launch, as a tuple of views of one
// tensor, or None.  Arguments as for linear; weights and biases: tuples (a bias may be None).
PyObject* py_linears(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (intercepted() || n != 5 || !is_tensor(a[0]) || !PyTuple_Check(a[1]) || !PyTuple_Check(a[2])) return none();
  const Py_ssize_t count = PyTuple_GET_SIZE(a[1]);
  if (count < 1 || count > daisy::kMaxSegments || PyTuple_GET_SIZE(a[2]) != count) return none();
  const Tensor& x = THPVariable_Unpack(a[0]);
  const int max_rows = (int)PyLong_AsLong(a[3]), tile = (int)PyLong_AsLong(a[4]);
  const int dev = gpu_of(x);
  Rows r;
  if (dev < 0 || !as_rows(x, dev, r)) return none();
  daisy::ProjSegment seg[daisy::kMaxSegments];
  int64_t pitch = 0;
  for (Py_ssize_t i = 0; i < count; ++i) {
    PyObject *wo = PyTuple_GET_ITEM(a[1], i), *bo = PyTuple_GET_ITEM(a[2], i);
    if (!is_tensor(wo) || !tensor_or_none(bo)) return none();
    const Tensor& w = THPVariable_Unpack(wo);
    const Tensor* bias = opt_tensor(bo);
    if (!rows_bf16(w, 2, dev) || w.size(1) != r.K || w.stride(0) < r.K || needs_autograd({&x, &w, bias})) return none();
    if (bias && (!on_gpu(*bias, dev) || !bf16(*bias) || bias->numel() != w.size(0) || !bias->is_contiguous())) return none();
    seg[i] = daisy::ProjSegment{r.p, r.stride, (const uint16_t*)ptr(w), w.stride(0), (const uint16_t*)ptr(bias), nullptr, 0, (int)w.size(0), 0};
    pitch += (w.size(0) + 7) / 8 * 8;
  }
  if (!tile && (max_rows <= 0 || (r.M > max_rows && !daisy::proj_segments_wanted(r.M, (int)pitch, r.K)))) return none();
  Unlocked unlocked;
  Tensor y = empty({(int64_t)r.M, pitch}, at::kBFloat16, x);
  int64_t at = 0;
  for (Py_ssize_t i = 0; i < count; ++i) {
    seg[i].y = (uint16_t*)ptr(y) + at;
    seg[i].y_sm = pitch;
    at += (seg[i].N + 7) / 8 * 8;
  }
  const hipStream_t s = stream_of(dev);
  const int rc = r.M <= max_rows && !tile ? daisy::linear_segments(seg, (int)count, r.M, r.K, s) : daisy::proj_segments(seg, (int)count, r.M, r.K, s, tile);
  if (rc != DAISY_OK) return none();
  unlocked.end();
  PyObject* res = PyTuple_New(count);
  c10::SmallVector<int64_t, 5> sizes(x.sizes().begin(), x.sizes().end()), strides(x.dim(), 1);
  at = 0;
  for (Py_ssize_t i = 0; i < count; ++i) {
    sizes.back() = seg[i].N;
    for (int64_t d = x.dim() - 2, step = pitch; d >= 0; step *= sizes[d--]) strides[d] = step;
    PyTuple_SET_ITEM(res, i, wrap(y.as_strided(sizes, strides, at)));
    at += (seg[i].N + 7) / 8 * 8;
  }
  return res;
  END_HANDLE_TH_ERRORS
}

// ---- attention ----------------------------------------------------------------------------------------------------
// prefill_attention(q, k, v, window, scale, cos, sin, doc_start, out, k_out) -> (out, k_out)
PyObject* py_prefill_attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (intercepted() || n != 10) return none();
  for (int i : {0, 1, 2})
    if (!is_tensor(a[i])) return none();
  for (int i : {5, 6, 7, 8, 9})
    if (!tensor_or_none(a[i])) return none();
  const Tensor &q = THPVariable_Unpack(a[0]), &k = THPVariable_Unpack(a[1]), &v = THPVariable_Unpack(a[2]);
  const int window = (int)PyLong_AsLong(a[3]);
  const float scale = (float)PyFloat_AsDouble(a[4]);
  if (PyErr_Occurred()) { PyErr_Clear(); return none(); }
  const Tensor *cos = opt_tensor(a[5]), *sin = opt_tensor(a[6]), *doc = opt_tensor(a[7]), *out = opt_tensor(a[8]), *ko = opt_tensor(a[9]);
  const int dev = gpu_of(q);
  if (dev < 0) return none();
  for (const Tensor* t : {&q, &k, &v})
    if (!rows_bf16(*t, 4, dev) || t->sizes() != q.sizes()) return none();
  const int64_t B = q.size(0), T = q.size(1), H = q.size(2), D = q.size(3);
  if ((cos == nullptr) != (sin == nullptr) || (ko && !cos)) return none();
  if (cos && (!rotary_table(*cos, T, D / 2, dev) || !rotary_table(*sin, T, D / 2, dev))) return none();
  if (doc && !(int32_vector(*doc, T, dev) && doc->dim() == 1)) return none();
  for (const Tensor* t : {out, ko})
    if (t && (!rows_bf16(*t, 4, dev) || t->sizes() != q.sizes())) return none();
  Unlocked unlocked;
  Tensor o = out ? *out : empty(q.sizes(), at::kBFloat16, q), kr;
  if (ko) kr = *ko;
  else if (cos) kr = empty(q.sizes(), at::kBFloat16, q);
  const Strides3 qs(q), ks(k), vs(v), os(o), kos = kr.defined() ? Strides3(kr) : Strides3();
  const int rc = daisy_prefill_fwd(ptr(q), qs.s, ptr(k), ks.s, ptr(v), vs.s, (const float*)ptr(cos), (const float*)ptr(sin),
                                   (const int32_t*)ptr(doc), ptr(o), os.s, kr.defined() ? ptr(kr) : nullptr, kos.s,
                                   (int)B, (int)T, (int)H, (int)D, window, scale, 0, stream_of(dev));
  if (rc != DAISY_OK) return none();
  unlocked.end();
  PyObject* r = PyTuple_New(2);
  PyTuple_SET_ITEM(r, 0, wrap(o));
  PyTuple_SET_ITEM(r, 1, kr.defined() ? wrap(kr) : new_none());
  return r;
  END_HANDLE_TH_ERRORS
}

// layer_prefill(x, qkvo_w, cos, sin, H, D, window, doc_start, ve, g_ve, k_out, v_out, scale, eps, max_rows, want_q)
//   -> (y [B, T, dim], q [B, T, H, D] or None, k, v [B, H, T, D])   (rows of a token side by side in memory all the same)
// CausalSelfAttention.prefill on bf16 weights: QKV projection, norm + RoPE + value mix, attention, output projection.
PyObject* py_layer_prefill(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (intercepted() || n != 16) return none();
  for (int i : {0, 1, 2, 3})
    if (!is_tensor(a[i])) return none();
  for (int i : {7, 8, 9, 10, 11})
    if (!tensor_or_none(a[i])) return none();
  const Tensor &x = THPVariable_Unpack(a[0]), &w = THPVariable_Unpack(a[1]), &cos = THPVariable_Unpack(a[2]), &sin = THPVariable_Unpack(a[3]);
  const int H = (int)PyLong_AsLong(a[4]), D = (int)PyLong_AsLong(a[5]), window = (int)PyLong_AsLong(a[6]);
  const Tensor *doc = opt_tensor(a[7]), *ve = opt_tensor(a[8]), *g_ve = opt_tensor(a[9]), *k_out = opt_tensor(a[10]), *v_out = opt_tensor(a[11]);
  const float scale = (float)PyFloat_AsDouble(a[12]), eps = (float)PyFloat_AsDouble(a[13]);
  const int max_rows = (int)PyLong_AsLong(a[14]);
  const bool want_q = a[15] == Py_True;
  if (PyErr_Occurred()) { PyErr_Clear(); return none(); }
  const int dev = gpu_of(x);
  if (dev < 0) return none();
  const int dim = H * D;
  Rows r;
  if (x.dim() != 3 || !as_rows(x, dev, r) || r.K != dim) return none();
  if (!rows_bf16(w, 3, dev) || !w.is_contiguous() || w.size(0) != 4 || w.size(1) != dim || w.size(2) != dim) return none();
  const int64_t B = x.size(0), T = x.size(1);
  if (!rotary_table(cos, T, D / 2, dev) || !rotary_table(sin, T, D / 2, dev)) return none();
  if (doc && !(int32_vector(*doc, T, dev) && doc->dim() == 1)) return none();
  if ((ve == nullptr) != (g_ve == nullptr) || (k_out == nullptr) != (v_out == nullptr)) return none();
  if (needs_autograd({&x, &w, ve, g_ve})) return none();
  GateSource gate{nullptr, 0};
  if (ve && !(gate_source(*g_ve, dev, gate) && on_gpu(*ve, dev) && bf16(*ve) && ve->is_contiguous() && ve->numel() == B * T * dim)) return none();
  for (const Tensor* t : {k_out, v_out})
    if (t && (!rows_bf16(*t, 4, dev) || t->size(0) != B || t->size(1) != T || t->size(2) != H || t->size(3) != D)) return none();

  Unlocked unlocked;
  const hipStream_t s = stream_of(dev);
  const uint16_t* wp = (const uint16_t*)ptr(w);
  const std::array<int64_t, 4> shape{B, T, H, D};
  const int64_t full[3] = {T * dim, dim, D};
  // (made as the caller gets them: two views from Python cost the host a sixth of a small layer's call)
  const std::array<int64_t, 4> by_head{B, H, T, D}, by_head_strides{T * dim, D, dim, 1};
  auto rows = [&] { return Tensor(at::detail::empty_strided_cuda(by_head, by_head_strides, at::kBFloat16, x.device())); };
  Tensor k = k_out ? *k_out : rows(), v = v_out ? *v_out : rows();
  Strides3 ks, vs;
  for (int i = 0; i < 3; ++i) {
    ks.s[i] = k_out ? k_out->stride(i) : full[i];
    vs.s[i] = v_out ? v_out->stride(i) : full[i];
  }
  Tensor q = empty(shape, at::kBFloat16, x);
  if (max_rows > 0 && r.M > max_rows && daisy::proj_qkv_wanted(r.M, 3 * dim, dim)) {
    daisy::QkvEpilogue e{(uint16_t*)ptr(q), full[0], full[1], full[2], (uint16_t*)ptr(k), ks.s[0], ks.s[1], ks.s[2],
                         (uint16_t*)ptr(v), vs.s[0], vs.s[1], vs.s[2], (const uint16_t*)ptr(ve), full[0], full[1], full[2],
                         gate, (const float*)ptr(cos), (const float*)ptr(sin), 0, H, (int)T, eps};
    if (daisy::proj_qkv(r.p, r.stride, wp, dim, e, (int)B, dim, D, s) != DAISY_OK) return none();
  } else {
    Tensor qkv;
    if (max_rows > 0 && r.M <= max_rows) {
      qkv = empty({B, T, 3 * (int64_t)dim}, at::kBFloat16, x);
      if (daisy_linear_rows_fwd(r.p, r.stride, wp, dim, ptr(qkv), 3 * dim, r.M, 3 * dim, dim, s) != DAISY_OK) return none();
    } else {
      qkv = at::linear(x, w.narrow(0, 0, 3).view({3 * (int64_t)dim, dim}));
    }
    const uint16_t* base = (const uint16_t*)ptr(qkv);
    const int64_t in[3] = {T * 3 * dim, 3 * (int64_t)dim, D};
    if (daisy::prep_launch(base, in, base + dim, in, base + 2 * dim, in, ptr(ve), full, gate, (const float*)ptr(cos),
                           (const float*)ptr(sin), 0, nullptr, 0, nullptr, ptr(q), full, ptr(k), ks.s, ptr(v), vs.s,
                           (int)B, (int)T, H, D, eps, s) != DAISY_OK) return none();
  }
  // A workgroup reads its query rows before it writes its output rows, and no other workgroup touches either: the
  // output may take the queries' place when the caller does not want them.
  Tensor o = want_q ? empty(shape, at::kBFloat16, x) : q;
  if (daisy_prefill_fwd(ptr(q), full, ptr(k), ks.s, ptr(v), vs.s, nullptr, nullptr, (const int32_t*)ptr(doc), ptr(o), full,
                        nullptr, nullptr, (int)B, (int)T, H, D, window, scale, 0, s) != DAISY_OK) return none();
  const Rows orow{(const uint16_t*)ptr(o), dim, r.M, dim};
  const uint16_t* wo = wp + 3 * (int64_t)dim * dim;
  Tensor y;
  if (max_rows > 0 && r.M > max_rows && daisy::proj_wanted(r.M, dim, dim)) {
    y = empty(x.sizes(), at::kBFloat16, x);
    if (daisy::proj_linear(orow.p, dim, wo, dim, nullptr, (uint16_t*)ptr(y), dim, r.M, dim, dim, s) != DAISY_OK) return none();
  } else {
    y = at::linear(o.view({B, T, (int64_t)dim}), w.select(0, 3));
  }
  unlocked.end();
  PyObject* res = PyTuple_New(4);
  PyTuple_SET_ITEM(res, 0, wrap(y));
  PyTuple_SET_ITEM(res, 1, want_q ? wrap(q) : new_none());
  PyTuple_SET_ITEM(res, 2, wrap(k_out ? k.transpose(1, 2) : k));
  PyTuple_SET_ITEM(res, 3, wrap(v_out ? v.transpose(1, 2) : v));
  return res;
  END_HANDLE_TH_ERRORS
}

// layer_step(x, qkvo_w, k_ring, v_ring, pos, cos, sin, ve, g_ve, status, scale, eps, max_rows)
//   -> (y [B, 1, dim], k_new, v_new [B, 1, H, D])   (k_new, v_new None with the position in device memory)
// CausalSelfAttention.step on a ring: QKV projection, the one-launch attention step, output projection.
PyObject* py_layer_step(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (intercepted() || n != 13) return none();
  for (int i : {0, 1, 2, 3, 5, 6})
    if (!is_tensor(a[i])) return none();
  for (int i : {7, 8, 9})
    if (!tensor_or_none(a[i])) return none();
  const Tensor &x = THPVariable_Unpack(a[0]), &w = THPVariable_Unpack(a[1]), &kr = THPVariable_Unpack(a[2]), &vr = THPVariable_Unpack(a[3]);
  const Tensor* pos_dev = is_tensor(a[4]) ? &THPVariable_Unpack(a[4]) : nullptr;
  const int pos = pos_dev ? 0 : (int)PyLong_AsLong(a[4]);
  const Tensor &cos = THPVariable_Unpack(a[5]), &sin = THPVariable_Unpack(a[6]);
  const Tensor *ve = opt_tensor(a[7]), *g_ve = opt_tensor(a[8]), *status = opt_tensor(a[9]);
  const float scale = (float)PyFloat_AsDouble(a[10]), eps = (float)PyFloat_AsDouble(a[11]);
  const int max_rows = (int)PyLong_AsLong(a[12]);
  if (PyErr_Occurred()) { PyErr_Clear(); return none(); }
  const int dev = gpu_of(x);
  if (dev < 0) return none();
  const bool f16 = kr.scalar_type() == at::kHalf;
  for (const Tensor* t : {&kr, &vr})
    if (!on_gpu(*t, dev) || t->dim() != 4 || t->stride(3) != 1 || t->sizes() != kr.sizes() || t->scalar_type() != kr.scalar_type() || !(f16 || bf16(*t)))
      return none();
  const int64_t B = kr.size(0), H = kr.size(1), W = kr.size(2), D = kr.size(3), dim = H * D;
  Rows r;
  if (x.dim() != 3 || !as_rows(x, dev, r) || r.K != dim || r.M != B || x.size(0) != B) return none();
  if (!rows_bf16(w, 3, dev) || !w.is_contiguous() || w.size(0) != 4 || w.size(1) != dim || w.size(2) != dim) return none();
  if (!rotary_table(cos, 1, D / 2, dev) || !rotary_table(sin, cos.size(0), D / 2, dev)) return none();
  if (pos_dev ? !int32_vector(*pos_dev, 1, dev) : (pos < 0 || pos >= cos.size(0))) return none();
  if (status && !int32_vector(*status, 1, dev)) return none();
  if ((ve == nullptr) != (g_ve == nullptr) || needs_autograd({&x, &w, ve, g_ve})) return none();
  GateSource gate{nullptr, 0};
  if (ve && !(gate_source(*g_ve, dev, gate) && on_gpu(*ve, dev) && bf16(*ve) && ve->is_contiguous() && ve->numel() == B * dim)) return none();

  Unlocked unlocked;
  const hipStream_t s = stream_of(dev);
  const uint16_t* wp = (const uint16_t*)ptr(w);
  Tensor qkv;
  // projection rows and, beside them, the attention's output
  const bool own_qkv = max_rows > 0 && (B <= max_rows || daisy::proj_wanted((int)B, (int)(3 * dim), (int)dim));
  if (own_qkv) {
    qkv = empty({B, 3 * dim}, at::kBFloat16, x);
    if (!own_linear(r, wp, dim, (int)(3 * dim), nullptr, (uint16_t*)ptr(qkv), 3 * dim, max_rows, s)) return none();
  } else {
    qkv = at::linear(x, w.narrow(0, 0, 3).view({3 * dim, dim}));
  }
  Tensor o, y, k_new, v_new;
  if (f16 && !pos_dev) {
    k_new = empty({B, 1, H, D}, at::kBFloat16, x);
    v_new = empty({B, 1, H, D}, at::kBFloat16, x);
  }
  const int live = pos_dev ? (int)W : (int)std::min<int64_t>((int64_t)pos + 1, W);
  const size_t need = daisy_decode_workspace_bytes((int)B, (int)H, (int)D, live, 0);
  Tensor ws;
  if (need) ws = empty({(int64_t)need}, at::kByte, x);
  const uint16_t* base = (const uint16_t*)ptr(qkv);
  const uint16_t* wo = wp + 3 * dim * dim;
  // one sequence with a split ring: the output projection combines the splits itself, and no attention row is written
  const bool projects = max_rows > 0 && daisy::step_projects((int)B, (int)H, (int)D, live);
  if (projects) y = empty({B, 1, dim}, at::kBFloat16, x);
  else o = empty({B, 1, dim}, at::kBFloat16, x);
  const int64_t rs[2] = {3 * dim, D}, os[2] = {dim, D};
  const Strides3 krs(kr), vrs(vr);
  const daisy::StepPrep prep{pos, (const float*)ptr(cos), (const float*)ptr(sin), (int)cos.size(0), eps, ptr(ve), os, gate, f16,
                             (int32_t*)ptr(status), k_new.defined() ? (uint16_t*)ptr(k_new) : nullptr,
                             v_new.defined() ? (uint16_t*)ptr(v_new) : nullptr,
                             projects ? daisy::StepProjection{wo, dim, (uint16_t*)ptr(y), (int)dim} : daisy::StepProjection{nullptr, 0, nullptr, 0}};
  if (daisy::attn_step_launch(base, rs, base + dim, rs, base + 2 * dim, rs, ptr(kr), krs.s, ptr(vr), vrs.s, projects ? ptr(qkv) : ptr(o), os, (int)B, (int)H,
                              (int)D, (int)W, pos_dev ? (const int32_t*)ptr(*pos_dev) : nullptr, scale, 0, need ? ptr(ws) : nullptr, need, s,
                              prep) != DAISY_OK) return none();
  if (!projects) {
    const Rows orow{(const uint16_t*)ptr(o), dim, (int)B, (int)dim};
    if (max_rows > 0 && (B <= max_rows || daisy::proj_wanted((int)B, (int)dim, (int)dim))) {
      y = empty({B, 1, dim}, at::kBFloat16, x);
      if (!own_linear(orow, wo, dim, (int)dim, nullptr, (uint16_t*)ptr(y), dim, max_rows, s)) return none();
    } else {
      y = at::linear(o, w.select(0, 3));
    }
  }
  unlocked.end();
  PyObject* res = PyTuple_New(3);
  PyTuple_SET_ITEM(res, 0, wrap(y));
  if (pos_dev) {
    PyTuple_SET_ITEM(res, 1, new_none());
    PyTuple_SET_ITEM(res, 2, new_none());
  } else {
    if (!f16) {
      const int64_t slot = pos % W;
      auto row = [&](const Tensor& t) {
        return t.as_strided({B, 1, H, D}, {t.stride(0), t.stride(1), t.stride(1), 1}, t.storage_offset() + slot * t.stride(2));
      };
      k_new = row(kr);
      v_new = row(vr);
    }
    PyTuple_SET_ITEM(res, 1, wrap(k_new));
    PyTuple_SET_ITEM(res, 2, wrap(v_new));
  }
  return res;
  END_HANDLE_TH_ERRORS
}

// ---- KDA ------------------------------------------------------------------------------------------------------------
// kda_chunk(q, k, v, g, beta, scale, initial_state, want_state, l2norm, l2_eps, cu_seqlens) -> (o, state or None)
PyObject* py_kda_chunk(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (intercepted() || n != 11) return none();
  for (int i : {0, 1, 2, 3, 4})
    if (!is_tensor(a[i])) return none();
  if (!tensor_or_none(a[6]) || !tensor_or_none(a[10])) return none();
  const Tensor &q = THPVariable_Unpack(a[0]), &k = THPVariable_Unpack(a[1]), &v = THPVariable_Unpack(a[2]), &g = THPVariable_Unpack(a[3]),
               &beta = THPVariable_Unpack(a[4]);
  const Tensor *s0 = opt_tensor(a[6]), *cu = opt_tensor(a[10]);
  const bool want_state = a[7] == Py_True, l2norm = a[8] == Py_True;
  const int dev = gpu_of(q);
  if (dev < 0) return none();
  for (const Tensor* t : {&q, &k, &v})
    if (!rows_bf16(*t, 4, dev) || !t->is_contiguous()) return none();
  if (!on_gpu(g, dev) || !(f32(g) || bf16(g)) || !g.is_contiguous() || !on_gpu(beta, dev) || !f32(beta) || !beta.is_contiguous()) return none();
  const int64_t B = q.size(0), T = q.size(1), H = q.size(2), Dk = q.size(3), Dv = v.size(3);
  if (k.sizes() != q.sizes() || g.sizes() != q.sizes() || v.size(0) != B || v.size(1) != T || v.size(2) != H) return none();
  if (beta.dim() != 3 || beta.size(0) != B || beta.size(1) != T || beta.size(2) != H) return none();
  const float scale = a[5] == Py_None ? (float)(1.0 / std::sqrt((double)Dk)) : (float)PyFloat_AsDouble(a[5]);
  const float l2_eps = (float)PyFloat_AsDouble(a[9]);
  if (PyErr_Occurred()) { PyErr_Clear(); return none(); }
  int64_t n_seq = 0;
  if (cu) {
    if (B != 1 || cu->dim() != 1 || cu->numel() < 2 || !int32_vector(*cu, cu->numel(), dev)) return none();
    n_seq = cu->numel() - 1;
  }
  const int64_t states = n_seq ? n_seq : B;
  if (s0 && !(on_gpu(*s0, dev) && f32(*s0) && s0->is_contiguous() && s0->dim() == 4 && s0->size(0) == states && s0->size(1) == H &&
              s0->size(2) == Dk && s0->size(3) == Dv)) return none();
  const size_t need = n_seq ? daisy_kda_varlen_workspace_bytes((int)T, (int)n_seq, (int)H, (int)Dk, (int)Dv, 64)
                            : daisy_kda_workspace_bytes((int)B, (int)T, (int)H, (int)Dk, (int)Dv, 64);
  if (need == 0) return none();
  Unlocked unlocked;
  Tensor o = empty({B, T, H, Dv}, at::kBFloat16, q), st;
  if (want_state) st = empty({states, H, Dk, Dv}, at::kFloat, q);
  Tensor ws = empty({(int64_t)need}, at::kByte, q);
  const hipStream_t s = stream_of(dev);
  const int rc = n_seq ? daisy_kda_chunk_varlen_fwd(ptr(q), ptr(k), ptr(v), ptr(g), bf16(g), (const float*)ptr(beta), (const int32_t*)ptr(*cu),
                                                    (int)n_seq, (const float*)ptr(s0), ptr(o), want_state ? (float*)ptr(st) : nullptr, (int)T,
                                                    (int)H, (int)Dk, (int)Dv, 64, scale, l2norm, l2_eps, ptr(ws), need, s)
                       : daisy_kda_chunk_fwd(ptr(q), ptr(k), ptr(v), ptr(g), bf16(g), (const float*)ptr(beta), (const float*)ptr(s0), ptr(o),
                                             want_state ? (float*)ptr(st) : nullptr, (int)B, (int)T, (int)H, (int)Dk, (int)Dv, 64, scale,
                                             l2norm, l2_eps, ptr(ws), need, s);
  if (rc != DAISY_OK) return none();
  unlocked.end();
  PyObject* r = PyTuple_New(2);
  PyTuple_SET_ITEM(r, 0, wrap(o));
  PyTuple_SET_ITEM(r, 1, want_state ? wrap(st) : new_none());
  return r;
  END_HANDLE_TH_ERRORS
}

// kda_layer(x, weights, H, Dk, Dv, taps, state, windows, homes, keep, norm_eps, max_rows) -> (y, state, wq, wk, wv)
// KimiLinearSelfAttention on bf16 weights without value embeddings or padding.  weights: tuple of q, k, v, f0, g0, b, f1, g1
// projections, g1's bias, output projection, the three convolutions' weights and biases, A_log, dt_bias, norm weight.
// state / windows (tuple of three): what the layer carries, or None.  keep: return the states after the last token; homes: tuple of
// four tensors (state, windows) to store them in where they fit, or None each.  One token with carried states updates them in place.
PyObject* py_kda_layer(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  constexpr int kWeights = 19;
  if (intercepted() || n != 12 || !is_tensor(a[0]) || !PyTuple_Check(a[1]) || PyTuple_GET_SIZE(a[1]) != kWeights || !tensor_or_none(a[6])) return none();
  if (!PyTuple_Check(a[7]) || PyTuple_GET_SIZE(a[7]) != 3 || !PyTuple_Check(a[8]) || PyTuple_GET_SIZE(a[8]) != 4) return none();
  const Tensor* w[kWeights];
  for (int i = 0; i < kWeights; ++i) {
    PyObject* o = PyTuple_GET_ITEM(a[1], i);
    const bool optional = i == 8 || i == 13 || i == 14 || i == 15;
    if (!(is_tensor(o) || (optional && o == Py_None))) return none();
    w[i] = opt_tensor(o);
  }
  const Tensor* win[3]; const Tensor* home[4];
  for (int i = 0; i < 3; ++i) {
    PyObject* o = PyTuple_GET_ITEM(a[7], i);
    if (!tensor_or_none(o)) return none();
    win[i] = opt_tensor(o);
  }
  for (int i = 0; i < 4; ++i) {
    PyObject* o = PyTuple_GET_ITEM(a[8], i);
    if (!tensor_or_none(o)) return none();
    home[i] = opt_tensor(o);
  }
  const Tensor& x = THPVariable_Unpack(a[0]);
  const Tensor* state = opt_tensor(a[6]);
  const int64_t H = PyLong_AsLong(a[2]), Dk = PyLong_AsLong(a[3]), Dv = PyLong_AsLong(a[4]), taps = PyLong_AsLong(a[5]);
  const bool keep = a[9] == Py_True;
  const float norm_eps = (float)PyFloat_AsDouble(a[10]);
  const int max_rows = (int)PyLong_AsLong(a[11]);
  if (PyErr_Occurred()) { PyErr_Clear(); return none(); }
  const int dev = gpu_of(x);
  if (dev < 0 || max_rows <= 0 || taps < 2 || taps > 4) return none();
  Rows r;
  if (x.dim() != 3 || !as_rows(x, dev, r)) return none();
  const int64_t B = x.size(0), T = x.size(1), dim = r.K, M = r.M, kd = H * Dk, vd = H * Dv;
  if (c10::GradMode::is_enabled()) {
    if (x.requires_grad()) return none();
    for (const Tensor* t : w)
      if (t && t->requires_grad()) return none();
  }
  auto matrix = [&](const Tensor* t, int64_t rows, int64_t cols) {
    return rows_bf16(*t, 2, dev) && t->is_contiguous() && t->size(0) == rows && t->size(1) == cols && (reinterpret_cast<uintptr_t>(t->data_ptr()) & 15) == 0;
  };
  auto vector = [&](const Tensor* t, int64_t len, at::ScalarType type) {
    return on_gpu(*t, dev) && t->scalar_type() == type && t->numel() == len && t->is_contiguous();
  };
  const int64_t widths[6] = {kd, kd, vd, Dv, Dv, H};
  for (int i = 0; i < 6; ++i)
    if (!matrix(w[i], widths[i], dim)) return none();
  if (!matrix(w[6], kd, Dv) || !matrix(w[7], vd, Dv) || (w[8] && !vector(w[8], vd, at::kBFloat16)) || !matrix(w[9], dim, vd)) return none();
  for (int i = 0; i < 3; ++i) {
    if (!vector(w[10 + i], widths[i] * taps, at::kBFloat16) || (w[13 + i] && !vector(w[13 + i], widths[i], at::kBFloat16))) return none();
    if (win[i] && !(vector(win[i], B * widths[i] * taps, at::kBFloat16) && win[i]->dim() == 3 && win[i]->size(0) == B && win[i]->size(1) == widths[i])) return none();
  }
  if (!vector(w[16], H, at::kFloat) || !vector(w[17], kd, at::kFloat) || !vector(w[18], Dv, at::kBFloat16) ||
      (reinterpret_cast<uintptr_t>(ptr(w[18])) & 15) != 0) return none();
  if (state && !(vector(state, B * kd * Dv, at::kFloat) && state->dim() == 4 && state->size(0) == B && state->size(1) == H && state->size(2) == Dk)) return none();
  const bool step = keep && T == 1 && state;
  const size_t need = step ? 0 : daisy_kda_workspace_bytes((int)B, (int)T, (int)H, (int)Dk, (int)Dv, 64);
  if (step ? !(win[0] && win[1] && win[2] && daisy::kda_layer_step_serves((int)Dk, (int)Dv, (int)taps)) : (need == 0 || dim % 64 != 0 || Dv % 64 != 0 || !daisy::gated_rmsnorm_serves((int)Dv)))
    return none();

  // ---- the projections of the input ---------------------------------------------------------------------------------
  Unlocked unlocked;
  const hipStream_t s = stream_of(dev);
  const uint16_t* W[kWeights];
  for (int i = 0; i < kWeights; ++i) W[i] = (const uint16_t*)ptr(w[i]);
  const int64_t pitch = (2 * kd + vd + 2 * Dv + H + 7) / 8 * 8, small = (2 * Dv + H + 7) / 8 * 8;
  const bool rows_kernel = M <= max_rows, together = rows_kernel || daisy::proj_layer_wanted((int)M, (int)pitch, (int)dim);
  Tensor proj, big[3];
  daisy::ProjSegment seg[6];
  proj = empty({M, together ? pitch : small}, at::kBFloat16, x);
  {
    uint16_t* y = (uint16_t*)ptr(proj);
    for (int i = 0; i < 6; ++i) {
      seg[i] = daisy::ProjSegment{r.p, r.stride, W[i], dim, nullptr, y, together ? pitch : small, (int)widths[i], 0};
      if (together || i >= 3) y += widths[i];
    }
  }
  if (rows_kernel) {
    if (daisy::linear_segments(seg, 6, (int)M, (int)dim, s) != DAISY_OK) return none();
  } else if (together) {
    if (daisy::proj_segments(seg, 6, (int)M, (int)dim, s) != DAISY_OK) return none();
  } else {
    for (int i = 0; i < 3; ++i) {
      if (daisy::proj_wanted((int)M, (int)widths[i], (int)dim)) {
        big[i] = empty({B, T, widths[i]}, at::kBFloat16, x);
        if (!own_linear(r, W[i], dim, (int)widths[i], nullptr, (uint16_t*)ptr(big[i]), widths[i], max_rows, s)) return none();
      } else {
        big[i] = at::linear(x, *w[i]);
      }
      seg[i].y = (uint16_t*)ptr(big[i]);
      seg[i].y_sm = widths[i];
    }
    if (daisy::proj_segments(seg + 3, 3, (int)M, (int)dim, s) != DAISY_OK) return none();
  }

  // ---- one token: everything up to the output projection in one launch; a prompt: the convolutions --------------------
  const float scale = (float)(1.0 / std::sqrt((double)Dk));
  constexpr float kL2Eps = 1e-6f;
  Tensor o, conv[3], new_win[3];
  // Where a state is kept: in its home when that has the shape, else in a new tensor.
  auto keeper = [&](const Tensor* h, at::IntArrayRef shape, at::ScalarType type) {
    return h && on_gpu(*h, dev) && h->scalar_type() == type && h->is_contiguous() && h->sizes() == shape ? *h : empty(shape, type, x);
  };
  if (step) {
    o = empty({B, 1, vd}, at::kBFloat16, x);
    daisy::KdaLayerStep p{seg[0].y, seg[1].y, seg[2].y, seg[3].y, seg[4].y, seg[5].y, seg[0].y_sm, seg[1].y_sm, seg[2].y_sm, seg[3].y_sm,
                          seg[4].y_sm, seg[5].y_sm, {W[10], W[11], W[12]}, {W[13], W[14], W[15]}, {}, (int)taps, W[6], W[7], W[8],
                          (const float*)ptr(w[16]), (const float*)ptr(w[17]), W[18], (float*)ptr(state), (uint16_t*)ptr(o), vd,
                          (int)H, (int)Dk, scale, kL2Eps, norm_eps};
    for (int i = 0; i < 3; ++i) p.window[i] = (uint16_t*)ptr(win[i]);
    if (daisy::kda_layer_step(p, (int)B, (int)Dv, s) != DAISY_OK) return none();
  } else {
    daisy::ConvPart parts[3];
    for (int i = 0; i < 3; ++i) {
      conv[i] = empty({B, T, widths[i]}, at::kBFloat16, x);
      const std::array<int64_t, 3> shape{B, widths[i], taps};
      // (a window is updated in place for short inputs only)
      if (keep) new_win[i] = win[i] && home[i + 1] && win[i]->data_ptr() == home[i + 1]->data_ptr() && T > 32 ? empty(shape, at::kBFloat16, x)
                                                                                                           : keeper(home[i + 1], shape, at::kBFloat16);
      parts[i] = daisy::ConvPart{seg[i].y, T * seg[i].y_sm, seg[i].y_sm, W[10 + i], W[13 + i], (const uint16_t*)ptr(win[i]), (uint16_t*)ptr(conv[i]),
                                 T * widths[i], widths[i], keep ? (uint16_t*)ptr(new_win[i]) : nullptr, (int)widths[i]};
    }
    if (daisy::short_conv_group(parts, 3, (int)B, (int)T, (int)taps, 1, s) != DAISY_OK) return none();
    for (Tensor& t : big) t = Tensor();
  }

  // ---- the rest.  The state of a step, the windows of a prompt may have changed in place by now: there is no way back to the
  // ---- caller's own path, which would apply the tokens a second time, so a refusal raises (and cannot be returned from here)
  auto rest = [&]() -> std::array<Tensor, 2> {
    Tensor st, y;
    if (!step) {
      // the low-rank products: with the decay gate and beta ahead of the delta rule, with the gated norm behind it
      const bool own_low = daisy::low_rank_wanted((int)M, (int)kd, (int)Dv) && (!w[8] || (reinterpret_cast<uintptr_t>(W[8]) & 15) == 0);
      Tensor g = empty({M, kd}, at::kBFloat16, x), gate, beta = empty({M, H}, at::kFloat, x);
      if (!own_low) gate = empty({M, vd}, at::kBFloat16, x);
      const daisy::ProjSegment low[2] = {{seg[3].y, seg[3].y_sm, W[6], Dv, nullptr, (uint16_t*)ptr(g), kd, (int)kd, 0},
                                         {seg[4].y, seg[4].y_sm, W[7], Dv, W[8], own_low ? nullptr : (uint16_t*)ptr(gate), vd, (int)vd, 0}};
      const daisy::KdaGates gates{(const float*)ptr(w[16]), (const float*)ptr(w[17]), (int)H, (int)Dk, seg[5].y, seg[5].y_sm, (float*)ptr(beta)};
      must(own_low ? daisy::low_rank_gate(seg[3].y, seg[3].y_sm, W[6], gates, (uint16_t*)ptr(g), (int)M, (int)kd, (int)Dv, s)
                   : daisy::proj_segments(low, 2, (int)M, (int)Dv, s, 0, &gates));
      o = empty({B, T, vd}, at::kBFloat16, x);
      if (keep) st = keeper(home[0], {B, H, Dk, Dv}, at::kFloat);
      Tensor ws = empty({(int64_t)need}, at::kByte, x);
      must(daisy_kda_chunk_fwd(ptr(conv[0]), ptr(conv[1]), ptr(conv[2]), ptr(g), 1, (const float*)ptr(beta), (const float*)ptr(state), ptr(o),
                               keep ? (float*)ptr(st) : nullptr, (int)B, (int)T, (int)H, (int)Dk, (int)Dv, 64, scale, 1, kL2Eps, ptr(ws), need, s));
      must(own_low ? daisy::low_rank_norm(seg[4].y, seg[4].y_sm, W[7], W[8], W[18], (uint16_t*)ptr(o), norm_eps, (int)M, (int)vd, (int)Dv, s)
                   : daisy_gated_rmsnorm_fwd(ptr(o), ptr(gate), W[18], ptr(o), M * H, (int)Dv, norm_eps, s));
    }
    if (M <= max_rows || daisy::proj_wanted((int)M, (int)dim, (int)vd)) {
      y = empty({B, T, dim}, at::kBFloat16, x);
      must(own_linear(Rows{(const uint16_t*)ptr(o), vd, (int)M, (int)vd}, W[9], vd, (int)dim, nullptr, (uint16_t*)ptr(y), dim, max_rows, s)
               ? DAISY_OK : DAISY_ERR_UNSUPPORTED);
    } else {
      y = at::linear(o, *w[9]);
    }
    return {y, st};
  };
  const auto [y, st] = rest();
  unlocked.end();
  PyObject* res = PyTuple_New(5);
  PyTuple_SET_ITEM(res, 0, wrap(y));
  PyTuple_SET_ITEM(res, 1, !keep ? new_none() : wrap(step ? *state : st));
  for (int i = 0; i < 3; ++i) PyTuple_SET_ITEM(res, 2 + i, !keep ? new_none() : wrap(step ? *win[i] : new_win[i]));
  return res;
  END_HANDLE_TH_ERRORS
}

template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t)>
PyObject* call(PyObject* self, PyObject* const* a, Py_ssize_t n) {
  PyObject* r = F(self, a, n);
  if (r == Py_None) Py_INCREF(r);
  return r;
}
#define FAST(name) {#name, (PyCFunction)(void (*)(void))call<py_##name>, METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {FAST(linear), FAST(norm), FAST(linears), FAST(prefill_attention), FAST(layer_prefill), FAST(layer_step), FAST(kda_chunk), FAST(kda_layer),
                          {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) { return PyModule_Create(&kModule); }
