// The package's call path from torch tensors to the kernels, as one CPython extension (daisy_amd/_native.so).
//
// A decode step of one sequence, or a prompt of a few hundred tokens, keeps the GPU busy for 20 to 60 us per layer;
// walking the same step through Python wrappers, ctypes and tensor views took the host 55 to 120 us.  The functions
// here take the tensors as they are, check shapes, types and strides in C++, allocate the outputs and launch.  Each
// returns None for anything out of the ordinary (other dtypes, layouts, devices, autograd, a kernel that refused its
// arguments): the Python function in front of it then runs its own path, which serves the case or raises.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/GradMode.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <array>
#include <cmath>

#include "internal.h"

namespace {

using at::Tensor;
using daisy::GateSource;

// ---- arguments ----------------------------------------------------------------------------------------------------
const Tensor* opt_tensor(PyObject* o) { return o == Py_None ? nullptr : &THPVariable_Unpack(o); }
bool is_tensor(PyObject* o) { return THPVariable_Check(o); }
bool tensor_or_none(PyObject* o) { return o == Py_None || THPVariable_Check(o); }

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

PyObject* none() { Py_RETURN_NONE; }
PyObject* wrap(const Tensor& t) { return THPVariable_Wrap(t); }

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
  if (n != 5 || !is_tensor(a[0]) || !is_tensor(a[1]) || !tensor_or_none(a[2])) return none();
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
  Tensor y = empty(sizes, at::kBFloat16, x);
  const uint16_t* wp = (const uint16_t*)ptr(w);
  const hipStream_t s = stream_of(dev);
  const bool ok = tile ? daisy::proj_linear(r.p, r.stride, wp, w.stride(0), (const uint16_t*)ptr(bias), (uint16_t*)ptr(y), N, r.M, N, r.K, s, tile) == DAISY_OK
                       : own_linear(r, wp, w.stride(0), N, (const uint16_t*)ptr(bias), (uint16_t*)ptr(y), N, max_rows, s);
  return ok ? wrap(y) : none();
  END_HANDLE_TH_ERRORS
}

// ---- attention ----------------------------------------------------------------------------------------------------
// prefill_attention(q, k, v, window, scale, cos, sin, doc_start, out, k_out) -> (out, k_out)
PyObject* py_prefill_attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 10) return none();
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
  Tensor o = out ? *out : empty(q.sizes(), at::kBFloat16, q), kr;
  if (ko) kr = *ko;
  else if (cos) kr = empty(q.sizes(), at::kBFloat16, q);
  const Strides3 qs(q), ks(k), vs(v), os(o), kos = kr.defined() ? Strides3(kr) : Strides3();
  const int rc = daisy_prefill_fwd(ptr(q), qs.s, ptr(k), ks.s, ptr(v), vs.s, (const float*)ptr(cos), (const float*)ptr(sin),
                                   (const int32_t*)ptr(doc), ptr(o), os.s, kr.defined() ? ptr(kr) : nullptr, kos.s,
                                   (int)B, (int)T, (int)H, (int)D, window, scale, 0, stream_of(dev));
  if (rc != DAISY_OK) return none();
  PyObject* r = PyTuple_New(2);
  PyTuple_SET_ITEM(r, 0, wrap(o));
  PyTuple_SET_ITEM(r, 1, kr.defined() ? wrap(kr) : none());
  return r;
  END_HANDLE_TH_ERRORS
}

// layer_prefill(x, qkvo_w, cos, sin, H, D, window, doc_start, ve, g_ve, k_out, v_out, scale, eps, max_rows, want_q)
//   -> (y [B, T, dim], q or None, k, v [B, T, H, D])
// CausalSelfAttention.prefill on bf16 weights: QKV projection, norm + RoPE + value mix, attention, output projection.
PyObject* py_layer_prefill(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 16) return none();
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
  if (doc && !int32_vector(*doc, T, dev)) return none();
  if ((ve == nullptr) != (g_ve == nullptr) || (k_out == nullptr) != (v_out == nullptr)) return none();
  if (needs_autograd({&x, &w, ve, g_ve})) return none();
  GateSource gate{nullptr, 0};
  if (ve && !(gate_source(*g_ve, dev, gate) && on_gpu(*ve, dev) && bf16(*ve) && ve->is_contiguous() && ve->numel() == B * T * dim)) return none();
  for (const Tensor* t : {k_out, v_out})
    if (t && (!rows_bf16(*t, 4, dev) || t->size(0) != B || t->size(1) != T || t->size(2) != H || t->size(3) != D)) return none();

  const hipStream_t s = stream_of(dev);
  const uint16_t* wp = (const uint16_t*)ptr(w);
  const std::array<int64_t, 4> shape{B, T, H, D};
  const int64_t full[3] = {T * dim, dim, D};
  Tensor k = k_out ? *k_out : empty(shape, at::kBFloat16, x), v = v_out ? *v_out : empty(shape, at::kBFloat16, x);
  const Strides3 ks(k), vs(v);
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
  PyObject* res = PyTuple_New(4);
  PyTuple_SET_ITEM(res, 0, wrap(y));
  PyTuple_SET_ITEM(res, 1, want_q ? wrap(q) : none());
  PyTuple_SET_ITEM(res, 2, wrap(k));
  PyTuple_SET_ITEM(res, 3, wrap(v));
  return res;
  END_HANDLE_TH_ERRORS
}

// layer_step(x, qkvo_w, k_ring, v_ring, pos, cos, sin, ve, g_ve, status, scale, eps, max_rows)
//   -> (y [B, 1, dim], k_new, v_new [B, 1, H, D])   (k_new, v_new None with the position in device memory)
// CausalSelfAttention.step on a ring: QKV projection, the one-launch attention step, output projection.
PyObject* py_layer_step(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 13) return none();
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
  Tensor o = empty({B, 1, dim}, at::kBFloat16, x), k_new, v_new;
  if (f16 && !pos_dev) {
    k_new = empty({B, 1, H, D}, at::kBFloat16, x);
    v_new = empty({B, 1, H, D}, at::kBFloat16, x);
  }
  const int live = pos_dev ? (int)W : (int)std::min<int64_t>((int64_t)pos + 1, W);
  const size_t need = daisy_decode_workspace_bytes((int)B, (int)H, (int)D, live, 0);
  Tensor ws;
  if (need) ws = empty({(int64_t)need}, at::kByte, x);
  const uint16_t* base = (const uint16_t*)ptr(qkv);
  const int64_t rs[2] = {3 * dim, D}, os[2] = {dim, D};
  const Strides3 krs(kr), vrs(vr);
  const daisy::StepPrep prep{pos, (const float*)ptr(cos), (const float*)ptr(sin), (int)cos.size(0), eps, ptr(ve), os, gate, f16,
                             (int32_t*)ptr(status), k_new.defined() ? (uint16_t*)ptr(k_new) : nullptr,
                             v_new.defined() ? (uint16_t*)ptr(v_new) : nullptr};
  if (daisy::attn_step_launch(base, rs, base + dim, rs, base + 2 * dim, rs, ptr(kr), krs.s, ptr(vr), vrs.s, ptr(o), os, (int)B, (int)H,
                              (int)D, (int)W, pos_dev ? (const int32_t*)ptr(*pos_dev) : nullptr, scale, 0, need ? ptr(ws) : nullptr, need, s,
                              prep) != DAISY_OK) return none();
  const Rows orow{(const uint16_t*)ptr(o), dim, (int)B, (int)dim};
  const uint16_t* wo = wp + 3 * dim * dim;
  Tensor y;
  if (max_rows > 0 && (B <= max_rows || daisy::proj_wanted((int)B, (int)dim, (int)dim))) {
    y = empty({B, 1, dim}, at::kBFloat16, x);
    if (!own_linear(orow, wo, dim, (int)dim, nullptr, (uint16_t*)ptr(y), dim, max_rows, s)) return none();
  } else {
    y = at::linear(o, w.select(0, 3));
  }
  PyObject* res = PyTuple_New(3);
  PyTuple_SET_ITEM(res, 0, wrap(y));
  if (pos_dev) {
    PyTuple_SET_ITEM(res, 1, none());
    PyTuple_SET_ITEM(res, 2, none());
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
  if (n != 11) return none();
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
  Tensor o = empty({B, T, H, Dv}, at::kBFloat16, q), st;
  if (n_seq) o.zero_();      // rows that belong to no sequence are not written by the kernels
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
  PyObject* r = PyTuple_New(2);
  PyTuple_SET_ITEM(r, 0, wrap(o));
  PyTuple_SET_ITEM(r, 1, want_state ? wrap(st) : none());
  return r;
  END_HANDLE_TH_ERRORS
}

#define FAST(name) {#name, (PyCFunction)(void (*)(void))py_##name, METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {FAST(linear), FAST(prefill_attention), FAST(layer_prefill), FAST(layer_step), FAST(kda_chunk),
                          {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) { return PyModule_Create(&kModule); }
