// The host side of the hot entry points in native code: argument checks, strides, the launch.
//
// An eager decode step at batch 1 spends its time on the host: ops.attn_decode_append took 27 us
// of Python (25 stride reads, 45 ctypes conversions, stream and workspace look-ups) around two
// kernels of 15 us. Each function here takes exactly the calls whose arguments need no conversion
// (tensors of the package's layouts and types on one device, outside graph capture) and returns
// None for every other one, which then goes the Python way, with its conversions and its errors;
// an int is the status of a launch that was rejected or failed. Nothing is kept between calls.
#include <Python.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/torch.h>

#include "../../include/forge_attn.h"

namespace {

using at::Tensor;

// A tensor as plain memory on a GPU: no subclass, functorch wrapper, fake tensor or forward-mode dual.
bool plain(const Tensor& t) {
  return t.defined() && t.is_cuda() && t.layout() == at::kStrided && !t.unsafeGetTensorImpl()->is_python_dispatch() &&
         t.has_storage() && !t.is_conj() && !t.is_neg() && !t._fw_grad(0).defined() &&
         !t.key_set().has_any(c10::DispatchKeySet({c10::DispatchKey::FuncTorchBatched,
                                                   c10::DispatchKey::FuncTorchGradWrapper,
                                                   c10::DispatchKey::Functionalize, c10::DispatchKey::Python}));
}

// The tensor behind a Python argument (a Parameter counts as one); false for anything that is no
// plain GPU tensor.
bool take(PyObject* o, Tensor& t) {
  if (!THPVariable_CheckExact(o)) return false;
  t = THPVariable_Unpack(o);
  return plain(t);
}

// The same where None is allowed (t stays undefined).
bool take_opt(PyObject* o, Tensor& t) { return o == Py_None || take(o, t); }

const void* ptr(const Tensor& t) { return t.defined() ? t.const_data_ptr() : nullptr; }

int dtype_of(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return FORGE_F32;
    case at::kBFloat16: return FORGE_BF16;
    case at::kHalf: return FORGE_F16;
    default: return -1;
  }
}

// fp32 norm gain of D values
bool gain_ok(const Tensor& w, int64_t D, c10::Device dev) {
  return !w.defined() ||
         (w.scalar_type() == at::kFloat && w.is_contiguous() && w.numel() == D && w.device() == dev);
}

struct Rope {
  const float* cos = nullptr;
  const float* sin = nullptr;
  int64_t sb = 0, st = 0;
};

// fp32 tables [T, D] or [1 or B, T, D] with equal strides
bool rope_ok(const Tensor& c, const Tensor& s, int64_t B, int64_t T, int64_t D, c10::Device dev, Rope& r) {
  if (!c.defined() && !s.defined()) return true;
  if (!c.defined() || !s.defined()) return false;
  const int64_t d = c.dim();
  if ((d != 2 && d != 3) || c.sizes() != s.sizes() || c.strides() != s.strides() || c.size(d - 1) != D ||
      c.size(d - 2) != T || c.stride(d - 1) != 1 || c.scalar_type() != at::kFloat || s.scalar_type() != at::kFloat ||
      c.device() != dev || s.device() != dev)
    return false;
  if (d == 3 && c.size(0) != 1 && c.size(0) != B) return false;
  r.cos = static_cast<const float*>(ptr(c));
  r.sin = static_cast<const float*>(ptr(s));
  r.sb = d == 3 && c.size(0) == B && B > 1 ? c.stride(0) : 0;
  r.st = c.stride(d - 2);
  return true;
}

bool as_int(PyObject* o, int64_t& v) {
  if (!PyLong_CheckExact(o)) return false;
  v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

bool as_float(PyObject* o, float& v) {
  if (!PyFloat_CheckExact(o)) return false;
  v = (float)PyFloat_AS_DOUBLE(o);
  return true;
}

bool capturing() {
  return c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None;
}

// Gives the GIL up for its scope (no Python object is touched there): an allocation may have to free
// and synchronise, and a launch waits while the stream's queue is full.
struct NoGil {
  PyThreadState* state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
};

// The buffer of (device, stream) from the caller's workspace table (ops._STREAM_WS: cleared buffers,
// the most recently used last), taken out of the table while a call uses it, so that no other thread
// launches on it in between, and put back once the call is launched.
struct StreamWorkspace {
  PyObject *table, *key = nullptr, *buf = nullptr;
  void* ptr = nullptr;
  size_t bytes = 0;

  StreamWorkspace(PyObject* table, int dev, hipStream_t stream, size_t need) : table(table) {
    if (!need) return;
    key = Py_BuildValue("(iK)", dev, (unsigned long long)(uintptr_t)stream);
    PyObject* b = key ? PyDict_GetItemWithError(table, key) : nullptr;
    if (b && THPVariable_CheckExact(b) && (size_t)THPVariable_Unpack(b).numel() >= need) {
      Py_INCREF(b);
      if (PyDict_DelItem(table, key) == 0) buf = b;
      else Py_DECREF(b);
    }
    if (PyErr_Occurred()) PyErr_Clear();
    if (!buf) return;
    ptr = THPVariable_Unpack(buf).data_ptr();
    bytes = (size_t)THPVariable_Unpack(buf).numel();
  }
  void put_back() {
    if (buf && PyDict_SetItem(table, key, buf) != 0) PyErr_Clear();
  }
  ~StreamWorkspace() {
    Py_XDECREF(buf);
    Py_XDECREF(key);
  }
};

PyObject* result(int st, const Tensor& out) {
  if (st != 0) return PyLong_FromLong(st);
  return THPVariable_Wrap(out);
}

// decode_append(table, q, k, v, k_cache, v_cache, scale, pos | None, pos_dev | None, row_pos | None,
//               max_kv_len | None, window, q_weight | None, k_weight | None, eps, norm_q, norm_k, norm_v,
//               cos | None, sin | None, chunk)
PyObject* decode_append_impl(PyObject* const* a) {
  Tensor q, k, v, kc, vc, pos_dev, row_pos, qw, kw, cos, sin;
  if (!take(a[1], q) || !take(a[2], k) || !take(a[3], v) || !take(a[4], kc) || !take(a[5], vc) ||
      !take_opt(a[8], pos_dev) || !take_opt(a[9], row_pos) || !take_opt(a[12], qw) || !take_opt(a[13], kw) ||
      !take_opt(a[18], cos) || !take_opt(a[19], sin))
    return nullptr;
  float scale, eps;
  int64_t window, chunk, pos = 0, max_kv = -1;
  if (!as_float(a[6], scale) || !as_float(a[14], eps) || !as_int(a[11], window) || !as_int(a[20], chunk) ||
      (a[7] != Py_None && !as_int(a[7], pos)) || (a[10] != Py_None && !as_int(a[10], max_kv)))
    return nullptr;
  const bool norm_q = a[15] == Py_True, norm_k = a[16] == Py_True, norm_v = a[17] == Py_True;
  if (q.dim() != 4 || k.dim() != 4 || kc.dim() != 4 || k.sizes() != v.sizes() || kc.sizes() != vc.sizes() ||
      kc.strides() != vc.strides())
    return nullptr;
  const int64_t B = q.size(0), H = q.size(1), T = q.size(2), D = q.size(3), K = kc.size(1), max_len = kc.size(2);
  const int dt = dtype_of(q);
  const c10::Device dev = q.device();
  if (dt < 0 || K <= 0 || H % K || kc.size(0) != B || kc.size(3) != D || k.size(0) != B || k.size(1) != K ||
      k.size(2) != T || k.size(3) != D)
    return nullptr;
  for (const Tensor* t : {&k, &v, &kc, &vc})
    if (t->scalar_type() != q.scalar_type() || t->device() != dev || t->stride(3) != 1) return nullptr;
  if (q.stride(3) != 1) return nullptr;
  if (row_pos.defined()) {
    if (row_pos.scalar_type() != at::kInt || row_pos.numel() != B || row_pos.device() != dev || !row_pos.is_contiguous())
      return nullptr;
    pos_dev.reset();
    pos = 0;
  } else if (pos_dev.defined()) {
    if (pos_dev.scalar_type() != at::kLong || pos_dev.device() != dev) return nullptr;
    pos = 0;
  }
  Rope r;
  if (!rope_ok(cos, sin, B, T, D, dev, r) || !gain_ok(qw, D, dev) || !gain_ok(kw, D, dev)) return nullptr;
  if (pos < 0 || pos > max_len) return nullptr;
  if (max_kv < 0) max_kv = !row_pos.defined() && !pos_dev.defined() ? pos + T : max_len;
  max_kv = std::max<int64_t>(1, std::min(max_kv, max_len));
  if (window < 0 || window > INT_MAX || chunk > INT_MAX || c10::hip::current_device() != dev.index()) return nullptr;
  if (chunk <= 0) {
    const int64_t span = window > 0 && window + 16 < max_len ? window + 16 : max_len;  // ops.decode_chunk
    chunk = (row_pos.defined() ? forge_attn_decode_chunk : forge_attn_decode_chunk_uniform)(dt, (int)B, (int)T, (int)H,
                                                                                          (int)K, (int)D, span);
  }
  const hipStream_t stream = c10::hip::getCurrentHIPStream(dev.index()).stream();
  const size_t need = forge_attn_decode_workspace_bytes(dt, (int)B, (int)T, (int)H, (int)K, (int)D, max_kv, (int)chunk);
  if (need && capturing()) return nullptr;
  StreamWorkspace ws(a[0], dev.index(), stream, need);
  if (need && !ws.ptr) return nullptr;
  const int rope = r.cos ? FORGE_ROPE : 0;
  Tensor out;
  int st;
  {
    NoGil unlocked;
    out = at::empty({B, T, H, D}, q.options().requires_grad(false));
    st = forge_attn_decode_append(
        dt, (int)B, (int)T, (int)H, (int)K, (int)D, ptr(q), q.stride(0), q.stride(1), q.stride(2),
        norm_q ? static_cast<const float*>(ptr(qw)) : nullptr, eps, (norm_q ? FORGE_NORM_QK : 0) | rope, ptr(k),
        k.stride(0), k.stride(1), k.stride(2), ptr(v), v.stride(0), v.stride(1), v.stride(2),
        norm_k ? static_cast<const float*>(ptr(kw)) : nullptr,
        (norm_k ? FORGE_NORM_QK : 0) | rope | (norm_v ? FORGE_NORM_V : 0), r.cos, r.sin, r.sb, r.st, kc.data_ptr(),
        vc.data_ptr(), kc.stride(0), kc.stride(1), kc.stride(2), max_len, static_cast<const int32_t*>(ptr(row_pos)),
        static_cast<const int64_t*>(ptr(pos_dev)), pos, max_kv, (int)window, scale, (int)chunk, out.data_ptr(),
        out.stride(0), out.stride(1), out.stride(2), ws.ptr, ws.bytes, ws.ptr ? FORGE_WS_ZEROED : 0, stream);
  }
  if (st == 0) ws.put_back();
  return result(st, out);
}

// kv_append(k, v, k_cache, v_cache, pos, k_weight | None, eps, norm_k, norm_v, cos | None, sin | None): host position
PyObject* kv_append_impl(PyObject* const* a) {
  Tensor k, v, kc, vc, kw, cos, sin;
  if (!take(a[0], k) || !take(a[1], v) || !take(a[2], kc) || !take(a[3], vc) || !take_opt(a[5], kw) ||
      !take_opt(a[9], cos) || !take_opt(a[10], sin))
    return nullptr;
  float eps;
  int64_t pos;
  if (!as_int(a[4], pos) || !as_float(a[6], eps)) return nullptr;
  const bool norm_k = a[7] == Py_True, norm_v = a[8] == Py_True;
  if (k.dim() != 4 || kc.dim() != 4 || k.sizes() != v.sizes() || kc.sizes() != vc.sizes() ||
      kc.strides() != vc.strides())
    return nullptr;
  const int64_t B = k.size(0), K = k.size(1), T = k.size(2), D = k.size(3);
  const int dt = dtype_of(kc);
  const c10::Device dev = k.device();
  if (dt < 0 || kc.size(0) != B || kc.size(1) != K || kc.size(3) != D || c10::hip::current_device() != dev.index())
    return nullptr;
  for (const Tensor* t : {&k, &v, &kc, &vc})
    if (t->scalar_type() != k.scalar_type() || t->device() != dev || t->stride(3) != 1) return nullptr;
  Rope r;
  if (!rope_ok(cos, sin, B, T, D, dev, r) || !gain_ok(kw, D, dev)) return nullptr;
  const int flags = (norm_k ? FORGE_NORM_QK : 0) | (r.cos ? FORGE_ROPE : 0) | (norm_v ? FORGE_NORM_V : 0);
  int st;
  {
    NoGil unlocked;
    st = forge_kv_append(
        dt, (int)B, (int)T, (int)K, (int)D, ptr(k), k.stride(0), k.stride(1), k.stride(2), ptr(v), v.stride(0),
        v.stride(1), v.stride(2), kc.data_ptr(), vc.data_ptr(), kc.stride(0), kc.stride(1), kc.stride(2), kc.size(2),
        nullptr, nullptr, pos, norm_k ? static_cast<const float*>(ptr(kw)) : nullptr, eps, flags, r.cos, r.sin, r.sb,
        r.st, c10::hip::getCurrentHIPStream(dev.index()).stream());
  }
  return PyLong_FromLong(st);
}

// prefill(q, k, v, scale, offset, window, q_weight | None, eps, norm_q, cos | None, sin | None): bf16/fp16 through
// forge_attn_prefill_ws, fp32 through forge_attn_prefill_f32
PyObject* prefill_impl(PyObject* const* a) {
  Tensor q, k, v, qw, cos, sin;
  if (!take(a[0], q) || !take(a[1], k) || !take(a[2], v) || !take_opt(a[6], qw) || !take_opt(a[9], cos) ||
      !take_opt(a[10], sin))
    return nullptr;
  float scale, eps;
  int64_t offset, window;
  if (!as_float(a[3], scale) || !as_int(a[4], offset) || !as_int(a[5], window) || !as_float(a[7], eps)) return nullptr;
  const bool norm_q = a[8] == Py_True;
  if (q.dim() != 4 || k.dim() != 4 || k.sizes() != v.sizes() || k.strides() != v.strides()) return nullptr;
  const int64_t B = q.size(0), H = q.size(1), T = q.size(2), D = q.size(3), K = k.size(1);
  const int dt = dtype_of(q);
  const c10::Device dev = q.device();
  if (dt < 0 || K <= 0 || H % K || k.size(0) != B || k.size(3) != D || offset < 0 || k.size(2) - T < offset ||
      window < 0 || window > INT_MAX || q.stride(3) != 1 || c10::hip::current_device() != dev.index())
    return nullptr;
  for (const Tensor* t : {&k, &v})
    if (t->scalar_type() != q.scalar_type() || t->device() != dev || t->stride(3) != 1) return nullptr;
  Rope r;
  if ((cos.defined() && cos.dim() != 2) || !rope_ok(cos, sin, B, T, D, dev, r) || !gain_ok(qw, D, dev)) return nullptr;
  const bool f32 = dt == FORGE_F32;
  if (f32 ? D != 32 && D != 64 && D != 128 : D != 64 && D != 128 && D != 256 && D != 512) return nullptr;
  const int flags = (norm_q ? FORGE_NORM_QK : 0) | (r.cos ? FORGE_ROPE : 0);
  const float* w = norm_q ? static_cast<const float*>(ptr(qw)) : nullptr;
  const auto opts = q.options().requires_grad(false);
  Tensor out, ws;
  int st;
  {
    NoGil unlocked;
    out = at::empty({B, T, H, D}, opts);
    const size_t need =
        f32 ? forge_attn_prefill_f32_workspace_bytes((int)B, (int)T, (int)H, (int)K, (int)D, offset, (int)window)
            : forge_attn_prefill_workspace_bytes(dt, (int)B, (int)T, (int)H, (int)K, (int)D, offset, (int)window);
    if (need) {
      try {
        ws = at::empty({(int64_t)need}, opts.dtype(at::kByte));
      } catch (const c10::OutOfMemoryError&) {   // the launch is not split then
      }
    }
    void* wp = ws.defined() ? ws.data_ptr() : nullptr;
    const hipStream_t stream = c10::hip::getCurrentHIPStream(dev.index()).stream();
    st = f32 ? forge_attn_prefill_f32((int)B, (int)T, (int)H, (int)K, (int)D, ptr(q), q.stride(0), q.stride(1),
                                      q.stride(2), w, eps, flags, r.cos, r.sin, r.st, ptr(k), ptr(v), k.stride(0),
                                      k.stride(1), k.stride(2), offset, (int)window, scale, out.data_ptr(),
                                      out.stride(0), out.stride(1), out.stride(2), wp, need, stream)
             : forge_attn_prefill_ws(dt, (int)B, (int)T, (int)H, (int)K, (int)D, ptr(q), q.stride(0), q.stride(1),
                                     q.stride(2), w, eps, flags, r.cos, r.sin, r.st, ptr(k), ptr(v), k.stride(0),
                                     k.stride(1), k.stride(2), offset, (int)window, scale, nullptr, 0, out.data_ptr(),
                                     out.stride(0), out.stride(1), out.stride(2), wp, need, stream);
  }
  return result(st, out);
}

// linear_small(x, w, bias | None, w_up | None, gain | None, eps, norm, residual | None): contiguous x [..., K] of at
// most 16 rows, w and w_up [N, K], residual [..., N]
PyObject* linear_small_impl(PyObject* const* a) {
  Tensor x, w, b, up, gain, res;
  if (!take(a[0], x) || !take(a[1], w) || !take_opt(a[2], b) || !take_opt(a[3], up) || !take_opt(a[4], gain) ||
      !take_opt(a[7], res))
    return nullptr;
  float eps;
  if (!as_float(a[5], eps) || x.dim() < 1 || w.dim() != 2) return nullptr;
  const bool norm = a[6] == Py_True;
  const int64_t K = x.size(-1), N = w.size(0);
  const int dt = dtype_of(x);
  const c10::Device dev = x.device();
  if (K <= 0 || K % 32 || (dt != FORGE_BF16 && dt != FORGE_F16) || !x.is_contiguous() || x.numel() < K ||
      x.numel() > 16 * K || w.size(1) != K || !w.is_contiguous() || c10::hip::current_device() != dev.index())
    return nullptr;
  for (const Tensor* t : {&w, &b, &up, &res})
    if (t->defined() && (t->scalar_type() != x.scalar_type() || t->device() != dev || !t->is_contiguous())) return nullptr;
  if ((b.defined() && b.numel() != N) || (up.defined() && up.sizes() != w.sizes())) return nullptr;
  if (norm && !gain.defined()) return nullptr;
  if (gain.defined() && ((gain.scalar_type() != at::kFloat && gain.scalar_type() != x.scalar_type()) ||
                         gain.device() != dev || !gain.is_contiguous() || gain.numel() != K))
    return nullptr;
  const int64_t M = x.numel() / K;
  if (res.defined() && res.numel() != M * N) return nullptr;
  if (N > INT_MAX || K > INT_MAX || M > forge_linear_small_rows((int)N, (int)K, norm, up.defined(), res.defined()))
    return nullptr;   // torch's calls are faster there
  if (((uintptr_t)ptr(x) | (uintptr_t)ptr(w) | (uintptr_t)ptr(up) | (uintptr_t)ptr(gain)) % 16) return nullptr;
  auto shape = x.sizes().vec();
  shape.back() = N;
  Tensor out;
  int st;
  {
    NoGil unlocked;
    out = at::empty(shape, x.options().requires_grad(false));
    st = forge_linear_small(dt, (int)M, (int)N, (int)K, ptr(x), K, ptr(w), ptr(up), K, ptr(b), ptr(gain),
                            gain.defined() ? dtype_of(gain) : FORGE_F32, norm, eps, ptr(res), N, out.data_ptr(), N,
                            c10::hip::getCurrentHIPStream(dev.index()).stream());
  }
  return result(st, out);
}

// tensors_are(tensors, ids, state, w): whether the tuple of tensors is the recorded one, by id and by
// (data_ptr, version) each, of w's dtype and device (w: Attention's fused q/k/v weights)
PyObject* tensors_are_impl(PyObject* const* a) {
  if (!PyTuple_CheckExact(a[0]) || !PyTuple_CheckExact(a[1]) || !PyTuple_CheckExact(a[2])) return nullptr;
  Tensor w;
  if (!take(a[3], w)) return nullptr;
  const Py_ssize_t n = PyTuple_GET_SIZE(a[0]);
  if (PyTuple_GET_SIZE(a[1]) != n || PyTuple_GET_SIZE(a[2]) != n) Py_RETURN_FALSE;
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* o = PyTuple_GET_ITEM(a[0], i);
    PyObject* st = PyTuple_GET_ITEM(a[2], i);
    if (!THPVariable_Check(o) || !PyTuple_CheckExact(st) || PyTuple_GET_SIZE(st) < 2) return nullptr;
    const Tensor& t = THPVariable_Unpack(o);
    if (!plain(t) || t.is_inference()) return nullptr;
    if (t.scalar_type() != w.scalar_type() || t.device() != w.device()) Py_RETURN_FALSE;
    if (PyLong_AsVoidPtr(PyTuple_GET_ITEM(a[1], i)) != o ||
        PyLong_AsUnsignedLongLong(PyTuple_GET_ITEM(st, 0)) != (unsigned long long)(uintptr_t)t.const_data_ptr() ||
        PyLong_AsLongLong(PyTuple_GET_ITEM(st, 1)) != (long long)t._version()) {
      PyErr_Clear();
      Py_RETURN_FALSE;
    }
  }
  Py_RETURN_TRUE;
}

// An exception on the way (out of memory, for one) goes the Python way too, which raises it there.
template <PyObject* (*F)(PyObject* const*), Py_ssize_t N>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != N) {
    PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", N, n);
    return nullptr;
  }
  try {
    PyObject* r = F(args);
    if (r) return r;
    if (PyErr_Occurred()) PyErr_Clear();
  } catch (...) {
    PyErr_Clear();
  }
  Py_RETURN_NONE;
}

#define FORGE_ENTRY(NAME, N) \
  {#NAME, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(&entry<NAME##_impl, N>)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    FORGE_ENTRY(decode_append, 21), FORGE_ENTRY(kv_append, 11), FORGE_ENTRY(prefill, 11),
    FORGE_ENTRY(linear_small, 8),   FORGE_ENTRY(tensors_are, 4), {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_forge_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__forge_host(void) { return PyModule_Create(&module); }
