// The host side of the ops in ops.py, in C++: what a valid call spends between Python and the launch.
//
// A launch takes ~4 us of host time, but checking a dozen tensors, reading their shapes, strides and addresses one
// attribute at a time and converting twenty arguments through ctypes took 9-13 us more per call -- a decode step issued call
// by call (24 layers, 123 calls) spent 1690 us on the host for 670 us of GPU work. Each function here takes the
// arguments of its namesake in ops.py, does the same checks and the same launch, and returns None as soon as anything is not
// the ordinary case (another dtype, a strided operand, a wrong shape, a CPU tensor, arguments that the entry point refuses):
// ops.py then runs its own checks, which make the copy or raise the error. Only a call that has launched nothing is answered
// so (the norm ahead of a QKV projection that is then refused aside: it fills a pool buffer, and ops.py fills it again); what the
// runtime reports at a launch is raised here. Nothing is remembered between calls but the scratch pool.
#include <Python.h>

#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Device.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/autocast_mode.h>

#include <stdexcept>
#include <string>
#include <unordered_map>

#include "tllm_hip.h"

namespace {

using at::Tensor;

// ---- arguments ------------------------------------------------------------------------------------------------------------
inline bool is_none(PyObject* o) { return o == Py_None; }
inline const Tensor& tensor(PyObject* o) { return THPVariable_Unpack(o); }

inline bool gpu_tensor(PyObject* o) { return THPVariable_Check(o) && tensor(o).is_cuda(); }
inline bool bf16(const Tensor& t) { return t.scalar_type() == at::kBFloat16; }
inline bool fp8(const Tensor& t) { return t.scalar_type() == at::kFloat8_e4m3fn; }
// the norm's scale: fp32 or bf16, dense, of the given length
inline bool norm_scale_ok(const Tensor& t, int64_t n) {
  return t.dim() == 1 && t.size(0) == n && t.stride(0) == 1 && (bf16(t) || t.scalar_type() == at::kFloat);
}
inline bool bias_ok(PyObject* o, int64_t n) {
  if (is_none(o)) return true;
  if (!gpu_tensor(o)) return false;
  const Tensor& t = tensor(o);
  return bf16(t) && t.dim() == 1 && t.size(0) == n && t.stride(0) == 1;
}
// a dense weight [n, k], bf16 without scales or fp8 e4m3 with one fp32 scale per row
inline bool weight_ok(PyObject* w, PyObject* ws) {
  if (!gpu_tensor(w)) return false;
  const Tensor& t = tensor(w);
  if (t.dim() != 2 || !t.is_contiguous()) return false;
  if (is_none(ws)) return bf16(t);
  if (!gpu_tensor(ws)) return false;
  const Tensor& s = tensor(ws);
  return fp8(t) && s.scalar_type() == at::kFloat && s.dim() == 1 && s.size(0) == t.size(0) && s.stride(0) == 1;
}
inline const void* ptr(PyObject* o) { return is_none(o) ? nullptr : tensor(o).const_data_ptr(); }
inline void* mut(const Tensor& t) { return t.mutable_data_ptr(); }

inline bool to_i64(PyObject* o, int64_t* v) {
  if (!PyLong_Check(o)) return false;
  *v = PyLong_AsLongLong(o);
  if (*v == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}
inline bool to_f64(PyObject* o, double* v) {
  if (!PyFloat_Check(o) && !PyLong_Check(o)) return false;
  *v = PyFloat_AsDouble(o);
  if (*v == -1.0 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

inline void* stream() { return c10::hip::getCurrentHIPStream().stream(); }
PyObject* none() { Py_RETURN_NONE; }

// Ahead of a launch and of an allocation the interpreter lock is given up, as ctypes and torch's own bindings do: both may wait
// (a full queue, a kernel's first load, memory that has to be freed first), and what they wait for may need the lock.
struct Unlocked {
  PyThreadState* const state = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(state); }
};
Tensor empty(at::IntArrayRef shape, const at::TensorOptions& options) {
  Unlocked u;
  return at::empty(shape, options);
}

// Calls an entry point: true behind a launch, false where it refused its arguments and launched nothing. An error of the
// runtime's is raised and the call not made again: the kernel may be on its way (the error that an earlier call left is
// reported by the next launch), and an op that writes in place would be applied twice.
template <class F>
bool launch(const char* what, F entry_point) {
  const int rc = [&] {
    Unlocked u;
    return entry_point();
  }();
  if (rc == TLLM_E_LAUNCH) throw std::runtime_error(std::string(what) + " failed (code " + std::to_string(rc) + "): " + tllm_last_error());
  return rc == TLLM_OK;
}
inline PyObject* wrap(const Tensor& t) { return THPVariable_Wrap(t); }

// ---- scratch pool -----------------------------------------------------------------------------------------------------------
// One buffer per (shape, dtype, device), kept until clear() (scratch_pool.py:17-22 of the reference); it is touched under the
// interpreter lock only, which makes it safe to share between threads.
std::unordered_map<std::string, Tensor>& pool() {
  static auto* p = new std::unordered_map<std::string, Tensor>();   // never destroyed: tensors outlive the interpreter otherwise
  return *p;
}

Tensor pool_get(at::IntArrayRef shape, at::ScalarType dtype, at::Device device) {
  std::string key(reinterpret_cast<const char*>(shape.data()), shape.size() * 8);
  for (int v : {static_cast<int>(dtype), static_cast<int>(device.type()), static_cast<int>(device.index())}) key.push_back(static_cast<char>(v));
  auto it = pool().find(key);
  if (it != pool().end()) return it->second;
  const Tensor t = empty(shape, at::TensorOptions().dtype(dtype).device(device));
  return pool().emplace(std::move(key), t).first->second;   // (another thread's, if it was first)
}

// An output the kernel writes while other workgroups still read `in`: not a pool buffer that is that very memory.
Tensor pooled_output(at::IntArrayRef shape, const Tensor& in) {
  Tensor t = pool_get(shape, at::kBFloat16, in.device());
  const char *a = static_cast<const char*>(t.const_data_ptr()), *b = static_cast<const char*>(in.const_data_ptr());
  if (t.numel() && in.numel() && a < b + in.numel() * in.element_size() && b < a + t.numel() * t.element_size())
    return empty(shape, in.options().dtype(at::kBFloat16));
  return t;
}

// pool_get(shape tuple, dtype, device)
PyObject* pool_buffer(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 3 || !PyTuple_Check(a[0]) || !THPDtype_Check(a[1]) || !THPDevice_Check(a[2])) return none();
  at::DimVector dims(PyTuple_GET_SIZE(a[0]));
  for (size_t i = 0; i < dims.size(); ++i)
    if (!to_i64(PyTuple_GET_ITEM(a[0], i), &dims[i])) return none();
  return wrap(pool_get(dims, reinterpret_cast<THPDtype*>(a[1])->scalar_type, reinterpret_cast<THPDevice*>(a[2])->device));
}

PyObject* py_pool_clear(PyObject*, PyObject*) {
  pool().clear();
  return none();
}

PyObject* py_pool_stats(PyObject*, PyObject*) {
  long long bytes = 0;
  for (auto& kv : pool()) bytes += kv.second.numel() * kv.second.element_size();
  return Py_BuildValue("nL", static_cast<Py_ssize_t>(pool().size()), bytes);
}

// ---- rotary source ------------------------------------------------------------------------------------------------------------
PyObject* g_c_address;   // interned "_c_address": the address of a YarnParams object's C struct (yarn.py)

// yarn: a YarnParams object; positions / offset: None or int64 tensors. Tables of cos / sin values take the Python path.
bool rope_of(PyObject* yarn, PyObject* positions, PyObject* offset, int64_t rows, int64_t tokens_per_batch, int64_t max_ctx, TllmRope* r) {
  if (is_none(yarn)) return false;
  PyObject* addr = PyObject_GetAttr(yarn, g_c_address);
  if (addr == nullptr) {
    PyErr_Clear();
    return false;
  }
  *r = TllmRope{};
  r->yarn = static_cast<const TllmYarn*>(PyLong_AsVoidPtr(addr));
  Py_DECREF(addr);
  if (r->yarn == nullptr) return false;
  if (!is_none(positions)) {
    if (!gpu_tensor(positions)) return false;
    const Tensor& p = tensor(positions);
    if (p.scalar_type() != at::kLong || !p.is_contiguous() || p.numel() != rows) return false;
    r->positions = static_cast<const int64_t*>(p.const_data_ptr());
  }
  if (!is_none(offset)) {
    if (!gpu_tensor(offset)) return false;
    const Tensor& o = tensor(offset);
    if (o.scalar_type() != at::kLong || o.numel() != 1) return false;
    r->offset = static_cast<const int64_t*>(o.const_data_ptr());
  }
  r->tokens_per_batch = tokens_per_batch;
  r->max_ctx = max_ctx;
  return true;
}

// ---- ops ----------------------------------------------------------------------------------------------------------------------
bool rmsnorm_into(const Tensor& x, const Tensor& scale, double eps, const Tensor& out) {
  const int64_t hidden = x.size(-1);
  return launch("rmsnorm_forward", [&] {
    return tllm_rmsnorm_bf16(x.const_data_ptr(), scale.const_data_ptr(), bf16(scale), mut(out), hidden ? x.numel() / hidden : 0, hidden,
                             static_cast<float>(eps), stream());
  });
}

// rmsnorm(x, scale, eps, out)
PyObject* rmsnorm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  double eps;
  if (n != 4 || !gpu_tensor(a[0]) || !gpu_tensor(a[1]) || !to_f64(a[2], &eps)) return none();
  const Tensor &x = tensor(a[0]), &scale = tensor(a[1]);
  if (!bf16(x) || x.dim() < 1 || !x.is_contiguous() || !norm_scale_ok(scale, x.size(-1))) return none();
  if (is_none(a[3])) {
    const Tensor out = pool_get(x.sizes(), at::kBFloat16, x.device());
    return rmsnorm_into(x, scale, eps, out) ? wrap(out) : none();
  }
  if (!gpu_tensor(a[3])) return none();
  const Tensor& out = tensor(a[3]);
  if (!bf16(out) || out.sizes() != x.sizes() || !out.is_contiguous() || !rmsnorm_into(x, scale, eps, out)) return none();
  Py_INCREF(a[3]);
  return a[3];
}

inline bool ids_ok(const Tensor& ids) { return (ids.scalar_type() == at::kInt || ids.scalar_type() == at::kLong) && ids.is_contiguous(); }
inline bool table_ok(const Tensor& t) { return bf16(t) && t.dim() == 2 && t.is_contiguous(); }
inline bool flag_ok(PyObject* o) {
  return is_none(o) || (gpu_tensor(o) && tensor(o).scalar_type() == at::kInt && tensor(o).numel() == 1);
}
at::DimVector with_last(const Tensor& t, int64_t last) {
  at::DimVector s(t.sizes().begin(), t.sizes().end());
  s.push_back(last);
  return s;
}
inline int* flag(PyObject* o) { return is_none(o) ? nullptr : static_cast<int*>(mut(tensor(o))); }

// embedding(ids, table, out, oob_flag)
PyObject* embedding(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 4 || !gpu_tensor(a[0]) || !gpu_tensor(a[1]) || !flag_ok(a[3])) return none();
  const Tensor &ids = tensor(a[0]), &table = tensor(a[1]);
  if (!ids_ok(ids) || !table_ok(table)) return none();
  const auto shape = with_last(ids, table.size(1));
  Tensor out;
  if (is_none(a[2])) {
    out = empty(shape, table.options());
  } else {
    if (!gpu_tensor(a[2])) return none();
    out = tensor(a[2]);
    if (!bf16(out) || out.sizes() != at::IntArrayRef(shape) || !out.is_contiguous()) return none();
  }
  const bool done = launch("embedding_forward", [&] {
    return tllm_embedding_bf16(table.const_data_ptr(), ids.const_data_ptr(), ids.scalar_type() == at::kLong, mut(out), ids.numel(), table.size(1),
                          table.size(0), flag(a[3]), stream());
  });
  if (!done) return none();
  return wrap(out);
}

// embedding_rmsnorm(ids, table, scale, eps, x_out, out, oob_flag)
PyObject* embedding_rmsnorm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  double eps;
  if (n != 7 || !gpu_tensor(a[0]) || !gpu_tensor(a[1]) || !gpu_tensor(a[2]) || !to_f64(a[3], &eps) || !flag_ok(a[6])) return none();
  const Tensor &ids = tensor(a[0]), &table = tensor(a[1]), &scale = tensor(a[2]);
  if (!ids_ok(ids) || !table_ok(table)) return none();
  const int64_t hidden = table.size(1);
  if (hidden % 8 != 0 || hidden > 8192 || !norm_scale_ok(scale, hidden)) return none();
  const auto shape = with_last(ids, hidden);
  Tensor got[2];
  for (int i = 0; i < 2; ++i) {
    if (is_none(a[4 + i])) {
      got[i] = i == 0 ? empty(shape, table.options()) : pool_get(shape, at::kBFloat16, table.device());
    } else {
      if (!gpu_tensor(a[4 + i])) return none();
      got[i] = tensor(a[4 + i]);
      if (!bf16(got[i]) || got[i].sizes() != at::IntArrayRef(shape) || !got[i].is_contiguous()) return none();
    }
  }
  if (got[0].const_data_ptr() == got[1].const_data_ptr()) return none();
  const bool done = launch("embedding_rmsnorm_forward", [&] {
    return tllm_embed_rmsnorm_bf16(table.const_data_ptr(), ids.const_data_ptr(), ids.scalar_type() == at::kLong, mut(got[0]), scale.const_data_ptr(),
                              bf16(scale), mut(got[1]), ids.numel(), hidden, table.size(0), static_cast<float>(eps), flag(a[6]), stream());
  });
  if (!done) return none();
  PyObject *x = wrap(got[0]), *y = wrap(got[1]);
  PyObject* r = PyTuple_Pack(2, x, y);
  Py_XDECREF(x);
  Py_XDECREF(y);
  return r;
}

// swiglu(x, alpha, limit, interleaved, out)
PyObject* swiglu(PyObject*, PyObject* const* a, Py_ssize_t n) {
  double alpha, limit = 0.0;
  if (n != 5 || !gpu_tensor(a[0]) || !to_f64(a[1], &alpha) || !(is_none(a[2]) || to_f64(a[2], &limit)) || !PyBool_Check(a[3])) return none();
  const Tensor& x = tensor(a[0]);
  if (!bf16(x) || x.dim() < 1 || !x.is_contiguous() || x.size(-1) % 2 != 0 || x.numel() == 0) return none();
  const int64_t n_out = x.size(-1) / 2;
  at::DimVector shape(x.sizes().begin(), x.sizes().end());
  shape.back() = n_out;
  Tensor out;
  if (is_none(a[4])) {
    out = empty(shape, x.options());
  } else {
    if (!gpu_tensor(a[4])) return none();
    out = tensor(a[4]);
    if (!bf16(out) || out.sizes() != at::IntArrayRef(shape) || !out.is_contiguous()) return none();
  }
  const bool done = launch("swiglu", [&] {
    return tllm_swiglu_bf16(x.const_data_ptr(), mut(out), x.numel() / (2 * n_out), n_out, 2 * n_out, static_cast<float>(alpha), static_cast<float>(limit),
                       !is_none(a[2]), a[3] == Py_True, stream());
  });
  if (!done) return none();
  return wrap(out);
}

// The QKV launch behind both forms: the norm inside the decode kernel where it can be, a launch ahead otherwise.
bool launch_qkv(bool decode, const Tensor& x_in, const Tensor& w, PyObject* bias, PyObject* w_scale, PyObject* norm_scale, bool fuse_norm, double eps,
                void* q, void* k, void* v, int64_t q_rs, int64_t k_rs, int64_t v_rs, int64_t kv_slot, int nq, int nkv, int hd, const TllmRope* rope) {
  Tensor x = x_in;
  const int64_t rows = x.size(0), hidden = x.size(1);
  const void *ns = nullptr, *ws = ptr(w_scale);
  int ns_bf16 = 0;
  if (!is_none(norm_scale)) {
    const Tensor& s = tensor(norm_scale);
    if (fuse_norm) {
      ns = s.const_data_ptr();
      ns_bf16 = bf16(s);
    } else {
      const Tensor t = pool_get(x.sizes(), at::kBFloat16, x.device());
      if (!rmsnorm_into(x, s, eps, t)) return false;
      x = t;
    }
  }
  const float e = static_cast<float>(eps);
  if (ws != nullptr) {
    if (!decode || hidden % 32 != 0 || hd % 16 != 0) return false;
    return launch("qkv_rope_decode_w8", [&] {
      return tllm_qkv_rope_decode_w8_bf16(x.const_data_ptr(), ns, ns_bf16, e, w.const_data_ptr(), static_cast<const float*>(ws), ptr(bias), q, k, v,
                                          q_rs, k_rs, v_rs, kv_slot, rows, hidden, nq, nkv, hd, rope, stream());
    });
  }
  if (ns != nullptr)
    return launch("norm_qkv_rope_decode", [&] {
      return tllm_norm_qkv_rope_decode_bf16(x.const_data_ptr(), ns, ns_bf16, e, w.const_data_ptr(), ptr(bias), q, k, v, q_rs, k_rs, v_rs, kv_slot,
                                            rows, hidden, nq, nkv, hd, rope, stream());
    });
  return launch(decode ? "qkv_rope_decode" : "qkv_rope_prefill", [&] {
    return (decode ? tllm_qkv_rope_decode_bf16 : tllm_qkv_rope_prefill_bf16)(x.const_data_ptr(), w.const_data_ptr(), ptr(bias), q, k, v, q_rs, k_rs, v_rs,
                                                                            kv_slot, rows, hidden, nq, nkv, hd, rope, stream());
  });
}

bool heads_of(PyObject* const* a, int64_t total_out, int* nq, int* nkv, int* hd) {
  int64_t v[3];
  for (int i = 0; i < 3; ++i)
    if (!to_i64(a[i], &v[i]) || v[i] < 0 || v[i] > (1 << 20)) return false;
  if (v[2] == 0 || total_out != (v[0] + 2 * v[1]) * v[2]) return false;
  *nq = static_cast<int>(v[0]);
  *nkv = static_cast<int>(v[1]);
  *hd = static_cast<int>(v[2]);
  return true;
}

// qkv_rope(x, weight, bias, num_q_heads, num_kv_heads, head_dim, yarn, positions, offset, tokens_per_batch, max_context_length,
//          rotate, kind, out, norm_scale, norm_eps, weight_scale, fuse_norm, cos, sin)
// (the tables are looked at for their device alone: yarn are the parameters that they carry)
PyObject* qkv_rope(PyObject*, PyObject* const* a, Py_ssize_t n) {
  int nq, nkv, hd;
  int64_t tpb, max_ctx;
  double eps;
  if (n != 20 || !PyBool_Check(a[17]) || !gpu_tensor(a[0]) || !weight_ok(a[1], a[16]) || !to_i64(a[10], &max_ctx) || !to_f64(a[15], &eps) || !PyBool_Check(a[11])) return none();
  for (int i : {7, 8, 18, 19})                     // used or not: a tensor of another device is the caller's mistake
    if (!is_none(a[i]) && !gpu_tensor(a[i])) return none();
  const Tensor &x = tensor(a[0]), &w = tensor(a[1]);
  if (!bf16(x) || x.dim() != 2 || !x.is_contiguous() || x.size(1) != w.size(1) || x.size(0) == 0 || !bias_ok(a[2], w.size(0)) ||
      !heads_of(a + 3, w.size(0), &nq, &nkv, &hd))
    return none();
  const int64_t rows = x.size(0), q_dim = static_cast<int64_t>(nq) * hd, kv_dim = static_cast<int64_t>(nkv) * hd;
  if (!is_none(a[14]) && !(gpu_tensor(a[14]) && norm_scale_ok(tensor(a[14]), x.size(1)))) return none();
  tpb = rows;
  if (!is_none(a[9]) && !to_i64(a[9], &tpb)) return none();
  if (tpb == 0) tpb = rows;
  bool decode;
  if (!PyUnicode_Check(a[12])) return none();
  if (PyUnicode_CompareWithASCIIString(a[12], "decode") == 0) decode = true;
  else if (PyUnicode_CompareWithASCIIString(a[12], "prefill") == 0) decode = false;
  else return none();
  TllmRope r;
  const bool rotate = a[11] == Py_True;
  if (rotate && !rope_of(a[6], a[7], a[8], rows, tpb, max_ctx, &r)) return none();
  Tensor q, k, v;
  PyObject* result;
  if (is_none(a[13])) {
    q = pooled_output({rows, nq, hd}, x).view({rows, q_dim});
    const Tensor kv = pooled_output({2, rows, kv_dim}, x);
    k = kv.select(0, 0);
    v = kv.select(0, 1);
    result = nullptr;
  } else {
    if (!PyTuple_Check(a[13]) || PyTuple_GET_SIZE(a[13]) != 3) return none();
    for (int i = 0; i < 3; ++i) {
      PyObject* o = PyTuple_GET_ITEM(a[13], i);
      if (!gpu_tensor(o)) return none();
      const Tensor& t = tensor(o);
      if (!bf16(t) || t.dim() != 2 || t.size(0) != rows || t.size(1) != (i == 0 ? q_dim : kv_dim) || t.stride(1) != 1) return none();
      (i == 0 ? q : i == 1 ? k : v) = t;
    }
    result = a[13];
  }
  if (!launch_qkv(decode, x, w, a[2], a[16], a[14], a[17] == Py_True, eps, mut(q), mut(k), mut(v), q.stride(0), k.stride(0), v.stride(0), 0, nq, nkv, hd,
                  rotate ? &r : nullptr))
    return none();
  if (result != nullptr) {
    Py_INCREF(result);
    return result;
  }
  PyObject *pq = wrap(q), *pk = wrap(k), *pv = wrap(v);
  result = PyTuple_Pack(3, pq, pk, pv);
  Py_XDECREF(pq);
  Py_XDECREF(pk);
  Py_XDECREF(pv);
  return result;
}

// qkv_rope_cache(hidden, weight, bias, yarn, max_context_length, cache_k, cache_v, offset, num_q_heads, num_kv_heads, head_dim,
//                weight_scale, positions, norm_scale, norm_eps, fuse_norm)
PyObject* qkv_rope_cache(PyObject*, PyObject* const* a, Py_ssize_t n) {
  int nq, nkv, hd;
  int64_t max_ctx;
  double eps;
  if (n != 16 || !PyBool_Check(a[15]) || !gpu_tensor(a[0]) || !weight_ok(a[1], a[11]) || !gpu_tensor(a[2]) || !to_i64(a[4], &max_ctx) || !gpu_tensor(a[5]) ||
      !gpu_tensor(a[6]) || !gpu_tensor(a[7]) || !to_f64(a[14], &eps))
    return none();
  const Tensor &h = tensor(a[0]), &w = tensor(a[1]), &ck = tensor(a[5]), &cv = tensor(a[6]), &off = tensor(a[7]);
  if (!bf16(h) || h.dim() != 3 || h.size(1) != 1 || h.size(0) == 0 || !h.is_contiguous() || h.size(2) != w.size(1) || !bias_ok(a[2], w.size(0)) ||
      !heads_of(a + 8, w.size(0), &nq, &nkv, &hd))
    return none();
  const int64_t batch = h.size(0);
  if (!bf16(ck) || !bf16(cv) || ck.dim() != 4 || ck.sizes() != cv.sizes() || ck.strides() != cv.strides() || ck.size(0) != batch ||
      ck.size(2) != nkv || ck.size(3) != hd || ck.stride(3) != 1 || ck.stride(2) != hd || off.dim() != 1)
    return none();
  if (!is_none(a[13]) && !(gpu_tensor(a[13]) && norm_scale_ok(tensor(a[13]), h.size(2)))) return none();
  TllmRope r;
  if (!rope_of(a[3], a[12], a[7], batch, 1, max_ctx, &r)) return none();
  const Tensor x = h.view({batch, h.size(2)});
  const Tensor q = pooled_output({batch, nq, hd}, x);
  if (!launch_qkv(true, x, w, a[2], a[11], a[13], a[15] == Py_True, eps, mut(q), mut(ck), mut(cv), static_cast<int64_t>(nq) * hd, ck.stride(0), cv.stride(0),
                  ck.stride(1), nq, nkv, hd, &r))
    return none();
  return wrap(q.view({batch, 1, static_cast<int64_t>(nq) * hd}));
}

// F.linear is an operator of torch's that everything hooks into: what a raw launch would pass by -- a tensor subclass, vmap,
// forward-mode derivatives, autocast, tracing, function and dispatch modes, a gradient -- stays with it.
bool only_eager() {
  const c10::DispatchKeySet now = c10::impl::tls_local_dispatch_key_set().included_;
  return (now.raw_repr() & ~c10::default_included_set.raw_repr()) == 0 && !at::impl::torch_function_mode_enabled() &&
         !at::autocast::is_autocast_enabled(at::kCUDA);
}
bool plain_operand(PyObject* o, c10::DeviceIndex device) {
  if (!THPVariable_CheckExact(o)) return false;
  const Tensor& t = tensor(o);
  const c10::DispatchKeySet ordinary({c10::DispatchKey::CUDA, c10::DispatchKey::AutogradCUDA, c10::DispatchKey::ADInplaceOrView,
                                      c10::DispatchKey::AutocastCUDA});
  return t.is_cuda() && t.device().index() == device && (t.key_set().raw_repr() & ~ordinary.raw_repr()) == 0 &&
         !(c10::GradMode::is_enabled() && t.requires_grad()) && !t._fw_grad(0).defined();
}

// Whether a GEMM tile is ahead of the library's GEMM. Up to tiles of 128 x 224 covering the result in one round of the 256 CUs
// and about 2500 rows it mostly is ([2880, 4096] weight, us: 97 rows 13.8 and 15.5, 192 rows 16.5 and 32, 999 rows 29.8 and 35.4,
// 2400 rows 53.2 and 55.6; behind two rounds 2700 68.6 and 58.5, 4096 94 and 75; other weights 3000 rows 0.84 - 0.92 of the
// library's rate). Tiles of 128 x 256 are ahead as long as they are one round if the outputs are no multiple of 128, which the library's
// own tiles would fit ([2880, 4096] 2500 rows 55.3 and 58.5, K = 2048 33.0 and 36.3, 512 17.0 and 21.5; [4400, 4096] 1664 55.9 and 59.7; [8176,
// 2880] 1024 44.5 and 47.8; but [3072, 4096] 2500 55.7 and 53.9, [2048, 4096] 2560 43.8 and 41.4), up to weights of about 25 M elements
// ([6000, 4096] 1280 rows 55.9 and 59.4, [6992, 4096] 1092 62.1 and 58.6). Where the tiles are few and K is long the library shares K out between workgroups: from a K of
// 50 per tile on (32 above 4096) it is ahead ([512, 2048] 48 rows 5.7 and 7.4, [1024, 8192] 48 rows 11.9 and 17.2, [2880, 5120]
// 8 rows 10.5 and 15.5), with 25 - 64 rows of a K of 2900 and more from 30 on ([2880, 4096] 48 rows 13.1 and 14.9). And it has
// a kernel for a few rows of a small weight ([512, 512] 16 rows 4.1 and 4.7, [1024, 1024] 4.6 and 5.8). Of 1600 calls of a K of
// 64 .. 8192 and 128 .. 8192 outputs measured, 85 are 3 % slower so than with the library, 353 without the latter three.
bool linear_in_tiles(int64_t rows, int64_t k, int64_t out) {
  const int64_t widest = out % 128 && out * k <= 25000000 ? 256 : 224;
  if (rows > 2560 || ((rows + 127) / 128) * ((out + widest - 1) / widest) > 256) return false;
  const int tile = tllm_linear_gemm_tile(rows, k, out);
  const int64_t bm = tile >> 16, bn = tile & 0xffff, tiles = ((rows + bm - 1) / bm) * ((out + bn - 1) / bn);
  if (k >= 1024 && k >= (k > 4096 ? 32 : 50) * tiles) return false;
  if (rows > 24 && rows <= 64 && k >= 2900 && k >= 30 * tiles) return false;
  return !(rows > 1 && rows <= 24 && k >= 512 && k < 2048 && out <= 2048);
}

// linear(x, weight, bias): F.linear for plain bf16 tensors, K a multiple of 64 and outputs of 16, where a tile is ahead
PyObject* linear(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 3 || !only_eager() || !THPVariable_CheckExact(a[0]) || !tensor(a[0]).is_cuda()) return none();
  const c10::DeviceIndex device = c10::hip::current_device();
  for (int i = 0; i < 3; ++i)
    if (!(i == 2 && is_none(a[2])) && !plain_operand(a[i], device)) return none();
  if (!weight_ok(a[1], Py_None)) return none();
  const Tensor &x = tensor(a[0]), &w = tensor(a[1]);
  const int64_t out = w.size(0), k = w.size(1);
  if (!bf16(x) || x.dim() < 1 || x.size(-1) != k || x.numel() == 0 || !bias_ok(a[2], out) || k % 64 || out % 16 || out * k >= (1ll << 31))
    return none();
  const int64_t rows = x.numel() / k;
  if (!linear_in_tiles(rows, k, out)) return none();
  at::DimVector shape(x.sizes().begin(), x.sizes().end());
  shape.back() = out;
  const Tensor xc = x.is_contiguous() ? x : [&] {
    Unlocked u;
    return x.contiguous();
  }();
  const Tensor y = empty(shape, xc.options());
  const bool done = launch("linear", [&] {
    return tllm_linear_bf16(xc.const_data_ptr(), w.const_data_ptr(), ptr(a[2]), mut(y), out, rows, k, out, stream());
  });
  if (!done) return none();
  return wrap(y);
}

// out_residual(hidden, weight, bias, residual, weight_scale)
PyObject* out_residual(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 5 || !gpu_tensor(a[0]) || !weight_ok(a[1], a[4]) || !gpu_tensor(a[2]) || !gpu_tensor(a[3])) return none();
  const Tensor &h = tensor(a[0]), &w = tensor(a[1]), &res = tensor(a[3]);
  const int64_t out = w.size(0), in = w.size(1);
  if (!bf16(h) || h.dim() != 3 || h.size(1) != 1 || h.size(2) != in || !h.is_contiguous() || !bias_ok(a[2], out)) return none();
  const int64_t batch = h.size(0);
  if (!bf16(res) || res.dim() != 3 || res.size(0) != batch || res.size(1) != 1 || res.size(2) != out || !res.is_contiguous()) return none();
  const bool done = launch("out_residual_decode_forward", [&] {
    return tllm_out_residual_decode_bf16(h.const_data_ptr(), w.const_data_ptr(), static_cast<const float*>(ptr(a[4])), ptr(a[2]), mut(res), mut(res), out, out,
                                    batch, in, out, stream());
  });
  if (!done) return none();
  return wrap(res.view({batch, 1, out}));
}

// unembedding(hidden, weight, weight_scale)
PyObject* unembedding(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 3 || !gpu_tensor(a[0]) || !weight_ok(a[1], a[2])) return none();
  const Tensor &h = tensor(a[0]), &w = tensor(a[1]);
  if (!bf16(h) || h.dim() != 3 || h.size(1) != 1 || h.size(2) != w.size(1) || !h.is_contiguous()) return none();
  const Tensor logits = pool_get({h.size(0), w.size(0)}, at::kBFloat16, h.device());
  const bool done = launch("unembedding_decode_forward", [&] {
    return tllm_unembedding_decode_bf16(h.const_data_ptr(), w.const_data_ptr(), static_cast<const float*>(ptr(a[2])), mut(logits), w.size(0), h.size(0),
                                   w.size(1), w.size(0), stream());
  });
  if (!done) return none();
  return wrap(logits.unsqueeze(1));
}

struct Attn {
  const Tensor *q, *k, *v;
  int64_t bs, n_ctx, n_kv_ctx, start_is_i64, window;
  int nkv, group;
  float scale;
  const void *sinks, *start;
};

// (q, k, v, sinks, sm_scale, bandwidth, start_q): the operands both attention kernels take as they are
bool attn_of(PyObject* const* a, Attn* t) {
  double scale;
  if (!gpu_tensor(a[0]) || !gpu_tensor(a[1]) || !gpu_tensor(a[2]) || !to_f64(a[4], &scale) || !gpu_tensor(a[6])) return false;
  const Tensor &q = tensor(a[0]), &k = tensor(a[1]), &v = tensor(a[2]), &s = tensor(a[6]);
  if (!bf16(q) || !bf16(k) || !bf16(v) || q.dim() != 5 || k.dim() != 4 || q.size(4) != 64 || k.sizes() != v.sizes() || k.strides() != v.strides())
    return false;
  if (k.size(0) != q.size(0) || k.size(2) != q.size(2) || k.size(3) != 64 || k.stride(3) != 1 || k.stride(2) != 64 || k.stride(1) % 8 ||
      k.stride(0) % 8)
    return false;
  if (s.dim() != 1 || s.size(0) != 1 || (s.scalar_type() != at::kInt && s.scalar_type() != at::kLong)) return false;
  t->window = 0;
  if (!is_none(a[5]) && (!to_i64(a[5], &t->window) || t->window < 0 || t->window > INT32_MAX)) return false;
  t->q = &q;
  t->k = &k;
  t->v = &v;
  t->bs = q.size(0);
  t->n_ctx = q.size(1);
  t->nkv = static_cast<int>(q.size(2));
  t->group = static_cast<int>(q.size(3));
  t->n_kv_ctx = k.size(1);
  t->scale = static_cast<float>(scale);
  t->start = s.const_data_ptr();
  t->start_is_i64 = s.scalar_type() == at::kLong;
  t->sinks = nullptr;
  if (!is_none(a[3])) {
    if (!gpu_tensor(a[3])) return false;
    const Tensor& z = tensor(a[3]);
    if (!bf16(z) || z.dim() != 1 || z.size(0) != q.size(2) * q.size(3) || z.stride(0) != 1) return false;
    t->sinks = z.const_data_ptr();
  }
  return t->bs > 0 && t->n_ctx > 0;
}

// attention_decode(q, k, v, sinks, sm_scale, bandwidth, start_q, kv_len_hint)
PyObject* attention_decode(PyObject*, PyObject* const* a, Py_ssize_t n) {
  Attn t;
  int64_t hint = 0;
  if (n != 8 || !attn_of(a, &t) || !(is_none(a[7]) || to_i64(a[7], &hint))) return none();
  if (t.n_ctx != 1 || t.group > 16 || !t.q->is_contiguous()) return none();
  if (!is_none(a[7]) && hint < 1) hint = 1;
  const int64_t width = static_cast<int64_t>(t.nkv) * t.group * 64;
  const int64_t plan = hint && hint < t.n_kv_ctx ? hint : t.n_kv_ctx;
  const int64_t bytes = tllm_attention_decode_workspace_bytes(t.bs, t.nkv * t.group, t.nkv, plan, static_cast<int>(t.window));
  const Tensor o = pool_get({t.bs, width}, at::kBFloat16, t.q->device());
  Tensor work;
  if (bytes) work = pool_get({bytes / 4 > 1 ? bytes / 4 : 1}, at::kFloat, t.q->device());
  const bool done = launch("attention_decode", [&] {
    return tllm_attention_decode_bf16(t.q->const_data_ptr(), t.k->const_data_ptr(), t.v->const_data_ptr(), t.sinks, mut(o), width, width, t.k->stride(0),
                                 t.k->stride(1), t.bs, t.n_kv_ctx, t.nkv, t.group, 64, t.scale, static_cast<int>(t.window), t.start,
                                 static_cast<int>(t.start_is_i64), hint, bytes ? mut(work) : nullptr, bytes, stream());
  });
  if (!done) return none();
  return wrap(o.view({t.bs, 1, width}));
}

// attention(q, k, v, sinks, sm_scale, bandwidth, start_q)
PyObject* attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
  Attn t;
  if (n != 7 || !attn_of(a, &t)) return none();
  const Tensor& q = *t.q;
  auto al16 = [](const Tensor& x) { return reinterpret_cast<uintptr_t>(x.const_data_ptr()) % 16 == 0; };
  if (q.stride(4) != 1 || q.stride(3) != 64 || q.stride(2) != 64 * t.group || q.stride(1) % 8 || q.stride(0) % 8 || !al16(q) || !al16(*t.k) ||
      !al16(*t.v))
    return none();
  const int64_t width = static_cast<int64_t>(t.nkv) * t.group * 64;
  const Tensor o = pool_get({t.bs, t.n_ctx, width}, at::kBFloat16, q.device());
  const bool done = launch("attention", [&] {
    return tllm_attention_prefill_bf16(q.const_data_ptr(), t.k->const_data_ptr(), t.v->const_data_ptr(), t.sinks, mut(o), q.stride(0), q.stride(1),
                                  o.stride(0), o.stride(1), t.k->stride(0), t.k->stride(1), t.bs, t.n_ctx, t.n_kv_ctx, t.nkv, t.group, 64, t.scale,
                                  static_cast<int>(t.window), t.start, static_cast<int>(t.start_is_i64), stream());
  });
  if (!done) return none();
  return wrap(o);
}

// Whatever ATen throws (out of memory, ...) reaches Python as the RuntimeError it would be there.
template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t)>
PyObject* guarded(PyObject* self, PyObject* const* a, Py_ssize_t n) {
  try {
    return F(self, a, n);
  } catch (const c10::OutOfMemoryError& e) {
    PyObject* torch = PyImport_ImportModule("torch");
    PyObject* type = torch ? PyObject_GetAttrString(torch, "OutOfMemoryError") : nullptr;
    PyErr_SetString(type ? type : PyExc_RuntimeError, e.what_without_backtrace());
    Py_XDECREF(type);
    Py_XDECREF(torch);
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
  }
  return nullptr;
}

#define TLLM_OP(f) {#f, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(guarded<f>)), METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {
    TLLM_OP(rmsnorm), TLLM_OP(embedding), TLLM_OP(embedding_rmsnorm), TLLM_OP(swiglu), TLLM_OP(qkv_rope), TLLM_OP(qkv_rope_cache), TLLM_OP(linear),
    TLLM_OP(out_residual), TLLM_OP(unembedding), TLLM_OP(attention_decode), TLLM_OP(attention),
    {"pool_get", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(guarded<pool_buffer>)), METH_FASTCALL, nullptr},
    {"pool_clear", py_pool_clear, METH_NOARGS, nullptr},
    {"pool_stats", py_pool_stats, METH_NOARGS, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "tllm_host", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_tllm_host(void) {
  g_c_address = PyUnicode_InternFromString("_c_address");
  return PyModule_Create(&kModule);
}
