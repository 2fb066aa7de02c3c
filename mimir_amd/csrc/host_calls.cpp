// The host side of the common calls in native code: argument checks, output
// allocation, the parameter struct and the C-ABI launch of the forward, the
// backward, RoPE and the KV-cache attention.
//
// Through ctypes these cost 24 us (forward), 32 us (backward) and 17 us (decode) of
// Python per call, and the backward pays about twice that in a training step: the
// autograd engine runs it on a thread of its own, on a cold core.  A step on a few
// short documents (70 us of GPU work) went from 182 to 113 us with the calls here (64
// of which an autograd function of one multiplication takes too), a decode step of
// one row from 16.3 to 11.7.
//
// Every function here serves only well-formed calls: anything else (another device
// or dtype, a layout the kernels cannot read in place, metadata to convert, a failed
// allocation, arguments that the C ABI refuses) returns None, and the caller takes the
// general path in Python, which converts, falls back or raises.  An error of the launch
// itself raises here: kernels of the call may have run, and the general path would run
// them again (an in-place RoPE twice).
#include <Python.h>
#include <dlfcn.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <torch/csrc/DynamicTypes.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/mimir_prefixlm.h"

namespace {

struct Library {
  decltype(&mimir_prefixlm_fwd) fwd = nullptr;
  decltype(&mimir_prefixlm_fwd_workspace_size) fwd_workspace_size = nullptr;
  decltype(&mimir_prefixlm_fwd_workspace_bytes) fwd_workspace_bytes = nullptr;
  decltype(&mimir_prefixlm_bwd) bwd = nullptr;
  decltype(&mimir_prefixlm_bwd_workspace_size) bwd_workspace_size = nullptr;
  decltype(&mimir_prefixlm_bwd_dscore_bytes) bwd_dscore_bytes = nullptr;
  decltype(&mimir_prefixlm_rope) rope = nullptr;
  decltype(&mimir_prefixlm_cache_attn) cache_attn = nullptr;
  decltype(&mimir_prefixlm_cache_attn_workspace_bytes) cache_workspace = nullptr;
  decltype(&mimir_prefixlm_last_error) last_error = nullptr;
  c10::DeviceType device = c10::DeviceType::CUDA;  // of the tensors it takes
} lib;

// Where the general path takes over, a function returns nullptr without an error set: found
// out in 0.3 us (a C++ exception for it made it 1 to 2 us).
#define NEED(ok) \
  do {           \
    if (!(ok)) return nullptr; \
  } while (0)

const at::Tensor* tensor(PyObject* o) { return THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr; }
#define TENSOR(name, o)                       \
  const at::Tensor* const name##_ = tensor(o); \
  NEED(name##_ != nullptr);                   \
  const at::Tensor& name = *name##_
bool on_device(const at::Tensor& t) { return t.device().type() == lib.device; }
bool is_none(PyObject* o) { return o == Py_None; }
bool int32(PyObject* o, int32_t& out) {  // an int, or a one-element int64 CPU tensor (the reference's scalars)
  int64_t x;
  if (PyLong_CheckExact(o)) {
    x = PyLong_AsLongLong(o);
  } else {
    const at::Tensor* t = tensor(o);
    if (t == nullptr || !t->device().is_cpu() || t->scalar_type() != at::kLong || t->numel() != 1) return false;
    x = *t->const_data_ptr<int64_t>();
  }
  out = (int32_t)x;
  return x >= 0 && x <= 0x7fffffff;
}
bool truth(PyObject* o) { return PyObject_IsTrue(o) == 1; }
void* stream(PyObject* o) { return PyLong_AsVoidPtr(o); }

// A [.., heads, head_dim] operand the kernels read or write in place: unit stride on
// head_dim, 16-byte aligned rows that do not overlap.
bool in_place(const at::Tensor& t, const at::Tensor& like) {
  const int64_t vec = 16 / (int64_t)t.element_size(), d = t.dim();
  if (t.device() != like.device() || t.scalar_type() != like.scalar_type() || !t.has_storage()) return false;
  if (t.stride(d - 1) != 1 || t.stride(d - 3) < t.size(d - 1) || (uintptr_t)t.const_data_ptr() % 16 != 0) return false;
  for (int64_t i = 0; i < d - 1; ++i)
    if (t.stride(i) % vec != 0) return false;
  return true;
}
bool shaped(const at::Tensor& t, int64_t a, int64_t b, int64_t c) {
  return t.dim() == 3 && t.size(0) == a && t.size(1) == b && t.size(2) == c;
}
// A metadata operand's data, nullptr where it has to be converted or is too short.
const int32_t* metadata(PyObject* o, int64_t n, const at::Tensor& like) {
  TENSOR(t, o);
  NEED(t.dim() == 1 && t.size(0) >= n && t.scalar_type() == at::kInt && t.device() == like.device() && t.is_contiguous());
  return t.const_data_ptr<int32_t>();
}

at::Tensor empty(at::IntArrayRef shape, const at::Tensor& like, at::ScalarType type) {
  return at::empty(shape, at::TensorOptions().dtype(type).device(like.device()));
}

// Workspaces come from the caller's torch.empty (float32): it raises where there is no
// room, and the result is then undefined here.
at::Tensor workspace(PyObject* torch_empty, size_t bytes, PyObject* like) {
  const size_t n = bytes / 4 < 4 ? 4 : bytes / 4;
  PyObject* device = PyObject_GetAttrString(like, "device");
  PyObject* args = Py_BuildValue("(n)", (Py_ssize_t)n);
  PyObject* kw = Py_BuildValue("{s:O,s:N}", "dtype", (PyObject*)torch::getTHPDtype(at::kFloat), "device", device);
  PyObject* t = args && kw ? PyObject_Call(torch_empty, args, kw) : nullptr;
  Py_XDECREF(args);
  Py_XDECREF(kw);
  at::Tensor out;
  if (t != nullptr && THPVariable_Check(t)) out = THPVariable_Unpack(t);
  Py_XDECREF(t);
  return out;
}

// Whether the call was launched; after a HIP error `raised` and the Python error are set.
template <typename P>
bool launch(int (*entry)(const P*, void*), const P& p, void* s, bool& raised) {
  if (PyErr_Occurred() != nullptr) return false;  // an argument did not convert
  int status;
  Py_BEGIN_ALLOW_THREADS;
  status = entry(&p, s);
  Py_END_ALLOW_THREADS;
  if (status == MIMIR_ERR_HIP) {
    PyErr_SetString(PyExc_RuntimeError, lib.last_error());
    raised = true;
  }
  return status == MIMIR_OK;  // other failures are refusals: nothing launched
}

// The checks and fields the forward and the backward share.
struct Geometry {
  int64_t T, hq, hkv, d;
  int dtype;
};
bool geometry(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, Geometry& g) {
  if (!on_device(q) || q.dim() != 3 || k.dim() != 3 || v.dim() != 3) return false;
  if (q.scalar_type() != at::kBFloat16 && q.scalar_type() != at::kFloat) return false;
  g = {q.size(0), q.size(1), k.size(1), q.size(2),
       q.scalar_type() == at::kBFloat16 ? MIMIR_DTYPE_BFLOAT16 : MIMIR_DTYPE_FLOAT32};
  return g.T > 0 && g.T <= 0x7fffffff && g.hq > 0 && g.hkv > 0 && g.hq % g.hkv == 0 && g.d > 0 &&
         shaped(k, g.T, g.hkv, g.d) && shaped(v, g.T, g.hkv, g.d) && in_place(q, q) && in_place(k, q) && in_place(v, q);
}

#define STRIDES(p, name, t) (p).name##_stride_token = (t).stride(0), (p).name##_stride_head = (t).stride(1)

PyObject* wrap(std::initializer_list<at::Tensor> ts) {
  PyObject* out = PyTuple_New((Py_ssize_t)ts.size());
  Py_ssize_t i = 0;
  for (const at::Tensor& t : ts) PyTuple_SET_ITEM(out, i++, THPVariable_Wrap(t));
  return out;
}

template <typename F>
PyObject* guarded(Py_ssize_t given, Py_ssize_t wanted, F&& body) {
  if (given != wanted) {
    PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", wanted, given);
    return nullptr;
  }
  PyObject* out = nullptr;
  bool raised = false;
  try {
    out = body(raised);
  } catch (const std::exception&) {  // e.g. out of memory: the general path raises it
  }
  if (out != nullptr || raised) return out;
  PyErr_Clear();
  Py_RETURN_NONE;
}

// fwd(q, k, v, is_causal, prefix_lens, causal_lens, cu_seqlens, total_seqlen, numseqs, max_seqlen_all,
//     softmax_scale, split_mode, key_chunks, want_lo, gate, gated_out, torch_empty, stream)
//   -> (out, lse, out_lo, split_flag)
PyObject* py_fwd(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded(n, 18, [&](bool& raised) -> PyObject* {
    TENSOR(q, a[0]);
    TENSOR(k, a[1]);
    TENSOR(v, a[2]);
    Geometry g;
    NEED(geometry(q, k, v, g));
    MimirPrefixLMFwdParams p = {};
    p.is_causal = truth(a[3]);
    NEED(int32(a[7], p.total_seqlen));
    NEED(int32(a[8], p.numseqs));
    NEED(int32(a[9], p.max_seqlen_all));
    p.softmax_scale = (float)PyFloat_AsDouble(a[10]);
    NEED(int32(a[11], p.split_mode));
    NEED((p.prefix_lens = metadata(a[4], p.numseqs, q)) != nullptr);
    NEED((p.causal_lens = metadata(a[5], p.numseqs, q)) != nullptr);
    NEED((p.cu_seqlens = metadata(a[6], p.numseqs + 1, q)) != nullptr);
    p.total_tokens = (int32_t)g.T, p.num_q_heads = (int32_t)g.hq, p.num_kv_heads = (int32_t)g.hkv;
    p.head_dim = (int32_t)g.d, p.dtype = g.dtype;
    const bool bf16 = g.dtype == MIMIR_DTYPE_BFLOAT16;
    at::Tensor out = empty({g.T, g.hq, g.d}, q, q.scalar_type()), lse = empty({g.hq, g.T}, q, at::kFloat);
    at::Tensor lo = truth(a[13]) ? empty({g.T, g.hq, g.d}, q, q.scalar_type()) : empty({0}, q, q.scalar_type());
    at::Tensor flag = empty({bf16 ? 1 : 0}, q, at::kInt);
    p.q = q.const_data_ptr(), p.k = k.const_data_ptr(), p.v = v.const_data_ptr();
    p.out = out.mutable_data_ptr(), p.lse = (float*)lse.mutable_data_ptr();
    STRIDES(p, q, q), STRIDES(p, k, k), STRIDES(p, v, v), STRIDES(p, out, out);
    p.lse_stride_head = g.T;
    if (lo.numel() > 0) p.out_lo = lo.mutable_data_ptr(), STRIDES(p, out_lo, lo);
    if (bf16) p.split_flag = (int32_t*)flag.mutable_data_ptr();
    if (!is_none(a[14])) {
      TENSOR(gate, a[14]);
      TENSOR(gated, a[15]);
      NEED(shaped(gate, g.T, g.hq, g.d));
      NEED(shaped(gated, g.T, g.hq, g.d));
      NEED(in_place(gate, q));
      NEED(in_place(gated, q));
      p.gate = gate.const_data_ptr(), p.gated_out = gated.mutable_data_ptr();
      STRIDES(p, gate, gate), STRIDES(p, gated_out, gated);
    }
    p.workspace_bytes = truth(a[12]) ? lib.fwd_workspace_size(&p)
                                     : lib.fwd_workspace_bytes(p.total_tokens, p.numseqs, p.max_seqlen_all);
    at::Tensor ws = workspace(a[16], p.workspace_bytes, a[0]);
    NEED(ws.defined());
    p.workspace = ws.mutable_data_ptr();
    NEED(launch(lib.fwd, p, stream(a[17]), raised));
    return wrap({out, lse, lo, flag});
  });
}

// bwd(dout, q, k, v, out, lse, out_lo, split_flag, is_causal, prefix_lens, causal_lens, cu_seqlens, total_seqlen,
//     numseqs, max_seqlen_all, softmax_scale, split_mode, key_chunks, dscore_limit, region_limit, gate, grads,
//     torch_empty, stream) -> (dq, dk, dv)
// grads: None, or (dgate, dq, dk, dv) views to write.  A score-gradient region above
// region_limit needs the general path's look at the free memory.
PyObject* py_bwd(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded(n, 24, [&](bool& raised) -> PyObject* {
    TENSOR(dout, a[0]);
    TENSOR(q, a[1]);
    TENSOR(k, a[2]);
    TENSOR(v, a[3]);
    TENSOR(out, a[4]);
    TENSOR(lse, a[5]);
    TENSOR(lo, a[6]);
    TENSOR(flag, a[7]);
    Geometry g;
    NEED(geometry(q, k, v, g));
    NEED(shaped(dout, g.T, g.hq, g.d));
    NEED(shaped(out, g.T, g.hq, g.d));
    NEED(in_place(dout, q));
    NEED(in_place(out, q));
    NEED(lse.dim() == 2 && lse.size(0) == g.hq && lse.size(1) == g.T && lse.scalar_type() == at::kFloat &&
         lse.device() == q.device() && lse.is_contiguous());
    MimirPrefixLMBwdParams p = {};
    p.is_causal = truth(a[8]);
    NEED(int32(a[12], p.total_seqlen));
    NEED(int32(a[13], p.numseqs));
    NEED(int32(a[14], p.max_seqlen_all));
    p.softmax_scale = (float)PyFloat_AsDouble(a[15]);
    NEED(int32(a[16], p.split_mode));
    NEED((p.prefix_lens = metadata(a[9], p.numseqs, q)) != nullptr);
    NEED((p.causal_lens = metadata(a[10], p.numseqs, q)) != nullptr);
    NEED((p.cu_seqlens = metadata(a[11], p.numseqs + 1, q)) != nullptr);
    p.total_tokens = (int32_t)g.T, p.num_q_heads = (int32_t)g.hq, p.num_kv_heads = (int32_t)g.hkv;
    p.head_dim = (int32_t)g.d, p.dtype = g.dtype;
    at::Tensor dq, dk, dv;
    if (is_none(a[21])) {
      dq = empty({g.T, g.hq, g.d}, q, q.scalar_type());
      dk = empty({g.T, g.hkv, g.d}, q, q.scalar_type());
      dv = empty({g.T, g.hkv, g.d}, q, q.scalar_type());
    } else {
      NEED(PyTuple_Check(a[21]) && PyTuple_GET_SIZE(a[21]) == 4 && !is_none(a[20]));
      TENSOR(gate, a[20]);
      TENSOR(dgate, PyTuple_GET_ITEM(a[21], 0));
      TENSOR(dq_view, PyTuple_GET_ITEM(a[21], 1));
      TENSOR(dk_view, PyTuple_GET_ITEM(a[21], 2));
      TENSOR(dv_view, PyTuple_GET_ITEM(a[21], 3));
      dq = dq_view, dk = dk_view, dv = dv_view;
      NEED(shaped(gate, g.T, g.hq, g.d));
      NEED(shaped(dgate, g.T, g.hq, g.d));
      NEED(shaped(dq, g.T, g.hq, g.d));
      NEED(shaped(dk, g.T, g.hkv, g.d));
      NEED(shaped(dv, g.T, g.hkv, g.d));
      for (const at::Tensor* t : {&gate, &dgate, (const at::Tensor*)&dq, (const at::Tensor*)&dk, (const at::Tensor*)&dv})
        NEED(in_place(*t, q));
      p.gate = gate.const_data_ptr(), p.dgate = dgate.mutable_data_ptr();
      STRIDES(p, gate, gate), STRIDES(p, dgate, dgate);
    }
    p.q = q.const_data_ptr(), p.k = k.const_data_ptr(), p.v = v.const_data_ptr();
    p.out = out.const_data_ptr(), p.dout = dout.const_data_ptr(), p.lse = (const float*)lse.const_data_ptr();
    p.dq = dq.mutable_data_ptr(), p.dk = dk.mutable_data_ptr(), p.dv = dv.mutable_data_ptr();
    STRIDES(p, q, q), STRIDES(p, k, k), STRIDES(p, v, v), STRIDES(p, out, out), STRIDES(p, dout, dout);
    STRIDES(p, dq, dq), STRIDES(p, dk, dk), STRIDES(p, dv, dv);
    p.lse_stride_head = g.T;
    if (lo.numel() > 0) {
      NEED(shaped(lo, g.T, g.hq, g.d));
      NEED(in_place(lo, q));
      p.out_lo = lo.const_data_ptr(), STRIDES(p, out_lo, lo);
    }
    if (flag.numel() > 0) {
      NEED(flag.scalar_type() == at::kInt && flag.device() == q.device());
      p.split_flag = flag.const_data_ptr<int32_t>();
    }
    p.dq_key_chunks = truth(a[17]);
    p.dscore_limit_bytes = (size_t)PyLong_AsUnsignedLongLong(a[18]);
    if (p.dscore_limit_bytes > 0) NEED(lib.bwd_dscore_bytes(&p) <= (size_t)PyLong_AsUnsignedLongLong(a[19]));
    p.workspace_bytes = lib.bwd_workspace_size(&p);
    at::Tensor ws = workspace(a[22], p.workspace_bytes, a[1]);
    NEED(ws.defined());
    p.workspace = ws.mutable_data_ptr();
    NEED(launch(lib.bwd, p, stream(a[23]), raised));
    return wrap({dq, dk, dv});
  });
}

// rope(x, cos, sin, inverse, out_or_None, stream) -> out
PyObject* py_rope(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded(n, 6, [&](bool& raised) -> PyObject* {
    TENSOR(x, a[0]);
    TENSOR(cos, a[1]);
    TENSOR(sin, a[2]);
    NEED(on_device(x) && x.dim() == 3 && (x.scalar_type() == at::kBFloat16 || x.scalar_type() == at::kFloat));
    NEED(in_place(x, x));
    const int64_t T = x.size(0), d = x.size(2);
    NEED(T <= 0x7fffffff && x.size(1) > 0);
    for (const at::Tensor* t : {&cos, &sin})
      NEED(t->dim() == 2 && t->size(0) == T && t->size(1) == d && t->scalar_type() == at::kFloat &&
           t->device() == x.device() && t->stride(1) == 1 && t->stride(0) == cos.stride(0) && t->stride(0) % 4 == 0 &&
           (uintptr_t)t->const_data_ptr() % 16 == 0);
    at::Tensor out;
    if (is_none(a[4])) {
      out = empty({T, x.size(1), d}, x, x.scalar_type());
    } else {
      TENSOR(out_view, a[4]);
      out = out_view;
      NEED(shaped(out, T, x.size(1), d));
      NEED(in_place(out, x));
    }
    MimirRopeParams p = {};
    p.x = x.const_data_ptr(), p.y = out.mutable_data_ptr();
    p.cos = cos.const_data_ptr<float>(), p.sin = sin.const_data_ptr<float>();
    p.x_stride_token = x.stride(0), p.x_stride_head = x.stride(1);
    p.y_stride_token = out.stride(0), p.y_stride_head = out.stride(1);
    p.cs_stride_token = cos.stride(0);
    p.total_tokens = (int32_t)T, p.num_heads = (int32_t)x.size(1), p.head_dim = (int32_t)d;
    p.dtype = x.scalar_type() == at::kBFloat16 ? MIMIR_DTYPE_BFLOAT16 : MIMIR_DTYPE_FLOAT32;
    p.inverse = truth(a[3]);
    NEED(launch(lib.rope, p, stream(a[5]), raised));
    return THPVariable_Wrap(out);
  });
}

// cache_attn(query, key, value, cache_keys, cache_values, cache_lengths, causal, batch_indices, softmax_scale,
//            torch_empty, stream) -> out
PyObject* py_cache_attn(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded(n, 11, [&](bool& raised) -> PyObject* {
    TENSOR(q, a[0]);
    TENSOR(k, a[1]);
    TENSOR(v, a[2]);
    TENSOR(ck, a[3]);
    TENSOR(cv, a[4]);
    TENSOR(lens, a[5]);
    NEED(on_device(q) && q.scalar_type() == at::kBFloat16 && q.dim() == 4 && k.dim() == 4 && v.dim() == 4 &&
         ck.dim() == 4 && cv.dim() == 4);
    const int64_t B = q.size(0), S = q.size(1), hq = q.size(2), d = q.size(3), hkv = k.size(2), L = ck.size(1);
    NEED(B > 0 && S > 0 && hq > 0 && hkv > 0 && hq % hkv == 0 && L > 0 && B <= 0x7fffffff && S <= 0x7fffffff &&
         L <= 0x7fffffff && ck.size(0) <= 0x7fffffff);
    for (const at::Tensor* t : {&k, &v}) NEED(t->size(0) == B && t->size(1) == S && t->size(2) == hkv && t->size(3) == d);
    for (const at::Tensor* t : {&ck, &cv}) NEED(t->size(2) == hkv && t->size(3) == d && t->sizes() == ck.sizes());
    for (const at::Tensor* t : {&q, &k, &v, &ck, &cv}) NEED(in_place(*t, q));
    MimirCacheAttnParams p = {};
    for (PyObject* o : {a[5], a[7]}) {
      if (is_none(o)) continue;
      TENSOR(t, o);
      NEED(t.dim() == 1 && t.size(0) == B && t.device() == q.device() && t.is_contiguous() &&
           t.scalar_type() == lens.scalar_type() && (t.scalar_type() == at::kLong || t.scalar_type() == at::kInt));
    }
    p.cache_lengths = lens.const_data_ptr();
    if (!is_none(a[7])) p.batch_indices = tensor(a[7])->const_data_ptr();
    p.index_int64 = lens.scalar_type() == at::kLong;
    at::Tensor out = empty({B, S, hq, d}, q, at::kBFloat16);
    p.q = q.const_data_ptr(), p.k_new = k.const_data_ptr(), p.v_new = v.const_data_ptr();
    p.cache_k = ck.mutable_data_ptr(), p.cache_v = cv.mutable_data_ptr(), p.out = out.mutable_data_ptr();
#define STRIDES4(name, t) p.name##_stride_batch = (t).stride(0), p.name##_stride_token = (t).stride(1), p.name##_stride_head = (t).stride(2)
    STRIDES4(q, q), STRIDES4(kn, k), STRIDES4(vn, v), STRIDES4(ck, ck), STRIDES4(cv, cv), STRIDES4(out, out);
    p.batch = (int32_t)B, p.seqlen = (int32_t)S, p.cache_len = (int32_t)L, p.cache_rows = (int32_t)ck.size(0);
    p.max_kv_len = (int32_t)L, p.num_q_heads = (int32_t)hq, p.num_kv_heads = (int32_t)hkv, p.head_dim = (int32_t)d;
    p.causal = truth(a[6]);
    p.dtype = MIMIR_DTYPE_BFLOAT16;
    p.softmax_scale = (float)PyFloat_AsDouble(a[8]);
    p.workspace_bytes = lib.cache_workspace(&p);
    at::Tensor ws;
    if (p.workspace_bytes > 0) {
      ws = workspace(a[9], p.workspace_bytes, a[0]);
      NEED(ws.defined());
      p.workspace = ws.mutable_data_ptr();
    }
    NEED(launch(lib.cache_attn, p, stream(a[10]), raised));
    return THPVariable_Wrap(out);
  });
}

// bind(path, device="cuda"): the entry points of the (already loaded) C-ABI library, and
// the type of device whose tensors it takes.
PyObject* py_bind(PyObject*, PyObject* args) {
  const char *file, *device = "cuda";
  if (!PyArg_ParseTuple(args, "s|s", &file, &device)) return nullptr;
  try {
    lib.device = c10::Device(device).type();
  } catch (const std::exception&) {
    return PyErr_Format(PyExc_ValueError, "device %s", device);
  }
  void* h = dlopen(file, RTLD_NOW | RTLD_LOCAL);
  if (h == nullptr) return PyErr_Format(PyExc_ImportError, "%s", dlerror());
  bool ok = true;
  auto get = [&](auto& f, const char* name) {
    f = (std::remove_reference_t<decltype(f)>)dlsym(h, name);
    ok = ok && f != nullptr;
  };
  get(lib.fwd, "mimir_prefixlm_fwd");
  get(lib.fwd_workspace_size, "mimir_prefixlm_fwd_workspace_size");
  get(lib.fwd_workspace_bytes, "mimir_prefixlm_fwd_workspace_bytes");
  get(lib.bwd, "mimir_prefixlm_bwd");
  get(lib.bwd_workspace_size, "mimir_prefixlm_bwd_workspace_size");
  get(lib.bwd_dscore_bytes, "mimir_prefixlm_bwd_dscore_bytes");
  get(lib.rope, "mimir_prefixlm_rope");
  get(lib.cache_attn, "mimir_prefixlm_cache_attn");
  get(lib.cache_workspace, "mimir_prefixlm_cache_attn_workspace_bytes");
  get(lib.last_error, "mimir_prefixlm_last_error");
  if (!ok) return PyErr_Format(PyExc_ImportError, "%s lacks an entry point", file);
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", py_bind, METH_VARARGS, nullptr},
    {"fwd", (PyCFunction)(void*)py_fwd, METH_FASTCALL, nullptr},
    {"bwd", (PyCFunction)(void*)py_bwd, METH_FASTCALL, nullptr},
    {"rope", (PyCFunction)(void*)py_rope, METH_FASTCALL, nullptr},
    {"cache_attn", (PyCFunction)(void*)py_cache_attn, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host_calls", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__host_calls() {
  PyObject* m = PyModule_Create(&module);
  if (m != nullptr) PyModule_AddStringConstant(m, "built_for", MIMIR_BUILT_FOR);
  return m;
}
