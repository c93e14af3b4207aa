// Native front end of the per-layer kernels: the argument checks, output
// allocation and C-ABI call of one `nanovllm_amd.kernels` function in one
// CPython call.
//
// What bounds it: nothing on the GPU.  A layer makes nine kernel calls, and in
// Python each cost ~20 us of attribute reads, ctypes conversions (up to 34
// arguments) and stream look-ups, ~60 us while a torch default device is set
// (every attribute read and torch call then goes through a Python mode): a
// 1024-token prompt through Qwen3-0.6B's 28 layers took 8.8 ms for 3.3 ms of
// GPU work.  Here a call costs 2-4 us.
//
// Every function returns None, having done nothing, for any argument that is
// not of the ordinary form (exact tensors with storage on one GPU, the dtypes,
// strides and shapes the kernels take, a workspace that is large enough), for
// a refused launch and for any exception; the Python function that called it
// then runs its general path, which accepts the other forms or raises.
#include <Python.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/autocast_mode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/PyInterpreter.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <limits>

#include "nanovllm_amd.h"

namespace {

PyObject* g_current_device = nullptr;   // torch._C._cuda_getDevice
PyObject* g_raw_stream = nullptr;       // torch._C._cuda_getCurrentRawStream

// Thrown by the helpers for a form that the general path has to take.
struct Other {};

struct Args {
  PyObject* const* v;
  int64_t device = -1;      // of the tensors seen so far

  const at::Tensor& any(int i) const {
    if (!THPVariable_CheckExact(v[i])) throw Other{};
    const at::Tensor& t = THPVariable_Unpack(v[i]);
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || !t.has_storage()) throw Other{};
    return t;
  }
  const at::Tensor& tensor(int i) {
    const at::Tensor& t = any(i);
    const int64_t d = t.device().index();
    if (device >= 0 && d != device) throw Other{};
    device = d;
    return t;
  }
  bool none(int i) const { return v[i] == Py_None; }
  int32_t i32(int i) const {
    if (!PyLong_CheckExact(v[i])) throw Other{};
    int overflow = 0;
    const long x = PyLong_AsLongAndOverflow(v[i], &overflow);
    if (overflow || x < std::numeric_limits<int32_t>::min() || x > std::numeric_limits<int32_t>::max())
      throw Other{};
    return static_cast<int32_t>(x);
  }
  float f32(int i) const {
    if (!PyFloat_CheckExact(v[i])) throw Other{};
    return static_cast<float>(PyFloat_AS_DOUBLE(v[i]));
  }
  // one-element float32 tensor or None
  const float* scale(int i) const {
    if (none(i)) return nullptr;
    const at::Tensor& t = any(i);
    need(t.scalar_type() == at::kFloat && t.numel() == 1);
    return static_cast<const float*>(t.data_ptr());
  }
  static void need(bool ok) {
    if (!ok) throw Other{};
  }
};

void need(bool ok) { Args::need(ok); }

void need_rows(const at::Tensor& t) {
  need(t.scalar_type() == at::kBFloat16 && t.dim() == 2 && t.stride(1) == 1);
}

void need_i32(const at::Tensor& t) { need(t.scalar_type() == at::kInt && t.is_contiguous()); }

int32_t as_i32(int64_t x) {
  need(x >= std::numeric_limits<int32_t>::min() && x <= std::numeric_limits<int32_t>::max());
  return static_cast<int32_t>(x);
}

at::Tensor empty_bf16(at::IntArrayRef sizes, const at::Tensor& like) {
  return at::empty(sizes, at::TensorOptions().dtype(at::kBFloat16).device(like.device()));
}

// The current stream of the current device, as the Python path takes it;
// `only` >= 0 leaves another current device to the general path.
void* current_stream(int64_t only = -1) {
  PyObject* dev = PyObject_CallNoArgs(g_current_device);
  if (dev && only >= 0 && PyLong_AsLongLong(dev) != only) {
    Py_DECREF(dev);
    throw Other{};
  }
  PyObject* s = dev ? PyObject_CallOneArg(g_raw_stream, dev) : nullptr;
  Py_XDECREF(dev);
  void* p = s ? PyLong_AsVoidPtr(s) : nullptr;
  Py_XDECREF(s);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    throw Other{};
  }
  return p;
}

struct WithoutGil {
  PyThreadState* state = PyEval_SaveThread();
  ~WithoutGil() { PyEval_RestoreThread(state); }
};

// Runs a C-ABI call without the interpreter lock (taken again also where `f`
// throws); a refused call is the general path's to report.
template <typename F>
void launch(F&& f) {
  int status;
  {
    WithoutGil free;
    status = f();
  }
  need(status == NVA_OK);
}

template <typename F>
PyObject* guarded(Py_ssize_t n, Py_ssize_t want, F&& f) {
  if (n != want) {
    PyErr_SetString(PyExc_TypeError, "wrong number of arguments");
    return nullptr;
  }
  try {
    return f();
  } catch (...) {   // Other, and whatever the general path will raise again
    PyErr_Clear();
    Py_RETURN_NONE;
  }
}

struct Pages {
  int kv_dtype;
  void *k, *v;
  int64_t blk, tok, head;
  int32_t num_blocks, block_size, hkv, d;
};

Pages pages(Args& a, int ki, int vi) {
  const at::Tensor& k = a.tensor(ki);
  const at::Tensor& v = a.tensor(vi);
  need(k.dim() == 4 && k.sizes() == v.sizes() && k.strides() == v.strides() && k.stride(3) == 1 &&
       k.scalar_type() == v.scalar_type());
  Pages p;
  if (k.scalar_type() == at::kBFloat16)
    p.kv_dtype = NVA_KV_BF16;
  else if (k.scalar_type() == at::kFloat8_e4m3fn)
    p.kv_dtype = NVA_KV_FP8_E4M3;
  else
    throw Other{};
  p.k = k.data_ptr();
  p.v = v.data_ptr();
  p.blk = k.stride(0);
  p.tok = k.stride(1);
  p.head = k.stride(2);
  p.num_blocks = as_i32(k.size(0));
  p.block_size = as_i32(k.size(1));
  p.hkv = as_i32(k.size(2));
  p.d = as_i32(k.size(3));
  return p;
}

// The device's buffer in a {device index: uint8 tensor} dict, if it holds
// `bytes`; nothing is needed for 0 bytes.
struct Workspace {
  void* ptr = nullptr;
  size_t bytes = 0;
};
Workspace workspace(PyObject* bufs, int64_t device, size_t bytes) {
  Workspace w;
  if (bytes == 0) return w;
  need(PyDict_CheckExact(bufs));
  PyObject* key = PyLong_FromLongLong(device);
  PyObject* buf = key ? PyDict_GetItemWithError(bufs, key) : nullptr;   // borrowed
  Py_XDECREF(key);
  need(buf && THPVariable_CheckExact(buf));
  const at::Tensor& t = THPVariable_Unpack(buf);
  need(static_cast<size_t>(t.numel()) >= bytes);
  w.ptr = t.data_ptr();
  w.bytes = static_cast<size_t>(t.numel());
  return w;
}

// ---------------------------------------------------------------- functions

// (x, weight, eps, out | None) -> out
PyObject* rms_norm(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded(n, 4, [&]() -> PyObject* {
    Args a{v};
    const at::Tensor& x = a.tensor(0);
    const at::Tensor& w = a.tensor(1);
    need_rows(x);
    const int32_t rows = as_i32(x.size(0)), h = as_i32(x.size(1));
    need(w.numel() == h);
    at::Tensor out;
    if (a.none(3)) {
      out = empty_bf16({rows, h}, x);
    } else {
      out = a.tensor(3);
      need_rows(out);
      need(out.size(0) == rows && out.size(1) == h);
    }
    const float eps = a.f32(2);
    void* s = current_stream();
    launch([&] {
      return nva_rms_norm(x.data_ptr(), x.stride(0), w.data_ptr(), out.data_ptr(), out.stride(0), rows,
                          h, eps, s);
    });
    return THPVariable_Wrap(out);
  });
}

// (x, residual, weight, eps) -> (normed, sum)
template <bool THEN>
PyObject* add_rms_norm(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded(n, 4, [&]() -> PyObject* {
    Args a{v};
    const at::Tensor& x = a.tensor(0);
    const at::Tensor& r = a.tensor(1);
    const at::Tensor& w = a.tensor(2);
    need_rows(x);
    need_rows(r);
    need(x.sizes() == r.sizes() && w.numel() == x.size(1));
    const float eps = a.f32(3);
    const int32_t rows = as_i32(x.size(0)), h = as_i32(x.size(1));
    at::Tensor out = empty_bf16({rows, h}, x), sum = empty_bf16({rows, h}, x);
    void* s = current_stream();
    auto* fn = THEN ? nva_add_then_rms_norm : nva_add_rms_norm;
    launch([&] {
      return fn(x.data_ptr(), x.stride(0), r.data_ptr(), r.stride(0), w.data_ptr(), out.data_ptr(),
                h, sum.data_ptr(), h, rows, h, eps, s);
    });
    PyObject* o = THPVariable_Wrap(out);
    PyObject* t = THPVariable_Wrap(sum);
    PyObject* both = PyTuple_Pack(2, o, t);
    Py_XDECREF(o);
    Py_XDECREF(t);
    return both;
  });
}

// (x) -> out
PyObject* silu_mul(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded(n, 1, [&]() -> PyObject* {
    Args a{v};
    const at::Tensor& x = a.tensor(0);
    need_rows(x);
    const int32_t rows = as_i32(x.size(0)), inter = as_i32(x.size(1) / 2);
    at::Tensor out = empty_bf16({rows, inter}, x);
    void* s = current_stream();
    launch([&] {
      return nva_silu_mul(x.data_ptr(), x.stride(0), out.data_ptr(), inter, rows, inter, s);
    });
    return THPVariable_Wrap(out);
  });
}

// (qkv, positions, q_norm | None, k_norm | None, cos_sin, hq, hkv, d, eps, k_cache, v_cache,
//  slot_mapping, k_scale | None, v_scale | None) -> q
PyObject* qk_norm_rope_store(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded(n, 14, [&]() -> PyObject* {
    Args a{v};
    const at::Tensor& qkv = a.tensor(0);
    const at::Tensor& pos = a.tensor(1);
    const void* qw = a.none(2) ? nullptr : a.tensor(2).data_ptr();
    const void* kw = a.none(3) ? nullptr : a.tensor(3).data_ptr();
    const at::Tensor& cs = a.tensor(4);
    const int32_t hq = a.i32(5), hkv = a.i32(6), d = a.i32(7);
    const float eps = a.f32(8);
    const Pages p = pages(a, 9, 10);
    const at::Tensor& slots = a.tensor(11);
    const float* ks = a.scale(12);
    const float* vs = a.scale(13);
    need_rows(qkv);
    const int32_t t = as_i32(qkv.size(0));
    need(pos.scalar_type() == at::kLong && pos.is_contiguous() && pos.numel() == t);
    need(cs.scalar_type() == at::kFloat && cs.is_contiguous() && cs.dim() >= 1);
    const int32_t max_pos = as_i32(cs.size(0));
    need(p.hkv == hkv && p.d == d && hq >= 0 && hkv >= 0 && d >= 0);
    need(qkv.size(1) >= (static_cast<int64_t>(hq) + 2 * static_cast<int64_t>(hkv)) * d);
    need_i32(slots);
    need(slots.numel() == t);
    at::Tensor q = empty_bf16({t, hq, d}, qkv);
    void* s = current_stream();
    launch([&] {
      return nva_qk_norm_rope_store(
          qkv.data_ptr(), qkv.stride(0), static_cast<const int64_t*>(pos.data_ptr()), qw, kw,
          static_cast<const float*>(cs.data_ptr()), max_pos, t, hq, hkv, d, eps,
          q.data_ptr(), p.k, p.v, p.kv_dtype, p.blk, p.tok, p.head, p.num_blocks, p.block_size,
          static_cast<const int32_t*>(slots.data_ptr()), ks, vs, s);
    });
    return THPVariable_Wrap(q);
  });
}

// What the two attention entry points share.
struct Attention {
  Pages p;
  int32_t t, hq, bt_cols;
  at::Tensor out;
};
Attention attention(Args& a, const at::Tensor& q, int ki, int vi, const at::Tensor& bt, int out_i) {
  Attention r;
  r.p = pages(a, ki, vi);
  need(q.scalar_type() == at::kBFloat16 && q.dim() == 3 && q.stride(2) == 1 && q.size(2) == r.p.d &&
       r.p.hkv > 0 && q.size(1) % r.p.hkv == 0);
  need(bt.scalar_type() == at::kInt && bt.dim() == 2 && bt.stride(1) == 1);
  r.t = as_i32(q.size(0));
  r.hq = as_i32(q.size(1));
  r.bt_cols = as_i32(bt.size(1));
  if (a.none(out_i)) {
    r.out = empty_bf16(q.sizes(), q);
  } else {
    r.out = a.tensor(out_i);
    need(r.out.sizes() == q.sizes() && r.out.scalar_type() == at::kBFloat16 && r.out.stride(2) == 1);
  }
  return r;
}

// (q, k_cache, v_cache, cu_q, cu_k, max_q, max_k, softmax_scale, block_table, k_scale | None,
//  v_scale | None, out | None, workspaces) -> out
PyObject* paged_attention_varlen(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded(n, 13, [&]() -> PyObject* {
    Args a{v};
    const at::Tensor& q = a.tensor(0);
    const at::Tensor& cu_q = a.tensor(3);
    const at::Tensor& cu_k = a.tensor(4);
    const at::Tensor& bt = a.tensor(8);
    const int32_t max_q = a.i32(5), max_k = a.i32(6);
    const float scale = a.f32(7);
    const float* ks = a.scale(9);
    const float* vs = a.scale(10);
    need_i32(cu_q);
    need_i32(cu_k);
    const int32_t b = as_i32(cu_q.numel() - 1);
    const Attention r = attention(a, q, 1, 2, bt, 11);
    need(b >= 0 && cu_k.numel() == b + 1 && bt.size(0) >= b);
    const Workspace w = workspace(
        v[12], a.device,
        nva_paged_attention_workspace_size(b, r.t, r.hq, r.p.hkv, r.p.d, max_q, max_k));
    void* s = current_stream();
    launch([&] {
      return nva_paged_attention_varlen(
          q.data_ptr(), q.stride(0), q.stride(1), r.p.k, r.p.v, r.p.kv_dtype, r.p.blk, r.p.tok,
          r.p.head, r.p.num_blocks, r.p.block_size, static_cast<const int32_t*>(cu_q.data_ptr()),
          static_cast<const int32_t*>(cu_k.data_ptr()), static_cast<const int32_t*>(bt.data_ptr()),
          bt.stride(0), r.bt_cols, b, r.t, max_q, max_k, r.hq, r.p.hkv, r.p.d, scale, ks, vs,
          r.out.data_ptr(), r.out.stride(0), r.out.stride(1), w.ptr, w.bytes, s);
    });
    return THPVariable_Wrap(r.out);
  });
}

// (q, k_cache, v_cache, cache_seqlens, block_table, softmax_scale, max_k | None, k_scale | None,
//  v_scale | None, out | None, workspaces) -> out
PyObject* paged_attention_decode(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded(n, 11, [&]() -> PyObject* {
    Args a{v};
    const at::Tensor& q = a.tensor(0);
    const at::Tensor& lens = a.tensor(3);
    const at::Tensor& bt = a.tensor(4);
    const float scale = a.f32(5);
    const float* ks = a.scale(7);
    const float* vs = a.scale(8);
    need_i32(lens);
    const Attention r = attention(a, q, 1, 2, bt, 9);
    need(lens.numel() == r.t && bt.size(0) >= r.t);
    const int32_t max_k = a.none(6) ? as_i32(int64_t{r.bt_cols} * r.p.block_size) : a.i32(6);
    const Workspace w = workspace(
        v[10], a.device,
        nva_paged_attention_workspace_size(r.t, r.t, r.hq, r.p.hkv, r.p.d, 1, max_k));
    void* s = current_stream();
    launch([&] {
      return nva_paged_attention_decode(
          q.data_ptr(), q.stride(0), q.stride(1), r.p.k, r.p.v, r.p.kv_dtype, r.p.blk, r.p.tok,
          r.p.head, r.p.num_blocks, r.p.block_size, static_cast<const int32_t*>(lens.data_ptr()),
          static_cast<const int32_t*>(bt.data_ptr()), bt.stride(0), r.bt_cols, r.t, max_k,
          r.hq, r.p.hkv, r.p.d, scale, ks, vs, r.out.data_ptr(), r.out.stride(0), r.out.stride(1),
          w.ptr, w.bytes, s);
    });
    return THPVariable_Wrap(r.out);
  });
}

// (logits, index_map | None, out | None, workspaces) -> tokens
PyObject* argmax_rows(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded(n, 4, [&]() -> PyObject* {
    Args a{v};
    const at::Tensor& x = a.tensor(0);
    need_rows(x);
    const int32_t rows = as_i32(x.size(0)), vocab = as_i32(x.size(1));
    const int64_t* map = nullptr;
    if (!a.none(1)) {
      const at::Tensor& m = a.tensor(1);
      need(m.scalar_type() == at::kLong && m.numel() == vocab && m.is_contiguous());
      map = static_cast<const int64_t*>(m.data_ptr());
    }
    at::Tensor out;
    if (a.none(2)) {
      out = at::empty({rows}, at::TensorOptions().dtype(at::kLong).device(x.device()));
    } else {
      out = a.tensor(2);
      need(out.scalar_type() == at::kLong && out.is_contiguous() && out.dim() == 1 &&
           out.numel() >= rows);
      if (out.numel() > rows) out = out.narrow(0, 0, rows);
    }
    const size_t bytes = nva_argmax_workspace_size(rows, 0, vocab);
    need(bytes > 0);
    const Workspace w = workspace(v[3], a.device, bytes);
    void* s = current_stream();
    launch([&] {
      return nva_argmax_rows(x.data_ptr(), x.stride(0), vocab, rows, map,
                             static_cast<int64_t*>(out.data_ptr()), w.ptr, w.bytes, s);
    });
    return THPVariable_Wrap(out);
  });
}

// Whether something watches or rewrites torch calls (a function mode other than
// the default device's, a dispatch mode, a tracer, autocast): those see the
// Python path's calls.
PyTypeObject* g_device_context = nullptr;   // torch.utils._device.DeviceContext
bool watched() {
  const int64_t modes = at::impl::PythonTorchFunctionTLS::stack_len();
  for (int64_t i = 0; i < modes; ++i)
    if (Py_TYPE(at::impl::PythonTorchFunctionTLS::get_stack_at(i)->ptr(getPyInterpreter())) !=
        g_device_context)
      return true;
  return c10::impl::TorchDispatchModeTLS::any_modes_set() || torch::jit::tracer::isTracing() ||
         at::autocast::is_autocast_enabled(at::kCUDA);
}

// (x, weight, bias | None) -> x weight^T + bias: few rows without a bias on the
// kernel of linear.hip, everything else the library's product
PyObject* linear(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded(n, 3, [&]() -> PyObject* {
    Args a{v};
    const at::Tensor& x = a.tensor(0);
    const at::Tensor& w = a.tensor(1);
    need(!watched() && !x._fw_grad(0).defined() && !w._fw_grad(0).defined());
    if (a.none(2) && x.dim() == 2 && w.dim() == 2 && x.scalar_type() == at::kBFloat16 &&
        w.scalar_type() == at::kBFloat16 && x.size(1) == w.size(1) && x.stride(1) == 1 &&
        w.is_contiguous() && x.size(0) <= 64 &&
        !(at::GradMode::is_enabled() && (x.requires_grad() || w.requires_grad()))) {
      const int32_t rows = as_i32(x.size(0)), m = as_i32(w.size(0)), k = as_i32(x.size(1));
      if (nva_linear_preferred(rows, m, k) && x.stride(0) % 8 == 0 && x.stride(0) >= k &&
          reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0 &&
          reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 == 0) {
        void* s = current_stream(a.device);   // the library's product follows x's device
        at::Tensor out = empty_bf16({rows, m}, x);
        launch([&] {
          return nva_linear(x.data_ptr(), x.stride(0), w.data_ptr(), out.data_ptr(), m, rows, m, k, s);
        });
        return THPVariable_Wrap(out);
      }
    }
    at::Tensor out;
    {
      WithoutGil free;
      out = a.none(2) ? at::linear(x, w) : at::linear(x, w, a.any(2));
    }
    return THPVariable_Wrap(out);
  });
}

// (x [T, H, D]) -> its view [T, H * D]
PyObject* merge_heads(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded(n, 1, [&]() -> PyObject* {
    const at::Tensor& x = Args{v}.any(0);
    need(x.dim() == 3 && x.is_contiguous());
    return THPVariable_Wrap(x.view({x.size(0), x.size(1) * x.size(2)}));
  });
}

// (tensor) -> (device index, number of elements)
PyObject* place(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded(n, 1, [&]() -> PyObject* {
    const at::Tensor& x = Args{v}.any(0);
    return Py_BuildValue("(LL)", static_cast<long long>(x.device().index()),
                         static_cast<long long>(x.numel()));
  });
}

#define FAST(name, fn) {name, reinterpret_cast<PyCFunction>(fn), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    FAST("rms_norm", rms_norm),
    FAST("add_rms_norm", add_rms_norm<false>),
    FAST("add_then_rms_norm", add_rms_norm<true>),
    FAST("silu_mul", silu_mul),
    FAST("qk_norm_rope_store", qk_norm_rope_store),
    FAST("paged_attention_varlen", paged_attention_varlen),
    FAST("paged_attention_decode", paged_attention_decode),
    FAST("argmax_rows", argmax_rows),
    FAST("linear", linear),
    FAST("merge_heads", merge_heads),
    FAST("place", place),
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_front_end", nullptr, -1, methods};

}  // namespace

extern "C" __attribute__((visibility("default"))) PyObject* PyInit__front_end() {
  PyObject* torch_c = PyImport_ImportModule("torch._C");
  if (!torch_c) return nullptr;
  g_current_device = PyObject_GetAttrString(torch_c, "_cuda_getDevice");
  g_raw_stream = PyObject_GetAttrString(torch_c, "_cuda_getCurrentRawStream");
  Py_DECREF(torch_c);
  if (!g_current_device || !g_raw_stream) return nullptr;
  PyObject* device_module = PyImport_ImportModule("torch.utils._device");
  if (!device_module) return nullptr;
  g_device_context =
      reinterpret_cast<PyTypeObject*>(PyObject_GetAttrString(device_module, "DeviceContext"));
  Py_DECREF(device_module);
  if (!g_device_context) return nullptr;
  PyObject* m = PyModule_Create(&module);
  // what it was built against: the interpreter and torch whose ABI it uses
  if (m && (PyModule_AddIntConstant(m, "built_for_python", PY_VERSION_HEX >> 16) < 0 ||
            PyModule_AddStringConstant(m, "built_for_torch", NVA_TORCH_VERSION) < 0)) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
