// The call path from torch tensors to the C ABI (include/xmk.h): one CPython function per entry point,
// positional arguments only (the package's Python functions give them their names and defaults).
//
// What bounds it: nothing but host instructions.  Small products and attention shapes finish in less time
// than building a descriptor out of ctypes objects took (8-10 us per call through ctypes, of which the
// HIP launch itself is about 2): here a call reads sizes, strides and pointers straight from the tensors.
// The functions return the status code of the entry point (0: done), or their result.
//
// The kernels' library is bound at run time by path, so that this module has no state of its own besides
// the addresses of the entry points.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPStream.h>
#include <dlfcn.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/DynamicTypes.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>

#include "xmk.h"

namespace {

struct Api {
#define XMK_FUNCTIONS(F)                                                                                   \
  F(xmk_gemm) F(xmk_gemm_ws) F(xmk_gemm_qkv) F(xmk_fmha_fwd) F(xmk_fmha_bwd)   \
  F(xmk_fmha_bwd_workspace_bytes) F(xmk_fmha_bwd_best_workspace_bytes) F(xmk_fmha_decode) F(xmk_fmha_decode_static) F(xmk_int4_gemm)            \
  F(xmk_int4_gemm_ws) F(xmk_fp8_gemm_ex) F(xmk_gptj_decode_step)
#define XMK_DECLARE(name) decltype(&::name) name = nullptr;
  XMK_FUNCTIONS(XMK_DECLARE)
} api;

// Thrown after a Python exception has been set.
struct Raised {};

[[noreturn]] void raise(PyObject* type, const char* text) {
  PyErr_SetString(type, text);
  throw Raised{};
}

void need(Py_ssize_t got, Py_ssize_t want) {
  if (got != want) raise(PyExc_TypeError, "wrong number of arguments");
  if (!api.xmk_gemm) raise(PyExc_RuntimeError, "the kernel library is not bound");
}

const at::Tensor& tensor(PyObject* o) {
  if (!THPVariable_Check(o)) raise(PyExc_TypeError, "a torch tensor is expected");
  return THPVariable_Unpack(o);
}
const at::Tensor* tensor_or_null(PyObject* o) { return o == Py_None ? nullptr : &tensor(o); }
void* data(const at::Tensor& t) { return t.data_ptr(); }
void* data_or_null(PyObject* o) { return o == Py_None ? nullptr : data(tensor(o)); }

bool truth(PyObject* o) {
  if (o == Py_True) return true;
  if (o == Py_False || o == Py_None) return false;
  const int r = PyObject_IsTrue(o);
  if (r < 0) throw Raised{};
  return r != 0;
}
int64_t integer(PyObject* o) {
  const long long v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    PyObject* i = PyNumber_Index(o);  // numpy integers and the like
    if (!i) throw Raised{};
    const long long w = PyLong_AsLongLong(i);
    Py_DECREF(i);
    if (w == -1 && PyErr_Occurred()) throw Raised{};
    return w;
  }
  return v;
}
double real(PyObject* o) {
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) throw Raised{};
  return v;
}
void* address(PyObject* o) {
  void* p = PyLong_AsVoidPtr(o);
  if (!p && PyErr_Occurred()) throw Raised{};
  return p;
}

// None: torch's current stream on the current device.
void* stream(PyObject* o) {
  if (o == Py_None) return c10::hip::getCurrentHIPStream().stream();
  PyObject* s = PyObject_GetAttrString(o, "cuda_stream");
  if (!s) throw Raised{};
  void* p = PyLong_AsVoidPtr(s);
  Py_DECREF(s);
  if (!p && PyErr_Occurred()) throw Raised{};
  return p;
}

int32_t dtype_code(const at::Tensor& t) {
  switch (t.scalar_type()) {
    case at::kHalf: return XMK_F16;
    case at::kBFloat16: return XMK_BF16;
    case at::kFloat: return XMK_F32;
    case at::kFloat8_e4m3fn: return XMK_F8E4M3FN;
    case at::kChar: return XMK_S8;
    case at::kInt: return XMK_S32;
    default: PyErr_SetObject(PyExc_KeyError, (PyObject*)torch::getTHPDtype(t.scalar_type())); throw Raised{};
  }
}

int64_t dim(const at::Tensor& t, int64_t d) {
  if (d >= t.dim()) raise(PyExc_IndexError, "a tensor has too few dimensions");
  return t.sizes()[d];
}

// A 2-D (or batched 3-D) row-major tensor as an xmk_matrix.
xmk_matrix matrix(const at::Tensor& t, bool transpose) {
  const int64_t n = t.dim();
  if (n < 2) raise(PyExc_IndexError, "a matrix has at least two dimensions");
  return xmk_matrix{data(t), transpose, t.sizes()[n - 2], t.sizes()[n - 1], n == 3 ? t.strides()[0] : 0, t.strides()[n - 2]};
}

// Runs `call` without the interpreter lock.
template <class F>
auto unlocked(F&& call) {
  PyThreadState* state = PyEval_SaveThread();
  const auto r = call();
  PyEval_RestoreThread(state);
  return r;
}

template <class F>
PyObject* guarded(F&& body) {
  try {
    return body();
  } catch (const Raised&) {
    return nullptr;
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
}

PyObject* bind(PyObject*, PyObject* path) {
  return guarded([&]() -> PyObject* {
    const char* name = PyUnicode_AsUTF8(path);
    if (!name) throw Raised{};
    void* lib = dlopen(name, RTLD_NOW | RTLD_LOCAL);
    if (!lib) raise(PyExc_OSError, dlerror());
    Api a;
#define XMK_RESOLVE(name) \
  if (!(a.name = (decltype(a.name))dlsym(lib, #name))) raise(PyExc_OSError, "the kernel library lacks " #name);
    XMK_FUNCTIONS(XMK_RESOLVE)
    api = a;
    Py_RETURN_NONE;
  });
}

#define XMK_PY(name) PyObject* name(PyObject*, PyObject* const* a, Py_ssize_t n)

// (lhs, rhs, out, lhs_transpose, rhs_transpose, out_transpose, c, bias, alpha, beta, epilogue, stream, workspace)
XMK_PY(gemm) {
  return guarded([&]() -> PyObject* {
    need(n, 13);
    const at::Tensor &lhs = tensor(a[0]), &rhs = tensor(a[1]), &out = tensor(a[2]);
    xmk_gemm_desc d;
    d.lhs = matrix(lhs, truth(a[3]));
    d.rhs = matrix(rhs, truth(a[4]));
    d.out = matrix(out, truth(a[5]));
    d.c = data_or_null(a[6]);
    d.bias = data_or_null(a[7]);
    d.dtype_in = dtype_code(lhs);
    d.dtype_out = dtype_code(out);
    d.batch_size = lhs.dim() == 3 ? lhs.sizes()[0] : 1;
    d.alpha = (float)real(a[8]);
    d.beta = (float)real(a[9]);
    d.epilogue = (int32_t)integer(a[10]);
    void* st = stream(a[11]);
    const at::Tensor* ws = tensor_or_null(a[12]);
    void* scratch = ws ? data(*ws) : nullptr;
    const size_t bytes = ws ? ws->numel() * ws->element_size() : 0;
    return PyLong_FromLong(unlocked([&] { return ws ? api.xmk_gemm_ws(&d, scratch, bytes, st) : api.xmk_gemm(&d, st); }));
  });
}

// (lhs, weights, out_q, out_k, out_v, rhs_transpose, bias, epilogue, stream)
XMK_PY(gemm_qkv) {
  return guarded([&]() -> PyObject* {
    need(n, 9);
    const at::Tensor &lhs = tensor(a[0]), &w = tensor(a[1]), &out = tensor(a[2]);
    if (w.dim() != 3) raise(PyExc_IndexError, "the three weights are stacked in one tensor of three dimensions");
    xmk_gemm_desc d;
    d.lhs = matrix(lhs, false);
    d.rhs = matrix(w, truth(a[5]));
    d.out = matrix(out, false);
    d.c = nullptr;
    d.bias = data_or_null(a[6]);
    d.dtype_in = dtype_code(lhs);
    d.dtype_out = dtype_code(out);
    d.batch_size = 1;
    d.alpha = 1.0f;
    d.beta = 0.0f;
    d.epilogue = (int32_t)integer(a[7]);
    void *k = data_or_null(a[3]), *v = data_or_null(a[4]), *st = stream(a[8]);
    return PyLong_FromLong(unlocked([&] { return api.xmk_gemm_qkv(&d, k, v, st); }));
  });
}

struct Attention {
  uint32_t b, n, f, t, h;
  float scale;
};
Attention attention(const at::Tensor& q, const at::Tensor& k, PyObject* head_scale) {
  Attention s;
  s.b = (uint32_t)dim(q, 0); s.n = (uint32_t)dim(q, 1); s.f = (uint32_t)dim(q, 2); s.h = (uint32_t)dim(q, 3);
  s.t = (uint32_t)dim(k, 2);
  s.scale = (float)(head_scale == Py_None ? std::pow((double)s.h, -0.5) : real(head_scale));
  return s;
}

// (query, key, value, out, bias, lse, head_scale, causal, stream)
XMK_PY(fmha_forward) {
  return guarded([&]() -> PyObject* {
    need(n, 9);
    const at::Tensor &q = tensor(a[0]), &k = tensor(a[1]);
    const Attention s = attention(q, k, a[6]);
    void *v = data(tensor(a[2])), *o = data(tensor(a[3])), *bias = data_or_null(a[4]), *lse = data_or_null(a[5]);
    const int32_t dt = dtype_code(q), causal = truth(a[7]);
    void* st = stream(a[8]);
    return PyLong_FromLong(unlocked([&] {
      return api.xmk_fmha_fwd(data(q), data(k), v, bias, o, (float*)lse, dt, s.b, s.n, s.h, s.f, s.t, s.scale, causal, st);
    }));
  });
}

// Whether `bytes` of scratch that a call can do without are to be asked for: the allocator holds that much in whole unused
// segments, or the device has twice as much left.  A request that fails is no answer to that: torch then gives back every
// cached block and waits for the device, in each such call of a program whose memory is nearly full.  Under stream capture
// nothing is queried (the memory is the graph's, and asked for once).
bool spare_memory(const at::Tensor& like, int64_t bytes, void* st) {
  if (!like.is_cuda()) return false;
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing((hipStream_t)st, &capture) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  if (capture != hipStreamCaptureStatusNone) return true;
  try {
    const auto stats = c10::hip::HIPCachingAllocator::getDeviceStats(like.get_device());
    auto now = [](const c10::CachingDeviceAllocator::StatArray& of) { return of[0].current; };  // (0: all pools)
    if (now(stats.reserved_bytes) - now(stats.active_bytes) - now(stats.inactive_split_bytes) >= bytes) return true;
  } catch (const c10::Error&) {  // an allocator of the program's own, which keeps no such count
  }
  const c10::DeviceGuard on(like.device());
  size_t left = 0, total = 0;
  if (hipMemGetInfo(&left, &total) == hipSuccess) return left / 2 >= (size_t)bytes;
  (void)hipGetLastError();
  return false;
}

// (query, key, value, out, grad_out, lse, bias, head_scale, causal, stream) -> (dq, dk, dv), or the status code
XMK_PY(fmha_backward) {
  return guarded([&]() -> PyObject* {
    need(n, 10);
    const at::Tensor &q = tensor(a[0]), &k = tensor(a[1]), &v = tensor(a[2]);
    const Attention s = attention(q, k, a[7]);
    void *o = data(tensor(a[3])), *d_o = data(tensor(a[4])), *lse = data(tensor(a[5])), *bias = data_or_null(a[6]);
    const int32_t dt = dtype_code(q), causal = truth(a[8]);
    void* st = stream(a[9]);
    // The gradients first: what the call can do without must not take their memory.  Where memory is short, the least scratch.
    const at::Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v);
    size_t bytes = api.xmk_fmha_bwd_workspace_bytes(s.b, s.n, s.h, s.f, s.t);
    const size_t best = bias ? bytes : api.xmk_fmha_bwd_best_workspace_bytes(s.b, s.n, s.h, s.f, s.t, causal);
    auto scratch = [&](size_t size) { return at::empty({(int64_t)(size > 256 ? size : 256)}, q.options().dtype(at::kByte)); };
    at::Tensor ws;
    if (best > bytes && spare_memory(q, (int64_t)best, st)) {
      try {
        ws = scratch(best);
        bytes = best;
      } catch (const c10::OutOfMemoryError&) {
      }
    }
    if (!ws.defined()) ws = scratch(bytes);
    const int rc = unlocked([&] {
      return api.xmk_fmha_bwd(data(q), data(k), data(v), bias, o, d_o, (const float*)lse, data(dq), data(dk), data(dv), dt, s.b,
                              s.n, s.h, s.f, s.t, s.scale, causal, data(ws), bytes, st);
    });
    if (rc != XMK_OK) return PyLong_FromLong(rc);
    return Py_BuildValue("(NNN)", THPVariable_Wrap(dq), THPVariable_Wrap(dk), THPVariable_Wrap(dv));
  });
}

// What both decode calls share: their arguments are a[0 .. 3] and a[rest ..].
struct Decode {
  const at::Tensor &q, &k;
  uint32_t b, heads, h, t;
  int64_t stride;
  float scale;
  void *v, *o;
  int32_t dtype;
  void* st;
};
// (query, key, value, out, ..., num_keys, kv_head_stride, head_scale, stream)
Decode decode(PyObject* const* a, int rest) {
  const at::Tensor &q = tensor(a[0]), &k = tensor(a[1]);
  const uint32_t b = (uint32_t)dim(q, 0), heads = (uint32_t)dim(q, 1), h = (uint32_t)dim(q, q.dim() - 1);
  PyObject *keys = a[rest], *head_stride = a[rest + 1], *head_scale = a[rest + 2];
  const uint32_t t = (uint32_t)(keys == Py_None ? dim(k, 2) : integer(keys));
  if (k.dim() < 2) raise(PyExc_IndexError, "a tensor has too few dimensions");
  const int64_t stride = head_stride == Py_None ? k.strides()[1] : integer(head_stride);
  const float scale = (float)(head_scale == Py_None ? std::pow((double)h, -0.5) : real(head_scale));
  return Decode{q, k, b, heads, h, t, stride, scale, data(tensor(a[2])), data(tensor(a[3])), dtype_code(q), stream(a[rest + 3])};
}

// (query, key, value, out, workspace, num_keys, kv_head_stride, head_scale, stream).  The workspace is a tensor: a call without
// one would have to run on the array that calls on other streams may be using (fmha_decode_static).
XMK_PY(fmha_decode) {
  return guarded([&]() -> PyObject* {
    need(n, 9);
    const at::Tensor& ws = tensor(a[4]);
    const Decode d = decode(a, 5);
    void* scratch = data(ws);
    const size_t bytes = ws.numel() * ws.element_size();
    return PyLong_FromLong(unlocked([&] {
      return api.xmk_fmha_decode(data(d.q), data(d.k), d.v, d.o, d.dtype, d.b, d.heads, d.h, d.t, d.stride, d.scale, scratch, bytes, d.st);
    }));
  });
}

// (query, key, value, out, num_keys, kv_head_stride, head_scale, stream)
XMK_PY(fmha_decode_static) {
  return guarded([&]() -> PyObject* {
    need(n, 8);
    const Decode d = decode(a, 4);
    return PyLong_FromLong(unlocked([&] {
      return api.xmk_fmha_decode_static(data(d.q), data(d.k), d.v, d.o, d.dtype, d.b, d.heads, d.h, d.t, d.stride, d.scale, d.st);
    }));
  });
}

// (act, qweight, scales, zeros, out, workspace or None, group, bias, stream)
XMK_PY(int4_gemm) {
  return guarded([&]() -> PyObject* {
    need(n, 9);
    const at::Tensor &act = tensor(a[0]), &qw = tensor(a[1]);
    if (act.dim() != 2) raise(PyExc_ValueError, "act has two dimensions");
    const int64_t m = dim(act, 0), k = dim(act, 1), cols = dim(qw, 1), group = integer(a[6]);
    void *s = data(tensor(a[2])), *z = data(tensor(a[3])), *o = data(tensor(a[4])), *bias = data_or_null(a[7]);
    const at::Tensor* ws = tensor_or_null(a[5]);
    void* scratch = ws ? data(*ws) : nullptr;
    const size_t bytes = ws ? ws->numel() * ws->element_size() : 0;
    void* st = stream(a[8]);
    return PyLong_FromLong(unlocked([&] {
      return ws ? api.xmk_int4_gemm_ws(data(act), data(qw), s, z, bias, o, m, k, cols, group, scratch, bytes, st)
                : api.xmk_int4_gemm(data(act), data(qw), s, z, bias, o, m, k, cols, group, st);
    }));
  });
}

// (a, b, a_scale, b_scale, out, rhs_transpose, d_scale, bias, stream)
XMK_PY(fp8_gemm) {
  return guarded([&]() -> PyObject* {
    need(n, 9);
    const at::Tensor &x = tensor(a[0]), &w = tensor(a[1]);
    if (x.dim() != 2) raise(PyExc_ValueError, "a has two dimensions");
    const bool rhs_t = truth(a[5]);
    const int64_t m = dim(x, 0), k = dim(x, 1), cols = dim(w, rhs_t ? 0 : 1);
    void *sa = data(tensor(a[2])), *sb = data(tensor(a[3])), *o = data(tensor(a[4])), *sd = data_or_null(a[6]), *bias = data_or_null(a[7]);
    void* st = stream(a[8]);
    return PyLong_FromLong(unlocked([&] {
      return api.xmk_fp8_gemm_ex(data(x), data(w), (const float*)sa, (const float*)sb, (const float*)sd, bias, o, m, cols, k, rhs_t, st);
    }));
  });
}

// (config address, layers address, ln_f gamma, ln_f beta, lm_head address, hidden_in, position, logits, workspace, stream)
XMK_PY(gptj_decode_step) {
  return guarded([&]() -> PyObject* {
    need(n, 10);
    const auto* cfg = (const xmk_gptj_config*)address(a[0]);
    const auto* layers = (const xmk_gptj_layer*)address(a[1]);
    const auto* head = (const xmk_int4_linear*)address(a[4]);
    void *gamma = data_or_null(a[2]), *beta = data_or_null(a[3]), *in = data_or_null(a[5]), *logits = data_or_null(a[7]);
    const int32_t position = (int32_t)integer(a[6]);
    const at::Tensor& ws = tensor(a[8]);
    void *scratch = data(ws), *st = stream(a[9]);
    const size_t bytes = ws.numel() * ws.element_size();
    return PyLong_FromLong(unlocked([&] {
      return api.xmk_gptj_decode_step(cfg, layers, gamma, beta, head, in, position, logits, scratch, bytes, st);
    }));
  });
}

#define XMK_METHOD(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {{"bind", bind, METH_O, nullptr},
                         XMK_METHOD(gemm),
                         XMK_METHOD(gemm_qkv),
                         XMK_METHOD(fmha_forward),
                         XMK_METHOD(fmha_backward),
                         XMK_METHOD(fmha_decode),
                         XMK_METHOD(fmha_decode_static),
                         XMK_METHOD(int4_gemm),
                         XMK_METHOD(fp8_gemm),
                         XMK_METHOD(gptj_decode_step),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_xmk_native", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__xmk_native(void) { return PyModule_Create(&module); }
