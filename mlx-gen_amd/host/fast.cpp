// fast.cpp — native call path of the Python operators (module mlxq._fast).
//
// A decode-sized call spends more host time in Python than its kernel takes on the GPU: shape and
// dtype checks, one ctypes conversion per argument and the stream object came to ~14 us a call,
// against 5-7 us of kernel.  Each function here takes the call whose operands need no preparation
// (GPU tensors of the expected ranks, shapes and dtypes, contiguous and aligned), allocates the
// result and calls the C ABI; for anything else, and for a call that the library refuses, it returns
// None and the caller's general path prepares the operands or reports the error.  A device error is
// raised from here: the launch that failed is not made a second time.  Nothing is kept from one call to
// the next.
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ATen.h>

#include <string.h>

#include <vector>

#include "../../include/mlxq.h"

namespace {

int code_of(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return MLXQ_FLOAT32;
    case at::kBFloat16: return MLXQ_BFLOAT16;
    case at::kHalf: return MLXQ_FLOAT16;
    default: return -1;
  }
}

at::ScalarType type_of(int code) { return code == MLXQ_BFLOAT16 ? at::kBFloat16 : at::kFloat; }

// A plain GPU tensor in row-major order whose data starts at a multiple of `align` bytes (a nested tensor
// calls itself strided and contiguous too, and is for the general path to refuse).
const at::Tensor* plain(PyObject* o, size_t align) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.is_cuda() || t.layout() != at::kStrided || t.is_nested()) return nullptr;
  if (!t.is_contiguous() || t.is_conj() || t.is_neg()) return nullptr;
  if (reinterpret_cast<uintptr_t>(t.data_ptr()) % align != 0) return nullptr;
  return &t;
}

struct Pack {  // owns its tensors: the caller's list may change while the lock is released
  at::Tensor wq, s, b;
  int64_t N;
  int dt;
};

bool get_pack(PyObject* wq, PyObject* s, PyObject* b, int64_t K, long gs, long bits, Pack& p) {
  if ((bits != 4 && bits != 8) || (gs != 32 && gs != 64 && gs != 128) || K <= 0 || K % gs != 0) return false;
  const at::Tensor *w = plain(wq, 16), *ps = plain(s, 4), *pb = plain(b, 4);
  if (!w || !ps || !pb || w->dim() != 2 || ps->dim() != 2 || pb->dim() != 2) return false;
  if (w->scalar_type() != at::kInt && w->scalar_type() != at::kUInt32) return false;
  p.N = w->size(0);
  p.dt = code_of(ps->scalar_type());
  if ((p.dt != MLXQ_BFLOAT16 && p.dt != MLXQ_FLOAT32) || pb->scalar_type() != ps->scalar_type()) return false;
  const int64_t G = K / gs;
  if (p.N <= 0 || w->size(1) * 32 != K * bits || ps->size(0) != p.N || ps->size(1) != G || pb->size(0) != p.N ||
      pb->size(1) != G)
    return false;
  p.wq = *w;
  p.s = *ps;
  p.b = *pb;
  return true;
}

// Activations [..., K] of at least one row.
const at::Tensor* get_x(PyObject* o, int64_t& M, int64_t& K, int& dt) {
  const at::Tensor* x = plain(o, 16);
  if (!x || x->dim() < 1) return nullptr;
  K = x->size(-1);
  dt = code_of(x->scalar_type());
  if (dt < 0 || K <= 0 || x->numel() == 0) return nullptr;
  M = x->numel() / K;
  return x;
}

at::Tensor result(const at::Tensor& x, int64_t N, int dt) {
  if (x.dim() == 2) return at::empty({x.size(0), N}, x.options().dtype(type_of(dt)));
  at::DimVector shape(x.sizes().begin(), x.sizes().end());
  shape.back() = N;
  return at::empty(shape, x.options().dtype(type_of(dt)));
}

// torch's query of a device's raw current stream, looked up when the module is loaded: a lookup on first
// use under a static's guard could yield the interpreter lock to a thread that then waits for the guard.
PyObject* g_stream_query = nullptr;

void* stream_of(const at::Tensor& t, bool& ok) {
  ok = false;
  PyObject* index = PyLong_FromLong(t.get_device());
  PyObject* r = index ? PyObject_CallOneArg(g_stream_query, index) : nullptr;
  Py_XDECREF(index);
  if (!r) return nullptr;
  void* st = PyLong_AsVoidPtr(r);
  Py_DECREF(r);
  ok = !PyErr_Occurred();
  return st;
}

// MlxqError, given by the Python side when it loads the module.
PyObject* g_error = nullptr;

// A status that no second attempt may hide, raised as MlxqError(status, message).
struct DeviceError {
  int rc;
};

void refuse(int rc) {
  if (rc != MLXQ_OK && rc != MLXQ_EINVAL && rc != MLXQ_EUNSUPPORTED) throw DeviceError{rc};
}

// Calls the library without the interpreter lock, as ctypes does; its last error is this thread's.
template <typename F>
int unlocked(F&& call) {
  PyThreadState* save = PyEval_SaveThread();
  const int rc = call();
  PyEval_RestoreThread(save);
  refuse(rc);
  return rc;
}

// Runs f with C++ exceptions turned into "take the general path", which meets and reports them.
template <typename F>
PyObject* guarded(F&& f) {
  try {
    if (PyObject* r = f()) return r;
  } catch (const DeviceError& e) {
    if (g_error) {
      PyErr_Clear();
      if (PyObject* v = PyObject_CallFunction(g_error, "is", e.rc, mlxq_last_error())) {
        PyErr_SetObject(g_error, v);
        Py_DECREF(v);
      }
      return nullptr;
    }
  } catch (...) {
  }
  PyErr_Clear();
  Py_RETURN_NONE;
}

bool ints(PyObject* const* a, int n, long* out) {
  for (int i = 0; i < n; ++i) {
    if (!PyLong_CheckExact(a[i])) return false;
    out[i] = PyLong_AsLong(a[i]);
  }
  return !PyErr_Occurred();
}

// quantized_matmul(x, wq, scales, biases, group_size, bits)
PyObject* quantized_matmul(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    int64_t M, K;
    int dt;
    long v[2];
    Pack p;
    if (n != 6 || !ints(a + 4, 2, v)) return nullptr;
    const at::Tensor* x = get_x(a[0], M, K, dt);
    if (!x || !get_pack(a[1], a[2], a[3], K, v[0], v[1], p)) return nullptr;
    bool ok;
    void* st = stream_of(*x, ok);
    if (!ok) return nullptr;
    at::Tensor y = result(*x, p.N, dt == MLXQ_BFLOAT16 && p.dt == MLXQ_BFLOAT16 ? MLXQ_BFLOAT16 : MLXQ_FLOAT32);
    if (unlocked([&] { return mlxq_quantized_matmul(x->data_ptr(), dt, M, K, (const uint32_t*)p.wq.data_ptr(), p.s.data_ptr(),
                              p.b.data_ptr(), p.dt, p.N, 1, (int)v[0], (int)v[1], y.data_ptr(), st); }) != MLXQ_OK)
      return nullptr;
    return THPVariable_Wrap(std::move(y));
  });
}

// linear(x, wq, scales, biases, group_size, bits, bias, lora_a, lora_b, lora_scale, activation)
PyObject* linear(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    int64_t M, K;
    int dt;
    long v[2], act;
    Pack p;
    if (n != 11 || !ints(a + 4, 2, v) || !ints(a + 10, 1, &act)) return nullptr;
    const at::Tensor* x = get_x(a[0], M, K, dt);
    if (!x || !get_pack(a[1], a[2], a[3], K, v[0], v[1], p)) return nullptr;
    mlxq_epilogue ep = {};
    ep.activation = (int)act;
    ep.bias_dtype = ep.lora_dtype = dt;
    ep.lora_scale = (float)PyFloat_AsDouble(a[9]);
    if (PyErr_Occurred()) return nullptr;
    if (a[6] != Py_None) {
      const at::Tensor* bias = plain(a[6], 2);
      if (!bias || bias->dim() != 1 || bias->size(0) != p.N) return nullptr;
      ep.bias = bias->data_ptr();
      ep.bias_dtype = code_of(bias->scalar_type());
      if (ep.bias_dtype < 0) return nullptr;
    }
    if ((a[7] == Py_None) != (a[8] == Py_None)) return nullptr;
    if (a[7] != Py_None) {
      const at::Tensor *la = plain(a[7], 2), *lb = plain(a[8], 2);
      if (!la || !lb || la->dim() != 2 || lb->dim() != 2 || la->size(0) != K || lb->size(1) != p.N ||
          la->size(1) != lb->size(0) || la->scalar_type() != lb->scalar_type())
        return nullptr;
      ep.lora_a = la->data_ptr();
      ep.lora_b = lb->data_ptr();
      ep.lora_rank = la->size(1);
      ep.lora_dtype = code_of(la->scalar_type());
      if (ep.lora_dtype < 0) return nullptr;
    }
    const int odt = mlxq_linear_out_dtype(dt, p.dt, &ep);
    if (odt < 0) return nullptr;
    bool ok;
    void* st = stream_of(*x, ok);
    if (!ok) return nullptr;
    const size_t need = mlxq_linear_workspace_size(dt, p.dt, M, p.N, &ep);
    at::Tensor ws;
    if (need) ws = at::empty({(int64_t)need}, x->options().dtype(at::kByte));
    at::Tensor y = result(*x, p.N, odt);
    if (unlocked([&] { return mlxq_linear(x->data_ptr(), dt, M, K, (const uint32_t*)p.wq.data_ptr(), p.s.data_ptr(), p.b.data_ptr(), p.dt,
                    p.N, (int)v[0], (int)v[1], &ep, y.data_ptr(), need ? ws.data_ptr() : nullptr, need, st); }) != MLXQ_OK)
      return nullptr;
    return THPVariable_Wrap(std::move(y));
  });
}

// swiglu(x, gate, up, group_size, bits) with gate and up (wq, scales, biases) tuples or lists
PyObject* swiglu(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    int64_t M, K;
    int dt;
    long v[2];
    Pack p[2];
    if (n != 5 || !ints(a + 3, 2, v)) return nullptr;
    const at::Tensor* x = get_x(a[0], M, K, dt);
    if (!x) return nullptr;
    for (int i = 0; i < 2; ++i) {
      PyObject* t = a[1 + i];
      if ((!PyTuple_CheckExact(t) && !PyList_CheckExact(t)) || PySequence_Fast_GET_SIZE(t) != 3) return nullptr;
      PyObject** e = PySequence_Fast_ITEMS(t);
      if (!get_pack(e[0], e[1], e[2], K, v[0], v[1], p[i])) return nullptr;
    }
    if (p[0].N != p[1].N || p[0].dt != p[1].dt) return nullptr;
    bool ok;
    void* st = stream_of(*x, ok);
    if (!ok) return nullptr;
    at::Tensor h = result(*x, p[0].N, dt == MLXQ_BFLOAT16 && p[0].dt == MLXQ_BFLOAT16 ? MLXQ_BFLOAT16 : MLXQ_FLOAT32);
    if (unlocked([&] { return mlxq_swiglu(x->data_ptr(), dt, M, K, (const uint32_t*)p[0].wq.data_ptr(), p[0].s.data_ptr(),
                    p[0].b.data_ptr(), (const uint32_t*)p[1].wq.data_ptr(), p[1].s.data_ptr(), p[1].b.data_ptr(),
                    p[0].dt, p[0].N, (int)v[0], (int)v[1], h.data_ptr(), st); }) != MLXQ_OK)
      return nullptr;
    return THPVariable_Wrap(std::move(h));
  });
}

// embedding(ids, wq, scales, biases, group_size, bits, bf16): int32 ids
PyObject* embedding(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    long v[3];
    Pack p;
    if (n != 7 || !ints(a + 4, 3, v) || (v[1] != 4 && v[1] != 8)) return nullptr;
    const at::Tensor *ids = plain(a[0], 4), *wq = plain(a[1], 16);
    if (!ids || !wq || ids->scalar_type() != at::kInt || ids->numel() == 0 || wq->dim() != 2) return nullptr;
    const int64_t hidden = wq->size(1) * 32 / v[1];
    if (!get_pack(a[1], a[2], a[3], hidden, v[0], v[1], p)) return nullptr;
    bool ok;
    void* st = stream_of(*wq, ok);
    if (!ok) return nullptr;
    at::DimVector shape(ids->sizes().begin(), ids->sizes().end());
    shape.push_back(hidden);
    const int odt = v[2] ? MLXQ_BFLOAT16 : MLXQ_FLOAT32;
    at::Tensor out = at::empty(shape, wq->options().dtype(type_of(odt)));
    if (unlocked([&] { return mlxq_embedding(ids->data_ptr<int32_t>(), ids->numel(), (const uint32_t*)wq->data_ptr(), p.s.data_ptr(),
                       p.b.data_ptr(), p.dt, p.N, hidden, (int)v[0], (int)v[1], out.data_ptr(), odt, st); }) != MLXQ_OK)
      return nullptr;
    return THPVariable_Wrap(std::move(out));
  });
}

// dequantize(wq, scales, biases, group_size, bits)
PyObject* dequantize(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    long v[2];
    Pack p;
    if (n != 5 || !ints(a + 3, 2, v) || (v[1] != 4 && v[1] != 8)) return nullptr;
    const at::Tensor* wq = plain(a[0], 16);
    if (!wq || wq->dim() != 2) return nullptr;
    const int64_t K = wq->size(1) * 32 / v[1];
    if (!get_pack(a[0], a[1], a[2], K, v[0], v[1], p)) return nullptr;
    bool ok;
    void* st = stream_of(p.wq, ok);
    if (!ok) return nullptr;
    at::Tensor out = at::empty({p.N, K}, p.s.options());
    if (unlocked([&] {
          return mlxq_dequantize((const uint32_t*)p.wq.data_ptr(), p.s.data_ptr(), p.b.data_ptr(), p.dt, p.N, K,
                                 (int)v[0], (int)v[1], out.data_ptr(), st);
        }) != MLXQ_OK)
      return nullptr;
    return THPVariable_Wrap(std::move(out));
  });
}

// quantize_batched(weights, group_size, bits): a list of equal 2-D weights -> a list of (wq, scales,
// biases), the scales and biases of each two views of one allocation, the biases 256 to 511 bytes past
// the scales' end.
PyObject* quantize_batched(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    long v[2];
    if (n != 3 || !PyList_CheckExact(a[0]) || !ints(a + 1, 2, v)) return nullptr;
    const Py_ssize_t count = PyList_GET_SIZE(a[0]);
    const long gs = v[0], bits = v[1];
    if (count < 1 || (bits != 4 && bits != 8) || (gs != 32 && gs != 64 && gs != 128)) return nullptr;
    std::vector<at::Tensor> w;
    for (Py_ssize_t i = 0; i < count; ++i) {
      const at::Tensor* t = plain(PyList_GET_ITEM(a[0], i), 16);
      if (!t || t->dim() != 2 || t->numel() == 0) return nullptr;
      if (i && (t->sizes() != w[0].sizes() || t->scalar_type() != w[0].scalar_type() || t->device() != w[0].device()))
        return nullptr;
      w.push_back(*t);
    }
    const int64_t N = w[0].size(0), K = w[0].size(1), G = K / gs;
    const int dt = code_of(w[0].scalar_type());
    if ((dt != MLXQ_BFLOAT16 && dt != MLXQ_FLOAT32) || K % gs != 0) return nullptr;
    bool ok;
    void* st = stream_of(w[0], ok);
    if (!ok) return nullptr;
    const int64_t esz = dt == MLXQ_FLOAT32 ? 4 : 2, off = (N * G * esz + 511) / 256 * 256 / esz;
    std::vector<at::Tensor> q, s, b;
    std::vector<const void*> wp;
    std::vector<uint32_t*> qp;
    std::vector<void*> sp, bp;
    for (Py_ssize_t i = 0; i < count; ++i) {
      q.push_back(at::empty({N, K * bits / 32}, w[0].options().dtype(at::kInt)));
      at::Tensor sb = at::empty({off + N * G}, w[0].options());
      s.push_back(sb.as_strided({N, G}, {G, 1}, 0));
      b.push_back(sb.as_strided({N, G}, {G, 1}, off));
      wp.push_back(w[i].data_ptr());
      qp.push_back((uint32_t*)q[i].data_ptr());
      sp.push_back(s[i].data_ptr());
      bp.push_back(b[i].data_ptr());
    }
    if (unlocked([&] {
          return mlxq_quantize_batched(wp.data(), (int)count, dt, N, K, (int)gs, (int)bits, qp.data(), sp.data(),
                                       bp.data(), st);
        }) != MLXQ_OK)
      return nullptr;
    PyObject* out = PyList_New(count);
    for (Py_ssize_t i = 0; out && i < count; ++i) {
      PyObject* t = PyTuple_New(3);
      if (!t) {
        Py_CLEAR(out);
        break;
      }
      PyTuple_SET_ITEM(t, 0, THPVariable_Wrap(q[i]));
      PyTuple_SET_ITEM(t, 1, THPVariable_Wrap(s[i]));
      PyTuple_SET_ITEM(t, 2, THPVariable_Wrap(b[i]));
      PyList_SET_ITEM(out, i, t);
    }
    return out;
  });
}

// set_error_type(MlxqError)
PyObject* set_error_type(PyObject*, PyObject* type) {
  Py_INCREF(type);
  Py_XSETREF(g_error, type);
  Py_RETURN_NONE;
}

PyMethodDef kMethods[] = {
    {"set_error_type", (PyCFunction)set_error_type, METH_O, nullptr},
    {"quantized_matmul", (PyCFunction)(void*)quantized_matmul, METH_FASTCALL, nullptr},
    {"linear", (PyCFunction)(void*)linear, METH_FASTCALL, nullptr},
    {"swiglu", (PyCFunction)(void*)swiglu, METH_FASTCALL, nullptr},
    {"embedding", (PyCFunction)(void*)embedding, METH_FASTCALL, nullptr},
    {"dequantize", (PyCFunction)(void*)dequantize, METH_FASTCALL, nullptr},
    {"quantize_batched", (PyCFunction)(void*)quantize_batched, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_fast", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

// Built against one torch's headers: another one's objects may be laid out differently.
bool built_for_this_torch() {
  PyObject* torch = PyImport_ImportModule("torch");
  PyObject* v = torch ? PyObject_GetAttrString(torch, "__version__") : nullptr;
  const char* text = v ? PyUnicode_AsUTF8(v) : nullptr;
  const bool same = text && strcmp(text, MLXQ_TORCH_VERSION) == 0;
  if (text && !same) PyErr_Format(PyExc_ImportError, "mlxq._fast is built for torch %s, not %s", MLXQ_TORCH_VERSION, text);
  Py_XDECREF(v);
  Py_XDECREF(torch);
  return same;
}

}  // namespace

PyMODINIT_FUNC PyInit__fast(void) {
  if (!built_for_this_torch()) return nullptr;
  PyObject* c = PyImport_ImportModule("torch._C");
  Py_XSETREF(g_stream_query, c ? PyObject_GetAttrString(c, "_cuda_getCurrentRawStream") : nullptr);
  Py_XDECREF(c);
  return g_stream_query ? PyModule_Create(&kModule) : nullptr;
}
