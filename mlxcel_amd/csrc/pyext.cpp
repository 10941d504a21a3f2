// pyext.cpp — the Python entry points' common case in native code: exact
// torch tensors on a HIP device in, one C-ABI call (include/mlxq.h) on the
// current stream, tensors out.
//
// A call costs the host ~16 us through ctypes (argument structs, the device
// context manager, the shape query, the stream object), more than most decode
// kernels run; here it is the C call and one allocation per result.  Anything
// unusual returns None and takes the ctypes path in ops.py, which does the
// same and reports the errors: tensor subclasses, torch-function modes,
// tensors off the GPU, other Python types for numbers, more dimensions than
// the C ABI has.  A failed C call returns its status (an int).
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/mlxq.h"

namespace {

// dtype code of a tensor, -1 where the C ABI has none
int dtype_of(at::ScalarType t) {
  switch (t) {
    case at::kBool: return MLXQ_BOOL;
    case at::kByte: return MLXQ_UINT8;
    case at::kUInt16: return MLXQ_UINT16;
    case at::kUInt32: return MLXQ_UINT32;
    case at::kUInt64: return MLXQ_UINT64;
    case at::kChar: return MLXQ_INT8;
    case at::kShort: return MLXQ_INT16;
    case at::kInt: return MLXQ_INT32;
    case at::kLong: return MLXQ_INT64;
    case at::kHalf: return MLXQ_FLOAT16;
    case at::kFloat: return MLXQ_FLOAT32;
    case at::kDouble: return MLXQ_FLOAT64;
    case at::kBFloat16: return MLXQ_BFLOAT16;
    default: return -1;
  }
}

at::ScalarType scalar_of(int dt) {
  static const at::ScalarType t[] = {at::kBool, at::kByte, at::kUInt16, at::kUInt32, at::kUInt64, at::kChar, at::kShort,
                                     at::kInt,  at::kLong, at::kHalf,   at::kFloat,  at::kDouble, at::kBFloat16};
  return t[dt];
}

struct NotHandled {};  // the ctypes path takes the call
struct Status {
  int code;
};

struct Arr {
  mlxq_array a;
  bool on = false;
  const mlxq_array* p() const { return on ? &a : nullptr; }
};

void fill(Arr& r, const at::Tensor& t) {
  if (t.dim() > MLXQ_MAX_DIMS || !t.device().is_cuda()) throw NotHandled{};
  const int dt = dtype_of(t.scalar_type());
  if (dt < 0) throw NotHandled{};
  r.on = true;
  r.a.data = t.numel() > 0 ? t.data_ptr() : nullptr;
  r.a.dtype = dt;
  r.a.ndim = (int32_t)t.dim();
  const auto sz = t.sizes(), st = t.strides();
  for (int64_t i = 0; i < t.dim(); i++) {
    r.a.shape[i] = sz[i];
    r.a.strides[i] = st[i];
  }
}

const at::Tensor& tensor(PyObject* o) {
  if (!THPVariable_CheckExact(o)) throw NotHandled{};
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || t.layout() != at::kStrided || !t.device().is_cuda()) throw NotHandled{};
  return t;
}

Arr arr(PyObject* o) {
  Arr r;
  if (o != Py_None) fill(r, tensor(o));
  return r;
}

int integer(PyObject* o, int none = -1) {
  if (o == Py_None) return none;
  if (!PyLong_CheckExact(o)) throw NotHandled{};
  int over = 0;
  const long v = PyLong_AsLongAndOverflow(o, &over);
  if (over || v < INT32_MIN || v > INT32_MAX) throw NotHandled{};
  return (int)v;
}

bool boolean(PyObject* o) {
  if (!PyBool_Check(o)) throw NotHandled{};
  return o == Py_True;
}

const char* text(PyObject* o) {
  if (!PyUnicode_CheckExact(o)) throw NotHandled{};
  const char* s = PyUnicode_AsUTF8(o);
  if (!s) {
    PyErr_Clear();
    throw NotHandled{};
  }
  return s;
}

at::Tensor make(int ndim, const int64_t* shape, int dt, const at::Device& dev) {
  return at::empty(at::IntArrayRef(shape, ndim), at::TensorOptions().dtype(scalar_of(dt)).device(dev));
}

// The C call on the device's current stream, without the GIL (as ctypes calls it).
template <class F>
void call(const at::Device& dev, F&& f) {
  const c10::DeviceGuard guard(dev);
  void* stream = c10::hip::getCurrentHIPStream(dev.index()).stream();
  int st;
  Py_BEGIN_ALLOW_THREADS
  st = f(stream);
  Py_END_ALLOW_THREADS
  if (st != MLXQ_OK) throw Status{st};
}

// Runs a wrapper's body: its result, None (not handled), or the status.
template <class F>
PyObject* entry(Py_ssize_t n, Py_ssize_t want, F&& f) {
  if (n != want) {
    PyErr_SetString(PyExc_TypeError, "wrong number of arguments");
    return nullptr;
  }
  if (at::impl::torch_function_mode_enabled()) Py_RETURN_NONE;
  try {
    return f();
  } catch (const NotHandled&) {
    Py_RETURN_NONE;
  } catch (const Status& s) {
    return PyLong_FromLong(s.code);
  } catch (const std::exception&) {
    // torch's own (out of memory, or Python code that an allocation runs under
    // a dispatch mode): the ctypes path meets it again and raises it
    PyErr_Clear();
    Py_RETURN_NONE;
  }
}

PyObject* keep(PyObject* given, const at::Tensor& t) {
  if (given != Py_None) {
    Py_INCREF(given);
    return given;
  }
  return THPVariable_Wrap(t);
}

// (x, w, scales, biases, linear_bias, linear, transpose, group_size, bits, mode, out)
PyObject* quantized_matmul(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return entry(n, 11, [&]() -> PyObject* {
    const at::Tensor& xt = tensor(v[0]);
    const Arr x = arr(v[0]), w = arr(v[1]), s = arr(v[2]), b = arr(v[3]), lb = arr(v[4]);
    const bool linear = boolean(v[5]), tr = boolean(v[6]);
    const int gs = integer(v[7]), bits = integer(v[8]);
    const char* mode = text(v[9]);
    at::Tensor out;
    Arr o;
    if (v[10] == Py_None) {
      int32_t nd, dt;
      int64_t sh[MLXQ_MAX_DIMS];
      const int st = mlxq_quantized_matmul_shape(x.p(), w.p(), s.p(), b.p(), tr, gs, bits, mode, &nd, sh, &dt);
      if (st) throw Status{st};
      out = make(nd, sh, dt, xt.device());
      fill(o, out);
    } else {
      o = arr(v[10]);
    }
    call(xt.device(), [&](void* stream) {
      return linear ? mlxq_quantized_linear(x.p(), w.p(), s.p(), b.p(), lb.p(), gs, bits, mode, &o.a, stream)
                    : mlxq_quantized_matmul(x.p(), w.p(), s.p(), b.p(), tr, gs, bits, mode, &o.a, stream);
    });
    return keep(v[10], out);
  });
}

constexpr int kMulti = 4;

// A reference of the call's own: another thread may change the caller's list
// while the GIL is released.
struct Held {
  PyObject* o = nullptr;
  ~Held() { Py_XDECREF(o); }
};

// items of a list or tuple of at most kMulti tensors
int items(PyObject* o, Held* to) {
  const bool l = PyList_CheckExact(o), t = PyTuple_CheckExact(o);
  if (!l && !t) throw NotHandled{};
  const Py_ssize_t n = l ? PyList_GET_SIZE(o) : PyTuple_GET_SIZE(o);
  if (n < 1 || n > kMulti) throw NotHandled{};
  for (Py_ssize_t i = 0; i < n; i++) {
    to[i].o = l ? PyList_GET_ITEM(o, i) : PyTuple_GET_ITEM(o, i);
    Py_INCREF(to[i].o);
  }
  return (int)n;
}

// (x, ws, scales, biases, group_size, bits, mode, out)
PyObject* quantized_matmul_multi(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return entry(n, 8, [&]() -> PyObject* {
    const at::Tensor& xt = tensor(v[0]);
    const Arr x = arr(v[0]);
    Held wo[kMulti], so[kMulti], bo[kMulti], oo[kMulti];
    const int cnt = items(v[1], wo);
    if (items(v[2], so) != cnt) throw NotHandled{};
    const bool biases = v[3] != Py_None, given = v[7] != Py_None;
    if ((biases && items(v[3], bo) != cnt) || (given && items(v[7], oo) != cnt)) throw NotHandled{};
    const int gs = integer(v[4]), bits = integer(v[5]);
    const char* mode = text(v[6]);
    Arr w[kMulti], s[kMulti], b[kMulti], o[kMulti];
    const mlxq_array *pw[kMulti], *ps[kMulti], *pb[kMulti];
    mlxq_array* po[kMulti];
    at::Tensor out[kMulti];
    for (int i = 0; i < cnt; i++) {
      w[i] = arr(wo[i].o);
      s[i] = arr(so[i].o);
      if (!w[i].on || !s[i].on) throw NotHandled{};
      if (biases) b[i] = arr(bo[i].o);
      pw[i] = w[i].p();
      ps[i] = s[i].p();
      pb[i] = b[i].p();
      if (given) {
        o[i] = arr(oo[i].o);
        if (!o[i].on) throw NotHandled{};
      } else {
        int32_t nd, dt;
        int64_t sh[MLXQ_MAX_DIMS];
        const int st = mlxq_quantized_matmul_shape(x.p(), pw[i], ps[i], pb[i], true, gs, bits, mode, &nd, sh, &dt);
        if (st) throw Status{st};
        out[i] = make(nd, sh, dt, xt.device());
        fill(o[i], out[i]);
      }
      po[i] = &o[i].a;
    }
    call(xt.device(), [&](void* stream) {
      return mlxq_quantized_matmul_multi(x.p(), cnt, pw, ps, biases ? pb : nullptr, gs, bits, mode, po, stream);
    });
    PyObject* r = PyList_New(cnt);
    if (!r) return nullptr;
    for (int i = 0; i < cnt; i++) PyList_SET_ITEM(r, i, keep(given ? oo[i].o : Py_None, out[i]));
    return r;
  });
}

// (x, w, scales, biases, lhs_indices, rhs_indices, transpose, group_size, bits, mode, sorted_indices, out)
PyObject* gather_qmm(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return entry(n, 12, [&]() -> PyObject* {
    const at::Tensor& xt = tensor(v[0]);
    const Arr x = arr(v[0]), w = arr(v[1]), s = arr(v[2]), b = arr(v[3]), l = arr(v[4]), r = arr(v[5]);
    const bool tr = boolean(v[6]), sorted = boolean(v[10]);
    const int gs = integer(v[7]), bits = integer(v[8]);
    const char* mode = text(v[9]);
    at::Tensor out;
    Arr o;
    if (v[11] == Py_None) {
      int32_t nd, dt;
      int64_t sh[MLXQ_MAX_DIMS];
      const int st =
          mlxq_gather_qmm_shape(x.p(), w.p(), s.p(), b.p(), l.p(), r.p(), tr, gs, bits, mode, &nd, sh, &dt);
      if (st) throw Status{st};
      out = make(nd, sh, dt, xt.device());
      fill(o, out);
    } else {
      o = arr(v[11]);
    }
    call(xt.device(), [&](void* stream) {
      return mlxq_gather_qmm(x.p(), w.p(), s.p(), b.p(), l.p(), r.p(), tr, gs, bits, sorted, mode, nullptr, &o.a,
                             stream);
    });
    return keep(v[11], out);
  });
}

// (w, scales, biases, group_size, bits, mode, dtype code or -1, out): `out` allocated by the caller
PyObject* dequantize(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return entry(n, 8, [&]() -> PyObject* {
    const at::Tensor& wt = tensor(v[0]);
    const Arr w = arr(v[0]), s = arr(v[1]), b = arr(v[2]), o = arr(v[7]);
    if (!s.on || !o.on) throw NotHandled{};
    const int gs = integer(v[3]), bits = integer(v[4]), dt = integer(v[6]);
    const char* mode = text(v[5]);
    Arr oc = o;
    call(wt.device(), [&](void* stream) { return mlxq_dequantize(w.p(), s.p(), b.p(), gs, bits, mode, dt, &oc.a, stream); });
    Py_INCREF(v[7]);
    return v[7];
  });
}

// (w, group_size, bits, mode, wq, scales, biases): results allocated by the caller
PyObject* quantize(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return entry(n, 7, [&]() -> PyObject* {
    const at::Tensor& wt = tensor(v[0]);
    const Arr w = arr(v[0]);
    const int gs = integer(v[1]), bits = integer(v[2]);
    const char* mode = text(v[3]);
    Arr q = arr(v[4]), s = arr(v[5]), b = arr(v[6]);
    if (!q.on || !s.on) throw NotHandled{};
    call(wt.device(), [&](void* stream) { return mlxq_quantize(w.p(), gs, bits, mode, &q.a, &s.a, b.on ? &b.a : nullptr, stream); });
    Py_RETURN_TRUE;
  });
}

// (geglu, x, indices, gate_w, gate_s, gate_b, up_w, up_s, up_b, down_w, down_s, down_b, scores,
//  din, dff, k, gu_bits, d_bits, group_size, out)
PyObject* fused_moe(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return entry(n, 20, [&]() -> PyObject* {
    const bool geglu = boolean(v[0]);
    const at::Tensor& xt = tensor(v[1]);
    Arr a[12];
    for (int i = 0; i < 12; i++) a[i] = arr(v[1 + i]);
    int d[6];
    for (int i = 0; i < 6; i++) {
      if (v[13 + i] == Py_None) throw NotHandled{};
      d[i] = integer(v[13 + i]);
    }
    at::Tensor out;
    Arr o;
    if (v[19] == Py_None) {
      const int64_t din = d[0] > 0 ? d[0] : 0;
      out = at::empty({din}, xt.options().requires_grad(false));
      fill(o, out);
    } else {
      o = arr(v[19]);
    }
    call(xt.device(), [&](void* stream) {
      return (geglu ? mlxq_fused_moe_geglu : mlxq_fused_moe_expert)(
          a[0].p(), a[1].p(), a[2].p(), a[3].p(), a[4].p(), a[5].p(), a[6].p(), a[7].p(), a[8].p(), a[9].p(), a[10].p(),
          a[11].p(), d[0], d[1], d[2], d[3], d[4], d[5], &o.a, stream);
    });
    return keep(v[19], out);
  });
}

#define FAST(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {FAST(quantized_matmul), FAST(quantized_matmul_multi), FAST(gather_qmm), FAST(dequantize),
                         FAST(quantize),         FAST(fused_moe),              {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_mlxq_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__mlxq_native() {
  PyObject* m = PyModule_Create(&module);
  // the torch it was compiled against: ops.py takes no other
  if (m && PyModule_AddStringConstant(m, "torch_version", MLXQ_TORCH_VERSION) < 0) Py_CLEAR(m);
  return m;
}
