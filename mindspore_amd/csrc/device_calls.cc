// The device-tensor calls of mindspore_amd/kernels.py as one native call each.
//
// A call on device tensors is a few checks, an output allocation, the current stream and one call of the C ABI.  Through
// Python objects and ctypes that took the host about 9.5 us (FullConnection 128 x 768 x 768, whose kernel takes 4.7),
// so that small shapes ran at the host's pace; here the same steps act on the tensors directly.
// The library is reached through the addresses that lib.py hands over (bind), so a process holds one copy of it,
// whichever file it was loaded from.  The interpreter lock is released while the library is in a call, as ctypes does.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/mi355x_int8.h"

namespace {

struct Api {
  decltype(&mi_matmul_run) matmul_run;
  decltype(&mi_matmul_run_group) matmul_run_group;
  decltype(&mi_conv_out_shape) conv_out_shape;
  decltype(&mi_conv_run) conv_run;
  decltype(&mi_dynquant_run) dynquant_run;
  decltype(&mi_dynquant_await_params) dynquant_await_params;
  decltype(&mi_dynquant_run_segments) dynquant_run_segments;
  decltype(&mi_dynmm_run) dynmm_run;
  decltype(&mi_dynmm_run_chained) dynmm_run_chained;
  decltype(&mi_dynmm_run_rows) dynmm_run_rows;
  decltype(&mi_dynmm_run_group) dynmm_run_group;
} api;
PyObject *check_fn = nullptr;  // lib.check(code, what): raises MiError
PyObject *address_fn = nullptr;  // lib.address(pointer): the address a ctypes pointer holds
PyObject *memory_error = nullptr;  // torch.OutOfMemoryError
PyObject *name_raw = nullptr, *name_n = nullptr, *name_scale = nullptr, *name_zero_point = nullptr;

// Runs `call` without the interpreter lock; false with a Python error set when it failed.
template <typename F>
bool call_library(const char *what, F &&call) {
  int rc;
  Py_BEGIN_ALLOW_THREADS;
  rc = call();
  Py_END_ALLOW_THREADS;
  if (rc == MI_OK) return true;
  PyObject *r = PyObject_CallFunction(check_fn, "is", rc, what);
  if (r != nullptr) {
    Py_DECREF(r);
    PyErr_Format(PyExc_RuntimeError, "%s failed with status %d", what, rc);
  }
  return false;
}

void *stream() { return static_cast<void *>(c10::hip::getCurrentHIPStream().stream()); }

bool as_handle(PyObject *o, void **h) {
  *h = PyLong_AsVoidPtr(o);
  return !(*h == nullptr && PyErr_Occurred());
}

// A contiguous device tensor of `type` whose last extent is `last` (< 0: any); null with a ValueError otherwise.
const at::Tensor *operand(PyObject *o, at::ScalarType type, int64_t last, const char *kind) {
  const at::Tensor &t = THPVariable_Unpack(o);
  if (t.scalar_type() == type && t.is_cuda() && t.is_contiguous() && (last < 0 || (t.dim() > 0 && t.size(-1) == last)))
    return &t;
  if (last < 0) PyErr_Format(PyExc_ValueError, "expected a contiguous CUDA %s tensor", kind);
  else PyErr_Format(PyExc_ValueError, "expected a contiguous CUDA %s tensor [..., %lld]", kind, (long long)last);
  return nullptr;
}

at::Tensor empty(at::IntArrayRef size, at::ScalarType type, const at::Device &device) {
  return at::Tensor(at::detail::empty_cuda(size, type, device, std::nullopt));
}

at::Tensor empty_rows(const at::Tensor &a, int64_t n, at::ScalarType type) {
  c10::SmallVector<int64_t, 8> size(a.sizes().begin(), a.sizes().end());
  size.back() = n;
  return empty(size, type, a.device());
}

// The caller's output tensor; null with a ValueError when it does not fit.
const at::Tensor *given_out(PyObject *o, int64_t elements) {
  if (THPVariable_Check(o)) {
    const at::Tensor &t = THPVariable_Unpack(o);
    if (t.scalar_type() == at::kChar && t.is_cuda() && t.is_contiguous() && t.numel() == elements) return &t;
  }
  PyErr_Format(PyExc_ValueError, "out must be a contiguous CUDA int8 tensor with %lld elements", (long long)elements);
  return nullptr;
}

// A device address: a whole number, or whatever ctypes takes for a void pointer.
bool as_address(PyObject *o, const void **p) {
  if (PyLong_Check(o)) {
    *p = PyLong_AsVoidPtr(o);
    return !PyErr_Occurred();
  }
  PyObject *v = PyObject_CallOneArg(address_fn, o);
  if (v == nullptr) return false;
  *p = PyLong_AsVoidPtr(v);
  Py_DECREF(v);
  return !PyErr_Occurred();
}

// float(o) and int(o), the latter into 32 bits as ctypes narrows it
bool as_float(PyObject *o, double *x) {
  PyObject *f = PyNumber_Float(o);
  if (f == nullptr) return false;
  *x = PyFloat_AS_DOUBLE(f);
  Py_DECREF(f);
  return true;
}
bool as_int32(PyObject *o, int32_t *x) {
  PyObject *i = PyNumber_Long(o);
  if (i == nullptr) return false;
  *x = (int32_t)PyLong_AsUnsignedLongLongMask(i);
  Py_DECREF(i);
  return !PyErr_Occurred();
}

bool count_args(Py_ssize_t nargs, Py_ssize_t want) {
  if (nargs == want) return true;
  PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", want, nargs);
  return false;
}

// No C++ exception may cross into the interpreter (an allocation can throw).
template <typename F>
PyObject *guarded(F &&f) {
  try {
    return f();
  } catch (const c10::OutOfMemoryError &e) {
    PyErr_SetString(memory_error, e.what_without_backtrace());
  } catch (const std::exception &e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
  }
  return nullptr;
}

template <typename T>
bool take(PyObject *addresses, const char *name, T *fn) {
  PyObject *v = PyDict_GetItemString(addresses, name);
  if (v == nullptr) {
    PyErr_Format(PyExc_KeyError, "%s", name);
    return false;
  }
  *fn = reinterpret_cast<T>(PyLong_AsVoidPtr(v));
  return !PyErr_Occurred();
}

// bind({entry point: address}, check, torch.OutOfMemoryError, address)
PyObject *bind(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  if (!count_args(nargs, 4)) return nullptr;
  PyObject *d = args[0];
  if (!take(d, "mi_matmul_run", &api.matmul_run) || !take(d, "mi_matmul_run_group", &api.matmul_run_group) ||
      !take(d, "mi_conv_out_shape", &api.conv_out_shape) || !take(d, "mi_conv_run", &api.conv_run) ||
      !take(d, "mi_dynquant_run", &api.dynquant_run) || !take(d, "mi_dynquant_await_params", &api.dynquant_await_params) ||
      !take(d, "mi_dynquant_run_segments", &api.dynquant_run_segments) || !take(d, "mi_dynmm_run", &api.dynmm_run) ||
      !take(d, "mi_dynmm_run_chained", &api.dynmm_run_chained) || !take(d, "mi_dynmm_run_rows", &api.dynmm_run_rows) ||
      !take(d, "mi_dynmm_run_group", &api.dynmm_run_group))
    return nullptr;
  Py_INCREF(args[1]);
  Py_XSETREF(check_fn, args[1]);
  Py_INCREF(args[2]);
  Py_XSETREF(memory_error, args[2]);
  Py_INCREF(args[3]);
  Py_XSETREF(address_fn, args[3]);
  Py_RETURN_NONE;
}

// Every call below returns NotImplemented when its operand is not a torch tensor (the caller then takes the host path).

// matmul_run(handle, a, n, k, out or None) -> int8 [..., n]
PyObject *matmul_run(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  if (!count_args(nargs, 5)) return nullptr;
  if (!THPVariable_Check(args[1])) Py_RETURN_NOTIMPLEMENTED;
  return guarded([&]() -> PyObject * {
    void *h;
    const int64_t n = PyLong_AsLongLong(args[2]), k = PyLong_AsLongLong(args[3]);
    if (!as_handle(args[0], &h) || PyErr_Occurred()) return nullptr;
    const at::Tensor *a = operand(args[1], at::kChar, k, "int8");
    if (a == nullptr) return nullptr;
    const int64_t rows = a->numel() / k;
    at::Tensor made;
    const at::Tensor *out = &made;
    if (args[4] == Py_None) made = empty_rows(*a, n, at::kChar);
    else if ((out = given_out(args[4], rows * n)) == nullptr) return nullptr;
    const int8_t *ap = static_cast<const int8_t *>(a->data_ptr());
    int8_t *cp = static_cast<int8_t *>(out->data_ptr());
    void *s = stream();
    if (!call_library("mi_matmul_run", [&] { return api.matmul_run(static_cast<mi_matmul *>(h), ap, (int32_t)rows, cp, s); }))
      return nullptr;
    if (args[4] == Py_None) return THPVariable_Wrap(std::move(made));
    Py_INCREF(args[4]);
    return args[4];
  });
}

// The members of a group call: handles, and the outputs given or made.
struct Group {
  int count = 0;
  c10::SmallVector<void *, 8> handle, out;
  PyObject *outs = nullptr;  // what the call returns: the caller's sequence, or a new list
  ~Group() { Py_XDECREF(outs); }
  bool fill(PyObject *kernels, PyObject *given, const at::Tensor &a, at::ScalarType type) {
    PyObject *seq = PySequence_Fast(kernels, "expected a sequence of kernels");
    if (seq == nullptr) return false;
    const bool ok = fill_from(seq, given, a, type);
    Py_DECREF(seq);
    return ok;
  }

 private:
  bool fill_from(PyObject *seq, PyObject *given, const at::Tensor &a, at::ScalarType type) {
    const Py_ssize_t members = PySequence_Fast_GET_SIZE(seq);
    if (members > INT_MAX) {
      PyErr_SetString(PyExc_ValueError, "too many kernels");
      return false;
    }
    count = (int)members;
    handle.resize(members);
    out.resize(members);
    if (given == Py_None) {
      outs = PyList_New(count);
      if (outs == nullptr) return false;
    } else {
      Py_INCREF(given);
      outs = given;
    }
    for (int i = 0; i < count; ++i) {
      PyObject *kernel = PySequence_Fast_GET_ITEM(seq, i);
      PyObject *raw = PyObject_GetAttr(kernel, name_raw);
      if (raw == nullptr) return false;
      const bool ok = as_handle(raw, &handle[i]);
      Py_DECREF(raw);
      if (!ok) return false;
      if (given == Py_None) {
        PyObject *no = PyObject_GetAttr(kernel, name_n);
        if (no == nullptr) return false;
        const int64_t n = PyLong_AsLongLong(no);
        Py_DECREF(no);
        if (n < 0) return false;
        at::Tensor t = empty_rows(a, n, type);
        out[i] = t.data_ptr();
        PyObject *w = THPVariable_Wrap(std::move(t));
        if (w == nullptr) return false;
        PyList_SET_ITEM(outs, i, w);
      } else {
        PyObject *o = PySequence_GetItem(given, i);
        if (o == nullptr) return false;
        const bool tensor = THPVariable_Check(o);
        if (tensor) out[i] = THPVariable_Unpack(o).data_ptr();
        Py_DECREF(o);
        if (!tensor) {
          PyErr_SetString(PyExc_TypeError, "outs must hold tensors");
          return false;
        }
      }
    }
    return true;
  }
};

// matmul_run_group(kernels, a, k, outs or None) -> outs
PyObject *matmul_run_group(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  if (!count_args(nargs, 4)) return nullptr;
  if (!THPVariable_Check(args[1])) Py_RETURN_NOTIMPLEMENTED;
  return guarded([&]() -> PyObject * {
    const int64_t k = PyLong_AsLongLong(args[2]);
    if (PyErr_Occurred()) return nullptr;
    const at::Tensor *a = operand(args[1], at::kChar, k, "int8");
    Group g;
    if (a == nullptr || !g.fill(args[0], args[3], *a, at::kChar)) return nullptr;
    const int8_t *ap = static_cast<const int8_t *>(a->data_ptr());
    const int32_t rows = (int32_t)(a->numel() / k);
    void *s = stream();
    if (!call_library("mi_matmul_run_group", [&] {
          return api.matmul_run_group(reinterpret_cast<mi_matmul *const *>(g.handle.data()), g.count, ap, rows,
                                      reinterpret_cast<int8_t *const *>(g.out.data()), s);
        }))
      return nullptr;
    Py_INCREF(g.outs);
    return g.outs;
  });
}

// Input quantisation of a dynamic MatMul, from kernels.py's (in_quant, params_dev, row_params): the first that is given,
// from the last to the first.
struct InQuant {
  double scale = 0.0;
  int32_t zp = 0, per_row = 0;
  int64_t row_bytes = 0;
  const mi_dq_params *dev = nullptr;
  bool chained = false;  // an address was given (a null one is the library's to refuse)
  bool fill(PyObject *const *args) {
    if (args[2] != Py_None) {  // the tensor of parameter blocks that dynquant_run_rows made
      if (!THPVariable_Check(args[2])) {
        PyErr_SetString(PyExc_TypeError, "row_params must be a tensor");
        return false;
      }
      const at::Tensor &t = THPVariable_Unpack(args[2]);
      dev = static_cast<const mi_dq_params *>(t.data_ptr());
      row_bytes = t.numel();
      per_row = 1;
    } else if (args[1] != Py_None) {
      const void *p = nullptr;
      if (!as_address(args[1], &p)) return false;
      dev = static_cast<const mi_dq_params *>(p);
      chained = true;
    } else {
      PyObject *so = PyObject_GetAttr(args[0], name_scale);
      PyObject *zo = so == nullptr ? nullptr : PyObject_GetAttr(args[0], name_zero_point);
      const bool ok = zo != nullptr && as_float(so, &scale) && as_int32(zo, &zp);
      Py_XDECREF(so);
      Py_XDECREF(zo);
      return ok;
    }
    return true;
  }
};

// dynmm_run(handle, a, n, k, in_quant, params_dev, row_params) -> fp32 [..., n]
PyObject *dynmm_run(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  if (!count_args(nargs, 7)) return nullptr;
  if (!THPVariable_Check(args[1])) Py_RETURN_NOTIMPLEMENTED;
  return guarded([&]() -> PyObject * {
    void *h;
    const int64_t n = PyLong_AsLongLong(args[2]), k = PyLong_AsLongLong(args[3]);
    InQuant q;
    if (!as_handle(args[0], &h) || !q.fill(args + 4)) return nullptr;
    const at::Tensor *a = operand(args[1], at::kChar, k, "int8");
    if (a == nullptr) return nullptr;
    const int64_t rows = a->numel() / k;
    if (q.per_row && q.row_bytes != rows * (int64_t)sizeof(mi_dq_params)) {
      PyErr_Format(PyExc_ValueError, "row_params does not hold %lld parameter blocks", (long long)rows);
      return nullptr;
    }
    at::Tensor out = empty_rows(*a, n, at::kFloat);
    const int8_t *ap = static_cast<const int8_t *>(a->data_ptr());
    float *cp = static_cast<float *>(out.data_ptr());
    mi_dynmm *mm = static_cast<mi_dynmm *>(h);
    void *s = stream();
    const char *what = q.per_row ? "mi_dynmm_run_rows" : q.chained ? "mi_dynmm_run_chained" : "mi_dynmm_run";
    if (!call_library(what, [&] {
          if (q.per_row) return api.dynmm_run_rows(mm, ap, (int32_t)rows, q.dev, cp, s);
          if (q.chained) return api.dynmm_run_chained(mm, ap, (int32_t)rows, q.dev, cp, s);
          return api.dynmm_run(mm, ap, (int32_t)rows, q.scale, q.zp, cp, s);
        }))
      return nullptr;
    return THPVariable_Wrap(std::move(out));
  });
}

// dynmm_run_group(kernels, a, k, outs or None, in_quant, params_dev, row_params) -> outs
PyObject *dynmm_run_group(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  if (!count_args(nargs, 7)) return nullptr;
  if (!THPVariable_Check(args[1])) Py_RETURN_NOTIMPLEMENTED;
  return guarded([&]() -> PyObject * {
    const int64_t k = PyLong_AsLongLong(args[2]);
    InQuant q;
    if (PyErr_Occurred() || !q.fill(args + 4)) return nullptr;
    const at::Tensor *a = operand(args[1], at::kChar, k, "int8");
    Group g;
    if (a == nullptr || !g.fill(args[0], args[3], *a, at::kFloat)) return nullptr;
    const int8_t *ap = static_cast<const int8_t *>(a->data_ptr());
    const int32_t rows = (int32_t)(a->numel() / k);
    void *s = stream();
    if (!call_library("mi_dynmm_run_group", [&] {
          return api.dynmm_run_group(reinterpret_cast<mi_dynmm *const *>(g.handle.data()), g.count, ap, rows, q.scale, q.zp, q.dev,
                                     q.per_row, reinterpret_cast<float *const *>(g.out.data()), s);
        }))
      return nullptr;
    Py_INCREF(g.outs);
    return g.outs;
  });
}

// conv_run(handle, x, oc, out or None) -> int8 [batch, oh, ow, oc]; the caller has checked x's rank and channels
PyObject *conv_run(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  if (!count_args(nargs, 5)) return nullptr;
  if (!THPVariable_Check(args[1])) Py_RETURN_NOTIMPLEMENTED;
  return guarded([&]() -> PyObject * {
    void *h;
    const int64_t ic = PyLong_AsLongLong(args[2]), oc = PyLong_AsLongLong(args[3]);
    if (!as_handle(args[0], &h) || PyErr_Occurred()) return nullptr;
    const at::Tensor &any = THPVariable_Unpack(args[1]);
    if (any.dim() != 4 || any.size(3) != ic) {
      PyObject *shape = PyObject_GetAttrString(args[1], "shape");
      PyObject *tuple = shape == nullptr ? nullptr : PySequence_Tuple(shape);
      if (tuple != nullptr) PyErr_Format(PyExc_ValueError, "expected NHWC with %lld channels, got %R", (long long)ic, tuple);
      Py_XDECREF(shape);
      Py_XDECREF(tuple);
      return nullptr;
    }
    mi_conv *conv = static_cast<mi_conv *>(h);
    const int32_t b = (int32_t)any.size(0), ih = (int32_t)any.size(1), iw = (int32_t)any.size(2);
    int32_t oh = 0, ow = 0;
    if (!call_library("mi_conv_out_shape", [&] { return api.conv_out_shape(conv, ih, iw, &oh, &ow); })) return nullptr;
    const at::Tensor *x = operand(args[1], at::kChar, -1, "int8");
    if (x == nullptr) return nullptr;
    at::Tensor made;
    const at::Tensor *out = &made;
    if (args[4] == Py_None) made = empty({b, oh, ow, oc}, at::kChar, x->device());
    else if ((out = given_out(args[4], (int64_t)b * oh * ow * oc)) == nullptr) return nullptr;
    const int8_t *xp = static_cast<const int8_t *>(x->data_ptr());
    int8_t *cp = static_cast<int8_t *>(out->data_ptr());
    void *s = stream();
    if (!call_library("mi_conv_run", [&] { return api.conv_run(conv, xp, b, ih, iw, cp, s); })) return nullptr;
    if (args[4] == Py_None) return THPVariable_Wrap(std::move(made));
    Py_INCREF(args[4]);
    return args[4];
  });
}

// dynquant_run(handle, x, address of a host parameter block or 0) -> int8 tensor; with an address the call waits
// until the parameters of the run are known and fills the block
PyObject *dynquant_run(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  if (!count_args(nargs, 3)) return nullptr;
  if (!THPVariable_Check(args[1])) Py_RETURN_NOTIMPLEMENTED;
  return guarded([&]() -> PyObject * {
    void *h, *host;
    if (!as_handle(args[0], &h) || !as_handle(args[2], &host)) return nullptr;
    const at::Tensor *x = operand(args[1], at::kFloat, -1, "float32");
    if (x == nullptr) return nullptr;
    at::Tensor q = empty(x->sizes(), at::kChar, x->device());
    const float *xp = static_cast<const float *>(x->data_ptr());
    int8_t *qp = static_cast<int8_t *>(q.data_ptr());
    const int64_t n = x->numel();
    mi_dynquant *dq = static_cast<mi_dynquant *>(h);
    void *s = stream();
    if (!call_library("mi_dynquant_run", [&] { return api.dynquant_run(dq, xp, n, qp, s); })) return nullptr;
    if (host != nullptr && !call_library("mi_dynquant_await_params", [&] {
          return api.dynquant_await_params(dq, s, static_cast<mi_dq_params *>(host));
        }))
      return nullptr;
    return THPVariable_Wrap(std::move(q));
  });
}

// dynquant_run_rows(handle, x) -> (int8 tensor, uint8 tensor of one parameter block per row)
PyObject *dynquant_run_rows(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  if (!count_args(nargs, 2)) return nullptr;
  if (!THPVariable_Check(args[1])) Py_RETURN_NOTIMPLEMENTED;
  return guarded([&]() -> PyObject * {
    void *h;
    if (!as_handle(args[0], &h)) return nullptr;
    const at::Tensor *x = operand(args[1], at::kFloat, -1, "float32");
    if (x == nullptr) return nullptr;
    if (x->dim() == 0 || x->size(-1) == 0) {
      PyErr_SetString(PyExc_ValueError, "expected a tensor of rows");
      return nullptr;
    }
    const int64_t unit = x->size(-1), rows = x->numel() / unit;
    at::Tensor q = empty(x->sizes(), at::kChar, x->device());
    at::Tensor params = empty({rows * (int64_t)sizeof(mi_dq_params)}, at::kByte, x->device());
    const float *xp = static_cast<const float *>(x->data_ptr());
    int8_t *qp = static_cast<int8_t *>(q.data_ptr());
    mi_dq_params *pp = static_cast<mi_dq_params *>(params.data_ptr());
    void *s = stream();
    if (!call_library("mi_dynquant_run_segments", [&] {
          return api.dynquant_run_segments(static_cast<mi_dynquant *>(h), xp, rows, unit, qp, pp, s);
        }))
      return nullptr;
    PyObject *qo = THPVariable_Wrap(std::move(q)), *po = THPVariable_Wrap(std::move(params));
    PyObject *both = qo != nullptr && po != nullptr ? PyTuple_Pack(2, qo, po) : nullptr;
    Py_XDECREF(qo);
    Py_XDECREF(po);
    return both;
  });
}

#define MI_METHOD(f) {#f, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(f)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {MI_METHOD(bind),          MI_METHOD(matmul_run), MI_METHOD(matmul_run_group),
                         MI_METHOD(dynmm_run),     MI_METHOD(dynmm_run_group), MI_METHOD(conv_run),
                         MI_METHOD(dynquant_run),  MI_METHOD(dynquant_run_rows), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_device_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__device_calls(void) {
  name_raw = PyUnicode_InternFromString("_raw");
  name_n = PyUnicode_InternFromString("n");
  name_scale = PyUnicode_InternFromString("scale");
  name_zero_point = PyUnicode_InternFromString("zero_point");
  if (name_raw == nullptr || name_n == nullptr || name_scale == nullptr || name_zero_point == nullptr) return nullptr;
  return PyModule_Create(&module);
}
