// The common call of the Python classes' Run in one native function each: arguments checked, output allocated, current
// stream looked up, library entry point called.  A small layer runs for 4 - 5 us on the device, and the same steps in
// Python (attributes of the tensors, torch.empty, ctypes) take 2 - 3 us beside the launch itself.  Anything out of the
// ordinary - another type of tensor or argument, a shape or device that does not fit, a status below zero - returns
// None with nothing done, and the Python code behind it decides.
#define PY_SSIZE_T_CLEAN
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>

#include <cstdint>

namespace {

typedef int (*ConvRun)(void*, const void*, void*, int32_t, int32_t, void*);
typedef int (*DwRun)(void*, const int8_t*, void*, int32_t, int32_t, int32_t, void*);
typedef int (*PairRun)(void*, void*, const void*, void*, int32_t, int32_t, int32_t, void*);

// A plain contiguous 4-D device tensor of the type, or nullptr.
const at::Tensor* Plain(PyObject* o, at::ScalarType type) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  return t.defined() && t.is_cuda() && t.layout() == at::kStrided && t.scalar_type() == type && t.dim() == 4 && t.is_contiguous() ? &t : nullptr;
}

bool Int32(int64_t v) { return v >= 0 && v <= INT32_MAX; }

// The output: the caller's, or a new one.  False where the caller's does not fit.
bool Output(PyObject* out, const at::Tensor& x, at::ScalarType type, at::IntArrayRef shape, at::Tensor* own, void** ptr) {
  if (out == Py_None) {
    *own = at::empty(shape, x.options().dtype(type));
    *ptr = own->data_ptr();
    return true;
  }
  const at::Tensor* t = Plain(out, type);
  if (!t || t->sizes() != shape || t->device() != x.device()) return false;
  *ptr = t->data_ptr();
  return true;
}

bool Stream(PyObject* stream, const at::Tensor& x, void** raw) {
  if (stream == Py_None) {
    *raw = c10::hip::getCurrentHIPStream(x.get_device()).stream();
    return true;
  }
  if (!PyLong_CheckExact(stream)) return false;
  *raw = PyLong_AsVoidPtr(stream);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

PyObject* Result(int rc, PyObject* out, const at::Tensor& own) {
  if (rc < 0) Py_RETURN_NONE;
  if (out == Py_None) return THPVariable_Wrap(own);
  Py_INCREF(out);
  return out;
}

// Whether the arguments from `first` to `last` are all Python integers, as the classes pass them.
bool Ints(PyObject* const* args, int first, int last) {
  for (int i = first; i <= last; ++i)
    if (!PyLong_CheckExact(args[i])) return false;
  return true;
}

template <typename F>
PyObject* Guarded(F&& f) {
  try {
    return f();
  } catch (const std::exception&) {  // an allocation that fails, for one: the Python code meets it again
    PyErr_Clear();
    Py_RETURN_NONE;
  }
}

// conv(entry, handle, input type, output type, ic, oc, x, out, stream)
PyObject* Conv(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return Guarded([&]() -> PyObject* {
    if (n != 9 || !Ints(a, 0, 5)) Py_RETURN_NONE;
    const at::Tensor* x = Plain(a[6], static_cast<at::ScalarType>(PyLong_AsLong(a[2])));
    const int64_t ic = PyLong_AsLong(a[4]), oc = PyLong_AsLong(a[5]);
    if (!x || x->size(1) != ic || !Int32(x->size(0)) || !Int32(x->size(2) * x->size(3))) Py_RETURN_NONE;
    const int64_t shape[4] = {x->size(0), oc, x->size(2), x->size(3)};
    at::Tensor own;
    void *to = nullptr, *stream = nullptr;
    if (!Stream(a[8], *x, &stream) || !Output(a[7], *x, static_cast<at::ScalarType>(PyLong_AsLong(a[3])), shape, &own, &to)) Py_RETURN_NONE;
    const ConvRun run = reinterpret_cast<ConvRun>(PyLong_AsVoidPtr(a[0]));
    void* const handle = PyLong_AsVoidPtr(a[1]);
    const void* const from = x->data_ptr();
    int rc;
    Py_BEGIN_ALLOW_THREADS;
    rc = run(handle, from, to, static_cast<int32_t>(shape[0]), static_cast<int32_t>(shape[2] * shape[3]), stream);
    Py_END_ALLOW_THREADS;
    return Result(rc, a[7], own);
  });
}

// The output shape of a 3x3 layer behind `channels` planes of x.
struct DwShape {
  int64_t dims[4];
  DwShape(const at::Tensor& x, int64_t channels, int64_t stride, int64_t pad) : dims{x.size(0), channels, (x.size(2) + 2 * pad - 3) / stride + 1, (x.size(3) + 2 * pad - 3) / stride + 1} {}
  static bool Fits(const at::Tensor& x, int64_t stride, int64_t pad) { return stride > 0 && Int32(x.size(0)) && Int32(x.size(2)) && Int32(x.size(3)) && x.size(2) + 2 * pad >= 3 && x.size(3) + 2 * pad >= 3; }
};

// depthwise(entry, handle, output type, channels, stride, pad, current device, x, out, stream)
PyObject* Depthwise(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return Guarded([&]() -> PyObject* {
    if (n != 10 || !Ints(a, 0, 6)) Py_RETURN_NONE;
    const at::Tensor* x = Plain(a[7], at::kChar);
    const int64_t channels = PyLong_AsLong(a[3]), stride = PyLong_AsLong(a[4]), pad = PyLong_AsLong(a[5]);
    if (!x || x->size(1) != channels || x->get_device() != PyLong_AsLong(a[6]) || !DwShape::Fits(*x, stride, pad)) Py_RETURN_NONE;
    const DwShape shape(*x, channels, stride, pad);
    at::Tensor own;
    void *to = nullptr, *s = nullptr;
    if (!Stream(a[9], *x, &s) || !Output(a[8], *x, static_cast<at::ScalarType>(PyLong_AsLong(a[2])), shape.dims, &own, &to)) Py_RETURN_NONE;
    const DwRun run = reinterpret_cast<DwRun>(PyLong_AsVoidPtr(a[0]));
    void* const handle = PyLong_AsVoidPtr(a[1]);
    const int8_t* const from = static_cast<const int8_t*>(x->data_ptr());
    const int32_t batch = static_cast<int32_t>(x->size(0)), h = static_cast<int32_t>(x->size(2)), w = static_cast<int32_t>(x->size(3));
    int rc;
    Py_BEGIN_ALLOW_THREADS;
    rc = run(handle, from, to, batch, h, w, s);
    Py_END_ALLOW_THREADS;
    return Result(rc, a[8], own);
  });
}

// pair(entry, conv handle, depthwise handle, ic, oc, stride, pad, current device, x, out, stream)
PyObject* Pair(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return Guarded([&]() -> PyObject* {
    if (n != 11 || !Ints(a, 0, 7)) Py_RETURN_NONE;
    const at::Tensor* x = Plain(a[8], at::kChar);
    const int64_t ic = PyLong_AsLong(a[3]), oc = PyLong_AsLong(a[4]), stride = PyLong_AsLong(a[5]), pad = PyLong_AsLong(a[6]);
    if (!x || x->size(1) != ic || x->get_device() != PyLong_AsLong(a[7]) || !DwShape::Fits(*x, stride, pad)) Py_RETURN_NONE;
    const DwShape shape(*x, oc, stride, pad);
    at::Tensor own;
    void *to = nullptr, *s = nullptr;
    if (!Stream(a[10], *x, &s) || !Output(a[9], *x, at::kChar, shape.dims, &own, &to)) Py_RETURN_NONE;
    const PairRun run = reinterpret_cast<PairRun>(PyLong_AsVoidPtr(a[0]));
    void *const conv = PyLong_AsVoidPtr(a[1]), *const dw = PyLong_AsVoidPtr(a[2]);
    const void* const from = x->data_ptr();
    const int32_t batch = static_cast<int32_t>(x->size(0)), h = static_cast<int32_t>(x->size(2)), w = static_cast<int32_t>(x->size(3));
    int rc;
    Py_BEGIN_ALLOW_THREADS;
    rc = run(conv, dw, from, to, batch, h, w, s);
    Py_END_ALLOW_THREADS;
    return Result(rc, a[9], own);
  });
}

// type_code(tensor): the number the functions above know its element type by
PyObject* TypeCode(PyObject*, PyObject* t) {
  if (!THPVariable_Check(t)) Py_RETURN_NONE;
  return PyLong_FromLong(static_cast<long>(THPVariable_Unpack(t).scalar_type()));
}

PyMethodDef kMethods[] = {
    {"conv", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(Conv)), METH_FASTCALL, nullptr},
    {"depthwise", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(Depthwise)), METH_FASTCALL, nullptr},
    {"pair", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(Pair)), METH_FASTCALL, nullptr},
    {"type_code", TypeCode, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "pl_python_run", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_pl_python_run() { return PyModule_Create(&kModule); }
