// What the Python side of a call does with its tensors, in C++: looks each of
// them over and hands back their addresses.
//
// A call on a small matrix or a few tokens takes as long as Python needs for it, and a
// layer of 128 experts has 768 tensors.  Looking at a tensor's type, device, strides and
// size from Python costs 0.4 us, here 0.03: the operator's six tensors 2.3 -> 0.4 us, a
// layer's 768 112 -> 22.
//
// Nothing is decided here: whatever is not plainly in order (no tensor, a subclass of
// one, another device, type, size or layout, no memory of its own) is answered with
// None or False, and the caller then takes its slow way, which raises the error that
// belongs to it.  No state is kept.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>

namespace {

// The address of a plain contiguous tensor on GPU `device`, of this type and (unless negative)
// this number of elements and dimensions; null if it is anything else.  An empty tensor has
// no address to find: the caller learns that it is in order through `fine`.
void *address_of(PyObject *object, PyObject *dtype, int64_t numel, int64_t dims, int64_t device, bool *fine) {
  *fine = false;
  if (!THPVariable_CheckExact(object) || !THPDtype_Check(dtype)) return nullptr;
  try {
    const at::Tensor &t = THPVariable_Unpack(object);
    if (!t.defined() || !t.is_cuda() || t.device().index() != device ||
        t.scalar_type() != reinterpret_cast<THPDtype *>(dtype)->scalar_type || !t.is_contiguous() ||
        (numel >= 0 && t.numel() != numel) || (dims >= 0 && t.dim() != dims))
      return nullptr;
    void *p = t.data_ptr();
    *fine = true;
    return p;
  } catch (...) {   // a tensor without memory: the slow way has the error for it
    return nullptr;
  }
}

bool integer(PyObject *object, int64_t *out) {
  if (!PyLong_Check(object)) return false;
  *out = PyLong_AsLongLong(object);
  if (*out == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

// addresses(spec, tensors, numels, device): spec[i] = (dtype, name, dims), all of them tuples.
PyObject *addresses(PyObject *, PyObject *const *args, Py_ssize_t n) {
  if (n != 4) {
    PyErr_SetString(PyExc_TypeError, "addresses(spec, tensors, numels, device)");
    return nullptr;
  }
  PyObject *spec = args[0], *tensors = args[1], *numels = args[2];
  int64_t device;
  if (!PyTuple_Check(spec) || !PyTuple_Check(tensors) || !PyTuple_Check(numels) || !integer(args[3], &device) ||
      PyTuple_GET_SIZE(spec) != PyTuple_GET_SIZE(tensors) || PyTuple_GET_SIZE(numels) != PyTuple_GET_SIZE(tensors))
    Py_RETURN_NONE;
  const Py_ssize_t count = PyTuple_GET_SIZE(tensors);
  PyObject *out = PyTuple_New(count);
  if (!out) return nullptr;
  for (Py_ssize_t i = 0; i < count; i++) {
    PyObject *what = PyTuple_GET_ITEM(spec, i);
    int64_t numel, dims;
    bool fine = PyTuple_Check(what) && PyTuple_GET_SIZE(what) == 3 &&
                integer(PyTuple_GET_ITEM(numels, i), &numel) && integer(PyTuple_GET_ITEM(what, 2), &dims);
    void *p = fine ? address_of(PyTuple_GET_ITEM(tensors, i), PyTuple_GET_ITEM(what, 0), numel, dims, device, &fine)
                   : nullptr;
    if (!fine) {
      Py_DECREF(out);
      Py_RETURN_NONE;
    }
    PyObject *address = PyLong_FromUnsignedLongLong(reinterpret_cast<uintptr_t>(p));
    if (!address) {
      Py_DECREF(out);
      return nullptr;
    }
    PyTuple_SET_ITEM(out, i, address);
  }
  return out;
}

// layer_addresses(table, row, layers, spec, numels, device): the addresses of layers[e][c] into
// table[row + c][e], an int64 tensor in host memory with a column per layer; False if some are not
// in order (what the table then holds is not to be used).
PyObject *layer_addresses(PyObject *, PyObject *const *args, Py_ssize_t n) {
  if (n != 6) {
    PyErr_SetString(PyExc_TypeError, "layer_addresses(table, row, layers, spec, numels, device)");
    return nullptr;
  }
  PyObject *layers = args[2], *spec = args[3], *numels = args[4];
  int64_t row, device, want[8], dims[8];
  if (!THPVariable_CheckExact(args[0]) || !integer(args[1], &row) || !PyList_Check(layers) || !PyTuple_Check(spec) ||
      !PyTuple_Check(numels) || !integer(args[5], &device) || PyTuple_GET_SIZE(spec) > 8 ||
      PyTuple_GET_SIZE(numels) != PyTuple_GET_SIZE(spec))
    Py_RETURN_FALSE;
  const Py_ssize_t count = PyList_GET_SIZE(layers), columns = PyTuple_GET_SIZE(spec);
  int64_t *table = nullptr;
  try {
    const at::Tensor &t = THPVariable_Unpack(args[0]);
    if (!t.defined() || !t.is_cpu() || t.scalar_type() != at::kLong || t.dim() != 2 || !t.is_contiguous() ||
        t.size(1) != count || row < 0 || row > t.size(0) - columns)
      Py_RETURN_FALSE;
    table = static_cast<int64_t *>(t.data_ptr()) + row * count;
  } catch (...) {
    Py_RETURN_FALSE;
  }
  for (Py_ssize_t c = 0; c < columns; c++) {
    PyObject *what = PyTuple_GET_ITEM(spec, c);
    if (!PyTuple_Check(what) || PyTuple_GET_SIZE(what) != 3 || !integer(PyTuple_GET_ITEM(numels, c), &want[c]) ||
        !integer(PyTuple_GET_ITEM(what, 2), &dims[c]))
      Py_RETURN_FALSE;
  }
  for (Py_ssize_t e = 0; e < count; e++) {
    PyObject *layer = PyList_GET_ITEM(layers, e);
    if (!PyTuple_Check(layer) || PyTuple_GET_SIZE(layer) != columns) Py_RETURN_FALSE;
    for (Py_ssize_t c = 0; c < columns; c++) {
      bool fine;
      void *p = address_of(PyTuple_GET_ITEM(layer, c), PyTuple_GET_ITEM(PyTuple_GET_ITEM(spec, c), 0), want[c],
                           dims[c], device, &fine);
      if (!fine) Py_RETURN_FALSE;
      table[c * count + e] = static_cast<int64_t>(reinterpret_cast<uintptr_t>(p));
    }
  }
  Py_RETURN_TRUE;
}

PyMethodDef kMethods[] = {
    {"addresses", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(addresses)), METH_FASTCALL, nullptr},
    {"layer_addresses", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(layer_addresses)), METH_FASTCALL,
     nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_tensor_args", nullptr, -1, kMethods,
                       nullptr,               nullptr,        nullptr, nullptr};

}  // namespace

#ifndef SUB1_TORCH_VERSION
#error "the build says which torch these headers are of"
#endif
// The classes behind a tensor differ from one torch to the next and nothing in the library's symbols
// says so: whoever loads the module compares this with the torch it has.
PyMODINIT_FUNC PyInit__tensor_args() {
  PyObject *module = PyModule_Create(&kModule);
  if (module && PyModule_AddStringConstant(module, "built_against", "qmoe_amd, built against torch " SUB1_TORCH_VERSION) < 0) {
    Py_DECREF(module);
    return nullptr;
  }
  return module;
}
