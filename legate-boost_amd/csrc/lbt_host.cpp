// lbtree._host: what calls of a few microseconds would spend in Python, as a Python extension: the per-tree part of the calls that take
// a whole ensemble, and the prediction with an ensemble that is packed.
//
// Such a call hands over three arrays per tree. Looking at three tensors from Python (type, device, layout, shape, address)
// takes about 1.4 us a tree: of the 162 us that a prediction of 1000 x 10 with 100 trees took, 140, while the kernels need
// 25. Here it is a few nanoseconds a tensor.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>
#include <cstring>
#include <exception>
#include <vector>

namespace {

// address of a dense, contiguous device tensor of `type` with the rows of the others; false: not of this form
bool take(PyObject* o, at::ScalarType type, int64_t* rows, int64_t columns, uint64_t* address)
{
  if (!THPVariable_CheckExact(o)) return false;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || t.layout() != at::kStrided || !t.is_cuda() || t.scalar_type() != type || t.dim() < 1 || !t.is_contiguous())
    return false;
  if (columns > 0 && (t.dim() != 2 || t.size(1) != columns)) return false;
  if (*rows < 0) *rows = t.size(0);
  if (t.size(0) != *rows || *rows < 1 || *rows > INT32_MAX) return false;
  *address = reinterpret_cast<uint64_t>(t.data_ptr());
  return true;
}

// The host arrays of an ensemble, tree by tree: addresses of the three device arrays, node counts.
struct Arrays {
  PyObject* out[4] = {};
  ~Arrays()
  {
    for (PyObject* o : out) Py_XDECREF(o);
  }
  bool open(Py_ssize_t n)
  {
    for (int i = 0; i < 4; i++)
      if ((out[i] = PyBytes_FromStringAndSize(nullptr, n * (i < 3 ? 8 : 4))) == nullptr) return false;
    return true;
  }
  // false: an array has to be converted or is not as it should be
  bool put(Py_ssize_t t, PyObject* leaf, PyObject* feature, PyObject* split, int64_t n_outputs)
  {
    int64_t rows = -1;
    uint64_t address[3];
    if (!take(leaf, at::kDouble, &rows, n_outputs, &address[0]) || !take(feature, at::kInt, &rows, 0, &address[1]) ||
        !take(split, at::kDouble, &rows, 0, &address[2]))
      return false;
    for (int i = 0; i < 3; i++) std::memcpy(PyBytes_AS_STRING(out[i]) + 8 * t, &address[i], 8);
    const int32_t nodes = static_cast<int32_t>(rows);
    std::memcpy(PyBytes_AS_STRING(out[3]) + 4 * t, &nodes, 4);
    return true;
  }
};

// tree_arrays(trees, n_outputs): trees is a list or tuple of (leaf_value [nodes, n_outputs] f64, feature [nodes] i32,
// split_value [nodes] f64). Returns the addresses of the three and the node counts as bytes (uint64, uint64, uint64,
// int32), or None when some array has to be converted or is not as it should be: the caller then looks closer.
PyObject* tree_arrays(PyObject*, PyObject* args)
{
  PyObject* trees;
  long long n_outputs;
  if (!PyArg_ParseTuple(args, "OL", &trees, &n_outputs)) return nullptr;
  if ((!PyList_CheckExact(trees) && !PyTuple_CheckExact(trees)) || n_outputs < 1) Py_RETURN_NONE;
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(trees);
  Arrays a;
  if (!a.open(n)) return nullptr;
  bool plain = true;
  try {
    for (Py_ssize_t t = 0; t < n && plain; t++) {
      PyObject* tree = PySequence_Fast_GET_ITEM(trees, t);
      plain = PyTuple_CheckExact(tree) && PyTuple_GET_SIZE(tree) == 3 &&
              a.put(t, PyTuple_GET_ITEM(tree, 0), PyTuple_GET_ITEM(tree, 1), PyTuple_GET_ITEM(tree, 2), n_outputs);
    }
  } catch (const std::exception&) {
    plain = false;  // whatever it is, the caller meets it again in Python
  }
  if (!plain) Py_RETURN_NONE;
  return PyTuple_Pack(4, a.out[0], a.out[1], a.out[2], a.out[3]);
}

// References that are given back when they are left
struct Held {
  std::vector<PyObject*> objects;
  ~Held()
  {
    for (PyObject* o : objects) Py_DECREF(o);
  }
};

// model_arrays(models, type, names, n_outputs): the same for a list or tuple of objects of `type` whose three attributes `names` are the
// arrays, and a fifth value: a list of the arrays, which keeps the addresses valid. (100 trees, 1000 rows: a call takes 24 us; through the tuples
// above, gathered in Python, 29.) An attribute may be code that changes the list or looks at what the collector knows: None where the
// list has another length at the end, and the arrays are no list before they are complete. What such code raises the caller meets
// again in Python, but for what is no Exception (an interrupt): that is passed on.
PyObject* model_arrays(PyObject*, PyObject* args)
{
  PyObject *models, *type, *names;
  long long n_outputs;
  if (!PyArg_ParseTuple(args, "OOOL", &models, &type, &names, &n_outputs)) return nullptr;
  if ((!PyList_CheckExact(models) && !PyTuple_CheckExact(models)) || !PyType_Check(type) || !PyTuple_CheckExact(names) ||
      PyTuple_GET_SIZE(names) != 3 || n_outputs < 1)
    Py_RETURN_NONE;
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(models);
  Arrays a;
  if (!a.open(n)) return nullptr;
  Held keep;
  bool plain = true;
  try {
    keep.objects.reserve(3 * n);
    for (Py_ssize_t t = 0; t < n && plain; t++) {
      plain = t < PySequence_Fast_GET_SIZE(models) &&
              PyObject_TypeCheck(PySequence_Fast_GET_ITEM(models, t), reinterpret_cast<PyTypeObject*>(type));
      if (!plain) break;
      PyObject* model = PySequence_Fast_GET_ITEM(models, t);
      Py_INCREF(model);
      PyObject* got[3] = {};
      for (int i = 0; i < 3 && plain; i++) {
        got[i] = PyObject_GetAttr(model, PyTuple_GET_ITEM(names, i));
        plain  = got[i] != nullptr;
        if (plain) keep.objects.push_back(got[i]);
      }
      Py_DECREF(model);
      plain = plain && a.put(t, got[0], got[1], got[2], n_outputs);
    }
  } catch (const std::exception&) {
    plain = false;
  }
  if (PyErr_Occurred()) {
    if (!PyErr_ExceptionMatches(PyExc_Exception)) return nullptr;
    PyErr_Clear();
  }
  if (!plain || PySequence_Fast_GET_SIZE(models) != n) Py_RETURN_NONE;
  PyObject* list = PyList_New(3 * n);
  if (list == nullptr) return nullptr;
  for (Py_ssize_t i = 0; i < 3 * n; i++) PyList_SET_ITEM(list, i, keep.objects[static_cast<size_t>(i)]);
  keep.objects.clear();  // (the list has the references)
  PyObject* result = PyTuple_Pack(5, a.out[0], a.out[1], a.out[2], a.out[3], list);
  Py_DECREF(list);
  return result;
}

// predict_packed(X, entry, stream, ensemble, dtype, n_outputs): lbt_predict_packed, whose address is `entry`, on a dense float (dtype 0) or
// double (1) matrix on the device. Returns the predictions, or the status where that is not 0, or None where X is something else or torch is
// being listened to: the caller then goes through Python.
using PredictPacked = int (*)(void*, const void*, int32_t, int64_t, int32_t, const void*, double*);
PyObject* predict_packed(PyObject*, PyObject* const* args, Py_ssize_t n_args)
{
  if (n_args != 6) {
    PyErr_SetString(PyExc_TypeError, "predict_packed takes six arguments");
    return nullptr;
  }
  if (!THPVariable_CheckExact(args[0])) Py_RETURN_NONE;
  uint64_t number[5];
  for (int i = 0; i < 5; i++) {
    number[i] = PyLong_AsUnsignedLongLong(args[1 + i]);
    if (number[i] == static_cast<uint64_t>(-1) && PyErr_Occurred()) return nullptr;
  }
  try {
    if (at::impl::torch_function_mode_enabled() || c10::impl::TorchDispatchModeTLS::any_modes_set()) Py_RETURN_NONE;
    const at::Tensor& x = THPVariable_Unpack(args[0]);
    if (!x.defined() || x.layout() != at::kStrided || !x.is_cuda() || x.dim() != 2 || !x.is_contiguous() ||
        x.scalar_type() != (number[3] == 0 ? at::kFloat : at::kDouble) || x.size(1) > INT32_MAX)
      Py_RETURN_NONE;
    at::Tensor out = at::empty({x.size(0), static_cast<int64_t>(number[4])}, x.options().dtype(at::kDouble));
    const auto entry = reinterpret_cast<PredictPacked>(number[0]);
    const void* from = x.const_data_ptr();
    double* const to = out.mutable_data_ptr<double>();
    int status       = 0;
    Py_BEGIN_ALLOW_THREADS
    status = entry(reinterpret_cast<void*>(number[1]), from, static_cast<int32_t>(number[3]), x.size(0), static_cast<int32_t>(x.size(1)),
                   reinterpret_cast<const void*>(number[2]), to);
    Py_END_ALLOW_THREADS
    if (status != 0) return PyLong_FromLong(status);
    return THPVariable_Wrap(std::move(out));
  } catch (const std::exception&) {
    Py_RETURN_NONE;  // whatever it is, the caller meets it again in Python
  }
}

PyMethodDef methods[] = {{"tree_arrays", tree_arrays, METH_VARARGS, "addresses and node counts of an ensemble's arrays"},
                         {"model_arrays", model_arrays, METH_VARARGS, "the same from the attributes of an ensemble's models"},
                         {"predict_packed", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(predict_packed)), METH_FASTCALL,
                          "prediction with a packed ensemble"},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// torch_version: what this was compiled against; the layout of a tensor is that of this version alone
PyMODINIT_FUNC PyInit__host()
{
  PyObject* m = PyModule_Create(&module);
  if (m != nullptr && PyModule_AddStringConstant(m, "torch_version", LBT_TORCH_VERSION) != 0) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
