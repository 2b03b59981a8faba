// lbtree._host: the per-tree part of the calls that take a whole ensemble, as a Python extension.
//
// Such a call hands over three arrays per tree. Looking at three tensors from Python (type, device, layout, shape, address)
// takes about 1.4 us a tree: of the 162 us that a prediction of 1000 x 10 with 100 trees took, 140, while the kernels need
// 25. Here it is a few nanoseconds a tensor.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>
#include <cstring>
#include <exception>

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
  PyObject* out[4]   = {};
  for (int i = 0; i < 4; i++) {
    out[i] = PyBytes_FromStringAndSize(nullptr, n * (i < 3 ? 8 : 4));
    if (out[i] == nullptr) {
      for (int j = 0; j < i; j++) Py_DECREF(out[j]);
      return nullptr;
    }
  }
  bool plain = true;
  try {
    for (Py_ssize_t t = 0; t < n && plain; t++) {
      PyObject* tree = PySequence_Fast_GET_ITEM(trees, t);
      if (!PyTuple_CheckExact(tree) || PyTuple_GET_SIZE(tree) != 3) {
        plain = false;
        break;
      }
      int64_t rows = -1;
      uint64_t address[3];
      plain = take(PyTuple_GET_ITEM(tree, 0), at::kDouble, &rows, n_outputs, &address[0]) &&
              take(PyTuple_GET_ITEM(tree, 1), at::kInt, &rows, 0, &address[1]) &&
              take(PyTuple_GET_ITEM(tree, 2), at::kDouble, &rows, 0, &address[2]);
      if (!plain) break;
      for (int i = 0; i < 3; i++) std::memcpy(PyBytes_AS_STRING(out[i]) + 8 * t, &address[i], 8);
      const int32_t nodes = static_cast<int32_t>(rows);
      std::memcpy(PyBytes_AS_STRING(out[3]) + 4 * t, &nodes, 4);
    }
  } catch (const std::exception&) {
    plain = false;  // whatever it is, the caller meets it again in Python
  }
  PyObject* result = plain ? PyTuple_Pack(4, out[0], out[1], out[2], out[3]) : nullptr;
  for (int i = 0; i < 4; i++) Py_DECREF(out[i]);
  if (plain) return result;
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {{"tree_arrays", tree_arrays, METH_VARARGS, "addresses and node counts of an ensemble's arrays"},
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
