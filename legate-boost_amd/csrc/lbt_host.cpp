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
#include <torch/csrc/Device.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>
#include <cstring>
#include <exception>
#include <vector>

#include "../../include/lbtree.h"

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

// The library's entries run with Python's lock given back. An exception that leaves one (it has vectors of its own) takes the lock again on
// its way to the handler, which gives references back and looks at Python's error. (Python ends a thread that asks for the
// lock while it shuts down by unwinding it, hence noexcept(false).)
struct Unlocked {
  PyThreadState* const state = PyEval_SaveThread();
  ~Unlocked() noexcept(false) { PyEval_RestoreThread(state); }
};
template <typename Call>
int unlocked(Call call)
{
  const Unlocked free;
  return call();
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
    const int64_t n = x.size(0), f = x.size(1);
    const int status = unlocked([&] {
      return entry(reinterpret_cast<void*>(number[1]), from, static_cast<int32_t>(number[3]), n, static_cast<int32_t>(f),
                   reinterpret_cast<const void*>(number[2]), to);
    });
    if (status != 0) return PyLong_FromLong(status);
    return THPVariable_Wrap(std::move(out));
  } catch (const std::exception&) {
    Py_RETURN_NONE;  // whatever it is, the caller meets it again in Python
  }
}

// Whether torch is being listened to: the calls below then go through Python
bool listened_to() { return at::impl::torch_function_mode_enabled() || c10::impl::TorchDispatchModeTLS::any_modes_set(); }

// A dense, contiguous device tensor of `type` and `dims` dimensions; null: something else
const at::Tensor* dense(PyObject* o, at::ScalarType type, int64_t dims)
{
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || t.layout() != at::kStrided || !t.is_cuda() || t.scalar_type() != type || t.dim() != dims || !t.is_contiguous()) return nullptr;
  return &t;
}

bool integers(PyObject* const* args, int n, int64_t* out)
{
  for (int i = 0; i < n; i++) {
    out[i] = PyLong_AsLongLong(args[i]);
    if (out[i] == -1 && PyErr_Occurred()) return false;
  }
  return true;
}
bool numbers(PyObject* const* args, int n, double* out)
{
  for (int i = 0; i < n; i++) {
    out[i] = PyFloat_AsDouble(args[i]);
    if (out[i] == -1.0 && PyErr_Occurred()) return false;
  }
  return true;
}

// After a number that is none: the caller meets it again in Python, which says what is wrong as it always did; what is no Exception (an
// interrupt) is passed on.
PyObject* not_a_number()
{
  if (!PyErr_ExceptionMatches(PyExc_Exception)) return nullptr;
  PyErr_Clear();
  Py_RETURN_NONE;
}

// build_tree(X, g, h, mask, workspace, entry, size_entry, stream, row_offset, max_depth, split_samples, seed, cache, row_leaf, l1, l2, gain):
// lbt_build_tree_async and lbt_build_tree_workspace_bytes, whose addresses are `entry` and `size_entry`, for a float or double matrix and gradients as they
// have to be on the device; mask: a uint8 tensor there or None; workspace(bytes, device): the scratch tensor. Returns (leaf_value, feature,
// split_value, gain, hessian, row_leaf or None), or the status where that is not 0, or None, with nothing done, for anything else: the
// caller then goes through Python. A round of boosting on 1000 x 10 took its host 57 us, with this, the two calls below and no copy of a plain learner 36.
using BuildTree      = decltype(&lbt_build_tree_async);
using WorkspaceBytes = decltype(&lbt_build_tree_workspace_bytes);
PyObject* build_tree(PyObject*, PyObject* const* args, Py_ssize_t n_args)
{
  if (n_args != 17) {
    PyErr_SetString(PyExc_TypeError, "build_tree takes 17 arguments");
    return nullptr;
  }
  int64_t v[9];
  double r[3];
  if (!integers(args + 5, 9, v) || !numbers(args + 14, 3, r)) return not_a_number();
  const int64_t row_offset = v[3], max_depth = v[4], samples = v[5], seed = v[6], cache = v[7];
  const bool row_leaf = v[8] != 0;
  try {
    if (listened_to()) Py_RETURN_NONE;
    const at::Tensor* x = dense(args[0], at::kFloat, 2);
    const bool wide     = x == nullptr;
    if (wide) x = dense(args[0], at::kDouble, 2);
    const at::Tensor *g = dense(args[1], at::kDouble, 2), *h = dense(args[2], at::kDouble, 2);
    if (x == nullptr || g == nullptr || h == nullptr || g->sizes() != h->sizes() || g->size(0) != x->size(0) || g->device() != x->device() ||
        h->device() != x->device() || max_depth < 0 || max_depth > 24 || samples < INT32_MIN || samples > INT32_MAX || seed < INT32_MIN ||
        seed > INT32_MAX || x->size(1) > INT32_MAX || g->size(1) > INT32_MAX)
      Py_RETURN_NONE;
    const at::Tensor* mask = nullptr;
    if (args[3] != Py_None) {
      mask = dense(args[3], at::kByte, 1);
      if (mask == nullptr || mask->size(0) != x->size(1) || mask->device() != x->device()) Py_RETURN_NONE;
    }
    const int64_t n = x->size(0);
    const int32_t f = static_cast<int32_t>(x->size(1)), k = static_cast<int32_t>(g->size(1));
    const int32_t type = wide ? LBT_F64 : LBT_F32, nodes = (1 << (max_depth + 1)) - 1;
    lbt_build_params prm{};
    prm.struct_bytes = sizeof(prm);
    prm.max_depth = static_cast<int32_t>(max_depth), prm.max_nodes = nodes, prm.split_samples = static_cast<int32_t>(samples);
    prm.seed = static_cast<int32_t>(seed), prm.dataset_rows = n;
    prm.l1_regularization = r[0], prm.l2_regularization = r[1], prm.min_split_gain = r[2];
    prm.hist_cache_bytes = cache;
    const size_t bytes = reinterpret_cast<WorkspaceBytes>(v[1])(n, f, k, prm.max_depth, prm.split_samples, type, cache);
    if (bytes == 0) Py_RETURN_NONE;  // an argument that is refused
    PyObject* device  = THPDevice_New(x->device());
    PyObject* scratch = device != nullptr ? PyObject_CallFunction(args[4], "KO", static_cast<unsigned long long>(bytes), device) : nullptr;
    Py_XDECREF(device);
    if (scratch == nullptr) {
      if (!PyErr_ExceptionMatches(PyExc_Exception)) return nullptr;
      PyErr_Clear();
      Py_RETURN_NONE;
    }
    Held keep;
    keep.objects.push_back(scratch);
    const at::Tensor* ws = dense(scratch, at::kByte, 1);
    if (ws == nullptr || ws->device() != x->device()) Py_RETURN_NONE;
    const auto real = x->options().dtype(at::kDouble), whole = x->options().dtype(at::kInt);
    at::Tensor leaf = at::empty({nodes, k}, real), feature = at::empty({nodes}, whole), split = at::empty({nodes}, real),
               gain = at::empty({nodes}, real), hessian = at::empty({nodes, k}, real), rows;
    lbt_build_taps taps{};
    if (row_leaf) {
      rows          = at::empty({n}, whole);
      taps.row_leaf = rows.mutable_data_ptr<int32_t>();
    }
    const void* const from       = x->const_data_ptr();
    const double* const grad     = g->const_data_ptr<double>();
    const double* const hess     = h->const_data_ptr<double>();
    const uint8_t* const allowed = mask != nullptr ? mask->const_data_ptr<uint8_t>() : nullptr;
    double* const to_leaf = leaf.mutable_data_ptr<double>();
    int32_t* const to_feature = feature.mutable_data_ptr<int32_t>();
    double* const to_split = split.mutable_data_ptr<double>();
    double* const to_gain = gain.mutable_data_ptr<double>();
    double* const to_hessian = hessian.mutable_data_ptr<double>();
    void* const room = ws->data_ptr();
    const size_t has = static_cast<size_t>(ws->numel());
    const int status = unlocked([&] {
      return reinterpret_cast<BuildTree>(v[0])(reinterpret_cast<void*>(v[2]), from, type, row_offset, n, f, grad, hess, k, allowed, &prm, to_leaf,
                                               to_feature, to_split, to_gain, to_hessian, room, has, row_leaf ? &taps : nullptr);
    });
    if (status != 0) return PyLong_FromLong(status);
    PyObject* out = PyTuple_New(6);
    if (out == nullptr) return nullptr;
    at::Tensor* const all[5] = {&leaf, &feature, &split, &gain, &hessian};
    for (int i = 0; i < 5; i++) PyTuple_SET_ITEM(out, i, THPVariable_Wrap(std::move(*all[i])));
    if (!row_leaf) Py_INCREF(Py_None);
    PyTuple_SET_ITEM(out, 5, row_leaf ? THPVariable_Wrap(std::move(rows)) : Py_None);
    return out;
  } catch (const std::exception&) {
    if (PyErr_Occurred()) PyErr_Clear();
    Py_RETURN_NONE;  // whatever it is, the caller meets it again in Python
  }
}

// weighted_gradient(y, pred, weight, entry, stream, objective, learning_rate): lbt_weighted_gradient on device doubles; weight: [rows] or None.
// Returns (g, h), a status that is not 0, or None as above.
PyObject* weighted_gradient(PyObject*, PyObject* const* args, Py_ssize_t n_args)
{
  if (n_args != 7) {
    PyErr_SetString(PyExc_TypeError, "weighted_gradient takes seven arguments");
    return nullptr;
  }
  int64_t v[3];
  double rate;
  if (!integers(args + 3, 3, v) || !numbers(args + 6, 1, &rate)) return not_a_number();
  try {
    if (listened_to()) Py_RETURN_NONE;
    const at::Tensor *y = dense(args[0], at::kDouble, 2), *pred = dense(args[1], at::kDouble, 2);
    if (y == nullptr || pred == nullptr || y->device() != pred->device() || pred->size(1) > INT32_MAX) Py_RETURN_NONE;
    const int64_t n = pred->size(0), k = pred->size(1);
    if (y->numel() != (v[2] == LBT_OBJ_LOG_LOSS && k > 1 ? n : n * k)) Py_RETURN_NONE;
    const at::Tensor* w = nullptr;
    if (args[2] != Py_None) {
      w = dense(args[2], at::kDouble, 1);
      if (w == nullptr || w->numel() != n || w->device() != pred->device()) Py_RETURN_NONE;
    }
    const auto real = pred->options().requires_grad(false);
    at::Tensor g = at::empty({n, k}, real), h = at::empty({n, k}, real);
    const double *const at = pred->const_data_ptr<double>(), *const target = y->const_data_ptr<double>();
    const double* const weight = w != nullptr ? w->const_data_ptr<double>() : nullptr;
    double *const to_g = g.mutable_data_ptr<double>(), *const to_h = h.mutable_data_ptr<double>();
    const int status = unlocked([&] {
      return reinterpret_cast<decltype(&lbt_weighted_gradient)>(v[0])(reinterpret_cast<void*>(v[1]), static_cast<int32_t>(v[2]), at, target, weight,
                                                                      rate, n, static_cast<int32_t>(k), to_g, to_h);
    });
    if (status != 0) return PyLong_FromLong(status);
    PyObject* out = PyTuple_New(2);
    if (out == nullptr) return nullptr;
    PyTuple_SET_ITEM(out, 0, THPVariable_Wrap(std::move(g)));
    PyTuple_SET_ITEM(out, 1, THPVariable_Wrap(std::move(h)));
    return out;
  } catch (const std::exception&) {
    Py_RETURN_NONE;
  }
}

// add_leaf_values(pred, leaf_value, row_leaf, entry, stream): lbt_add_leaf_values. Returns the status, or None as above.
PyObject* add_leaf_values(PyObject*, PyObject* const* args, Py_ssize_t n_args)
{
  if (n_args != 5) {
    PyErr_SetString(PyExc_TypeError, "add_leaf_values takes five arguments");
    return nullptr;
  }
  int64_t v[2];
  if (!integers(args + 3, 2, v)) return not_a_number();
  try {
    if (listened_to()) Py_RETURN_NONE;
    const at::Tensor *pred = dense(args[0], at::kDouble, 2), *leaf = dense(args[1], at::kDouble, 2), *rows = dense(args[2], at::kInt, 1);
    if (pred == nullptr || leaf == nullptr || rows == nullptr || leaf->size(1) != pred->size(1) || rows->size(0) != pred->size(0) ||
        leaf->device() != pred->device() || rows->device() != pred->device() || pred->size(1) > INT32_MAX || leaf->size(0) > INT32_MAX)
      Py_RETURN_NONE;
    const double* const from   = leaf->const_data_ptr<double>();
    const int32_t* const nodes = rows->const_data_ptr<int32_t>();
    double* const to           = static_cast<double*>(pred->data_ptr());
    const int64_t n = pred->size(0), k = pred->size(1), n_nodes = leaf->size(0);
    const int status = unlocked([&] {
      return reinterpret_cast<decltype(&lbt_add_leaf_values)>(v[0])(reinterpret_cast<void*>(v[1]), from, static_cast<int32_t>(n_nodes), nodes, n,
                                                                    static_cast<int32_t>(k), to);
    });
    return PyLong_FromLong(status);
  } catch (const std::exception&) {
    Py_RETURN_NONE;
  }
}

// next_gradient(pred, leaf_value, row_leaf, y, weight, g, h, sums, entry, stream, objective, learning_rate): lbt_next_gradient; weight: [rows] or
// None, sums: [2][chunks] or None. Returns the status, or None as above.
PyObject* next_gradient(PyObject*, PyObject* const* args, Py_ssize_t n_args)
{
  if (n_args != 12) {
    PyErr_SetString(PyExc_TypeError, "next_gradient takes twelve arguments");
    return nullptr;
  }
  int64_t v[3];
  double rate;
  if (!integers(args + 8, 3, v) || !numbers(args + 11, 1, &rate)) return not_a_number();
  try {
    if (listened_to()) Py_RETURN_NONE;
    const at::Tensor *pred = dense(args[0], at::kDouble, 2), *leaf = dense(args[1], at::kDouble, 2), *rows = dense(args[2], at::kInt, 1),
                     *y = dense(args[3], at::kDouble, 2), *g = dense(args[5], at::kDouble, 2), *h = dense(args[6], at::kDouble, 2);
    if (pred == nullptr || leaf == nullptr || rows == nullptr || y == nullptr || g == nullptr || h == nullptr) Py_RETURN_NONE;
    const int64_t n = pred->size(0), k = pred->size(1);
    for (const at::Tensor* t : {leaf, rows, y, g, h})
      if (t->device() != pred->device()) Py_RETURN_NONE;
    if (k > INT32_MAX || leaf->size(0) > INT32_MAX || leaf->size(1) != k || rows->size(0) != n || g->sizes() != pred->sizes() ||
        h->sizes() != pred->sizes() || y->numel() != (v[2] == LBT_OBJ_LOG_LOSS && k > 1 ? n : n * k))
      Py_RETURN_NONE;
    const at::Tensor *w = nullptr, *sums = nullptr;
    if (args[4] != Py_None) {
      w = dense(args[4], at::kDouble, 1);
      if (w == nullptr || w->numel() != n || w->device() != pred->device()) Py_RETURN_NONE;
    }
    if (args[7] != Py_None) {
      sums = dense(args[7], at::kDouble, 2);
      if (sums == nullptr || sums->numel() != 2 * ((n * k + 4095) / 4096) || sums->device() != pred->device()) Py_RETURN_NONE;
    }
    const double *const from = leaf->const_data_ptr<double>(), *const target = y->const_data_ptr<double>();
    const double* const weight = w != nullptr ? w->const_data_ptr<double>() : nullptr;
    const int32_t* const nodes = rows->const_data_ptr<int32_t>();
    double *const at = static_cast<double*>(pred->data_ptr()), *const to_g = g->mutable_data_ptr<double>(), *const to_h = h->mutable_data_ptr<double>();
    double* const to_sums = sums != nullptr ? sums->mutable_data_ptr<double>() : nullptr;
    const int64_t n_nodes = leaf->size(0);
    const int status      = unlocked([&] {
      return reinterpret_cast<decltype(&lbt_next_gradient)>(v[0])(reinterpret_cast<void*>(v[1]), static_cast<int32_t>(v[2]), from,
                                                                  static_cast<int32_t>(n_nodes), nodes, at, target, weight, rate, n,
                                                                  static_cast<int32_t>(k), to_g, to_h, to_sums);
    });
    return PyLong_FromLong(status);
  } catch (const std::exception&) {
    Py_RETURN_NONE;
  }
}

PyMethodDef methods[] = {{"tree_arrays", tree_arrays, METH_VARARGS, "addresses and node counts of an ensemble's arrays"},
                         {"model_arrays", model_arrays, METH_VARARGS, "the same from the attributes of an ensemble's models"},
                         {"predict_packed", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(predict_packed)), METH_FASTCALL,
                          "prediction with a packed ensemble"},
                         {"build_tree", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(build_tree)), METH_FASTCALL, "one tree"},
                         {"weighted_gradient", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(weighted_gradient)), METH_FASTCALL,
                          "gradients and hessians of a round"},
                         {"add_leaf_values", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(add_leaf_values)), METH_FASTCALL,
                          "prediction update of a round"},
                         {"next_gradient", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(next_gradient)), METH_FASTCALL,
                          "prediction update of a round, gradients and hessians of the next one"},
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
