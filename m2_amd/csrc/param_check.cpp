// CPython extension m2_amd._param_check: "are these still the tensors a plan was made from?"
//
// A plan of the native schedule (m2_amd/schedule.py) holds device addresses of some fifty tensors per layer and copies
// derived from four of them.  Before every use each tensor is looked up again where the modules keep it and its storage, address,
// type and shape (and, for those that copies were made from, its version counter) compared; so is every module on the way there, and
// every plain number that went into the plan (epsilons, filter constants, options).  For 12 layers that is about 1,300 look-ups: 0.1 ms in Python, 12 us here.  An address alone says little: the allocator gives it out
// again, and assigning to `.data` leaves the version counter where it was.  The weak reference keeps no memory alive but the
// storage's own record, so that no other storage can take its place.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <torch/csrc/autograd/python_variable.h>

#include <exception>
#include <type_traits>
#include <vector>

namespace {

struct ModuleSlot {
  PyObject *dict, *key, *expected;
  PyTypeObject* type;   // (a parametrisation changes the class of the module in its place)
};
struct TensorSlot {
  PyObject *dict, *key;
  c10::weak_intrusive_ptr<c10::StorageImpl> storage;
  const void* data;
  int64_t version;      // -1: not compared
  at::ScalarType dtype;
  c10::SmallVector<int64_t, 4> sizes, strides;
};
struct ValueSlot {
  PyObject *dict, *key, *expected;      // expected: null where the dict has no such key
};
struct Checker {
  PyObject_HEAD
  std::vector<ModuleSlot>* modules;
  std::vector<TensorSlot>* tensors;
  std::vector<ValueSlot>* values;
};

// The tensor at dict[key], or null (with or without a Python error).
const at::Tensor* look_up(PyObject* dict, PyObject* key) {
  PyObject* o = PyDict_GetItemWithError(dict, key);
  if (!o || !THPVariable_Check(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  return t.defined() && t.has_storage() ? &t : nullptr;
}
// Equal plain values: the object itself, or a number or text of the same type that compares equal.
bool same_value(PyObject* a, PyObject* b) {
  if (a == b) return true;
  if (!a || !b || Py_TYPE(a) != Py_TYPE(b) || !(PyFloat_CheckExact(a) || PyLong_CheckExact(a) || PyUnicode_CheckExact(a))) return false;
  return PyObject_RichCompareBool(a, b, Py_EQ) == 1;
}
int64_t version_of(const at::Tensor& t) { return t.is_inference() ? 0 : t._version(); }

bool same(const TensorSlot& s, const at::Tensor& t) {
  return t.storage().unsafeGetStorageImpl() == s.storage._unsafe_get_target() && t.const_data_ptr() == s.data &&
         t.scalar_type() == s.dtype && t.sizes().equals(s.sizes) && t.strides().equals(s.strides) && (s.version < 0 || version_of(t) == s.version);
}

// The dicts lead to modules, and those may lead back to the plan that holds this object: the garbage collector has to see them.
int checker_traverse(PyObject* self, visitproc visit, void* arg) {
  Checker* c = reinterpret_cast<Checker*>(self);
  if (c->modules)
    for (auto& m : *c->modules) { Py_VISIT(m.dict); Py_VISIT(m.key); Py_VISIT(m.expected); Py_VISIT(m.type); }
  if (c->tensors)
    for (auto& t : *c->tensors) { Py_VISIT(t.dict); Py_VISIT(t.key); }
  if (c->values)
    for (auto& v : *c->values) { Py_VISIT(v.dict); Py_VISIT(v.key); Py_VISIT(v.expected); }
  return 0;
}

// An emptied checker compares nothing: only the collector may call this.
int checker_clear(PyObject* self) {
  Checker* c = reinterpret_cast<Checker*>(self);
  std::vector<PyObject*> drop;                 // released when the slots are gone: a destructor may come back here
  if (c->modules)
    for (auto& m : *c->modules) drop.insert(drop.end(), {m.dict, m.key, m.expected, reinterpret_cast<PyObject*>(m.type)});
  if (c->tensors)
    for (auto& t : *c->tensors) drop.insert(drop.end(), {t.dict, t.key});
  if (c->values)
    for (auto& v : *c->values) drop.insert(drop.end(), {v.dict, v.key, v.expected});
  delete c->modules;
  delete c->tensors;
  delete c->values;
  c->modules = nullptr;
  c->tensors = nullptr;
  c->values = nullptr;
  for (PyObject* o : drop) Py_XDECREF(o);
  return 0;
}

void checker_dealloc(PyObject* self) {
  PyObject_GC_UnTrack(self);
  checker_clear(self);
  Py_TYPE(self)->tp_free(self);
}

// (dict, key) pairs and the object at each of them (a value may be absent)
template <typename Slot>
bool record(PyObject* list, std::vector<Slot>* slots) {
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(list); ++i) {
    PyObject *dict, *key;
    if (!PyArg_ParseTuple(PyList_GET_ITEM(list, i), "O!O", &PyDict_Type, &dict, &key)) return false;
    PyObject* o = PyDict_GetItemWithError(dict, key);
    if (!o && (PyErr_Occurred() || std::is_same<Slot, ModuleSlot>::value)) {
      if (!PyErr_Occurred()) PyErr_SetObject(PyExc_KeyError, key);
      return false;
    }
    if constexpr (std::is_same<Slot, ModuleSlot>::value) {
      slots->push_back({dict, key, o, Py_TYPE(o)});
      Py_INCREF(Py_TYPE(o));
    } else {
      slots->push_back({dict, key, o});
    }
    Py_INCREF(dict); Py_INCREF(key); Py_XINCREF(o);
  }
  return true;
}

// Checker(modules, tensors, values): lists of (dict, key), (dict, key, compare_version) and (dict, key); the present state is
// recorded.
PyObject* checker_new(PyTypeObject* type, PyObject* args, PyObject*) {
  PyObject *mods, *tens, *vals;
  if (!PyArg_ParseTuple(args, "O!O!O!", &PyList_Type, &mods, &PyList_Type, &tens, &PyList_Type, &vals)) return nullptr;
  Checker* c = reinterpret_cast<Checker*>(type->tp_alloc(type, 0));
  if (!c) return nullptr;
  c->modules = new std::vector<ModuleSlot>();
  c->tensors = new std::vector<TensorSlot>();
  c->values = new std::vector<ValueSlot>();
  if (!record(mods, c->modules) || !record(vals, c->values)) { Py_DECREF(c); return nullptr; }
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(tens); ++i) {
    PyObject *dict, *key;
    int ver;
    if (!PyArg_ParseTuple(PyList_GET_ITEM(tens, i), "O!Op", &PyDict_Type, &dict, &key, &ver)) { Py_DECREF(c); return nullptr; }
    try {                            // a tensor without memory behind it (fake, functional) throws: no exception may leave this entry
      const at::Tensor* t = look_up(dict, key);
      if (t) {
        c->tensors->push_back({dict, key, t->storage().getWeakStorageImpl(), t->const_data_ptr(), ver ? version_of(*t) : -1, t->scalar_type(),
                               {t->sizes().begin(), t->sizes().end()}, {t->strides().begin(), t->strides().end()}});
        Py_INCREF(dict); Py_INCREF(key);
        continue;
      }
      if (!PyErr_Occurred()) PyErr_SetObject(PyExc_KeyError, key);
    } catch (const std::exception& e) {
      PyErr_SetString(PyExc_ValueError, e.what());
    }
    Py_DECREF(c);
    return nullptr;
  }
  return reinterpret_cast<PyObject*>(c);
}

// unchanged() -> bool
PyObject* checker_unchanged(PyObject* self, PyObject*) {
  Checker* c = reinterpret_cast<Checker*>(self);
  if (!c->modules || !c->tensors || !c->values) Py_RETURN_FALSE;
  for (const auto& m : *c->modules)
    if (PyDict_GetItemWithError(m.dict, m.key) != m.expected || Py_TYPE(m.expected) != m.type) {
      if (PyErr_Occurred()) return nullptr;
      Py_RETURN_FALSE;
    }
  for (const auto& v : *c->values)
    if (!same_value(PyDict_GetItemWithError(v.dict, v.key), v.expected)) {
      if (PyErr_Occurred()) return nullptr;
      Py_RETURN_FALSE;
    }
  for (const auto& s : *c->tensors) {
    bool unchanged = false;
    try {
      const at::Tensor* t = look_up(s.dict, s.key);
      unchanged = t && same(s, *t);
    } catch (const std::exception&) {      // not a tensor with memory any more
    }
    if (!unchanged) {
      if (PyErr_Occurred()) return nullptr;
      Py_RETURN_FALSE;
    }
  }
  Py_RETURN_TRUE;
}

PyMethodDef checker_methods[] = {{"unchanged", checker_unchanged, METH_NOARGS, "True if every module, tensor and value is as recorded."},
                                 {nullptr, nullptr, 0, nullptr}};
PyTypeObject CheckerType = {PyVarObject_HEAD_INIT(nullptr, 0) "m2_amd._param_check.Checker"};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_param_check", nullptr, -1, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__param_check() {
  CheckerType.tp_basicsize = sizeof(Checker);
  CheckerType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_GC;
  CheckerType.tp_traverse = checker_traverse;
  CheckerType.tp_clear = checker_clear;
  CheckerType.tp_new = checker_new;
  CheckerType.tp_dealloc = checker_dealloc;
  CheckerType.tp_methods = checker_methods;
  if (PyType_Ready(&CheckerType) < 0) return nullptr;
  PyObject* m = PyModule_Create(&module_def);
  if (!m) return nullptr;
  Py_INCREF(&CheckerType);
  PyModule_AddObject(m, "Checker", reinterpret_cast<PyObject*>(&CheckerType));
  return m;
}
