// The Python side of a launch, natively: what Triton's JIT calls for every `kernel[grid](...)`.
//
// `Launcher` is the base of HIPLauncher (backend/driver.py).  Called with the launcher arguments of the reference
// (backend/driver.py:262-265) it turns the ordinary ones -- exact ints and floats, torch tensors on the GPU, None -- into
// tts_arg records on the stack and calls tts_launch with the GIL released; anything else (hooks, objects with a data_ptr
// method, numpy scalars, empty grids, every error) goes to the Python method `_generic`, before anything has happened, so
// that there is one place that says what such calls do.
// What bounds a small launch is the host.  With this work in Python and ctypes a call of vector add took 12.5 us of it and one
// of LayerNorm (nine arguments) 14.1, now 8.0 and 7.7: 3.8 in tts_launch, the rest Triton's own.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <climits>
#include <cstdint>

#include "../../include/tts_hip.h"

namespace {

using LaunchFn = tts_status (*)(tts_plan *, int, int, int, void *, const tts_arg *, int);
LaunchFn g_launch = nullptr;
PyObject *g_plan_type = nullptr, *g_raise = nullptr;            // _native.PlanHandle, _native._raise
PyObject *g_tensor_type = nullptr, *g_parameter_type = nullptr;  // torch.Tensor, torch.nn.Parameter: no overridden attributes
PyObject *g_chain_type = nullptr;                                // triton.knobs.HookChain, or None
PyObject *s_generic, *s_handle, *s_kinds, *s_is_cuda, *s_data_ptr, *s_calls;

constexpr int MAX_ARGS = 64, FIXED = 9;

struct Launcher {
  PyObject_HEAD
  int n;
  int pos[MAX_ARGS];      // positions of the runtime arguments among the kernel's arguments
  char is_ptr[MAX_ARGS];
};

// _bind(slots): [(position, is a pointer), ...]
PyObject *launcher_bind(PyObject *self, PyObject *slots) {
  Launcher *l = (Launcher *)self;
  l->n = -1;  // (until all is well: every call goes the general way)
  PyObject *seq = PySequence_Fast(slots, "slots");
  if (!seq) return nullptr;
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(seq);
  for (Py_ssize_t i = 0; i < n && i < MAX_ARGS; i++) {
    int p = 0, ptr = 0;
    if (!PyArg_ParseTuple(PySequence_Fast_GET_ITEM(seq, i), "ip", &p, &ptr)) {
      Py_DECREF(seq);
      return nullptr;
    }
    l->pos[i] = p;
    l->is_ptr[i] = (char)ptr;
  }
  if (n <= MAX_ARGS) l->n = (int)n;
  Py_DECREF(seq);
  Py_RETURN_NONE;
}

// a non-negative int that fits a grid extent
bool extent(PyObject *o, int *out) {
  if (!PyLong_CheckExact(o)) return false;
  int over = 0;
  const long long v = PyLong_AsLongLongAndOverflow(o, &over);
  if (over || v <= 0 || v > INT_MAX) return false;
  *out = (int)v;
  return true;
}

// the address of a tensor in device memory; false: leave it to `_generic` (no Python error is set)
bool device_address(PyObject *o, void **out) {
  if ((PyObject *)Py_TYPE(o) != g_tensor_type && (PyObject *)Py_TYPE(o) != g_parameter_type) return false;
  PyObject *cuda = PyObject_GetAttr(o, s_is_cuda);
  const bool on_gpu = cuda == Py_True;
  Py_XDECREF(cuda);
  PyObject *p = on_gpu ? PyObject_CallMethodNoArgs(o, s_data_ptr) : nullptr;
  const bool ok = p && PyLong_CheckExact(p);
  if (ok) *out = (void *)(uintptr_t)PyLong_AsUnsignedLongLongMask(p);
  Py_XDECREF(p);
  if (!ok) PyErr_Clear();
  return ok;
}

// Is there nothing to call: None, or Triton's chain of hooks (an exact triton.knobs.HookChain) with none in it?
bool no_hook(PyObject *hook) {
  if (hook == Py_None) return true;
  if ((PyObject *)Py_TYPE(hook) != g_chain_type) return false;
  PyObject *calls = PyObject_GetAttr(hook, s_calls);
  const bool none = calls && PyList_CheckExact(calls) && PyList_GET_SIZE(calls) == 0;
  Py_XDECREF(calls);
  if (!calls) PyErr_Clear();
  return none;
}

PyObject *launcher_call(PyObject *self, PyObject *args, PyObject *kwargs) {
  Launcher *l = (Launcher *)self;
  const Py_ssize_t given = PyTuple_GET_SIZE(args);
  auto general = [&]() -> PyObject * {
    PyObject *f = PyObject_GetAttr(self, s_generic);
    if (!f) return nullptr;
    PyObject *r = PyObject_Call(f, args, kwargs);
    Py_DECREF(f);
    return r;
  };
  if (kwargs || given < FIXED || l->n < 0 || !g_launch) return general();
  PyObject *const *a = &PyTuple_GET_ITEM(args, 0);
  int g[3];
  if (!extent(a[0], &g[0]) || !extent(a[1], &g[1]) || !extent(a[2], &g[2]) || !PyLong_CheckExact(a[3]) || (PyObject *)Py_TYPE(a[4]) != g_plan_type || !no_hook(a[7]) ||
      !no_hook(a[8]))
    return general();
  // the plan: its address and the kinds of its arguments, as PlanHandle keeps them
  PyObject *handle = PyObject_GetAttr(a[4], s_handle), *kinds = handle ? PyObject_GetAttr(a[4], s_kinds) : nullptr;
  tts_plan *plan = nullptr;
  tts_arg packed[MAX_ARGS];
  bool plain = kinds && PyLong_CheckExact(handle) && PyBytes_CheckExact(kinds) && PyBytes_GET_SIZE(kinds) == l->n;
  if (plain) plan = (tts_plan *)(uintptr_t)PyLong_AsUnsignedLongLongMask(handle);
  plain = plain && plan;
  for (int i = 0; plain && i < l->n; i++) {
    if (l->pos[i] < 0 || FIXED + l->pos[i] >= given) { plain = false; break; }
    PyObject *v = a[FIXED + l->pos[i]];
    tts_arg &t = packed[i];
    t.kind = PyBytes_AS_STRING(kinds)[i];
    t.reserved = 0;
    t.v.i = 0;
    if ((t.kind == TTS_ARG_PTR) != (l->is_ptr[i] != 0)) plain = false;
    else if (t.kind == TTS_ARG_PTR) {
      if (PyLong_CheckExact(v)) t.v.ptr = (void *)(uintptr_t)PyLong_AsUnsignedLongLongMask(v);
      else if (v != Py_None) plain = device_address(v, &t.v.ptr);
    } else if (t.kind == TTS_ARG_INT) {
      if (PyLong_Check(v)) t.v.i = (int64_t)PyLong_AsUnsignedLongLongMask(v);  // (bool too)
      else plain = false;
    } else {
      if (PyFloat_CheckExact(v)) t.v.f = PyFloat_AS_DOUBLE(v);
      else plain = false;
    }
  }
  Py_XDECREF(handle);
  Py_XDECREF(kinds);
  if (!plain) {
    PyErr_Clear();
    return general();
  }
  void *stream = (void *)(uintptr_t)PyLong_AsUnsignedLongLongMask(a[3]);
  const int n = l->n;
  tts_status st;
  Py_BEGIN_ALLOW_THREADS  // (args holds a reference to the plan and to every tensor)
  st = g_launch(plan, g[0], g[1], g[2], stream, packed, n);
  Py_END_ALLOW_THREADS
  if (st != TTS_OK) return PyObject_CallFunction(g_raise, "i", (int)st);
  Py_RETURN_NONE;
}

PyMethodDef launcher_methods[] = {{"_bind", launcher_bind, METH_O, "takes the runtime arguments' positions: [(position, is a pointer), ...]"}, {nullptr, nullptr, 0, nullptr}};
PyType_Slot launcher_slots[] = {{Py_tp_call, (void *)launcher_call}, {Py_tp_methods, launcher_methods}, {Py_tp_new, (void *)PyType_GenericNew}, {0, nullptr}};
PyType_Spec launcher_spec = {"tts_launch.Launcher", sizeof(Launcher), 0, Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE, launcher_slots};

// setup(address of tts_launch, PlanHandle, _raise, torch.Tensor, torch.nn.Parameter, the type of Triton's hook chains)
PyObject *setup(PyObject *, PyObject *args) {
  unsigned long long address = 0;
  PyObject *o[5];
  if (!PyArg_ParseTuple(args, "KOOOOO", &address, &o[0], &o[1], &o[2], &o[3], &o[4])) return nullptr;
  PyObject **to[5] = {&g_plan_type, &g_raise, &g_tensor_type, &g_parameter_type, &g_chain_type};
  for (int i = 0; i < 5; i++) {
    Py_INCREF(o[i]);
    Py_XSETREF(*to[i], o[i]);
  }
  g_launch = (LaunchFn)(uintptr_t)address;
  Py_RETURN_NONE;
}

PyMethodDef module_methods[] = {{"setup", setup, METH_VARARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "tts_launch", nullptr, -1, module_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_tts_launch(void) {
  s_generic = PyUnicode_InternFromString("_generic");
  s_handle = PyUnicode_InternFromString("_address");
  s_kinds = PyUnicode_InternFromString("_kinds");
  s_is_cuda = PyUnicode_InternFromString("is_cuda");
  s_calls = PyUnicode_InternFromString("calls");
  s_data_ptr = PyUnicode_InternFromString("data_ptr");
  PyObject *m = PyModule_Create(&module_def);
  if (!m) return nullptr;
  PyObject *type = PyType_FromSpec(&launcher_spec);
  if (!type || PyModule_AddObject(m, "Launcher", type) < 0) {
    Py_XDECREF(type);
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
