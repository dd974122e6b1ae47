// Python entry to libpikv_hip.so: one function per entry point of include/pikv_hip.h, typed by its declaration.
//
// A call of one launch spends about 2.5 us in the launch; through ctypes the conversion of its 12 to 25 arguments, a Python call
// per tensor for its address among them, took 5 us more, which is what bounded the small calls (a decode step of 1 x 700
// tokens: three calls, 31 addresses).  Arguments here: for a pointer into GPU memory a GPU tensor (anything with is_cuda and
// data_ptr()), an address as int or as a ctypes pointer, None; for a host array a list of such or of numbers, a ctypes array, or
// an object with a buffer of the parameter's element type (numpy).  A list, a buffer or a CPU tensor where a kernel would read it is
// refused; whether a tensor is on the GPU is not asked again in the module `of_checked`, the same functions for callers that have
// checked theirs (31 addresses of a decode step of 1 x 700 tokens: 25.3 us, 26.7 with the question).
// Beside them the two checks that run for every tensor of a call (56 and 47 times in an evaluation pass of the
// mixture-of-experts model).  The symbols come from the library that load() is given; the GIL is released around each call.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <dlfcn.h>

#include <cstdint>
#include <cstring>
#include <tuple>
#include <type_traits>
#include <utility>

#include "../../include/pikv_hip.h"

namespace {

PyObject *g_data_ptr, *g_is_cuda, *g_is_contiguous, *g_dtype, *g_device, *g_dim, *g_value, *g_from_param;
PyObject *g_cast, *g_void_p;             // ctypes.cast, ctypes.c_void_p
PyObject *g_pointers;                    // (c_void_p, the base of ctypes' pointer classes)
PyObject *g_pointer_to[4];               // POINTER(c_void_p), POINTER(c_int32), POINTER(c_int64), POINTER(c_float)
PyObject *g_tensor, *g_parameter;        // torch.Tensor, torch.nn.Parameter
PyObject *g_refuse, *g_has_storage;      // ops._refuse, torch._C._has_storage

// Host arrays of one call.
struct Arena {
  alignas(16) unsigned char bytes[4096];
  size_t used = 0;
  void* take(size_t n) {
    const size_t at = (used + 15) / 16 * 16;
    if (n > sizeof(bytes) - at) {
      PyErr_SetString(PyExc_ValueError, "argument lists are too long");
      return nullptr;
    }
    used = at + n;
    return bytes + at;
  }
};

bool tensor_address(PyObject* t, void*& p) {
  PyObject* a = PyObject_CallMethodNoArgs(t, g_data_ptr);
  if (!a) return false;
  p = PyLong_AsVoidPtr(a);
  Py_DECREF(a);
  return !PyErr_Occurred();
}

// The value of a ctypes pointer, or the address of a ctypes array.
bool ctypes_address(PyObject* o, void*& p) {
  PyObject* c = PyObject_CallFunctionObjArgs(g_cast, o, g_void_p, nullptr);
  PyObject* v = c ? PyObject_GetAttr(c, g_value) : nullptr;
  Py_XDECREF(c);
  if (!v) return false;
  p = v == Py_None ? nullptr : PyLong_AsVoidPtr(v);
  Py_DECREF(v);
  return !PyErr_Occurred();
}

// A pointer into GPU memory.  CHECKED: the caller has seen that its tensors are there.
template <bool CHECKED>
bool address(PyObject* o, void*& p) {
  if (o == Py_None) {
    p = nullptr;
    return true;
  }
  if (PyLong_Check(o)) {
    p = PyLong_AsVoidPtr(o);
    return !PyErr_Occurred();
  }
  bool refused = PyList_Check(o) || PyTuple_Check(o);
  if (!refused && PyObject_CheckBuffer(o)) {             // host memory, but for the pointers of ctypes
    const int r = PyObject_IsInstance(o, g_pointers);
    if (r != 0) return r > 0 && ctypes_address(o, p);
    refused = true;
  }
  if (!refused && CHECKED) return tensor_address(o, p);
  if (!refused) {
    PyObject* cuda = PyObject_GetAttr(o, g_is_cuda);
    const int r = cuda ? PyObject_IsTrue(cuda) : -1;
    Py_XDECREF(cuda);
    if (r != 0) return r > 0 && tensor_address(o, p);
  }
  PyErr_Format(PyExc_TypeError, "a pointer into GPU memory is a GPU tensor, an address or None, not a %s%s",
               refused ? "" : "CPU ", Py_TYPE(o)->tp_name);
  return false;
}

template <typename T>
bool number(PyObject* o, T& v) {
  if constexpr (std::is_floating_point_v<T>) {
    const double d = PyFloat_AsDouble(o);
    if (d == -1.0 && PyErr_Occurred()) return false;
    v = (T)d;
  } else {
    PyObject* i = PyNumber_Index(o);
    if (!i) return false;
    const long long n = PyLong_AsLongLong(i);
    Py_DECREF(i);
    if (n == -1 && PyErr_Occurred()) return false;
    v = (T)n;
    if ((long long)v != n) {
      PyErr_SetString(PyExc_OverflowError, "an integer argument does not fit its parameter");
      return false;
    }
  }
  return true;
}

// A host array of E from an object with a buffer of that element type.
template <typename E>
bool host_buffer(PyObject* o, E*& a, Arena& arena) {
  Py_buffer b;
  if (PyObject_GetBuffer(o, &b, PyBUF_CONTIG_RO | PyBUF_FORMAT) != 0) return false;
  const char* f = b.format ? b.format : "B";
  if (*f == '@' || *f == '=' || *f == '<') ++f;
  const char* const kinds = std::is_pointer_v<E> ? "PlLqQnN" : std::is_floating_point_v<E> ? "fd" : "ilqn";
  bool ok = b.ndim == 1 && b.itemsize == (Py_ssize_t)sizeof(E) && f[0] != 0 && f[1] == 0 && std::strchr(kinds, f[0]);
  if (!ok) {
    PyErr_Format(PyExc_TypeError, "a host array of another element type or shape (format %s)", b.format ? b.format : "B");
  } else {
    a = static_cast<E*>(arena.take((size_t)b.len));
    ok = a != nullptr;
    if (ok) std::memcpy(a, b.buf, (size_t)b.len);
  }
  PyBuffer_Release(&b);
  return ok;
}

template <bool CHECKED, typename E>
bool host_array(PyObject* o, E*& a, Arena& arena) {
  static_assert(std::is_pointer_v<E> || std::is_same_v<E, int32_t> || std::is_same_v<E, int64_t> || std::is_same_v<E, float>);
  a = nullptr;
  if (o == Py_None) return true;
  if (PyList_Check(o) || PyTuple_Check(o)) {
    const Py_ssize_t n = PySequence_Fast_GET_SIZE(o);
    a = static_cast<E*>(arena.take((size_t)n * sizeof(E)));
    if (!a) return false;
    for (Py_ssize_t i = 0; i < n; ++i) {
      PyObject* e = PySequence_Fast_GET_ITEM(o, i);
      if constexpr (std::is_pointer_v<E>) {
        void* p = nullptr;
        if (!address<CHECKED>(e, p)) return false;
        a[i] = static_cast<E>(p);
      } else if (!number(e, a[i])) {
        return false;
      }
    }
    return true;
  }
  constexpr int kind = std::is_pointer_v<E> ? 0 : std::is_same_v<E, int32_t> ? 1 : std::is_same_v<E, int64_t> ? 2 : 3;
  PyObject* c = PyObject_CallMethodOneArg(g_pointer_to[kind], g_from_param, o);   // a ctypes array or pointer of that type
  if (c) {
    void* p = nullptr;
    const bool ok = ctypes_address(c, p);
    Py_DECREF(c);
    a = static_cast<E*>(p);
    return ok;
  }
  if (!PyErr_ExceptionMatches(PyExc_TypeError) || !PyObject_CheckBuffer(o)) return false;
  PyErr_Clear();
  return host_buffer(o, a, arena);
}

// HOST: a pointer parameter that is a host array (every pointer to pointers is one).
template <bool CHECKED, bool HOST, typename T>
bool convert(PyObject* o, T& v, Arena& arena) {
  if constexpr (!std::is_pointer_v<T>) {
    static_assert(!HOST, "a host array is a pointer");
    return number(o, v);
  } else {
    using E = std::remove_cv_t<std::remove_pointer_t<T>>;
    if constexpr (HOST || std::is_pointer_v<E>) {
      E* a = nullptr;
      if (!host_array<CHECKED, E>(o, a, arena)) return false;
      v = a;
      return true;
    } else {
      void* p = nullptr;
      if (!address<CHECKED>(o, p)) return false;
      v = static_cast<T>(p);
      return true;
    }
  }
}

// HOSTS: the parameters that are host arrays of numbers, a bit each.
template <bool CHECKED, uint32_t HOSTS, typename R, typename... A, size_t... I>
PyObject* invoke(R (*f)(A...), const char* name, PyObject* const* args, Py_ssize_t n, std::index_sequence<I...>) {
  if (!f) return PyErr_Format(PyExc_RuntimeError, "%s: no library loaded", name);
  if (n != (Py_ssize_t)sizeof...(A)) return PyErr_Format(PyExc_TypeError, "%s takes %d arguments, got %zd", name, (int)sizeof...(A), n);
  Arena arena;
  std::tuple<std::decay_t<A>...> v{};
  if (!(convert<CHECKED, (I < 32 && (HOSTS >> I % 32 & 1) != 0)>(args[I], std::get<I>(v), arena) && ...)) return nullptr;
  R r;
  Py_BEGIN_ALLOW_THREADS
  r = f(std::get<I>(v)...);
  Py_END_ALLOW_THREADS
  return PyLong_FromLongLong((long long)r);
}
template <bool CHECKED, uint32_t HOSTS, typename R, typename... A>
PyObject* invoke(R (*f)(A...), const char* name, PyObject* const* args, Py_ssize_t n) {
  return invoke<CHECKED, HOSTS>(f, name, args, n, std::index_sequence_for<A...>());
}

struct Entry {
  const char* name;
  void** slot;
};

// name, and the positions of its host arrays of numbers
#define PIKV_ENTRIES(X)                                                                                                       \
  X(pikv_abi_version, 0) X(pikv_router_fused, 0) X(pikv_router_tail, 0) X(pikv_capacity_slots, 0)                             \
  X(pikv_capacity_slots_static, 0) X(pikv_capacity_slots_static_max, 0) X(pikv_router_workspace_bytes, 0)                     \
  X(pikv_router_fused_workspace_bytes, 0) X(pikv_quant_scatter, 0) X(pikv_cache_advance, 0) X(pikv_quant_gather, 0)           \
  X(pikv_quant_append, 0) X(pikv_quantize_rows, 0) X(pikv_quant8_minshift, 0) X(pikv_gather_dequant, 0)                       \
  X(pikv_gather_dequant_scores, 0) X(pikv_h2o_accumulate, 0) X(pikv_attend_values, 0) X(pikv_attend_workspace_bytes, 0)       \
  X(pikv_decode_attend, 0) X(pikv_decode_attend_workspace_bytes, 0) X(pikv_prefill_attend, 0)                                 \
  X(pikv_prefill_attend_workspace_bytes, 0) X(pikv_evict_select, 0) X(pikv_evict_select_h2o, 0)                               \
  X(pikv_evict_workspace_bytes, 0) X(pikv_h2o_budget, 0) X(pikv_cache_make_room, bits(16)) X(pikv_compact_rows, bits(1))      \
  X(pikv_linear_group, bits(6, 7, 11)) X(pikv_linear_group_workspace_bytes, 0) X(pikv_linear_tiled, bits(6))                  \
  X(pikv_cache_mean, 0) X(pikv_cache_mean_workspace_bytes, 0) X(pikv_value_lora, bits(6)) X(pikv_expert_combine, bits(2))     \
  X(pikv_expert_combine_factors, bits(4)) X(pikv_adaptive_router, 0) X(pikv_quant_scatter_routed, 0)                          \
  X(pikv_fakequant_colblocks, 0) X(pikv_fakequant_workspace_bytes, 0) X(pikv_fakequant_preset, 0)

template <typename... P>
constexpr uint32_t bits(P... p) { return ((1u << p) | ...); }

#define PIKV_DEFINE(name, hosts)                                                              \
  decltype(&::name) f_##name = nullptr;                                                       \
  template <bool CHECKED>                                                                     \
  PyObject* c_##name(PyObject*, PyObject* const* args, Py_ssize_t n) { return invoke<CHECKED, hosts>(f_##name, #name, args, n); }
PIKV_ENTRIES(PIKV_DEFINE)

#define PIKV_SLOT(name, hosts) {#name, reinterpret_cast<void**>(&f_##name)},
const Entry g_entries[] = {PIKV_ENTRIES(PIKV_SLOT)};

PyObject* load(PyObject*, PyObject* path) {
  const char* p = PyUnicode_AsUTF8(path);
  if (!p) return nullptr;
  void* lib = dlopen(p, RTLD_NOW | RTLD_LOCAL);
  if (!lib) return PyErr_Format(PyExc_OSError, "%s", dlerror());
  const auto version = reinterpret_cast<decltype(&::pikv_abi_version)>(dlsym(lib, "pikv_abi_version"));
  if (!version || version() != PIKV_ABI_VERSION)         // its functions may have other arguments
    return PyErr_Format(PyExc_OSError, "%s has ABI version %d, this extension was built for %d", p, version ? version() : 0, PIKV_ABI_VERSION);
  for (const Entry& e : g_entries) {
    void* s = dlsym(lib, e.name);
    if (!s) return PyErr_Format(PyExc_OSError, "%s: no symbol %s", p, e.name);
    *e.slot = s;
  }
  Py_RETURN_NONE;
}

// -1: an exception is set
int is_true(PyObject* o) {
  if (!o) return -1;
  const int r = PyObject_IsTrue(o);
  Py_DECREF(o);
  return r;
}
int is_same(PyObject* o, PyObject* want) {
  if (!o) return -1;
  Py_DECREF(o);
  return o == want;
}

PyObject* setup(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 4) return PyErr_Format(PyExc_TypeError, "setup takes 4 arguments");
  PyObject** const to[] = {&g_tensor, &g_parameter, &g_refuse, &g_has_storage};
  for (int i = 0; i < 4; ++i) {
    Py_INCREF(args[i]);
    Py_XSETREF(*to[i], args[i]);
  }
  Py_RETURN_NONE;
}

// need(t, name, *, dtype=None, ndim=None, optional=False): t, if it is a contiguous GPU tensor of that dtype and number of
// dimensions (or None and optional); what it is not, g_refuse(t, name, dtype, ndim) says in an exception.
PyObject* need(PyObject*, PyObject* const* args, Py_ssize_t n, PyObject* kw) {
  if (n != 2 || !g_tensor) return PyErr_Format(PyExc_TypeError, "need(t, name, *, dtype, ndim, optional)");
  PyObject *t = args[0], *dtype = Py_None, *ndim = Py_None;
  bool optional = false;
  for (Py_ssize_t i = 0; kw && i < PyTuple_GET_SIZE(kw); ++i) {
    const char* k = PyUnicode_AsUTF8(PyTuple_GET_ITEM(kw, i));
    if (!k) return nullptr;
    PyObject* v = args[n + i];
    if (std::strcmp(k, "dtype") == 0) dtype = v;
    else if (std::strcmp(k, "ndim") == 0) ndim = v;
    else if (std::strcmp(k, "optional") == 0) { const int o = PyObject_IsTrue(v); if (o < 0) return nullptr; optional = o; }
    else return PyErr_Format(PyExc_TypeError, "need: no argument %s", k);
  }
  int ok;
  if (t == Py_None) ok = optional;
  else ok = PyType_IsSubtype(Py_TYPE(t), reinterpret_cast<PyTypeObject*>(g_tensor));
  if (ok > 0 && t != Py_None) {
    ok = is_true(PyObject_GetAttr(t, g_is_cuda));
    if (ok > 0) ok = is_true(PyObject_CallMethodNoArgs(t, g_is_contiguous));
    if (ok > 0 && dtype != Py_None) ok = is_same(PyObject_GetAttr(t, g_dtype), dtype);
    if (ok > 0 && ndim != Py_None) {
      PyObject* d = PyObject_CallMethodNoArgs(t, g_dim);
      ok = d ? PyObject_RichCompareBool(d, ndim, Py_EQ) : -1;
      Py_XDECREF(d);
    }
  }
  if (ok < 0) return nullptr;
  if (ok) return Py_NewRef(t);
  PyObject* said = PyObject_CallFunctionObjArgs(g_refuse, t, args[1], dtype, ndim, nullptr);
  if (!said) return nullptr;
  Py_DECREF(said);
  return PyErr_Format(PyExc_ValueError, "%U is not what the operator needs", args[1]);
}

// ordinary(t, device, dtype, align): whether t is a dense tensor (no subclass but Parameter) of that device and dtype that a kernel
// may read by its address, `align` bytes at a time.
PyObject* ordinary(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 4 || !g_tensor) return PyErr_Format(PyExc_TypeError, "ordinary(t, device, dtype, align)");
  PyObject* t = args[0];
  PyObject* const type = reinterpret_cast<PyObject*>(Py_TYPE(t));
  if (type != g_tensor && type != g_parameter) Py_RETURN_FALSE;
  PyObject* d = PyObject_GetAttr(t, g_device);
  int ok = d ? PyObject_RichCompareBool(d, args[1], Py_EQ) : -1;
  Py_XDECREF(d);
  if (ok > 0) ok = is_same(PyObject_GetAttr(t, g_dtype), args[2]);
  if (ok > 0) ok = is_true(PyObject_CallMethodNoArgs(t, g_is_contiguous));
  if (ok > 0) ok = is_true(PyObject_CallOneArg(g_has_storage, t));     // a batched tensor has none
  if (ok > 0) {
    void* p = nullptr;
    const long long align = PyLong_AsLongLong(args[3]);
    ok = align < 1 || !tensor_address(t, p) ? -1 : reinterpret_cast<uintptr_t>(p) % (uintptr_t)align == 0;
    if (ok < 0 && !PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "align");
  }
  if (ok < 0) return nullptr;
  return PyBool_FromLong(ok);
}

#define PIKV_METHOD(name, hosts) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(c_##name<false>)), METH_FASTCALL, nullptr},
#define PIKV_METHOD_CHECKED(name, hosts) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(c_##name<true>)), METH_FASTCALL, nullptr},
PyMethodDef g_methods[] = {PIKV_ENTRIES(PIKV_METHOD){"load", load, METH_O, nullptr},
                          {"setup", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(setup)), METH_FASTCALL, nullptr},
                          {"need", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(need)), METH_FASTCALL | METH_KEYWORDS, nullptr},
                          {"ordinary", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(ordinary)), METH_FASTCALL, nullptr},
                          {nullptr, nullptr, 0, nullptr}};
PyMethodDef g_checked_methods[] = {PIKV_ENTRIES(PIKV_METHOD_CHECKED){nullptr, nullptr, 0, nullptr}};

PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_call", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};
PyModuleDef g_checked_module = {PyModuleDef_HEAD_INIT, "_call.of_checked", nullptr, -1, g_checked_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__call() {
  PyObject** const names[] = {&g_data_ptr, &g_is_cuda, &g_is_contiguous, &g_dtype, &g_device, &g_dim, &g_value, &g_from_param};
  const char* const text[] = {"data_ptr", "is_cuda", "is_contiguous", "dtype", "device", "dim", "value", "from_param"};
  for (int i = 0; i < 8; ++i)
    if (!(*names[i] = PyUnicode_InternFromString(text[i]))) return nullptr;
  PyObject* ctypes = PyImport_ImportModule("ctypes");
  if (!ctypes) return nullptr;
  g_cast = PyObject_GetAttrString(ctypes, "cast");
  g_void_p = PyObject_GetAttrString(ctypes, "c_void_p");
  PyObject* pointer = PyObject_GetAttrString(ctypes, "_Pointer");
  const char* const element[] = {"c_void_p", "c_int32", "c_int64", "c_float"};
  for (int i = 0; i < 4; ++i) {
    PyObject* e = PyObject_GetAttrString(ctypes, element[i]);
    g_pointer_to[i] = e ? PyObject_CallMethod(ctypes, "POINTER", "O", e) : nullptr;
    Py_XDECREF(e);
    if (!g_pointer_to[i]) return nullptr;
  }
  Py_DECREF(ctypes);
  if (!g_cast || !g_void_p || !pointer || !(g_pointers = PyTuple_Pack(2, g_void_p, pointer))) return nullptr;
  Py_DECREF(pointer);
  PyObject* module = PyModule_Create(&g_module);
  PyObject* checked = module ? PyModule_Create(&g_checked_module) : nullptr;
  if (!checked || PyModule_AddObject(module, "of_checked", checked) < 0) {   // (takes the reference when it succeeds)
    Py_XDECREF(checked);
    Py_XDECREF(module);
    return nullptr;
  }
  return module;
}
