// Call path from Python to the C ABI of libgdn_hip.so.
//
// A call through ctypes spends 20 to 28 us of host time on eight or nine
// tensors (a Python loop per descriptor, a pointer conversion per argument, the
// stream lookup), more than the kernels of a small call take.  This module
// fills the descriptors from the tensors themselves and calls the same entry
// points, whose addresses it gets from the loaded library, with the same
// arguments.  It takes plain tensors only; for anything else (subclasses,
// other objects) a function returns None and the caller goes through ctypes.
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <tuple>
#include <utility>

#include "../../include/gdn_hip.h"

namespace {

constexpr int kMaxDim = 4;

int32_t dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return GDN_DTYPE_F32;
    case at::kBFloat16: return GDN_DTYPE_BF16;
    case at::kHalf: return GDN_DTYPE_F16;
    case at::kInt: return GDN_DTYPE_I32;
    case at::kLong: return GDN_DTYPE_I64;
    default: return -1;
  }
}

bool plain(PyObject* o) { return THPVariable_CheckExact(o); }

// false for a tensor the descriptors cannot hold (the ctypes path raises for it)
bool describe(PyObject* o, gdn_tensor& d) {
  const at::Tensor& t = THPVariable_Unpack(o);
  const int64_t n = t.dim();
  if (n > kMaxDim) return false;
  d = gdn_tensor{};
  d.data = t.numel() > 0 ? t.data_ptr() : nullptr;
  d.dtype = dtype_code(t.scalar_type());
  d.ndim = (int32_t)n;
  for (int64_t i = 0; i < n; ++i) {
    d.shape[i] = t.size(i);
    d.stride[i] = t.stride(i);
  }
  return true;
}

template <typename X> bool convert(PyObject* o, X& x);
template <> bool convert<float>(PyObject* o, float& x) {
  x = (float)PyFloat_AsDouble(o);
  return !PyErr_Occurred();
}
template <> bool convert<int32_t>(PyObject* o, int32_t& x) {
  const long v = PyLong_AsLong(o);
  x = (int32_t)v;
  if (!PyErr_Occurred() && v != x) PyErr_SetString(PyExc_OverflowError, "argument does not fit 32 bits");
  return !PyErr_Occurred();
}
template <> bool convert<int64_t>(PyObject* o, int64_t& x) {
  x = PyLong_AsLongLong(o);
  return !PyErr_Occurred();
}

// One entry point of N tensors (a null one as None), then scalars X, then the
// stream: the current one of the first tensor's device.  Each entry is its own
// type ID, whose `fn` bind() sets.
template <int ID, int N, typename... X>
struct Entry {
  static void* fn;
  template <size_t... I, size_t... J>
  static PyObject* run(PyObject* const* args, std::index_sequence<I...>, std::index_sequence<J...>) {
    gdn_tensor d[N];
    bool null[N];
    for (int i = 0; i < N; ++i) {
      null[i] = args[i] == Py_None;
      if (!null[i] && (!plain(args[i]) || !describe(args[i], d[i]))) Py_RETURN_NONE;
    }
    if (null[0]) Py_RETURN_NONE;
    const at::Tensor& t = THPVariable_Unpack(args[0]);
    if (!t.is_cuda()) Py_RETURN_NONE;
    std::tuple<X...> x;
    if (!(convert<X>(args[N + J], std::get<J>(x)) && ...)) return nullptr;
    void* const stream = c10::hip::getCurrentHIPStream(t.device().index()).stream();
    typedef gdn_tensor* Ptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS  // (a launch may wait for room in its queue)
    rc = reinterpret_cast<int (*)(decltype((void)I, Ptr())..., X..., void*)>(fn)(
        (null[I] ? nullptr : &d[I])..., std::get<J>(x)..., stream);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
  }
  static PyObject* call(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != N + (Py_ssize_t)sizeof...(X) || !fn) {
      PyErr_SetString(PyExc_TypeError, fn ? "wrong number of arguments" : "the library is not bound");
      return nullptr;
    }
    try {
      return run(args, std::make_index_sequence<N>(), std::index_sequence_for<X...>());
    } catch (const std::exception& e) {
      PyErr_SetString(PyExc_RuntimeError, e.what());
      return nullptr;
    }
  }
};
template <int ID, int N, typename... X> void* Entry<ID, N, X...>::fn = nullptr;

// A workspace size: integers in, a 64-bit integer out.
template <int ID, typename... X>
struct Size {
  static void* fn;
  template <size_t... J>
  static PyObject* run(PyObject* const* args, std::index_sequence<J...>) {
    std::tuple<X...> x;
    if (!(convert<X>(args[J], std::get<J>(x)) && ...)) return nullptr;
    return PyLong_FromLongLong(reinterpret_cast<int64_t (*)(X...)>(fn)(std::get<J>(x)...));
  }
  static PyObject* call(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != (Py_ssize_t)sizeof...(X) || !fn) {
      PyErr_SetString(PyExc_TypeError, fn ? "wrong number of arguments" : "the library is not bound");
      return nullptr;
    }
    return run(args, std::index_sequence_for<X...>());
  }
};
template <int ID, typename... X> void* Size<ID, X...>::fn = nullptr;

// Index of the one HIP device that all tensors (None aside) live on, or -1.
PyObject* same_device(PyObject*, PyObject* const* args, Py_ssize_t n) {
  long dev = -1;
  for (Py_ssize_t i = 0; i < n; ++i) {
    if (args[i] == Py_None) continue;
    if (!plain(args[i])) return PyLong_FromLong(-1);
    const at::Device d = THPVariable_Unpack(args[i]).device();
    if (!d.is_cuda() || (dev >= 0 && d.index() != dev)) return PyLong_FromLong(-1);
    dev = d.index();
  }
  return PyLong_FromLong(dev);
}

// Whether the kernels can read a tensor with 16-byte accesses (unit inner
// stride, 16-byte aligned data and outer strides); None if it is not a plain one.
PyObject* vec16_ok(PyObject*, PyObject* o) {
  if (!plain(o)) Py_RETURN_NONE;
  const at::Tensor& t = THPVariable_Unpack(o);
  const int64_t n = t.dim();
  if (n == 0) Py_RETURN_NONE;
  try {
    bool ok = t.stride(n - 1) == 1 && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
    const int64_t es = (int64_t)t.element_size();
    for (int64_t i = 0; ok && i < n - 1; ++i) ok = t.stride(i) * es % 16 == 0;
    return PyBool_FromLong(ok);
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
}

typedef Entry<0, 8, float> RecurrentStep;
typedef Entry<1, 9, float, int32_t> ChunkPrefill;
typedef Entry<2, 10, float, int32_t> ChunkPrefillSplit;
typedef Entry<3, 9, float, int32_t, int32_t, int32_t, int32_t> ChunkPrefillEx;
typedef Entry<4, 6> ConvVarlen;
typedef Entry<5, 6, int64_t> ConvVarlenNorm;
typedef Entry<6, 5> ConvStep;
typedef Entry<7, 11, int32_t, float> DecodeFused;
typedef Entry<8, 4, float> RmsNorm;
typedef Entry<9, 6> Gating;
typedef Entry<10, 5, int64_t, float, int32_t> AttnVarlen;
typedef Entry<11, 5, int64_t, float, int32_t> AttnVarlenAny;
typedef Entry<12, 7, int64_t, float> PagedPrefill;
typedef Entry<13, 8, int64_t, float> PagedPrefillSplit;
typedef Entry<14, 7, int32_t, float> PagedDecode;
typedef Entry<15, 6, int32_t, float> PagedDecodeNoalloc;
typedef Entry<16, 13, int32_t, float, float> DecodeFusedNorm;
typedef Entry<17, 3> Linear;
typedef Entry<18, 10, float, int32_t, int32_t> ChunkPrefillSplitEx;
typedef Size<0, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t> ChunkPrefillSize;
typedef Size<1, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t> PagedPrefillSize;
typedef Size<2, int64_t, int64_t, int64_t, int32_t> PagedDecodeSize;

struct Bound {
  const char* name;
  void** fn;
  PyObject* (*call)(PyObject*, PyObject* const*, Py_ssize_t);
};
#define GDN_BOUND(NAME, E) {NAME, &E::fn, E::call}
const Bound kBound[] = {
    GDN_BOUND("gdn_recurrent_step", RecurrentStep),
    GDN_BOUND("gdn_chunk_prefill", ChunkPrefill),
    GDN_BOUND("gdn_chunk_prefill_split", ChunkPrefillSplit),
    GDN_BOUND("gdn_chunk_prefill_split_ex", ChunkPrefillSplitEx),
    GDN_BOUND("gdn_chunk_prefill_ex", ChunkPrefillEx),
    GDN_BOUND("causal_conv1d_varlen", ConvVarlen),
    GDN_BOUND("causal_conv1d_varlen_qknorm", ConvVarlenNorm),
    GDN_BOUND("causal_conv1d_step", ConvStep),
    GDN_BOUND("gdn_decode_step_fused", DecodeFused),
    GDN_BOUND("gdn_decode_step_fused_norm", DecodeFusedNorm),
    GDN_BOUND("gdn_linear", Linear),
    GDN_BOUND("gdn_rms_norm_gated", RmsNorm),
    GDN_BOUND("gdn_gating", Gating),
    GDN_BOUND("flash_attention_varlen", AttnVarlen),
    GDN_BOUND("flash_attention_varlen_any_dim", AttnVarlenAny),
    GDN_BOUND("paged_attention_prefill", PagedPrefill),
    GDN_BOUND("paged_attention_prefill_split", PagedPrefillSplit),
    GDN_BOUND("paged_attention_decode", PagedDecode),
    GDN_BOUND("paged_attention_decode_noalloc", PagedDecodeNoalloc),
    GDN_BOUND("gdn_chunk_prefill_workspace_size", ChunkPrefillSize),
    GDN_BOUND("paged_attention_prefill_workspace_size", PagedPrefillSize),
    GDN_BOUND("paged_attention_decode_workspace_size", PagedDecodeSize),
};
#undef GDN_BOUND
constexpr int kNumBound = sizeof(kBound) / sizeof(kBound[0]);

// bind({name: address}): the loaded library's entry points.
PyObject* bind(PyObject*, PyObject* dict) {
  for (const Bound& b : kBound) {
    PyObject* a = PyDict_Check(dict) ? PyDict_GetItemString(dict, b.name) : nullptr;
    if (!a) return PyErr_Format(PyExc_KeyError, "%s", b.name);
    *b.fn = PyLong_AsVoidPtr(a);
    if (PyErr_Occurred()) return nullptr;
  }
  Py_RETURN_NONE;
}

PyMethodDef g_methods[kNumBound + 4];
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_gdn_binding", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__gdn_binding() {
  int k = 0;
  auto add = [&](const char* name, void* f, int flags) {
    g_methods[k++] = PyMethodDef{name, reinterpret_cast<PyCFunction>(f), flags, nullptr};
  };
  for (const Bound& b : kBound) add(b.name, reinterpret_cast<void*>(b.call), METH_FASTCALL);
  add("same_device", reinterpret_cast<void*>(same_device), METH_FASTCALL);
  add("vec16_ok", reinterpret_cast<void*>(vec16_ok), METH_O);
  add("bind", reinterpret_cast<void*>(bind), METH_O);
  g_methods[k] = PyMethodDef{nullptr, nullptr, 0, nullptr};
  return PyModule_Create(&g_module);
}
