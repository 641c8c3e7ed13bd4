// CPython calls of the C-ABI (include/foldforge_amd.h): one function per entry point, its
// arguments converted by the entry point's own parameter types, so a call costs about a
// microsecond of host time where ctypes with 25 to 30 arguments takes eight. Checks stay in
// kernels.py; the one that runs over every parameter of every call (device, dtype, layout,
// shape) is params_ok below.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <array>
#include <tuple>
#include <type_traits>
#include <utility>

#include "foldforge_amd.h"

namespace {

// A pointer argument: a tensor's data, an address as int (a stream) or None (NULL).
void* pointer_from(PyObject* o) {
  if (o == Py_None) return nullptr;
  if (THPVariable_Check(o)) return THPVariable_Unpack(o).data_ptr();
  return PyLong_AsVoidPtr(o);  // sets TypeError for anything else
}

template <typename T>
T from(PyObject* o) {
  if constexpr (std::is_pointer_v<T>) {
    return static_cast<T>(pointer_from(o));
  } else if constexpr (std::is_floating_point_v<T>) {
    return static_cast<T>(PyFloat_AsDouble(o));
  } else if constexpr (std::is_same_v<T, size_t>) {
    return PyLong_AsSize_t(o);
  } else {
    const long long v = PyLong_AsLongLong(o);
    if (static_cast<long long>(static_cast<T>(v)) != v && !PyErr_Occurred())
      PyErr_SetString(PyExc_OverflowError, "integer argument out of range");
    return static_cast<T>(v);
  }
}

template <auto Fn>
struct Call;
template <typename R, typename... A, R (*Fn)(A...)>
struct Call<Fn> {
  template <size_t... I>
  static PyObject* apply(PyObject* const* args, std::index_sequence<I...>) {
    const std::tuple<A...> v{from<A>(args[I])...};
    if (PyErr_Occurred()) return nullptr;
    R r;
    // launches may wait for queue space: other Python threads run meanwhile, as under ctypes
    Py_BEGIN_ALLOW_THREADS;
    r = std::apply(Fn, v);
    Py_END_ALLOW_THREADS;
    if constexpr (std::is_same_v<R, size_t>)
      return PyLong_FromSize_t(r);
    else
      return PyLong_FromLong(r);
  }
  static PyObject* run(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != static_cast<Py_ssize_t>(sizeof...(A)))
      return PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", (Py_ssize_t)sizeof...(A), n);
    return apply(args, std::index_sequence_for<A...>{});
    END_HANDLE_TH_ERRORS
  }
};

// params_ok(x, tensors, shapes): whether every tensor is a contiguous fp32 strided tensor on
// x's device of the given shape (False: the caller looks closer, and raises or copies).
PyObject* params_ok(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 3 || !THPVariable_Check(args[0]) || !PyTuple_Check(args[1]) || !PyTuple_Check(args[2]) ||
      PyTuple_GET_SIZE(args[1]) != PyTuple_GET_SIZE(args[2]))
    return PyErr_Format(PyExc_TypeError, "params_ok(tensor, tuple of tensors, tuple of shapes)");
  const at::Device device = THPVariable_Unpack(args[0]).device();
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(args[1]); ++i) {
    PyObject* o = PyTuple_GET_ITEM(args[1], i);
    PyObject* shape = PyTuple_GET_ITEM(args[2], i);
    if (!THPVariable_Check(o) || !PyTuple_Check(shape)) Py_RETURN_FALSE;
    const at::Tensor& t = THPVariable_Unpack(o);
    if (t.scalar_type() != at::kFloat || t.layout() != at::kStrided || t.device() != device ||
        t.dim() != PyTuple_GET_SIZE(shape) || !t.is_contiguous())
      Py_RETURN_FALSE;
    for (int64_t d = 0; d < t.dim(); ++d) {
      const long long want = PyLong_AsLongLong(PyTuple_GET_ITEM(shape, d));
      if (want == -1 && PyErr_Occurred()) return nullptr;
      if (t.size(d) != want) Py_RETURN_FALSE;
    }
  }
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

#define FFK_CALL(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&Call<&name>::run)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    {"params_ok", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&params_ok)), METH_FASTCALL, nullptr},
    FFK_CALL(ffk_layer_norm),
    FFK_CALL(ffk_layer_norm_linear),
    FFK_CALL(ffk_swiglu_ffn_workspace),
    FFK_CALL(ffk_swiglu_ffn),
    FFK_CALL(ffk_triangle_multiplication_workspace),
    FFK_CALL(ffk_triangle_multiplication),
    FFK_CALL(ffk_triangle_attention_workspace),
    FFK_CALL(ffk_triangle_attention),
    FFK_CALL(ffk_triangle_attention_transition_workspace),
    FFK_CALL(ffk_triangle_attention_transition),
    FFK_CALL(ffk_flash_attention_bias),
    FFK_CALL(ffk_transition_workspace),
    FFK_CALL(ffk_transition),
    FFK_CALL(ffk_attention_pair_bias_workspace),
    FFK_CALL(ffk_attention_pair_bias),
    FFK_CALL(ffk_msa_pair_weighted_averaging_workspace),
    FFK_CALL(ffk_msa_pair_weighted_averaging),
    FFK_CALL(ffk_outer_product_mean_workspace),
    FFK_CALL(ffk_outer_product_mean),
    FFK_CALL(ffk_outer_product_mean_grouped_workspace),
    FFK_CALL(ffk_outer_product_mean_grouped),
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_bindings", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__bindings(void) { return PyModule_Create(&module_def); }
