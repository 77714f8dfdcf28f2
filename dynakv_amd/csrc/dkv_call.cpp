// CPython binding of the C ABI's per-call entry points (include/dynakv_amd.h): module _dkv_call.
//
// The Python wrappers make one to three of these calls per operation, with up to 40 arguments each.
// ctypes converts them one by one through Python objects, ~5 us a call beside a launch of ~3 us;
// here each argument is read straight into its C type, taken from the declaration of the function
// itself. Pointers and streams come as Python integers (None: NULL). The GIL is released around
// the call, as ctypes releases it.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <climits>
#include <tuple>
#include <type_traits>
#include <utility>

#include "../../include/dynakv_amd.h"

namespace {

template <class T>
bool read_arg(PyObject* o, T& v) {
  if constexpr (std::is_pointer_v<T>) {
    if (o == Py_None) {
      v = nullptr;
      return true;
    }
    v = static_cast<T>(PyLong_AsVoidPtr(o));
    return v || !PyErr_Occurred();
  } else if constexpr (std::is_floating_point_v<T>) {
    const double d = PyFloat_AsDouble(o);
    v = static_cast<T>(d);
    return d != -1.0 || !PyErr_Occurred();
  } else {
    static_assert(std::is_same_v<T, int> || std::is_same_v<T, long long>, "integer argument");
    const long long x = PyLong_AsLongLong(o);
    if (x == -1 && PyErr_Occurred()) return false;
    if (std::is_same_v<T, int> && (x < INT_MIN || x > INT_MAX)) {
      PyErr_SetString(PyExc_OverflowError, "argument does not fit a C int");
      return false;
    }
    v = static_cast<T>(x);
    return true;
  }
}

template <auto F>
struct Call;
template <class R, class... A, R (*F)(A...)>
struct Call<F> {
  static PyObject* run(PyObject*, PyObject* const* args, Py_ssize_t n) {
    return run_with(args, n, std::index_sequence_for<A...>{});
  }
  template <size_t... I>
  static PyObject* run_with(PyObject* const* args, Py_ssize_t n, std::index_sequence<I...>) {
    if (n != (Py_ssize_t)sizeof...(A))
      return PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd",
                          (Py_ssize_t)sizeof...(A), n);
    std::tuple<A...> a;
    if (!(read_arg(args[I], std::get<I>(a)) && ...)) return nullptr;
    R r;
    Py_BEGIN_ALLOW_THREADS;
    r = F(std::get<I>(a)...);
    Py_END_ALLOW_THREADS;
    return PyLong_FromLongLong(r);
  }
};

#define DKV_CALL(name) \
  {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(Call<name>::run)), METH_FASTCALL, nullptr}

PyMethodDef methods[] = {
    DKV_CALL(dkv_append_decode),
    DKV_CALL(dkv_append_decode_kv),
    DKV_CALL(dkv_append_prefill),
    DKV_CALL(dkv_append_prefill_kv),
    DKV_CALL(dkv_append_prefill_new_kv),
    DKV_CALL(dkv_decompress),
    DKV_CALL(dkv_decompress_kv),
    DKV_CALL(dkv_row_totals),
    DKV_CALL(dkv_scores),
    DKV_CALL(dkv_av),
    DKV_CALL(dkv_joint_scores),
    DKV_CALL(dkv_joint_scores_workspace_ints),
    DKV_CALL(dkv_joint_av_workspace_floats),
    DKV_CALL(dkv_joint_av),
    DKV_CALL(dkv_rope_table_floats),
    DKV_CALL(dkv_rope_table),
    DKV_CALL(dkv_splitk_workspace_floats),
    DKV_CALL(dkv_decode_splitk),
    DKV_CALL(dkv_decode_splitk_bt),
    DKV_CALL(dkv_dense_workspace_floats),
    DKV_CALL(dkv_dense_append),
    DKV_CALL(dkv_dense_choose_split),
    DKV_CALL(dkv_decode_dense),
    DKV_CALL(dkv_cutoff_workspace_bytes),
    DKV_CALL(dkv_cutoff_kv),
    DKV_CALL(dkv_rope_dense),
    DKV_CALL(dkv_prefill_attention),
    DKV_CALL(dkv_recon_kv),
    DKV_CALL(dkv_recon_kv_bt),
    DKV_CALL(dkv_rope_apply),
    DKV_CALL(dkv_decode_layer),
    DKV_CALL(dkv_add_rmsnorm),
    DKV_CALL(dkv_silu_mul),
    DKV_CALL(dkv_silu_mul_pairs),
    DKV_CALL(dkv_gemv),
    DKV_CALL(dkv_gemv_rmsnorm),
    DKV_CALL(dkv_gemv_glu),
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_dkv_call", nullptr, -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__dkv_call(void) { return PyModule_Create(&module); }
