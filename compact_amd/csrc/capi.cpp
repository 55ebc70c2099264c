// CPython binding of the C ABI: one vectorcall function per entry point, its
// arguments converted by their C types (None is a null pointer), the GIL
// released during the call.  A small LoRA step makes some 20 such calls: one of
// 30 arguments takes 0.2 us here and 2.5 through ctypes.

#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstdint>
#include <type_traits>
#include <tuple>
#include <utility>

#include "compact_amd.h"

namespace {

template <class T>
inline T from_py(PyObject* o) {
  if constexpr (std::is_pointer_v<T>) {
    if (o == Py_None) return nullptr;
    return reinterpret_cast<T>(static_cast<uintptr_t>(PyLong_AsUnsignedLongLong(o)));
  } else if constexpr (std::is_floating_point_v<T>) {
    return static_cast<T>(PyFloat_AsDouble(o));
  } else {
    return static_cast<T>(PyLong_AsLongLong(o));
  }
}

template <auto F>
struct Entry;

template <class R, class... A, R (*F)(A...)>
struct Entry<F> {
  template <size_t... I>
  static PyObject* go(PyObject* const* args, std::index_sequence<I...>) {
    std::tuple<A...> v{from_py<A>(args[I])...};
    if (PyErr_Occurred()) return nullptr;
    R r;
    Py_BEGIN_ALLOW_THREADS
    r = F(std::get<I>(v)...);
    Py_END_ALLOW_THREADS
    return PyLong_FromLongLong(static_cast<long long>(r));
  }
  static PyObject* call(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != static_cast<Py_ssize_t>(sizeof...(A))) {
      PyErr_Format(PyExc_TypeError, "%d arguments expected, got %zd", (int)sizeof...(A), n);
      return nullptr;
    }
    return go(args, std::index_sequence_for<A...>{});
  }
};

#define CPT_ENTRY(name) \
  {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(&Entry<&name>::call)), METH_FASTCALL, nullptr}

PyMethodDef methods[] = {
    CPT_ENTRY(cpt_silu_mul),
    CPT_ENTRY(cpt_swiglu_backward),
    CPT_ENTRY(cpt_swiglu_backward_glu),
    CPT_ENTRY(cpt_v3_quantize_group_absmax),
    CPT_ENTRY(cpt_v3_dequantize_group_absmax),
    CPT_ENTRY(cpt_silu_mul_quant),
    CPT_ENTRY(cpt_dequant_swiglu_backward),
    CPT_ENTRY(cpt_outlier_select_pair),
    CPT_ENTRY(cpt_silu_mul_quant_outlier),
    CPT_ENTRY(cpt_dequant_swiglu_backward_outlier),
    CPT_ENTRY(cpt_gemm_bf16),
    CPT_ENTRY(cpt_gemm_bf16_lora),
    CPT_ENTRY(cpt_gemm_bf16_ex),
    CPT_ENTRY(cpt_gemm16),
    CPT_ENTRY(cpt_gemm16_skinny),
    CPT_ENTRY(cpt_gemm16_skinny_small),
    CPT_ENTRY(cpt_gemm16_skinny_t),
    CPT_ENTRY(cpt_gemm16_skinny_dual),
    CPT_ENTRY(cpt_gemm16_skinny_dual2),
    CPT_ENTRY(cpt_gemm_bf16_skinny_dual_workspace_bytes),
    CPT_ENTRY(cpt_gemm_any),
    CPT_ENTRY(cpt_gemm_any_if),
    CPT_ENTRY(cpt_split_f32),
    CPT_ENTRY(cpt_gemm_f32x3),
    CPT_ENTRY(cpt_ffn_gate_up),
    CPT_ENTRY(cpt_ffn_gate_up_lora),
    CPT_ENTRY(cpt_ffn_gate_up16),
    CPT_ENTRY(cpt_ffn_down_dgrad),
    CPT_ENTRY(cpt_ffn_down_dgrad_lora),
    CPT_ENTRY(cpt_transpose_bf16),
    CPT_ENTRY(cpt_dora_scale),
    CPT_ENTRY(cpt_col_dot_div_rows),
    CPT_ENTRY(cpt_dora_col_norm),
    CPT_ENTRY(cpt_dora_col_norm_workspace_bytes),
    CPT_ENTRY(cpt_dora_col_norm16),
    CPT_ENTRY(cpt_dora_col_norm16_workspace_bytes),
    CPT_ENTRY(cpt_topk_abs),
    CPT_ENTRY(cpt_topk_scatter),
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_capi", "compact_amd's C ABI", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__capi(void) { return PyModule_Create(&module); }
