// The launchers as Python functions: one per status-returning entry point of
// include/rivoli_kvcache.h, taking the entry point's arguments in its order and returning its
// status. How an argument is converted follows from its C type in the header:
//   pointer       None, an int (an address) or an object with data_ptr() (a torch tensor)
//   void* (last)  the stream: None, an int or an object with cuda_stream (a torch.cuda.Stream)
//   int, ...      an int, narrowed as C would;   float: a number
// Short calls are bound by the host (a launch costs the runtime 2.6 us): through ctypes and its
// helpers a launcher took 1.7 us on top of that, here 0.5.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstdint>
#include <tuple>
#include <type_traits>
#include <utility>

#include "rivoli_kvcache.h"

namespace {

PyObject *kDataPtr, *kCudaStream;  // interned attribute names

bool address(PyObject* o, bool stream, void** out) {
    if (o == Py_None) {
        *out = nullptr;
        return true;
    }
    PyObject* v = nullptr;
    if (PyLong_Check(o)) {
        Py_INCREF(o);
        v = o;
    } else {
        v = stream ? PyObject_GetAttr(o, kCudaStream) : PyObject_CallMethodNoArgs(o, kDataPtr);
        if (!v) return false;
    }
    *out = reinterpret_cast<void*>(static_cast<uintptr_t>(PyLong_AsUnsignedLongLongMask(v)));
    Py_DECREF(v);
    return !PyErr_Occurred();
}

template <class T>
bool convert(PyObject* o, bool last, T* out) {
    if constexpr (std::is_pointer_v<T>) {
        void* p;
        if (!address(o, last && std::is_same_v<T, void*>, &p)) return false;
        *out = static_cast<T>(p);
        return true;
    } else if constexpr (std::is_floating_point_v<T>) {
        const double d = PyFloat_AsDouble(o);
        if (d == -1.0 && PyErr_Occurred()) return false;
        *out = static_cast<T>(d);
        return true;
    } else {
        if (PyFloat_Check(o)) {
            PyErr_SetString(PyExc_TypeError, "int expected instead of float");
            return false;
        }
        const unsigned long long v = PyLong_AsUnsignedLongLongMask(o);
        if (v == ~0ull && PyErr_Occurred()) return false;
        *out = static_cast<T>(v);
        return true;
    }
}

template <auto F>
struct Entry;
template <class... A, int (*F)(A...)>
struct Entry<F> {
    template <size_t... I>
    static PyObject* run(PyObject* const* args, std::index_sequence<I...>) {
        std::tuple<A...> a;
        if (!(convert(args[I], I + 1 == sizeof...(A), &std::get<I>(a)) && ...)) return nullptr;
        int code;
        Py_BEGIN_ALLOW_THREADS
        code = F(std::get<I>(a)...);
        Py_END_ALLOW_THREADS
        return PyLong_FromLong(code);
    }
    static PyObject* call(PyObject*, PyObject* const* args, Py_ssize_t n) {
        if (n != static_cast<Py_ssize_t>(sizeof...(A)))
            return PyErr_Format(PyExc_TypeError, "%zd arguments expected, %zd given",
                                static_cast<Py_ssize_t>(sizeof...(A)), n);
        return run(args, std::index_sequence_for<A...>{});
    }
};

#define ENTRY(name) \
    {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&Entry<&name>::call)), METH_FASTCALL, nullptr}
PyMethodDef kEntries[] = {
    ENTRY(rivoli_append_kv), ENTRY(rivoli_append_kv_rows), ENTRY(rivoli_index_append),
    ENTRY(rivoli_index_topk), ENTRY(rivoli_index_topk_batched), ENTRY(rivoli_index_score),
    ENTRY(rivoli_index_score_paged), ENTRY(rivoli_index_score_paged_hist),
    ENTRY(rivoli_dsa_select_gather_paged), ENTRY(rivoli_dsa_select_gather_paged_noalloc),
    ENTRY(rivoli_index_append_paged), ENTRY(rivoli_hash_rows), ENTRY(rivoli_device_sync),
    ENTRY(rivoli_kv_append_paged), ENTRY(rivoli_kv_gather_paged), ENTRY(rivoli_kv_gather_paged_packed),
    ENTRY(rivoli_kv_append_gather_paged), ENTRY(rivoli_kv_gather_rows_paged), ENTRY(rivoli_mla_attend),
    ENTRY(rivoli_mla_attend_paged), ENTRY(rivoli_act_quant_f8_prefix), ENTRY(rivoli_act_quant_f4_rotated),
    ENTRY(rivoli_index_score_blocks), ENTRY(rivoli_index_score_blocks_prefill),
    ENTRY(rivoli_index_select_blocks), ENTRY(rivoli_sel_shape), ENTRY(rivoli_sel_gather),
    ENTRY(rivoli_sel_gather_scored), ENTRY(rivoli_kv_ring_write), ENTRY(rivoli_gather_attn_shared_kv),
    ENTRY(rivoli_gather_attn_shared_kv_bounded), ENTRY(rivoli_gather_attn_shared_kv_split),
    ENTRY(rivoli_kv_compress_deposit), ENTRY(rivoli_kv_compress_prefill), ENTRY(rivoli_kv_compress_decode),
    ENTRY(rivoli_codec_e4m3_encode), ENTRY(rivoli_codec_e4m3_dequant_bf16), ENTRY(rivoli_codec_bf16_encode),
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "pylaunch", nullptr, -1, kEntries, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_pylaunch() {
    kDataPtr = PyUnicode_InternFromString("data_ptr");
    kCudaStream = PyUnicode_InternFromString("cuda_stream");
    return kDataPtr && kCudaStream ? PyModule_Create(&kModule) : nullptr;
}
