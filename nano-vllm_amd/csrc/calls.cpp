// CPython callables for the entry points of both libraries.
//
// A call of one token is bound by the host, and ctypes takes 0.8 to 1.3 us for an entry point of 13 to 24 arguments (that refuses its sizes; 0.3 us for
// five of them): an object and a converter an argument.  A callable here takes 0.2: a paged decode, which makes three such calls of 13, 6 and 23 arguments,
// 20.2 -> 18.2 us.  It knows its entry point's type from the header, takes Python integers, floats and None (a null
// pointer) straight into the arguments, and gives the interpreter lock away during the call, as ctypes does.  Anything else (a wrong number of
// arguments, a ctypes object, a number that does not fit) goes to the ctypes function that it stands for, with that one's
// conversions and errors.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <structmember.h>
#include <string.h>

#include <cstddef>
#include <tuple>
#include <type_traits>
#include <utility>

#include "../../include/nanovllm_hip.h"
#include "../../include/nanovllm_hip_mixers.h"

namespace {

struct Call {
    PyObject_HEAD
    vectorcallfunc vectorcall;
    PyObject* otherwise;          // the ctypes function
    void* entry;
};

template <typename T>
bool take(PyObject* o, T& v) {
    if constexpr (std::is_pointer_v<T>) {
        if (o == Py_None) {
            v = nullptr;
            return true;
        }
        if (!PyLong_CheckExact(o)) return false;
        v = (T)PyLong_AsVoidPtr(o);
        if (v != nullptr || !PyErr_Occurred()) return true;
    } else if constexpr (std::is_floating_point_v<T>) {
        if (!PyFloat_CheckExact(o)) return false;
        v = (T)PyFloat_AS_DOUBLE(o);
        return true;
    } else {
        if (!PyLong_Check(o)) return false;
        const long long x = PyLong_AsLongLong(o);
        v = (T)x;
        if ((long long)v == x && (x != -1 || !PyErr_Occurred())) return true;
    }
    PyErr_Clear();
    return false;
}

template <typename T>
constexpr char letter() {
    if constexpr (std::is_pointer_v<T>) return 'p';
    else if constexpr (std::is_floating_point_v<T>) return sizeof(T) == 4 ? 'f' : 'd';
    else return sizeof(T) == 4 ? 'i' : 'l';
}

template <typename F> struct Entry;
template <typename R, typename... A>
struct Entry<R(A...)> {
    static constexpr char signature[] = {letter<R>(), letter<A>()..., 0};          // result, arguments
    template <size_t... I>
    static bool all(PyObject* const* args, std::tuple<A...>& v, std::index_sequence<I...>) {
        return (take(args[I], std::get<I>(v)) && ...);
    }
    static PyObject* call(PyObject* self, PyObject* const* args, size_t nargsf, PyObject* names) {
        Call* c = (Call*)self;
        std::tuple<A...> v;
        if (PyVectorcall_NARGS(nargsf) != (Py_ssize_t)sizeof...(A) || (names != nullptr && PyTuple_GET_SIZE(names) != 0) ||
            !all(args, v, std::index_sequence_for<A...>{}))
            return PyObject_Vectorcall(c->otherwise, args, nargsf, names);
        R r;
        Py_BEGIN_ALLOW_THREADS
        r = std::apply((R (*)(A...))c->entry, v);
        Py_END_ALLOW_THREADS
        return PyLong_FromLongLong(r);
    }
};

struct Known {
    const char *name, *signature;
    vectorcallfunc call;
};
#define NV_ENTRY(NAME) {#NAME, Entry<decltype(NAME)>::signature, &Entry<decltype(NAME)>::call},
const Known known[] = {
    NV_ENTRY(nv_store_kvcache) NV_ENTRY(nv_attn_decode_workspace_bytes) NV_ENTRY(nv_attn_decode_paged)
    NV_ENTRY(nv_attn_decode_suggest_chunk) NV_ENTRY(nv_attn_decode_workspace_bytes_chunked) NV_ENTRY(nv_attn_decode_paged_chunked)
    NV_ENTRY(nv_attn_decode_paged_fused_chunked) NV_ENTRY(nv_attn_decode_static_scratch_bytes) NV_ENTRY(nv_attn_decode_paged_static)
    NV_ENTRY(nv_attn_decode_paged_fused) NV_ENTRY(nv_attn_prefill_workspace_bytes) NV_ENTRY(nv_attn_prefill_query_tiles)
    NV_ENTRY(nv_attn_prefill_varlen) NV_ENTRY(nv_rmsnorm) NV_ENTRY(nv_silu_and_mul) NV_ENTRY(nv_add_rmsnorm) NV_ENTRY(nv_rope)
    NV_ENTRY(nv_qknorm_rope_store) NV_ENTRY(nv_add_layernorm) NV_ENTRY(nv_gelu_tanh_and_mul) NV_ENTRY(nv_qk_prep_store)
    NV_ENTRY(nv_attn_scoremod_paged) NV_ENTRY(nv_attn_scoremod_paged_vld) NV_ENTRY(nv_attn_scoremod_step_workspace_bytes)
    NV_ENTRY(nv_attn_scoremod_workspace_bytes) NV_ENTRY(nv_causal_conv_silu) NV_ENTRY(nv_gated_delta_rule) NV_ENTRY(nv_stream_boundary)
    NV_ENTRY(nv_rms_norm_rows) NV_ENTRY(nv_causal_conv_add) NV_ENTRY(nv_token_gate) NV_ENTRY(nv_general_delta_rule)
    NV_ENTRY(nv_latent_prep_store) NV_ENTRY(nv_moe_route) NV_ENTRY(nv_moe_tile_rows_for) NV_ENTRY(nv_moe_tile_rows)
    NV_ENTRY(nv_moe_max_tiles) NV_ENTRY(nv_moe_align) NV_ENTRY(nv_moe_route_sort_words) NV_ENTRY(nv_moe_route_sort)
    NV_ENTRY(nv_moe_gate_up) NV_ENTRY(nv_moe_down) NV_ENTRY(nv_moe_gate_up_act) NV_ENTRY(nv_causal_conv_bias_silu)
    NV_ENTRY(nv_hashed_bigram_embed) NV_ENTRY(nv_stream_boundary_pair) NV_ENTRY(nv_relu_squared) NV_ENTRY(nv_decay_memory)
    NV_ENTRY(nv_state_space_scan) NV_ENTRY(nv_token_shift_mix) NV_ENTRY(nv_group_rms_norm) NV_ENTRY(nv_chunk_attn_prep_store)
    NV_ENTRY(nv_attn_chunk_sigmoid_tile_ok) NV_ENTRY(nv_attn_chunk_sigmoid_paged) NV_ENTRY(nv_causal_conv_act)
    NV_ENTRY(nv_stream_boundary_scaled) NV_ENTRY(nv_poly_norm) NV_ENTRY(nv_head_norm_rope_store) NV_ENTRY(nv_mlstm_memory)
    NV_ENTRY(nv_gated_write_memory) NV_ENTRY(nv_moe_route_grouped) NV_ENTRY(nv_moe_route_softmax) NV_ENTRY(nv_embed_positions)
    NV_ENTRY(nv_stream_layernorm_pair) NV_ENTRY(nv_silu_and_mul_rows) NV_ENTRY(nv_latent_store) NV_ENTRY(nv_head_linear)
    NV_ENTRY(nv_attn_latent_ok) NV_ENTRY(nv_attn_latent_workspace_bytes) NV_ENTRY(nv_attn_latent_paged)
    NV_ENTRY(nv_selective_scan_workspace_bytes) NV_ENTRY(nv_selective_scan) NV_ENTRY(nv_recurrence_workspace_bytes)
    NV_ENTRY(nv_gated_delta_rule_portions) NV_ENTRY(nv_general_delta_rule_portions) NV_ENTRY(nv_gated_write_memory_portions)
    NV_ENTRY(nv_fixed_decay_workspace_bytes) NV_ENTRY(nv_fixed_decay_memory) NV_ENTRY(nv_row_norm_rope_store) NV_ENTRY(nv_join_gated)
    NV_ENTRY(nv_clamped_glu_rows) NV_ENTRY(nv_scale_softcap) NV_ENTRY(nv_moe_up_relu2)
};

void call_dealloc(PyObject* self) {
    Py_XDECREF(((Call*)self)->otherwise);
    Py_TYPE(self)->tp_free(self);
}
PyTypeObject call_type = {PyVarObject_HEAD_INIT(nullptr, 0)};

PyMemberDef call_members[] = {
    {(char*)"otherwise", T_OBJECT, offsetof(Call, otherwise), READONLY, (char*)"the ctypes function"},
    {nullptr, 0, 0, 0, nullptr},
};

// bind(name, address, ctypes function) -> a callable, or None for an entry point that is not known here
PyObject* bind(PyObject*, PyObject* args) {
    const char* name;
    PyObject *address, *otherwise;
    if (!PyArg_ParseTuple(args, "sOO", &name, &address, &otherwise)) return nullptr;
    void* entry = PyLong_AsVoidPtr(address);
    if (entry == nullptr) {
        if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "bind: no address");
        return nullptr;
    }
    for (const Known& k : known) {
        if (strcmp(k.name, name) != 0) continue;
        Call* c = PyObject_New(Call, &call_type);
        if (c == nullptr) return nullptr;
        Py_INCREF(otherwise);
        c->vectorcall = k.call;
        c->otherwise = otherwise;
        c->entry = entry;
        return (PyObject*)c;
    }
    Py_RETURN_NONE;
}

// signature(name) -> what the header that this was built from says: a letter for the result and for each argument, or None
PyObject* signature(PyObject*, PyObject* name) {
    const char* wanted = PyUnicode_AsUTF8(name);
    if (wanted == nullptr) return nullptr;
    for (const Known& k : known)
        if (strcmp(k.name, wanted) == 0) return PyUnicode_FromString(k.signature);
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {{"bind", bind, METH_VARARGS, nullptr}, {"signature", signature, METH_O, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "nv_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_nv_calls() {
    call_type.tp_name = "nv_calls.Call";
    call_type.tp_basicsize = sizeof(Call);
    call_type.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL;
    call_type.tp_vectorcall_offset = offsetof(Call, vectorcall);
    call_type.tp_call = PyVectorcall_Call;
    call_type.tp_dealloc = call_dealloc;
    call_type.tp_members = call_members;
    if (PyType_Ready(&call_type) < 0) return nullptr;
    return PyModule_Create(&module);
}
