// The host side of the forward operators as one native call each: argument checks, output allocation, stride marshalling and
// the launch, for the calls a forward pass makes.
//
// What it is for: a pass over a few tokens is bound by the host (64 tokens, 8 experts, 128 -> 256 -> 128: seven launches that
// keep the GPU busy for 39 us took 131 us to issue, now 69), and most of that was Python: one interpreter call per tensor attribute,
// output and descriptor field.
//
// Every function here takes a call whole or returns None and has done nothing that matters: whatever it does not recognise
// (other dtypes, layouts, tensor subclasses, wrong shapes, an error status) is left to the Python code in ops.py, which
// handles it or raises.  Nothing is kept from one call for the next.  The C entry points are handed over as addresses once
// (init), so that this module works with whichever build of the library ctypes has loaded.
#include <Python.h>
#include <ATen/ATen.h>
#include <ATen/record_function.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>

#include "../../include/fast_moe_amd.h"

namespace {

decltype(&fmoe_route_workspace_bytes) route_workspace_bytes;
decltype(&fmoe_route_topk) c_route_topk;
decltype(&fmoe_grouped_gemm) c_grouped_gemm;
decltype(&fmoe_combine) c_combine;
decltype(&fmoe_quant_rows_e4m3) c_quant_rows;

constexpr int64_t kSlackRows = 128;      // ops.SLACK_ROWS

struct NoGil {
    PyThreadState* state = PyEval_SaveThread();
    ~NoGil() { PyEval_RestoreThread(state); }
};

// The tensor behind a plain tensor or parameter (no subclass) on the GPU, or an undefined one.  A copy: the GIL is released
// while it is used.
at::Tensor gpu_tensor(PyObject* o) {
    if (Py_TYPE(o) != (PyTypeObject*)THPVariableClass && Py_TYPE(o) != (PyTypeObject*)ParameterClass) return {};
    const at::Tensor& t = THPVariable_Unpack(o);
    return t.is_cuda() ? t : at::Tensor();
}

// None -> true with *out undefined; a plain GPU tensor -> true; anything else -> false
bool optional_tensor(PyObject* o, at::Tensor* out) {
    if (o == Py_None) return true;
    *out = gpu_tensor(o);
    return out->defined();
}

bool as_int(PyObject* o, int64_t* v) {
    if (!PyLong_CheckExact(o) && !PyBool_Check(o)) return false;
    *v = PyLong_AsLongLong(o);
    if (*v == -1 && PyErr_Occurred()) {
        PyErr_Clear();
        return false;
    }
    return true;
}

int dtype_code(at::ScalarType t) {
    return t == at::kFloat ? FMOE_F32 : t == at::kBFloat16 ? FMOE_BF16 : t == at::kFloat8_e4m3fn ? FMOE_E4M3 : -1;
}

at::Tensor empty(at::IntArrayRef shape, at::ScalarType dtype, const at::Tensor& like) {
    return at::empty(shape, at::TensorOptions(like.device()).dtype(dtype));
}

bool same_device(const at::Tensor& a, const at::Tensor& b) { return !b.defined() || b.device() == a.device(); }

bool i64_list(const at::Tensor& t, int64_t n) { return t.scalar_type() == at::kLong && t.is_contiguous() && t.numel() == n; }

struct Routing {
    at::Tensor topk_idx, gates, lengths, offsets, gate_index, token_index, reverse_index;
};

bool route(const at::Tensor& scores, int64_t k, int64_t mode, void* stream, Routing& r) {
    if (scores.dim() != 2 || !scores.is_contiguous()) return false;
    const int code = dtype_code(scores.scalar_type());
    if (code != FMOE_F32 && code != FMOE_BF16) return false;
    const int64_t T = scores.size(0), E = scores.size(1);
    if (k < 1 || k > E || E > INT32_MAX) return false;
    r.topk_idx = empty({T, k}, at::kLong, scores);
    r.gates = empty({T, k}, scores.scalar_type(), scores);
    r.lengths = empty({E}, at::kLong, scores);
    r.offsets = empty({E + 1}, at::kLong, scores);
    r.gate_index = empty({T * k}, at::kLong, scores);
    r.token_index = empty({T * k}, at::kLong, scores);
    r.reverse_index = empty({T, k}, at::kLong, scores);
    const size_t ws_bytes = route_workspace_bytes(T, (int)E, (int)k);
    const at::Tensor ws = empty({(int64_t)(ws_bytes ? ws_bytes : 1)}, at::kByte, scores);
    return c_route_topk(scores.data_ptr(), code, T, (int)E, (int)k, (int)mode, r.topk_idx.data_ptr<int64_t>(),
                        r.gates.data_ptr(), r.lengths.data_ptr<int64_t>(), r.offsets.data_ptr<int64_t>(),
                        r.gate_index.data_ptr<int64_t>(), r.token_index.data_ptr<int64_t>(),
                        r.reverse_index.data_ptr<int64_t>(), ws.data_ptr(), ws_bytes, stream) == FMOE_OK;
}

struct GemmArgs {
    at::Tensor offsets, a, b, row_index, bias, b2, bias2, a_scale, b_scale, b2_scale;
    int64_t total_rows = 0, index_div = 1, epilogue = FMOE_EPI_NONE, pow2 = 0;
};

bool gemm(const GemmArgs& g, void* stream, at::Tensor& out) {
    const at::Tensor &a = g.a, &b = g.b;
    const int code = dtype_code(a.scalar_type());
    if (code < 0 || b.scalar_type() != a.scalar_type() || a.dim() != 2 || b.dim() != 3) return false;
    const bool fp8 = code == FMOE_E4M3;
    const at::ScalarType out_dtype = code == FMOE_F32 ? at::kFloat : at::kBFloat16;
    const int64_t E = b.size(0), K = b.size(1), N = b.size(2);
    if (a.size(1) != K || a.stride(1) != 1 || g.total_rows < 1 || g.index_div < 1 || E > INT32_MAX || K > INT32_MAX ||
        N > INT32_MAX || g.index_div > INT32_MAX)
        return false;
    for (const at::Tensor* t : {&g.offsets, &g.b, &g.row_index, &g.bias, &g.b2, &g.bias2, &g.a_scale, &g.b_scale, &g.b2_scale})
        if (!same_device(a, *t)) return false;
    if (!i64_list(g.offsets, E + 1) || (g.row_index.defined() && !i64_list(g.row_index, g.total_rows))) return false;
    if (g.b2.defined() &&
        (g.b2.scalar_type() != b.scalar_type() || g.b2.sizes() != b.sizes() || g.b2.strides() != b.strides()))
        return false;
    if (b.stride(2) == 1 && b.stride(1) != 1) return false;     // ops.grouped_gemm asks for the plan of these first
    for (const at::Tensor* t : {&g.bias, &g.bias2})
        if (t->defined() &&
            (t->scalar_type() != out_dtype || t->dim() != 2 || t->size(0) != E || t->size(1) != N || t->stride(1) != 1))
            return false;
    if (g.bias.defined() && g.bias2.defined() && g.bias.stride(0) != g.bias2.stride(0)) return false;
    if (fp8) {
        if (!g.a_scale.defined() || !g.b_scale.defined() || (g.b2.defined() && !g.b2_scale.defined())) return false;
        for (const at::Tensor* t : {&g.a_scale, &g.b_scale, &g.b2_scale})
            if (t->defined() && (t->scalar_type() != at::kFloat || !t->is_contiguous() ||
                                 t->numel() != (t == &g.a_scale ? a.size(0) : E * N)))
                return false;
    } else if (g.a_scale.defined() || g.b_scale.defined() || g.b2_scale.defined()) {
        return false;
    }
    out = empty({g.total_rows + kSlackRows, N}, out_dtype, a).narrow(0, 0, g.total_rows);
    fmoe_gemm_desc d = {};
    d.num_experts = (int32_t)E;
    d.n = (int32_t)N;
    d.k = (int32_t)K;
    d.index_div = (int32_t)g.index_div;
    d.total_rows = g.total_rows;
    d.a_rows = a.size(0);
    auto data = [](const at::Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; };
    auto floats = [](const at::Tensor& t) { return t.defined() ? t.data_ptr<float>() : nullptr; };
    d.offsets = g.offsets.data_ptr<int64_t>();
    d.row_index = g.row_index.defined() ? g.row_index.data_ptr<int64_t>() : nullptr;
    d.a = a.data_ptr();
    d.a_dtype = code;
    d.a_stride_row = a.stride(0);
    d.a_scale = floats(g.a_scale);
    d.b = b.data_ptr();
    d.b2 = data(g.b2);
    d.b_stride_e = b.stride(0);
    d.b_stride_k = b.stride(1);
    d.b_stride_n = b.stride(2);
    d.b_scale = floats(g.b_scale);
    d.b2_scale = floats(g.b2_scale);
    d.scale_pow2 = fp8 && g.pow2;
    d.bias = data(g.bias);
    d.bias2 = data(g.bias2);
    d.bias_stride_e = g.bias.defined() ? g.bias.stride(0) : g.bias2.defined() ? g.bias2.stride(0) : 0;
    d.epilogue = (int32_t)g.epilogue;
    d.out_dtype = dtype_code(out_dtype);
    d.out = out.data_ptr();
    d.out_stride_row = out.stride(0);
    return c_grouped_gemm(&d, stream) == FMOE_OK;
}

bool combine(const at::Tensor& value, const at::Tensor& reverse, const at::Tensor& gates, const at::Tensor& gates_index,
             void* stream, at::Tensor& out) {
    const int code = dtype_code(value.scalar_type());
    if ((code != FMOE_F32 && code != FMOE_BF16) || value.dim() != 2 || value.stride(1) != 1 || reverse.dim() != 2)
        return false;
    if (!same_device(value, reverse) || !same_device(value, gates) || !same_device(value, gates_index)) return false;
    const int64_t T = reverse.size(0), K = reverse.size(1), D = value.size(1);
    if (!i64_list(reverse, T * K) || value.size(0) != T * K || K < 1 || K > INT32_MAX) return false;
    at::ScalarType out_dtype = value.scalar_type();
    int g_code = FMOE_F32;
    int64_t cols = 1, sr = 1, sc = 1;
    if (gates.defined()) {
        g_code = dtype_code(gates.scalar_type());
        if ((g_code != FMOE_F32 && g_code != FMOE_BF16) || gates.dim() != 2 || gates.numel() != T * K) return false;
        if (g_code == FMOE_F32) out_dtype = at::kFloat;
        cols = gates.size(1);
        sr = gates.stride(0);
        sc = gates.stride(1);
        if (gates_index.defined() && !i64_list(gates_index, T * K)) return false;
    }
    const bool indexed = gates.defined() && gates_index.defined();
    out = empty({T, D}, out_dtype, value);
    return c_combine(value.data_ptr(), code, T, (int)K, D, value.stride(0), reverse.data_ptr<int64_t>(),
                     gates.defined() ? gates.data_ptr() : nullptr, g_code, cols, sr, sc,
                     indexed ? gates_index.data_ptr<int64_t>() : nullptr, out.data_ptr(), dtype_code(out_dtype),
                     stream) == FMOE_OK;
}

PyObject* none() { Py_RETURN_NONE; }
PyObject* wrap(const at::Tensor& t) { return THPVariable_Wrap(t); }

// A C++ exception (a tensor that hides its storage, out of memory) also leaves the call to the Python code, which raises it
// as torch raises it there.
template <typename F>
bool guarded(F&& f) {
    NoGil nogil;
    try {
        return f();
    } catch (const std::exception&) {
        return false;
    }
}

// (scores, k, mode, stream) -> (topk_idx, gates, lengths, offsets, gate_index, token_index, reverse_index)
PyObject* py_route_topk(PyObject*, PyObject* const* args, Py_ssize_t n) {
    int64_t k, mode, stream;
    const at::Tensor scores = n == 4 ? gpu_tensor(args[0]) : at::Tensor();
    if (!scores.defined() || !as_int(args[1], &k) || !as_int(args[2], &mode) || !as_int(args[3], &stream)) return none();
    Routing r;
    if (!guarded([&] { return route(scores, k, mode, (void*)stream, r); })) return none();
    PyObject* out = PyTuple_New(7);
    if (!out) return nullptr;
    const at::Tensor* parts[7] = {&r.topk_idx, &r.gates, &r.lengths, &r.offsets, &r.gate_index, &r.token_index,
                                  &r.reverse_index};
    for (int i = 0; i < 7; ++i) PyTuple_SET_ITEM(out, i, wrap(*parts[i]));
    return out;
}

// (offsets, a, b, total_rows, row_index, index_div, bias, b2, bias2, epilogue, a_scale, b_scale, b2_scale, pow2, stream)
PyObject* py_grouped_gemm(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 15) return none();
    GemmArgs g;
    int64_t stream;
    g.offsets = gpu_tensor(args[0]);
    g.a = gpu_tensor(args[1]);
    g.b = gpu_tensor(args[2]);
    if (!g.offsets.defined() || !g.a.defined() || !g.b.defined() || !as_int(args[3], &g.total_rows) || !optional_tensor(args[4], &g.row_index) ||
        !as_int(args[5], &g.index_div) || !optional_tensor(args[6], &g.bias) || !optional_tensor(args[7], &g.b2) ||
        !optional_tensor(args[8], &g.bias2) || !as_int(args[9], &g.epilogue) || !optional_tensor(args[10], &g.a_scale) ||
        !optional_tensor(args[11], &g.b_scale) || !optional_tensor(args[12], &g.b2_scale) || !as_int(args[13], &g.pow2) ||
        !as_int(args[14], &stream))
        return none();
    at::Tensor out;
    return guarded([&] { return gemm(g, (void*)stream, out); }) ? wrap(out) : none();
}

// (value, reverse_index, gates, gates_index, stream)
PyObject* py_combine(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 5) return none();
    const at::Tensor value = gpu_tensor(args[0]), reverse = gpu_tensor(args[1]);
    at::Tensor gates, gates_index;
    int64_t stream;
    if (!value.defined() || !reverse.defined() || !optional_tensor(args[2], &gates) || !optional_tensor(args[3], &gates_index) ||
        !as_int(args[4], &stream))
        return none();
    at::Tensor out;
    return guarded([&] { return combine(value, reverse, gates, gates_index, (void*)stream, out); }) ? wrap(out) : none();
}

// (a, apply_silu, reciprocal, stream) -> (q, scale): a 2-D input with contiguous rows
PyObject* py_quant_rows(PyObject*, PyObject* const* args, Py_ssize_t n) {
    const at::Tensor a = n == 4 ? gpu_tensor(args[0]) : at::Tensor();
    int64_t silu, reciprocal, stream;
    if (!a.defined() || !as_int(args[1], &silu) || !as_int(args[2], &reciprocal) || !as_int(args[3], &stream)) return none();
    at::Tensor q, scale;
    const bool ok = guarded([&] {
        const int code = dtype_code(a.scalar_type());
        if ((code != FMOE_F32 && code != FMOE_BF16) || a.dim() != 2 || a.size(1) < 1 || a.stride(1) != 1) return false;
        const int64_t rows = a.size(0), cols = a.size(1);
        q = empty({rows, cols}, at::kFloat8_e4m3fn, a);
        scale = empty({rows}, at::kFloat, a);
        return c_quant_rows(a.data_ptr(), code, 1, rows, cols, rows * a.stride(0), a.stride(0), 1, (int)silu,
                            (uint8_t*)q.data_ptr(), rows * cols, cols, 1, scale.data_ptr<float>(), (int)reciprocal,
                            (void*)stream) == FMOE_OK;
    });
    return ok ? Py_BuildValue("(NN)", wrap(q), wrap(scale)) : none();
}

// (scores [T, E], x [T, D], w1 [E, D, H], bias1, w2 [E, H, O], bias2, k, mode, epilogue1, stream) -> [T, O]:
// routing, the gather GEMM with its activation, the second GEMM, the merge
PyObject* py_mlp_forward(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 10) return none();
    const at::Tensor scores = gpu_tensor(args[0]), x = gpu_tensor(args[1]), w1 = gpu_tensor(args[2]);
    const at::Tensor b1 = gpu_tensor(args[3]), w2 = gpu_tensor(args[4]), b2 = gpu_tensor(args[5]);
    int64_t k, mode, epilogue, stream;
    for (const at::Tensor* t : {&scores, &x, &w1, &b1, &w2, &b2})
        if (!t->defined()) return none();
    if (!as_int(args[6], &k) || !as_int(args[7], &mode) || !as_int(args[8], &epilogue) || !as_int(args[9], &stream))
        return none();
    at::Tensor y;
    const bool ok = guarded([&] {
        if (x.dim() != 2 || scores.dim() != 2 || scores.size(0) != x.size(0) || w1.dim() != 3 ||
            w1.size(0) != scores.size(1) || scores.device() != x.device())
            return false;
        Routing r;
        if (!route(scores, k, mode, (void*)stream, r)) return false;
        RECORD_USER_SCOPE("## expert_forward##");
        at::Tensor hidden, rows;
        GemmArgs g;
        g.offsets = r.offsets;
        g.a = x;
        g.b = w1;
        g.row_index = r.gate_index;
        g.bias = b1;
        g.total_rows = x.size(0) * k;
        g.index_div = k;
        g.epilogue = epilogue;
        if (!gemm(g, (void*)stream, hidden)) return false;
        GemmArgs down;
        down.offsets = r.offsets;
        down.a = hidden;
        down.b = w2;
        down.bias = b2;
        down.total_rows = hidden.size(0);
        return gemm(down, (void*)stream, rows) && combine(rows, r.reverse_index, r.gates, r.gate_index, (void*)stream, y);
    });
    return ok ? wrap(y) : none();
}

// init(addresses of the C entry points, in the order of the pointers above)
PyObject* py_init(PyObject*, PyObject* const* args, Py_ssize_t n) {
    int64_t v[5];
    if (n != 5) {
        PyErr_SetString(PyExc_TypeError, "init: five addresses expected");
        return nullptr;
    }
    for (int i = 0; i < 5; ++i)
        if (!as_int(args[i], &v[i])) {
            PyErr_SetString(PyExc_TypeError, "init: addresses are integers");
            return nullptr;
        }
    route_workspace_bytes = (decltype(route_workspace_bytes))v[0];
    c_route_topk = (decltype(c_route_topk))v[1];
    c_grouped_gemm = (decltype(c_grouped_gemm))v[2];
    c_combine = (decltype(c_combine))v[3];
    c_quant_rows = (decltype(c_quant_rows))v[4];
    return none();
}

#define FASTCALL(name, fn) {name, (PyCFunction)(void (*)(void))fn, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    FASTCALL("init", py_init),
    FASTCALL("route_topk", py_route_topk),
    FASTCALL("grouped_gemm", py_grouped_gemm),
    FASTCALL("combine", py_combine),
    FASTCALL("quant_rows", py_quant_rows),
    FASTCALL("mlp_forward", py_mlp_forward),
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) { return PyModule_Create(&module); }
