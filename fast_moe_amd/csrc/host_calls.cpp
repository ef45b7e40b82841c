// The host side of the operators, forward and backward, as one native call each: argument checks, output allocation, stride marshalling and
// the launch, for the calls a forward pass makes.
//
// What it is for: a pass over a few tokens is bound by the host (64 tokens, 8 experts, 128 -> 256 -> 128: seven launches that
// keep the GPU busy for 39 us took 131 us to issue, now 69), and most of that was Python: one interpreter call per tensor attribute,
// output and descriptor field.
//
// Every function here takes a call whole or returns None and has done nothing that matters: whatever it does not recognise
// (other dtypes, layouts, tensor subclasses, wrong shapes, a call the library refuses) is left to the Python code in ops.py,
// which handles it or raises.  What fails once work is being issued (no memory, a launch error) raises here: issued again it
// would run twice, and a launch error that the first attempt has read is gone for the second.  Nothing is kept from one call
// for the next.  The C entry points are handed over as addresses once (init), so that this module works with whichever build
// of the library ctypes has loaded.
#include <Python.h>
#include <ATen/ATen.h>
#include <ATen/record_function.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/version.h>

#include <cstdint>
#include <cstring>

#include "../../include/fast_moe_amd.h"

namespace {

decltype(&fmoe_route_workspace_bytes) route_workspace_bytes;
decltype(&fmoe_route_topk) c_route_topk;
decltype(&fmoe_grouped_gemm) c_grouped_gemm;
decltype(&fmoe_grouped_gemm_workspace_bytes) gemm_workspace_bytes;
decltype(&fmoe_grouped_gemm_ws) c_grouped_gemm_ws;
decltype(&fmoe_combine) c_combine;
decltype(&fmoe_quant_rows_e4m3) c_quant_rows;
decltype(&fmoe_gate_softmax) c_gate_softmax;
decltype(&fmoe_gate_softmax_pays) gate_softmax_pays;
decltype(&fmoe_gate_route_pays) gate_route_pays;
decltype(&fmoe_grouped_gemm_plan) c_gemm_plan;
decltype(&fmoe_combine_bwd) c_combine_bwd;
decltype(&fmoe_segment_colsum) c_segment_colsum;
decltype(&fmoe_swiglu_bwd) c_swiglu_bwd;
decltype(&fmoe_silu_mul) c_silu_mul;
decltype(&fmoe_gather_rows) c_gather_rows;
decltype(&fmoe_invert_index) c_invert_index;
decltype(&fmoe_gate_l1_bwd) c_gate_l1_bwd;
decltype(&fmoe_weight_grad) c_weight_grad;
decltype(&fmoe_weight_grad_pays) weight_grad_pays;
decltype(&fmoe_last_error) last_error;

constexpr int64_t kSlackRows = 128;      // ops.SLACK_ROWS

constexpr int kDeclined = -1;           // beside the C status codes: left to the Python code

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
    at::Tensor topk_idx, gates, lengths, offsets, gate_index, token_index, reverse_index, workspace;
};

bool route_ok(const at::Tensor& scores, int64_t k, const void** data) {
    if (scores.dim() != 2 || !scores.is_contiguous()) return false;
    const int code = dtype_code(scores.scalar_type());
    if (code != FMOE_F32 && code != FMOE_BF16) return false;
    const int64_t E = scores.size(1);
    *data = scores.data_ptr();
    return k >= 1 && k <= E && E <= INT32_MAX;
}

void allocate(const at::Tensor& scores, int64_t k, Routing& r) {
    const int64_t T = scores.size(0), E = scores.size(1);
    r.topk_idx = empty({T, k}, at::kLong, scores);
    r.gates = empty({T, k}, scores.scalar_type(), scores);
    r.lengths = empty({E}, at::kLong, scores);
    r.offsets = empty({E + 1}, at::kLong, scores);
    r.gate_index = empty({T * k}, at::kLong, scores);
    r.token_index = empty({T * k}, at::kLong, scores);
    r.reverse_index = empty({T, k}, at::kLong, scores);
    const size_t ws_bytes = route_workspace_bytes(T, (int)E, (int)k);
    r.workspace = empty({(int64_t)(ws_bytes ? ws_bytes : 1)}, at::kByte, scores);
}

int route(const at::Tensor& scores, const void* data, int64_t k, int64_t mode, void* stream, const Routing& r) {
    return c_route_topk(data, dtype_code(scores.scalar_type()), scores.size(0), (int)scores.size(1), (int)k, (int)mode,
                        r.topk_idx.data_ptr<int64_t>(), r.gates.data_ptr(), r.lengths.data_ptr<int64_t>(),
                        r.offsets.data_ptr<int64_t>(), r.gate_index.data_ptr<int64_t>(), r.token_index.data_ptr<int64_t>(),
                        r.reverse_index.data_ptr<int64_t>(), r.workspace.data_ptr(), r.workspace.numel(), stream);
}

// Intermediates of a call that is issued whole have no tensors of their own (one allocation holds them all): offsets and row_index are
// pointers then, and a stands for contiguous rows at a_data.
struct GemmArgs {
    at::Tensor offsets, a, b, row_index, bias, b2, bias2, a_scale, b_scale, b2_scale;
    int64_t total_rows = 0, index_div = 1, epilogue = FMOE_EPI_NONE, pow2 = 0;
    const int64_t *offsets_data = nullptr, *row_index_data = nullptr;
    const void* a_data = nullptr;
    int64_t a_rows = 0;
    bool n_contiguous = false;      // weights with n contiguous are taken
};

// Checks the operands and fills everything of the descriptor but the output.
bool gemm_ok(const GemmArgs& g, fmoe_gemm_desc& d) {
    const at::Tensor &a = g.a, &b = g.b;
    const int code = dtype_code(b.scalar_type());
    if (code < 0 || b.dim() != 3 || (!g.a_data && (a.scalar_type() != b.scalar_type() || a.dim() != 2))) return false;
    const bool fp8 = code == FMOE_E4M3;
    const at::ScalarType out_dtype = code == FMOE_F32 ? at::kFloat : at::kBFloat16;
    const int64_t E = b.size(0), K = b.size(1), N = b.size(2);
    if ((!g.a_data && (a.size(1) != K || a.stride(1) != 1)) || g.total_rows < 1 || g.index_div < 1 || E > INT32_MAX || K > INT32_MAX ||
        N > INT32_MAX || g.index_div > INT32_MAX)
        return false;
    for (const at::Tensor* t : {&g.offsets, &g.a, &g.row_index, &g.bias, &g.b2, &g.bias2, &g.a_scale, &g.b_scale, &g.b2_scale})
        if (!same_device(b, *t)) return false;
    if ((!g.offsets_data && !i64_list(g.offsets, E + 1)) || (g.row_index.defined() && !i64_list(g.row_index, g.total_rows))) return false;
    if (g.b2.defined() &&
        (g.b2.scalar_type() != b.scalar_type() || g.b2.sizes() != b.sizes() || g.b2.strides() != b.strides()))
        return false;
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
    d = {};
    d.num_experts = (int32_t)E;
    d.n = (int32_t)N;
    d.k = (int32_t)K;
    d.index_div = (int32_t)g.index_div;
    d.total_rows = g.total_rows;
    d.a_rows = g.a_data ? g.a_rows : a.size(0);
    auto data = [](const at::Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; };
    auto floats = [](const at::Tensor& t) { return t.defined() ? t.data_ptr<float>() : nullptr; };
    d.offsets = g.offsets_data ? g.offsets_data : g.offsets.data_ptr<int64_t>();
    d.row_index = g.row_index.defined() ? g.row_index.data_ptr<int64_t>() : g.row_index_data;
    d.a = g.a_data ? g.a_data : a.data_ptr();
    d.a_dtype = code;
    d.a_stride_row = g.a_data ? K : a.stride(0);
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
    // ... unless only the element-load kernel would read them in place: ops.grouped_gemm copies them first
    if (b.stride(2) == 1 && b.stride(1) != 1 && !g.n_contiguous) return false;
    if (b.stride(2) == 1 && b.stride(1) != 1 && K % 16 == 0 && N % 8 == 0 && g.total_rows * N >= (1 << 22)) {
        d.out = (void*)(uintptr_t)256;      // (where the allocator would put it, as far as alignment goes)
        d.out_stride_row = N;
        int plan;
        if (c_gemm_plan(&d, &plan) != FMOE_OK || plan == FMOE_PLAN_ELEMENT) return false;
    }
    return true;
}

at::Tensor allocate(fmoe_gemm_desc& d, const at::Tensor& like) {
    const at::Tensor out = empty({d.total_rows + kSlackRows, d.n}, d.out_dtype == FMOE_F32 ? at::kFloat : at::kBFloat16, like)
                               .narrow(0, 0, d.total_rows);
    d.out = out.data_ptr();
    d.out_stride_row = out.stride(0);
    return out;
}

// (the workspace may be handed out again as soon as the call is issued: what takes it runs behind the call on the stream)
int gemm(const fmoe_gemm_desc& d, const at::Tensor& like, void* stream) {
    const size_t bytes = gemm_workspace_bytes(&d);
    at::Tensor workspace;
    if (bytes) {
        try {
            workspace = empty({(int64_t)bytes}, at::kByte, like);
        } catch (const c10::OutOfMemoryError&) {    // it makes the call faster, not possible
        }
    }
    return workspace.defined() ? c_grouped_gemm_ws(&d, workspace.data_ptr(), bytes, stream) : c_grouped_gemm(&d, stream);
}

struct Combine {
    at::Tensor value, reverse, gates, gates_index;
    const void *value_data, *gates_data = nullptr;
    const int64_t *reverse_data, *index_data = nullptr;
    at::ScalarType out_dtype;
    int code, g_code = FMOE_F32;
    int64_t T, K, D, value_stride, cols = 1, sr = 1, sc = 1;
};

bool combine_ok(Combine& c) {
    c.code = dtype_code(c.value.scalar_type());
    if ((c.code != FMOE_F32 && c.code != FMOE_BF16) || c.value.dim() != 2 || c.value.stride(1) != 1 || c.reverse.dim() != 2)
        return false;
    if (!same_device(c.value, c.reverse) || !same_device(c.value, c.gates) || !same_device(c.value, c.gates_index)) return false;
    c.T = c.reverse.size(0);
    c.K = c.reverse.size(1);
    c.D = c.value.size(1);
    if (!i64_list(c.reverse, c.T * c.K) || c.value.size(0) != c.T * c.K || c.K < 1 || c.K > INT32_MAX) return false;
    c.out_dtype = c.value.scalar_type();
    if (c.gates.defined()) {
        c.g_code = dtype_code(c.gates.scalar_type());
        if ((c.g_code != FMOE_F32 && c.g_code != FMOE_BF16) || c.gates.dim() != 2 || c.gates.numel() != c.T * c.K) return false;
        if (c.g_code == FMOE_F32) c.out_dtype = at::kFloat;
        c.cols = c.gates.size(1);
        c.sr = c.gates.stride(0);
        c.sc = c.gates.stride(1);
        c.gates_data = c.gates.data_ptr();
        if (c.gates_index.defined()) {
            if (!i64_list(c.gates_index, c.T * c.K)) return false;
            c.index_data = c.gates_index.data_ptr<int64_t>();
        }
    }
    c.value_data = c.value.data_ptr();
    c.value_stride = c.value.stride(0);
    c.reverse_data = c.reverse.data_ptr<int64_t>();
    return true;
}

at::Tensor allocate(const Combine& c, const at::Tensor& like) { return empty({c.T, c.D}, c.out_dtype, like); }

int combine(const Combine& c, const at::Tensor& out, void* stream) {
    return c_combine(c.value_data, c.code, c.T, (int)c.K, c.D, c.value_stride, c.reverse_data, c.gates_data, c.g_code, c.cols,
                     c.sr, c.sc, c.index_data, out.data_ptr(), dtype_code(c.out_dtype), stream);
}

PyObject* none() { Py_RETURN_NONE; }
PyObject* wrap(const at::Tensor& t) { return THPVariable_Wrap(t); }

// check() looks at the operands (what throws there, a tensor that hides its storage say, is left to the Python code, which
// raises it as torch does), issue() allocates and launches (what throws there is the call's).  -> kDeclined or a C status.
template <typename Check, typename Issue>
int run(Check&& check, Issue&& issue) {
    NoGil nogil;
    try {
        if (!check()) return kDeclined;
    } catch (const std::exception&) {
        return kDeclined;
    }
    return issue();
}

// The library's other refusals come before its first launch: the Python code raises them, in its own words where it has any.
bool raised(int status, const char* what) {
    if (status != FMOE_ERR_LAUNCH) return false;
    PyErr_Format(PyExc_RuntimeError, "%s failed (status %d): %s", what, status, last_error());
    return true;
}

// (scores, k, mode, stream) -> (topk_idx, gates, lengths, offsets, gate_index, token_index, reverse_index)
PyObject* py_route_topk(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    int64_t k, mode, stream;
    const at::Tensor scores = n == 4 ? gpu_tensor(args[0]) : at::Tensor();
    if (!scores.defined() || !as_int(args[1], &k) || !as_int(args[2], &mode) || !as_int(args[3], &stream)) return none();
    Routing r;
    const void* data;
    const int status = run([&] { return route_ok(scores, k, &data); },
                           [&] {
                               allocate(scores, k, r);
                               return route(scores, data, k, mode, (void*)stream, r);
                           });
    if (raised(status, "fmoe_route_topk")) return nullptr;
    if (status != FMOE_OK) return none();
    PyObject* out = PyTuple_New(7);
    if (!out) return nullptr;
    const at::Tensor* parts[7] = {&r.topk_idx, &r.gates, &r.lengths, &r.offsets, &r.gate_index, &r.token_index,
                                  &r.reverse_index};
    for (int i = 0; i < 7; ++i) PyTuple_SET_ITEM(out, i, wrap(*parts[i]));
    return out;
    END_HANDLE_TH_ERRORS
}

// (offsets, a, b, total_rows, row_index, index_div, bias, b2, bias2, epilogue, a_scale, b_scale, b2_scale, pow2, stream)
template <bool N_CONTIGUOUS>
PyObject* py_grouped_gemm(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 15) return none();
    GemmArgs g;
    g.n_contiguous = N_CONTIGUOUS;
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
    fmoe_gemm_desc d;
    const int status = run([&] { return gemm_ok(g, d); },
                           [&] {
                               out = allocate(d, g.a);
                               return gemm(d, g.a, (void*)stream);
                           });
    if (raised(status, "fmoe_grouped_gemm")) return nullptr;
    return status == FMOE_OK ? wrap(out) : none();
    END_HANDLE_TH_ERRORS
}

// (value, reverse_index, gates, gates_index, stream)
PyObject* py_combine(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 5) return none();
    Combine c;
    c.value = gpu_tensor(args[0]);
    c.reverse = gpu_tensor(args[1]);
    int64_t stream;
    if (!c.value.defined() || !c.reverse.defined() || !optional_tensor(args[2], &c.gates) ||
        !optional_tensor(args[3], &c.gates_index) || !as_int(args[4], &stream))
        return none();
    at::Tensor out;
    const int status = run([&] { return combine_ok(c); },
                           [&] {
                               out = allocate(c, c.value);
                               return combine(c, out, (void*)stream);
                           });
    if (raised(status, "fmoe_combine")) return nullptr;
    return status == FMOE_OK ? wrap(out) : none();
    END_HANDLE_TH_ERRORS
}

// (a, apply_silu, reciprocal, stream) -> (q, scale): a 2-D input with contiguous rows
PyObject* py_quant_rows(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    const at::Tensor a = n == 4 ? gpu_tensor(args[0]) : at::Tensor();
    int64_t silu, reciprocal, stream;
    if (!a.defined() || !as_int(args[1], &silu) || !as_int(args[2], &reciprocal) || !as_int(args[3], &stream)) return none();
    at::Tensor q, scale;
    const void* data;
    int code;
    const int status = run(
        [&] {
            code = dtype_code(a.scalar_type());
            if ((code != FMOE_F32 && code != FMOE_BF16) || a.dim() != 2 || a.size(1) < 1 || a.stride(1) != 1) return false;
            data = a.data_ptr();
            return true;
        },
        [&] {
            const int64_t rows = a.size(0), cols = a.size(1);
            q = empty({rows, cols}, at::kFloat8_e4m3fn, a);
            scale = empty({rows}, at::kFloat, a);
            return c_quant_rows(data, code, 1, rows, cols, rows * a.stride(0), a.stride(0), 1, (int)silu,
                                (uint8_t*)q.data_ptr(), rows * cols, cols, 1, scale.data_ptr<float>(), (int)reciprocal,
                                (void*)stream);
        });
    if (raised(status, "fmoe_quant_rows_e4m3")) return nullptr;
    return status == FMOE_OK ? Py_BuildValue("(NN)", wrap(q), wrap(scale)) : none();
    END_HANDLE_TH_ERRORS
}

// What the launches that stand for the gate take: one type, rows of x and the weight at 16-byte boundaries.
bool gate_ok(const at::Tensor& x, const at::Tensor& w, const at::Tensor& bias, const void** x_data, const void** w_data, const void** b_data) {
    const int code = dtype_code(x.scalar_type());
    if ((code != FMOE_F32 && code != FMOE_BF16) || w.scalar_type() != x.scalar_type() || x.dim() != 2 || w.dim() != 2 ||
        x.size(1) != w.size(1) || x.stride(1) != 1 || !w.is_contiguous() || !same_device(x, w) || !same_device(x, bias) ||
        w.size(0) > INT32_MAX || w.size(1) > INT32_MAX)
        return false;
    if (bias.defined() && (bias.scalar_type() != x.scalar_type() || !bias.is_contiguous() || bias.numel() != w.size(0))) return false;
    if (!gate_softmax_pays(code, x.size(0), (int)x.size(1), (int)w.size(0)) || x.stride(0) < x.size(1) ||
        x.stride(0) % (code == FMOE_F32 ? 4 : 8))
        return false;
    *x_data = x.data_ptr();
    *w_data = w.data_ptr();
    *b_data = bias.defined() ? bias.data_ptr() : nullptr;
    return (uintptr_t)*x_data % 16 == 0 && (uintptr_t)*w_data % 16 == 0;
}

// (x [T, D], weight [E, D], bias [E] or None, stream) -> softmax(x weight^T + bias) [T, E], where fmoe_gate_softmax is the faster form
PyObject* py_gate_softmax(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 4) return none();
    const at::Tensor x = gpu_tensor(args[0]), w = gpu_tensor(args[1]);
    at::Tensor bias, scores;
    int64_t stream;
    if (!x.defined() || !w.defined() || !optional_tensor(args[2], &bias) || !as_int(args[3], &stream)) return none();
    const void *x_data, *w_data, *b_data = nullptr;
    const int status = run(
        [&] { return gate_ok(x, w, bias, &x_data, &w_data, &b_data); },
        [&] {
            scores = empty({x.size(0), w.size(0)}, x.scalar_type(), x);
            return c_gate_softmax(x_data, dtype_code(x.scalar_type()), x.size(0), (int)x.size(1), x.stride(0), w_data, b_data, (int)w.size(0),
                                  scores.data_ptr(), (void*)stream);
        });
    if (raised(status, "fmoe_gate_softmax")) return nullptr;
    return status == FMOE_OK ? wrap(scores) : none();
    END_HANDLE_TH_ERRORS
}

// (scores [T, E], x [T, D], w1 [E, D, H], bias1, w2 [E, H, O], bias2, k, mode, epilogue1, stream) -> [T, O]:
// routing, the gather GEMM with its activation, the second GEMM, the merge.  With scores None, a gate's weight [E, D] and its bias [E] or None
// behind the stream: the gate as fmoe_gate_softmax (where that pays), in the routing's launch where fmoe_gate_route_pays
PyObject* py_mlp_forward(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 10 && n != 12) return none();
    const bool gate = n == 12;
    const at::Tensor scores = gate ? gpu_tensor(args[10]) : gpu_tensor(args[0]);        // (gate: [E, D] in its place)
    const at::Tensor x = gpu_tensor(args[1]), w1 = gpu_tensor(args[2]);
    at::Tensor gate_bias;
    if (gate && (args[0] != Py_None || !optional_tensor(args[11], &gate_bias))) return none();
    const at::Tensor b1 = gpu_tensor(args[3]), w2 = gpu_tensor(args[4]), b2 = gpu_tensor(args[5]);
    int64_t k, mode, epilogue, stream;
    for (const at::Tensor* t : {&scores, &x, &w1, &b1, &w2, &b2})
        if (!t->defined()) return none();
    if (!as_int(args[6], &k) || !as_int(args[7], &mode) || !as_int(args[8], &epilogue) || !as_int(args[9], &stream))
        return none();
    at::Tensor scratch, y;
    const void *data = nullptr, *x_data = nullptr, *gate_bias_data = nullptr;
    char* base = nullptr;
    size_t at_ws = 0, ws_bytes = 0;
    int64_t *topk_idx = nullptr, *lengths = nullptr, *offsets = nullptr, *gate_index = nullptr, *token_index = nullptr, *reverse = nullptr;
    void *gates = nullptr, *gate_scores = nullptr;
    bool one_launch = false;
    fmoe_gemm_desc up, down;
    Combine merge;
    const char* what = "fmoe_route_topk";
    // All operands of the four launches, intermediates included, exist and are checked before the first launch: a call that
    // is declined has routed nothing.  One allocation holds the intermediates (twelve were 10 of the 30 us that the call took).
    const int status = run(
        [&] {
            if (x.dim() != 2 || scores.dim() != 2 || w1.dim() != 3 || w2.dim() != 3 || w2.size(1) != w1.size(2) ||
                w2.scalar_type() != w1.scalar_type() || scores.device() != x.device() || w1.device() != x.device() ||
                w2.device() != x.device())
                return false;
            const int64_t T = x.size(0), E = scores.size(gate ? 0 : 1);
            if (w1.size(0) != E || w2.size(0) != E) return false;
            if (gate) {
                if (!gate_ok(x, scores, gate_bias, &x_data, &data, &gate_bias_data) || k < 1 || k > E) return false;
                one_launch = gate_route_pays(dtype_code(x.scalar_type()), T, (int)x.size(1), (int)E, (int)k) != 0;
            } else if (scores.size(0) != T || !route_ok(scores, k, &data)) {
                return false;
            }
            const int64_t H = w1.size(2), O = w2.size(2), R = T * k;
            const int64_t row_size = w1.scalar_type() == at::kFloat ? 4 : 2;
            size_t bytes = 0;
            auto take = [&](int64_t n, int64_t size) {
                const size_t at = bytes;
                bytes += ((size_t)(n * size) + 255) & ~(size_t)255;
                return at;
            };
            ws_bytes = one_launch ? 0 : route_workspace_bytes(T, (int)E, (int)k);
            const size_t at_topk = take(R, 8), at_lengths = take(E, 8), at_offsets = take(E + 1, 8), at_gate = take(R, 8);
            const size_t at_token = take(R, 8), at_reverse = take(R, 8), at_gates = take(R, (int64_t)scores.element_size());
            at_ws = take((int64_t)ws_bytes, 1);
            const size_t at_scores = take(gate && !one_launch ? T * E : 0, (int64_t)scores.element_size());
            const size_t at_hidden = take((R + kSlackRows) * H, row_size), at_rows = take((R + kSlackRows) * O, row_size);
            scratch = empty({(int64_t)bytes}, at::kByte, x);
            base = (char*)scratch.data_ptr();
            topk_idx = (int64_t*)(base + at_topk);
            lengths = (int64_t*)(base + at_lengths);
            offsets = (int64_t*)(base + at_offsets);
            gate_index = (int64_t*)(base + at_gate);
            token_index = (int64_t*)(base + at_token);
            reverse = (int64_t*)(base + at_reverse);
            gates = base + at_gates;
            gate_scores = base + at_scores;
            GemmArgs g;
            g.offsets_data = offsets;
            g.a = x;
            g.b = w1;
            g.row_index_data = gate_index;
            g.bias = b1;
            g.total_rows = R;
            g.index_div = k;
            g.epilogue = epilogue;
            if (!gemm_ok(g, up)) return false;
            up.out = base + at_hidden;
            up.out_stride_row = H;
            g = GemmArgs();
            g.offsets_data = offsets;
            g.a_data = up.out;
            g.a_rows = R;
            g.b = w2;
            g.bias = b2;
            g.total_rows = R;
            if (!gemm_ok(g, down)) return false;
            down.out = base + at_rows;
            down.out_stride_row = O;
            merge.code = down.out_dtype;
            merge.g_code = dtype_code(scores.scalar_type());
            merge.out_dtype = merge.code == FMOE_F32 || merge.g_code == FMOE_F32 ? at::kFloat : at::kBFloat16;
            merge.T = T;
            merge.K = merge.cols = merge.sr = k;
            merge.D = merge.value_stride = O;
            merge.value_data = down.out;
            merge.reverse_data = reverse;
            merge.gates_data = gates;
            merge.index_data = gate_index;
            y = allocate(merge, x);
            return true;
        },
        [&] {
            const int code = dtype_code(scores.scalar_type());
            const fmoe_gate g = {x_data, data, gate_bias_data, x.stride(0), code, (int)x.size(1)};
            if (gate && !one_launch) {
                what = "fmoe_gate_softmax";
                if (const int rc = c_gate_softmax(x_data, code, merge.T, g.d, g.x_stride_row, data, gate_bias_data, (int)w1.size(0), gate_scores,
                                                  (void*)stream))
                    return rc;
                what = "fmoe_route_topk";
            }
            if (const int rc = c_route_topk(one_launch ? (const void*)&g : gate ? gate_scores : data, one_launch ? FMOE_SCORES_OF_GATE : code, merge.T,
                                            (int)w1.size(0), (int)k, (int)mode, topk_idx, gates, lengths, offsets, gate_index, token_index,
                                            reverse, base + at_ws, ws_bytes, (void*)stream))
                return rc;
            RECORD_USER_SCOPE("## expert_forward##");
            what = "fmoe_grouped_gemm";
            if (const int rc = gemm(up, x, (void*)stream)) return rc;
            if (const int rc = gemm(down, x, (void*)stream)) return rc;
            what = "fmoe_combine";
            return combine(merge, y, (void*)stream);
        });
    if (raised(status, what)) return nullptr;
    return status == FMOE_OK ? wrap(y) : none();
    END_HANDLE_TH_ERRORS
}

// ---- the backward pass's operators, as ops.py issues them
at::Tensor empty_rows(int64_t rows, int64_t cols, at::ScalarType dtype, const at::Tensor& like) {
    return empty({rows + kSlackRows, cols}, dtype, like).narrow(0, 0, rows);
}
bool float_matrix(const at::Tensor& t) {
    return (t.scalar_type() == at::kFloat || t.scalar_type() == at::kBFloat16) && t.dim() == 2 && t.size(1) > 0 && t.stride(1) == 1;
}
PyObject* wrap_or_none(const at::Tensor& t) { return t.defined() ? wrap(t) : none(); }

// (dy [T, D], value [T*K, D] or None, token_index, K, gates or None, gates_index or None, need_gate_grad, stream) -> (d_value, d_gates)
PyObject* py_combine_bwd(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 8) return none();
    const at::Tensor dy = gpu_tensor(args[0]), index = gpu_tensor(args[2]);
    at::Tensor value, gates, gates_index, d_value, d_gates;
    int64_t K, need, stream;
    if (!dy.defined() || !index.defined() || !optional_tensor(args[1], &value) || !as_int(args[3], &K) || !optional_tensor(args[4], &gates) ||
        !optional_tensor(args[5], &gates_index) || !as_int(args[6], &need) || !as_int(args[7], &stream))
        return none();
    const int status = run(
        [&] {
            if (!float_matrix(dy) || !dy.is_contiguous() || K < 1 || K > INT32_MAX) return false;
            const int64_t R = dy.size(0) * K;
            if (R < 1 || !same_device(dy, index) || !same_device(dy, value) || !same_device(dy, gates) || !same_device(dy, gates_index) ||
                !i64_list(index, R))
                return false;
            if (gates.defined() && (dtype_code(gates.scalar_type()) < 0 || gates.scalar_type() == at::kFloat8_e4m3fn || gates.dim() != 2 ||
                                    gates.numel() != R || (gates_index.defined() && !i64_list(gates_index, R))))
                return false;
            return !need || (value.defined() && float_matrix(value) && value.scalar_type() == dy.scalar_type() && value.size(0) == R &&
                             value.size(1) == dy.size(1));
        },
        [&] {
            const int64_t T = dy.size(0), D = dy.size(1);
            if (need) d_gates = at::zeros({T * K}, at::TensorOptions(dy.device()).dtype(at::kFloat));
            d_value = empty_rows(T * K, D, dy.scalar_type(), dy);
            const bool g = gates.defined();
            return c_combine_bwd(dy.data_ptr(), need ? value.data_ptr() : nullptr, dtype_code(dy.scalar_type()), T, (int)K, D,
                                 need ? value.stride(0) : D, index.data_ptr<int64_t>(), g ? gates.data_ptr() : nullptr,
                                 g ? dtype_code(gates.scalar_type()) : FMOE_F32, g ? gates.size(1) : 1, g ? gates.stride(0) : 1,
                                 g ? gates.stride(1) : 1, g && gates_index.defined() ? gates_index.data_ptr<int64_t>() : nullptr,
                                 d_value.data_ptr(), need ? d_gates.data_ptr<float>() : nullptr, (void*)stream);
        });
    if (raised(status, "fmoe_combine_bwd")) return nullptr;
    return status == FMOE_OK ? Py_BuildValue("(NN)", wrap(d_value), wrap_or_none(d_gates)) : none();
    END_HANDLE_TH_ERRORS
}

// (src [R, C], offsets, stream) -> [E, C]
PyObject* py_segment_colsum(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 3) return none();
    const at::Tensor src = gpu_tensor(args[0]), offsets = gpu_tensor(args[1]);
    at::Tensor out;
    int64_t stream;
    if (!src.defined() || !offsets.defined() || !as_int(args[2], &stream)) return none();
    const int status = run([&] { return float_matrix(src) && same_device(src, offsets) && offsets.numel() >= 2 && i64_list(offsets, offsets.numel()); },
                           [&] {
                               const int64_t E = offsets.numel() - 1;
                               out = empty({E, src.size(1)}, src.scalar_type(), src);
                               return c_segment_colsum(src.data_ptr(), dtype_code(src.scalar_type()), src.size(0), src.size(1), src.stride(0),
                                                       offsets.data_ptr<int64_t>(), (int)E, out.data_ptr(), (void*)stream);
                           });
    if (raised(status, "fmoe_segment_colsum")) return nullptr;
    return status == FMOE_OK ? wrap(out) : none();
    END_HANDLE_TH_ERRORS
}

// (g [R, C], u or None, dh, joint, stream) -> (dg, du)
PyObject* py_swiglu_bwd(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 5) return none();
    const at::Tensor g = gpu_tensor(args[0]), dh = gpu_tensor(args[2]);
    at::Tensor u, dg, du;
    int64_t joint, stream;
    if (!g.defined() || !dh.defined() || !optional_tensor(args[1], &u) || !as_int(args[3], &joint) || !as_int(args[4], &stream)) return none();
    const int status = run(
        [&] {
            for (const at::Tensor* t : {&g, &dh, (const at::Tensor*)&u})
                if (t->defined() && (!float_matrix(*t) || !t->is_contiguous() || t->scalar_type() != g.scalar_type() || t->sizes() != g.sizes() ||
                                     !same_device(g, *t)))
                    return false;
            return g.numel() > 0;
        },
        [&] {
            const int64_t rows = g.size(0), cols = g.size(1);
            int64_t pitch = 0;
            if (joint && u.defined() && g.scalar_type() == at::kBFloat16 && cols % 8 == 0) {
                const at::Tensor both = empty_rows(rows, 2 * cols, g.scalar_type(), g);
                dg = both.narrow(1, 0, cols);
                du = both.narrow(1, cols, cols);
                pitch = 2 * cols;
            } else {
                dg = empty_rows(rows, cols, g.scalar_type(), g);
                if (u.defined()) du = empty_rows(rows, cols, g.scalar_type(), g);
            }
            return c_swiglu_bwd(g.data_ptr(), u.defined() ? u.data_ptr() : nullptr, dh.data_ptr(), dg.data_ptr(),
                                du.defined() ? du.data_ptr() : nullptr, dtype_code(g.scalar_type()), g.numel(), cols, pitch, (void*)stream);
        });
    if (raised(status, "fmoe_swiglu_bwd")) return nullptr;
    return status == FMOE_OK ? Py_BuildValue("(NN)", wrap(dg), wrap_or_none(du)) : none();
    END_HANDLE_TH_ERRORS
}

// (a [R, C], with_slack, stream) -> silu(a)
PyObject* py_silu(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 3) return none();
    const at::Tensor a = gpu_tensor(args[0]);
    at::Tensor out;
    int64_t slack, stream;
    if (!a.defined() || !as_int(args[1], &slack) || !as_int(args[2], &stream)) return none();
    const int status = run([&] { return float_matrix(a) && a.is_contiguous() && a.numel() > 0; },
                           [&] {
                               out = slack ? empty_rows(a.size(0), a.size(1), a.scalar_type(), a) : empty(a.sizes(), a.scalar_type(), a);
                               return c_silu_mul(a.data_ptr(), nullptr, out.data_ptr(), dtype_code(a.scalar_type()), a.numel(), (void*)stream);
                           });
    if (raised(status, "fmoe_silu_mul")) return nullptr;
    return status == FMOE_OK ? wrap(out) : none();
    END_HANDLE_TH_ERRORS
}

// (src [T, C], index, index_div, stream) -> src[index / index_div] with slack rows
PyObject* py_gather_rows(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 4) return none();
    const at::Tensor src = gpu_tensor(args[0]), index = gpu_tensor(args[1]);
    at::Tensor out;
    int64_t div, stream;
    if (!src.defined() || !index.defined() || !as_int(args[2], &div) || !as_int(args[3], &stream)) return none();
    const int status = run([&] { return float_matrix(src) && same_device(src, index) && div >= 1 && div <= INT32_MAX && i64_list(index, index.numel()); },
                           [&] {
                               const int64_t es = src.element_size(), rows = index.numel();
                               out = empty_rows(rows, src.size(1), src.scalar_type(), src);
                               return c_gather_rows(src.data_ptr(), src.size(0), src.size(1) * es, src.stride(0) * es, index.data_ptr<int64_t>(),
                                                    (int)div, rows, out.data_ptr(), out.stride(0) * es, (void*)stream);
                           });
    if (raised(status, "fmoe_gather_rows")) return nullptr;
    return status == FMOE_OK ? wrap(out) : none();
    END_HANDLE_TH_ERRORS
}

// (index [T, K], stream) -> reverse [T, K]
PyObject* py_invert_index(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 2) return none();
    const at::Tensor index = gpu_tensor(args[0]);
    at::Tensor out;
    int64_t stream;
    if (!index.defined() || !as_int(args[1], &stream)) return none();
    const int status = run([&] { return index.dim() == 2 && i64_list(index, index.numel()) && index.size(1) <= INT32_MAX; },
                           [&] {
                               out = empty(index.sizes(), at::kLong, index);
                               return c_invert_index(index.data_ptr<int64_t>(), index.size(0), (int)index.size(1), out.data_ptr<int64_t>(), (void*)stream);
                           });
    if (raised(status, "fmoe_invert_index")) return nullptr;
    return status == FMOE_OK ? wrap(out) : none();
    END_HANDLE_TH_ERRORS
}

// (scores [T, E], topk_idx [T, K], d_gates [T, K], stream) -> d_scores
PyObject* py_gate_l1_bwd(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 4) return none();
    const at::Tensor scores = gpu_tensor(args[0]), topk = gpu_tensor(args[1]), d_gates = gpu_tensor(args[2]);
    at::Tensor out;
    int64_t stream;
    if (!scores.defined() || !topk.defined() || !d_gates.defined() || !as_int(args[3], &stream)) return none();
    const int status = run(
        [&] {
            return float_matrix(scores) && scores.is_contiguous() && d_gates.scalar_type() == scores.scalar_type() && d_gates.is_contiguous() &&
                   topk.dim() == 2 && i64_list(topk, topk.numel()) && d_gates.sizes() == topk.sizes() && topk.size(0) == scores.size(0) &&
                   same_device(scores, topk) && same_device(scores, d_gates) && scores.size(1) <= INT32_MAX && topk.size(1) <= INT32_MAX;
        },
        [&] {
            out = empty(scores.sizes(), scores.scalar_type(), scores);
            return c_gate_l1_bwd(scores.data_ptr(), dtype_code(scores.scalar_type()), scores.size(0), (int)scores.size(1), (int)topk.size(1),
                                 topk.data_ptr<int64_t>(), d_gates.data_ptr(), out.data_ptr(), (void*)stream);
        });
    if (raised(status, "fmoe_gate_l1_bwd")) return nullptr;
    return status == FMOE_OK ? wrap(out) : none();
    END_HANDLE_TH_ERRORS
}

// (dout [R, N], rows [R, K_in], offsets, halves, stream) -> [E, N, K_in], or two [E, N/2, K_in]: the calls fmoe_weight_grad takes
// (ops.jagged_weight_grad; its other route is left to it)
PyObject* py_weight_grad(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 5) return none();
    const at::Tensor a = gpu_tensor(args[0]), b = gpu_tensor(args[1]), offsets = gpu_tensor(args[2]);
    at::Tensor out, out2;
    int64_t halves, stream;
    if (!a.defined() || !b.defined() || !offsets.defined() || !as_int(args[3], &halves) || !as_int(args[4], &stream)) return none();
    const int status = run(
        [&] {
            if (!float_matrix(a) || !float_matrix(b) || a.scalar_type() != b.scalar_type() || a.size(0) != b.size(0) || !same_device(a, b) ||
                !same_device(a, offsets) || offsets.numel() < 2 || !i64_list(offsets, offsets.numel()))
                return false;
            const bool bf16 = a.scalar_type() == at::kBFloat16;
            const int64_t R = a.size(0), N = a.size(1), Kin = b.size(1), E = offsets.numel() - 1, chunk = bf16 ? 8 : 4;
            if (R < 1 || N % chunk || Kin % chunk || a.stride(0) % chunk || b.stride(0) % chunk || a.stride(0) < N || b.stride(0) < Kin ||
                (uintptr_t)a.data_ptr() % 16 || (uintptr_t)b.data_ptr() % 16 || E > INT32_MAX || Kin > INT32_MAX || E * N > INT32_MAX ||
                (halves && N % 64))
                return false;
            return (bf16 && R < 128) || weight_grad_pays(dtype_code(a.scalar_type()), (int)E, (int)N, (int)Kin, R) != 0;
        },
        [&] {
            const int64_t E = offsets.numel() - 1, N = a.size(1), Kin = b.size(1);
            out = empty({E, halves ? N / 2 : N, Kin}, a.scalar_type(), a);
            if (halves) out2 = empty({E, N / 2, Kin}, a.scalar_type(), a);
            return c_weight_grad(a.data_ptr(), b.data_ptr(), dtype_code(a.scalar_type()), (int)E, (int)N, (int)Kin, a.size(0), a.stride(0),
                                 b.stride(0), offsets.data_ptr<int64_t>(), out.data_ptr(), halves ? out2.data_ptr() : nullptr, (void*)stream);
        });
    if (raised(status, "fmoe_weight_grad")) return nullptr;
    if (status != FMOE_OK) return none();
    return halves ? Py_BuildValue("(NN)", wrap(out), wrap(out2)) : wrap(out);
    END_HANDLE_TH_ERRORS
}

// init(addresses of the C entry points, in the order of the pointers above)
PyObject* py_init(PyObject*, PyObject* const* args, Py_ssize_t n) {
    void* const entry[] = {&route_workspace_bytes, &c_route_topk, &c_grouped_gemm, &c_combine, &c_quant_rows, &c_gate_softmax, &gemm_workspace_bytes,
                           &c_grouped_gemm_ws, &c_gemm_plan, &c_combine_bwd, &c_segment_colsum, &c_swiglu_bwd, &c_silu_mul, &c_gather_rows,
                           &c_invert_index, &c_gate_l1_bwd, &c_weight_grad, &weight_grad_pays, &gate_softmax_pays,
                           &gate_route_pays, &last_error};
    constexpr Py_ssize_t count = sizeof(entry) / sizeof(entry[0]);
    if (n != count) {
        PyErr_Format(PyExc_TypeError, "init: %d addresses expected", (int)count);
        return nullptr;
    }
    int64_t v[count];
    for (int i = 0; i < count; ++i)
        if (!as_int(args[i], &v[i])) {
            PyErr_SetString(PyExc_TypeError, "init: addresses are integers");
            return nullptr;
        }
    static_assert(sizeof(c_combine) == sizeof(v[0]), "addresses of functions are 64 bits");
    for (int i = 0; i < count; ++i) std::memcpy(entry[i], &v[i], sizeof(v[i]));     // (each has a type of its own)
    return none();
}

#define FASTCALL(name, fn) {name, (PyCFunction)(void (*)(void))fn, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    FASTCALL("init", py_init),
    FASTCALL("route_topk", py_route_topk),
    FASTCALL("grouped_gemm", py_grouped_gemm<false>),
    FASTCALL("grouped_gemm_n", py_grouped_gemm<true>),
    FASTCALL("combine", py_combine),
    FASTCALL("quant_rows", py_quant_rows),
    FASTCALL("combine_bwd", py_combine_bwd),
    FASTCALL("segment_colsum", py_segment_colsum),
    FASTCALL("swiglu_bwd", py_swiglu_bwd),
    FASTCALL("silu", py_silu),
    FASTCALL("gather_rows", py_gather_rows),
    FASTCALL("invert_index", py_invert_index),
    FASTCALL("gate_l1_bwd", py_gate_l1_bwd),
    FASTCALL("weight_grad", py_weight_grad),
    FASTCALL("gate_softmax", py_gate_softmax),
    FASTCALL("mlp_forward", py_mlp_forward),
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) {
    PyObject* m = PyModule_Create(&module);
    if (m && PyModule_AddStringConstant(m, "torch_version", TORCH_VERSION) != 0) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
