// The autograd nodes of the Python surface in native code: one stage (NCNFunction), a stack of small groups
// (NCNNetFunction), levels of the radix grouping (NCNRadixNetFunction) and one stage behind a table
// (FusedLinearChunkNCNFunction), over the C ABI of libncn_hip.so (include/ncn_hip.h).
//
// A call on small tensors is host time: a node written in Python costs some 20 us forward and 25 to 75 us backward (autograd runs it
// in a thread of its own, whose core has slept), the kernels of a stage as little as 5.  Here a node allocates, checks and
// launches in about 7.  Training passes, Python nodes : these, us: x[1, 256, 32], 8 stages in one node 233 : 130; x[4, 256, 128], 3
// stages of groups of 32 rows 318 : 159; x[16, 1005, 160], 4 stages of groups of 5 rows 418 : 209 (its kernels).
//
// Every entry returns None for a call that it does not take, which the caller then hands to the Python node: wrong or
// unusual arguments (whose errors are raised there), copies that would have to be made, tensor subclasses, dispatch and function
// modes, function transforms, tracing, forward-mode gradients, and stacks large enough to look at the free memory.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <pybind11/pybind11.h>

#include <algorithm>
#include <cstring>

#include "../../include/ncn_hip.h"

#ifndef NCN_TORCH_ID_TEXT
#define NCN_TORCH_ID_TEXT "NCN_TORCH_ID=0000000000000000"
#endif
#ifndef NCN_TORCH_FOR_TEXT
#define NCN_TORCH_FOR_TEXT "NCN_TORCH_FOR=unknown;"
#endif

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// The entry points of the library that the Python side has loaded (bind()).
struct Library {
    decltype(&ncn_check_shape) check_shape;
    decltype(&ncn_kernel_path_scalars) kernel_path_scalars;
    decltype(&ncn_error_string) error_string;
    decltype(&ncn_workspace_bytes) workspace_bytes;
    decltype(&ncn_workspace_bytes_stages) workspace_bytes_stages;
    decltype(&ncn_forward) forward;
    decltype(&ncn_backward) backward;
    decltype(&ncn_forward_indexed) forward_indexed;
    decltype(&ncn_backward_indexed) backward_indexed;
    decltype(&ncn_stack_plan) stack_plan;
    decltype(&ncn_stack_forward) stack_forward;
    decltype(&ncn_stack_backward) stack_backward;
    decltype(&ncn_forward_radix) forward_radix;
    decltype(&ncn_backward_radix) backward_radix;
};
Library lib;
bool bound = false;

constexpr float kM = 0.9f;   // the m of the Python surface (ncn_cuda_module.M_DEFAULT)

void check(int rc, const char* what) {
    TORCH_CHECK(rc == 0, what, " failed: ", lib.error_string(rc), " (code ", rc, ")");
}
bool is_activation(at::ScalarType t) { return t == at::kFloat || t == at::kBFloat16; }
int code_of(at::ScalarType t) { return t == at::kFloat ? NCN_F32 : NCN_BF16; }
int weight_flag(const Tensor& W) { return W.scalar_type() == at::kBFloat16 ? NCN_W_BF16 : 0; }
void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
const float* f32(const Tensor& t) { return static_cast<const float*>(ptr(t)); }
Tensor empty(at::IntArrayRef size, at::ScalarType dtype, const Tensor& like) {
    return at::empty(size, like.options().dtype(dtype).requires_grad(false));
}
Tensor bytes(size_t n, const Tensor& like) { return empty({static_cast<int64_t>(n)}, at::kByte, like); }
bool aligned(const Tensor& t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15u) == 0; }
// what a gradient that arrives has to be for the library: contiguous and aligned, copied where it is not
Tensor prepared(const Tensor& t) {
    if (!t.defined()) return t;
    Tensor c = t.detach().contiguous();
    return aligned(c) ? c : c.clone(at::MemoryFormat::Contiguous);
}

// ---- what reaches a backward -------------------------------------------------------------------------------------
// Saved tensors come back from the caller's hooks, from anywhere and as anything, and a saved table or length is the caller's own
// tensor: what a kernel could not read, or would read past the end of, is refused with the errors of the Python nodes.
void on_device(const Tensor& t, const Tensor& like, const char* what) {
    TORCH_CHECK(t.is_cuda() && t.device() == like.device(), "all tensors must live on one GPU: ", what, " is on ", t.device(),
                ", the gradients on ", like.device());
}
Tensor returned(const Tensor& t, at::IntArrayRef sizes, const Tensor& like, const char* what) {
    on_device(t, like, what);
    TORCH_CHECK_VALUE(t.sizes().equals(sizes), what, " came back as ", t.sizes(), ", not as ", sizes);
    TORCH_CHECK_TYPE(is_activation(t.scalar_type()), what, " must be float32 or bfloat16, came back as ", t.scalar_type());
    return prepared(t);
}
// saved outputs of a call: [batch, N, E] of either type, or two bfloat16 planes of that
Tensor returned_output(const Tensor& t, at::IntArrayRef sizes, const Tensor& like, const char* what) {
    if (t.dim() != 4) return returned(t, sizes, like, what);
    TORCH_CHECK_TYPE(t.scalar_type() == at::kBFloat16, what, ": two planes must be bfloat16, came back as ", t.scalar_type());
    return returned(t, {2, sizes[0], sizes[1], sizes[2]}, like, what);
}
Tensor returned_weights(const Tensor& t, int64_t numel, const Tensor& like) {
    on_device(t, like, "W");
    TORCH_CHECK_VALUE(t.numel() == numel, "W must hold ", numel, " values, came back with ", t.numel());
    TORCH_CHECK_TYPE(is_activation(t.scalar_type()), "W must be float32 or bfloat16, came back as ", t.scalar_type());
    return prepared(t);
}
Tensor current_index(const Tensor& t, int64_t numel, const Tensor& like, const char* what) {
    if (!t.defined()) return t;
    on_device(t, like, what);
    TORCH_CHECK_VALUE(t.numel() == numel, what, " must hold ", numel, " values, now holds ", t.numel());
    TORCH_CHECK_TYPE(t.scalar_type() == at::kInt || t.scalar_type() == at::kLong, what, " must be int32 or int64, now is ", t.scalar_type());
    return prepared(t.to(at::kInt));
}

// ---- what a call is ---------------------------------------------------------------------------------------------
struct Call {
    ncn_shape shape;
    float alpha;
    int activation, first, count;   // stages (or radix levels) first .. first + count - 1
};

// Nothing between the caller and the kernels that a node in Python would have met.
bool plain_context() {
    using c10::DispatchKey;
    const c10::DispatchKeySet watched({DispatchKey::Python, DispatchKey::PythonTLSSnapshot, DispatchKey::Functionalize,
                                       DispatchKey::FuncTorchDynamicLayerFrontMode, DispatchKey::FuncTorchDynamicLayerBackMode,
                                       DispatchKey::FuncTorchBatched, DispatchKey::FuncTorchGradWrapper, DispatchKey::Tracer});
    return bound && !c10::impl::tls_local_dispatch_key_set().included_.has_any(watched) &&
           !c10::impl::TorchDispatchModeTLS::any_modes_set() && at::impl::PythonTorchFunctionTLS::stack_len() == 0 &&
           !torch::jit::tracer::isTracing();
}

// A tensor the library can read where it lies: a plain torch.Tensor or Parameter on the GPU, contiguous and aligned.
bool usable(PyObject* o, Tensor& out) {
    using c10::DispatchKey;
    if (!THPVariable_CheckExact(o)) return false;
    const Tensor& t = THPVariable_Unpack(o);
    const c10::DispatchKeySet odd({DispatchKey::Python, DispatchKey::Negative, DispatchKey::Conjugate, DispatchKey::ZeroTensor,
                                   DispatchKey::Functionalize, DispatchKey::FuncTorchBatched, DispatchKey::FuncTorchGradWrapper});
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || t.key_set().has_any(odd) || !t.is_contiguous() ||
        t.numel() == 0 || !aligned(t) || t._fw_grad(0).defined())
        return false;
    out = t;
    return true;
}

bool to_int(PyObject* o, int& out) {
    if (!PyLong_CheckExact(o)) return false;
    int overflow = 0;
    const long v = PyLong_AsLongAndOverflow(o, &overflow);
    if (overflow || v < INT32_MIN || v > INT32_MAX) return false;
    out = static_cast<int>(v);
    return true;
}
bool to_int64(PyObject* o, int64_t& out) {
    if (!PyLong_CheckExact(o)) return false;
    int overflow = 0;
    out = PyLong_AsLongLongAndOverflow(o, &overflow);
    return overflow == 0;
}
bool to_alpha(PyObject* o, float& out) {
    if (PyFloat_CheckExact(o)) {
        out = static_cast<float>(PyFloat_AS_DOUBLE(o));
        return true;
    }
    int i;
    if (!to_int(o, i)) return false;
    out = static_cast<float>(i);
    return true;
}

// x, xa [batch, N, E] of one type on one device, and scalars that the library takes.  `check_first`: the stage number that
// ncn_check_shape looks at.
bool read_call(PyObject* x_, PyObject* xa_, PyObject* alpha, PyObject* act, PyObject* n_cache, PyObject* n_head, PyObject* first,
               int64_t count, bool stages, Tensor& x, Tensor& xa, Call& c) {
    int nc, heads;
    if (!usable(x_, x) || !usable(xa_, xa) || x.dim() != 3 || !xa.sizes().equals(x.sizes()) || !is_activation(x.scalar_type()) ||
        xa.scalar_type() != x.scalar_type() || xa.device() != x.device())
        return false;
    if (!to_alpha(alpha, c.alpha) || !to_int(act, c.activation) || !to_int(n_cache, nc) || !to_int(n_head, heads) ||
        !to_int(first, c.first) || count < 1 || count > 1024)
        return false;
    c.count = static_cast<int>(count);
    c.shape = ncn_shape{x.size(0), x.size(1), x.size(2), heads, nc};
    return lib.check_shape(&c.shape, stages ? c.first : 0, c.count, c.activation) == NCN_OK &&
           lib.kernel_path_scalars(&c.shape, c.alpha, kM) != 0;
}
bool weight_of(PyObject* o, const Tensor& x, Tensor& W) {
    return usable(o, W) && is_activation(W.scalar_type()) && W.device() == x.device() && W.numel() == 2 * x.size(2);
}
bool wants_gradients(at::TensorList ts) {
    if (!at::GradMode::is_enabled()) return false;
    for (const Tensor& t : ts)
        if (t.requires_grad()) return true;
    return false;
}

PyObject* pair_of(const Tensor& a, const Tensor& b) {
    PyObject* t = PyTuple_New(2);
    if (!t) return nullptr;
    PyTuple_SET_ITEM(t, 0, THPVariable_Wrap(a));
    PyTuple_SET_ITEM(t, 1, THPVariable_Wrap(b));
    return t;
}

// the arguments of a call inside an autograd context (whose saved values are tensors, numbers and lists)
void keep(AutogradContext* ctx, const Call& c) {
    ctx->saved_data["call"] = std::vector<int64_t>{c.shape.batch, c.shape.N, c.shape.E, c.shape.n_head, c.shape.n_cache,
                                                   c.activation, c.first, c.count};
    ctx->saved_data["alpha"] = static_cast<double>(c.alpha);
}
Call kept(AutogradContext* ctx) {
    const std::vector<int64_t> v = ctx->saved_data["call"].toIntVector();
    return Call{ncn_shape{v[0], v[1], v[2], static_cast<int32_t>(v[3]), static_cast<int32_t>(v[4])},
                static_cast<float>(ctx->saved_data["alpha"].toDouble()), static_cast<int>(v[5]), static_cast<int>(v[6]),
                static_cast<int>(v[7])};
}
// dy, dya as they arrive: missing ones stay missing but for a missing dy, which is zeros; false: there is nothing to do
bool gradients(const variable_list& grads, const Call& c, Tensor& dy, Tensor& dya) {
    const Tensor& first = grads[0].defined() ? grads[0] : grads[1];
    if (!first.defined()) return false;
    const int64_t sizes[] = {c.shape.batch, c.shape.N, c.shape.E};
    if (grads[0].defined()) dy = returned(grads[0], sizes, first, "dy");
    if (grads[1].defined()) dya = returned(grads[1], sizes, first, "dya");
    if (!dy.defined()) dy = at::zeros_like(dya);
    TORCH_CHECK_TYPE(!dya.defined() || dya.scalar_type() == dy.scalar_type(), "dy and dya must both be float32 or bfloat16");
    return true;
}

// ---- one stage, with or without a table and context lengths -----------------------------------------------------
struct Grouping {
    Tensor table, lengths;   // int32, or undefined
    bool indexed() const { return table.defined() || lengths.defined(); }
    const int32_t* table_ptr() const { return static_cast<const int32_t*>(ptr(table)); }
    const int32_t* lengths_ptr() const { return static_cast<const int32_t*>(ptr(lengths)); }
};

struct StageOutputs {
    Tensor y, ya, saved_y, saved_ya;
};
// `saving`: with what a backward needs.  float32: the outputs themselves; bfloat16: also what their rounding took away, as a
// second plane on the register kernels, as float32 copies on the others.
StageOutputs run_stage(const Call& c, const Grouping& g, const Tensor& x, const Tensor& xa, const Tensor& W, bool saving) {
    const c10::DeviceGuard guard(x.device());
    const at::ScalarType dtype = x.scalar_type();
    StageOutputs o;
    Tensor copy, copy_a;
    int out_code = code_of(dtype);
    if (saving && dtype == at::kBFloat16 && lib.kernel_path_scalars(&c.shape, c.alpha, kM) == 2) {
        out_code = NCN_BF16X2;
        o.saved_y = empty({2, x.size(0), x.size(1), x.size(2)}, dtype, x);
        o.saved_ya = empty({2, x.size(0), x.size(1), x.size(2)}, dtype, x);
        o.y = o.saved_y.select(0, 0);
        o.ya = o.saved_ya.select(0, 0);
    } else {
        o.y = empty(x.sizes(), dtype, x);
        o.ya = empty(x.sizes(), dtype, x);
        if (saving && dtype == at::kBFloat16) {
            o.saved_y = copy = empty(x.sizes(), at::kFloat, x);
            o.saved_ya = copy_a = empty(x.sizes(), at::kFloat, x);
        } else {
            o.saved_y = o.y;
            o.saved_ya = o.ya;
        }
    }
    const int in_code = code_of(dtype) | weight_flag(W);
    float *const c32 = static_cast<float*>(ptr(copy)), *const ca32 = static_cast<float*>(ptr(copy_a));
    if (g.indexed())
        check(lib.forward_indexed(ptr(x), ptr(xa), in_code, ptr(o.y), ptr(o.ya), out_code, c32, ca32, f32(W), g.table_ptr(),
                                  g.lengths_ptr(), &c.shape, c.first, 1, c.alpha, kM, c.activation, stream_of(x)),
              "ncn_forward_indexed");
    else
        check(lib.forward(ptr(x), ptr(xa), in_code, ptr(o.y), ptr(o.ya), out_code, c32, ca32, f32(W), nullptr, 0, &c.shape,
                          c.first, 1, c.alpha, kM, c.activation, stream_of(x)),
              "ncn_forward");
    return o;
}

struct StageNode : torch::autograd::Function<StageNode> {
    static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& xa, const Tensor& W, const Call& c,
                                 const Grouping& g) {
        const StageOutputs o = run_stage(c, g, x, xa, W, true);
        ctx->save_for_backward({o.saved_y, o.saved_ya, W});
        // an output nobody differentiates arrives undefined instead of as zeros to fill and to read
        ctx->set_materialize_grads(false);
        keep(ctx, c);
        ctx->saved_data["bf16"] = x.scalar_type() == at::kBFloat16;
        if (g.table.defined()) ctx->saved_data["table"] = g.table;
        if (g.lengths.defined()) ctx->saved_data["lengths"] = g.lengths;
        return {o.y, o.ya};
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        Tensor dy, dya;
        const Call c = kept(ctx);
        if (!gradients(grads, c, dy, dya)) return variable_list(5);
        const variable_list saved = ctx->get_saved_variables();
        const Tensor y = returned_output(saved[0], dy.sizes(), dy, "y"), ya = returned_output(saved[1], dy.sizes(), dy, "ya");
        TORCH_CHECK_TYPE(y.sizes().equals(ya.sizes()) && y.scalar_type() == ya.scalar_type(), "y and ya came back as different kinds");
        const Tensor W = returned_weights(saved[2], 2 * c.shape.E, dy);
        Grouping g;
        if (ctx->saved_data.count("table")) g.table = current_index(ctx->saved_data["table"].toTensor(), c.shape.N, dy, "group_index");
        if (ctx->saved_data.count("lengths")) g.lengths = current_index(ctx->saved_data["lengths"].toTensor(), c.shape.batch, dy, "ctx_len");
        const c10::DeviceGuard guard(dy.device());
        const at::ScalarType dtype = ctx->saved_data["bf16"].toBool() ? at::kBFloat16 : at::kFloat;
        const Tensor dx = empty(dy.sizes(), dtype, dy), dxa = empty(dy.sizes(), dtype, dy);
        const Tensor dW = empty({2 * c.shape.E}, W.scalar_type(), dy);
        const int y_code = (y.dim() == 4 ? NCN_BF16X2 : code_of(y.scalar_type())) | weight_flag(W);
        const size_t ws_bytes = g.table.defined() ? lib.workspace_bytes(&c.shape)
                                                  : lib.workspace_bytes_stages(&c.shape, c.first, 1, c.activation, 2);
        const Tensor ws = bytes(ws_bytes, dy);
        float* const dw = static_cast<float*>(ptr(dW));
        if (g.indexed())
            check(lib.backward_indexed(ptr(y), ptr(ya), y_code, ptr(dy), ptr(dya), code_of(dy.scalar_type()), ptr(dx), ptr(dxa),
                                       code_of(dtype), nullptr, nullptr, f32(W), dw, ptr(ws), ws_bytes, g.table_ptr(),
                                       g.lengths_ptr(), &c.shape, c.first, 1, c.alpha, kM, c.activation, stream_of(dy)),
                  "ncn_backward_indexed");
        else
            check(lib.backward(ptr(y), ptr(ya), y_code, ptr(dy), ptr(dya), code_of(dy.scalar_type()), ptr(dx), ptr(dxa),
                               code_of(dtype), nullptr, nullptr, f32(W), dw, ptr(ws), ws_bytes, &c.shape, c.first, 1, c.alpha,
                               kM, c.activation, stream_of(dy)),
                  "ncn_backward");
        return {dx, dxa, dW.reshape(W.sizes()), Tensor(), Tensor()};
    }
};

PyObject* run_stage_call(const Call& c, const Grouping& g, const Tensor& x, const Tensor& xa, const Tensor& W) {
    variable_list out;
    {
        const pybind11::gil_scoped_release no_gil;
        if (wants_gradients({x, xa, W})) {
            out = StageNode::apply(x, xa, W, c, g);
        } else {   // nothing is kept: one plane of bfloat16 outputs, half the memory
            const at::NoGradGuard no_grad;
            const StageOutputs o = run_stage(c, g, x, xa, W, false);
            out = {o.y, o.ya};
        }
    }
    return pair_of(out[0], out[1]);
}

// stage(x, xa, W, alpha, activation, n_cache, n_head, module_l) -> (y, ya) or None
PyObject* stage(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Tensor x, xa, W;
    Call c;
    if (n != 8 || !plain_context() || !read_call(a[0], a[1], a[3], a[4], a[5], a[6], a[7], 1, true, x, xa, c) ||
        !weight_of(a[2], x, W))
        Py_RETURN_NONE;
    return run_stage_call(c, Grouping{}, x, xa, W);
    END_HANDLE_TH_ERRORS
}

// table_stage(x, xa, W, table, lengths, alpha, activation, n_cache, n_head) -> (y, ya) or None.  The caller has found the table to
// be a permutation; table and lengths: int32 on the device, or (lengths) None.
PyObject* table_stage(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Tensor x, xa, W;
    Grouping g;
    Call c;
    PyObject* const zero = PyLong_FromLong(0);
    const bool ok = n == 9 && plain_context() && read_call(a[0], a[1], a[5], a[6], a[7], a[8], zero, 1, true, x, xa, c) &&
                    weight_of(a[2], x, W);
    Py_DECREF(zero);
    if (!ok || !THPVariable_CheckExact(a[3]) || !usable(a[3], g.table) || g.table.scalar_type() != at::kInt ||
        g.table.device() != x.device() || g.table.numel() != x.size(1))
        Py_RETURN_NONE;
    if (a[4] != Py_None && (!usable(a[4], g.lengths) || g.lengths.scalar_type() != at::kInt || g.lengths.device() != x.device() ||
                            g.lengths.numel() != x.size(0)))
        Py_RETURN_NONE;
    return run_stage_call(c, g, x, xa, W);
    END_HANDLE_TH_ERRORS
}

// ---- stacks: weights as one [stages, 2E] copy, as the Python nodes keep them -------------------------------------
bool weights_of(PyObject* list, const Tensor& x, std::vector<Tensor>& Ws) {
    if (!PyList_CheckExact(list)) return false;
    const Py_ssize_t L = PyList_GET_SIZE(list);
    Ws.resize(L);
    for (Py_ssize_t k = 0; k < L; ++k)
        if (!weight_of(PyList_GET_ITEM(list, k), x, Ws[k]) || Ws[k].scalar_type() != Ws[0].scalar_type()) return false;
    return true;
}
Tensor stacked(at::TensorList Ws) {
    std::vector<Tensor> flat;
    flat.reserve(Ws.size());
    for (const Tensor& w : Ws) flat.push_back(w.dim() == 1 ? w : w.reshape(-1));
    return at::stack(flat);
}
// gradients of (x, xa, <others>, weights ..): `lead` entries before those of the weights, all but the first two empty
variable_list stack_gradients(const Tensor& dx, const Tensor& dxa, size_t lead, const Tensor& dW, const c10::IValue& sizes,
                              at::ScalarType w_dtype) {
    variable_list out(lead);
    out[0] = dx;
    out[1] = dxa;
    const std::vector<Tensor> rows = dW.unbind(0);
    const auto list = sizes.toList();
    for (size_t k = 0; k < rows.size(); ++k) {
        const std::vector<int64_t> s = list.get(k).toIntVector();
        const Tensor& r = rows[k];
        out.push_back((r.sizes().equals(s) ? r : r.reshape(s)).to(w_dtype));
    }
    return out;
}
c10::IValue sizes_value(at::TensorList Ws) {
    c10::List<c10::List<int64_t>> l;
    for (const Tensor& w : Ws) l.push_back(c10::List<int64_t>(w.sizes()));
    return c10::IValue(l);
}

struct StackPlan {
    int max_range, max_saves, ranges;
    int64_t forward_bytes, backward_bytes;
};

struct StackNode : torch::autograd::Function<StackNode> {
    static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& xa, const Call& c, const StackPlan& p,
                                 at::TensorList Ws) {
        const c10::DeviceGuard guard(x.device());
        const at::ScalarType dtype = x.scalar_type();
        const bool is_f32 = dtype == at::kFloat;
        const Tensor W = stacked(Ws);
        const Tensor y = empty(x.sizes(), dtype, x), ya = empty(x.sizes(), dtype, x);
        const int64_t n_saves = p.ranges - (is_f32 ? 1 : 0);
        Tensor saves, ws;
        if (n_saves) saves = empty({n_saves, 2, x.size(0), x.size(1), x.size(2)}, at::kFloat, x);
        if (p.forward_bytes) ws = bytes(p.forward_bytes, x);
        check(lib.stack_forward(ptr(x), ptr(xa), code_of(dtype) | weight_flag(W), ptr(y), ptr(ya), code_of(dtype),
                                static_cast<float*>(ptr(saves)), ptr(W), ptr(ws), p.forward_bytes, &c.shape, c.first, c.count,
                                p.max_range, p.max_saves, c.alpha, kM, c.activation, stream_of(x)),
              "ncn_stack_forward");
        ctx->set_materialize_grads(false);
        ctx->save_for_backward({W, saves, is_f32 ? y : Tensor(), is_f32 ? ya : Tensor()});
        keep(ctx, c);
        ctx->saved_data["plan"] = std::vector<int64_t>{p.max_range, p.max_saves, p.backward_bytes, is_f32, n_saves};
        ctx->saved_data["sizes"] = sizes_value(Ws);
        return {y, ya};
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        Tensor dy, dya;
        const Call c = kept(ctx);
        if (!gradients(grads, c, dy, dya)) return variable_list(4 + c.count);
        const variable_list saved = ctx->get_saved_variables();
        const std::vector<int64_t> p = ctx->saved_data["plan"].toIntVector();
        // (other types than the library's are read as float32, as the Python node does)
        const Tensor W = returned_weights(is_activation(saved[0].scalar_type()) ? saved[0] : saved[0].to(at::kFloat), 2 * c.shape.E * c.count, dy);
        Tensor saves, y, ya;
        if (p[4]) saves = returned(saved[1], {p[4], 2, dy.size(0), dy.size(1), dy.size(2)}, dy, "a kept activation");
        if (p[3]) {
            y = returned(saved[2], dy.sizes(), dy, "y");
            ya = returned(saved[3], dy.sizes(), dy, "ya");
        }
        for (const Tensor& t : {saves, y, ya})
            TORCH_CHECK_TYPE(!t.defined() || t.scalar_type() == at::kFloat, "a stack keeps float32, which came back as ", t.scalar_type());
        const c10::DeviceGuard guard(dy.device());
        const at::ScalarType dtype = p[3] ? at::kFloat : at::kBFloat16;
        const Tensor dx = empty(dy.sizes(), dtype, dy), dxa = empty(dy.sizes(), dtype, dy);
        const Tensor dW = empty({c.count, 2 * c.shape.E}, W.scalar_type(), dy), ws = bytes(p[2], dy);
        check(lib.stack_backward(f32(y), f32(ya), f32(saves), ptr(dy), ptr(dya), code_of(dy.scalar_type()), ptr(dx), ptr(dxa),
                                 code_of(dtype), ptr(W), ptr(dW), weight_flag(W), ptr(ws), p[2], &c.shape, c.first, c.count,
                                 static_cast<int>(p[0]), static_cast<int>(p[1]), c.alpha, kM, c.activation, stream_of(dy)),
              "ncn_stack_backward");
        return stack_gradients(dx, dxa, 4, dW, ctx->saved_data["sizes"], W.scalar_type());
    }
};

// stack(x, xa, weights, alpha, activation, n_cache, n_head, first_stage, max_range, budget, look) -> (y, ya) or None: a stack that is
// trained (ncn_cuda_module.stack_forward); `look`: saved bytes from which on the free memory has to be looked at.
PyObject* stack(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Tensor x, xa;
    std::vector<Tensor> Ws;
    Call c;
    StackPlan p;
    int64_t budget, look;
    if (n != 11 || !plain_context() || !PyList_CheckExact(a[2]) || PyList_GET_SIZE(a[2]) < 2 ||
        !read_call(a[0], a[1], a[3], a[4], a[5], a[6], a[7], PyList_GET_SIZE(a[2]), true, x, xa, c) || !weights_of(a[2], x, Ws) ||
        !to_int(a[8], p.max_range) || !to_int64(a[9], budget) || !to_int64(a[10], look) || p.max_range < 1)
        Py_RETURN_NONE;
    const int64_t pair = 8 * x.numel(), fewest = (c.count + p.max_range - 1) / p.max_range;
    if (std::min(budget, pair * c.count) > look || !(wants_gradients({x, xa}) || wants_gradients(Ws))) Py_RETURN_NONE;
    p.max_saves = static_cast<int>(std::min<int64_t>(std::max(budget / pair, fewest), c.count));
    int64_t out[2];
    p.ranges = lib.stack_plan(&c.shape, c.first, c.count, c.alpha, kM, c.activation, p.max_range, p.max_saves,
                              code_of(x.scalar_type()), out);
    if (p.ranges <= 0) Py_RETURN_NONE;
    p.forward_bytes = out[0];
    p.backward_bytes = out[1];
    variable_list y;
    try {
        const pybind11::gil_scoped_release no_gil;
        y = StackNode::apply(x, xa, c, p, at::TensorList(Ws));
    } catch (const c10::OutOfMemoryError&) {   // the Python node tries again with fewer activations kept
        Py_RETURN_NONE;
    }
    return pair_of(y[0], y[1]);
    END_HANDLE_TH_ERRORS
}

// ---- radix levels ------------------------------------------------------------------------------------------------
struct RadixNode : torch::autograd::Function<RadixNode> {
    static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& xa, const Call& c, at::TensorList Ws) {
        const c10::DeviceGuard guard(x.device());
        const Tensor W = stacked(Ws).to(at::kFloat);
        const Tensor y = empty(x.sizes(), at::kFloat, x), ya = empty(x.sizes(), at::kFloat, x);
        check(lib.forward_radix(ptr(x), ptr(xa), code_of(x.scalar_type()), ptr(y), ptr(ya), NCN_F32, nullptr, nullptr, f32(W),
                                &c.shape, c.first, c.count, c.alpha, kM, c.activation, stream_of(x)),
              "ncn_forward_radix");
        ctx->set_materialize_grads(false);
        ctx->save_for_backward({W, y, ya});
        keep(ctx, c);
        ctx->saved_data["bf16"] = x.scalar_type() == at::kBFloat16;
        ctx->saved_data["w_bf16"] = Ws[0].scalar_type() == at::kBFloat16;
        ctx->saved_data["sizes"] = sizes_value(Ws);
        return {y.to(x.scalar_type()), ya.to(x.scalar_type())};
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        Tensor dy, dya;
        const Call c = kept(ctx);
        if (!gradients(grads, c, dy, dya)) return variable_list(3 + c.count);
        const variable_list saved = ctx->get_saved_variables();
        const Tensor W = prepared(returned_weights(saved[0], 2 * c.shape.E * c.count, dy).to(at::kFloat));
        const Tensor y = returned(saved[1], dy.sizes(), dy, "y"), ya = returned(saved[2], dy.sizes(), dy, "ya");
        TORCH_CHECK_TYPE(y.scalar_type() == ya.scalar_type(), "y and ya came back as different types");
        const c10::DeviceGuard guard(dy.device());
        const Tensor dx = empty(dy.sizes(), at::kFloat, dy), dxa = empty(dy.sizes(), at::kFloat, dy);
        const Tensor dW = empty({c.count, 2 * c.shape.E}, at::kFloat, dy);
        // two float32 arrays (padded to 256 bytes) carry the state between the passes
        const size_t ws_bytes = lib.workspace_bytes(&c.shape) +
                                (c.count > 1 ? 2 * ((static_cast<size_t>(dy.numel()) * 4 + 255) / 256 * 256) : 0);
        const Tensor ws = bytes(ws_bytes, dy);
        check(lib.backward_radix(ptr(y), ptr(ya), code_of(y.scalar_type()), ptr(dy), ptr(dya), code_of(dy.scalar_type()), ptr(dx), ptr(dxa),
                                 NCN_F32, nullptr, nullptr, f32(W), static_cast<float*>(ptr(dW)), ptr(ws), ws_bytes, &c.shape,
                                 c.first, c.count, c.alpha, kM, c.activation, stream_of(dy)),
              "ncn_backward_radix");
        const at::ScalarType dtype = ctx->saved_data["bf16"].toBool() ? at::kBFloat16 : at::kFloat;
        return stack_gradients(dx.to(dtype), dxa.to(dtype), 3, dW, ctx->saved_data["sizes"],
                               ctx->saved_data["w_bf16"].toBool() ? at::kBFloat16 : at::kFloat);
    }
};

// radix(x, xa, weights, alpha, activation, n_cache, n_head, first_level) -> (y, ya) or None: all levels reversed from the outputs
PyObject* radix(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Tensor x, xa;
    std::vector<Tensor> Ws;
    Call c;
    if (n != 8 || !plain_context() || !PyList_CheckExact(a[2]) || PyList_GET_SIZE(a[2]) < 1 ||
        !read_call(a[0], a[1], a[3], a[4], a[5], a[6], a[7], PyList_GET_SIZE(a[2]), false, x, xa, c) || !weights_of(a[2], x, Ws) ||
        c.first < 0)
        Py_RETURN_NONE;
    int64_t span = 1;
    for (int k = 0; k < c.first + c.count; ++k) {
        span *= c.shape.n_cache;
        if (span > c.shape.N) Py_RETURN_NONE;
        if (c.shape.n_cache == 1 && k > 64) break;
    }
    if (c.shape.N % span != 0) Py_RETURN_NONE;
    variable_list y;
    {
        const pybind11::gil_scoped_release no_gil;
        y = RadixNode::apply(x, xa, c, at::TensorList(Ws));
    }
    return pair_of(y[0], y[1]);
    END_HANDLE_TH_ERRORS
}

// bind(addresses): the entry points of the loaded library, in the order of `Library`
PyObject* bind(PyObject*, PyObject* arg) {
    constexpr Py_ssize_t kEntries = sizeof(Library) / sizeof(void*);
    if (!PyTuple_CheckExact(arg) || PyTuple_GET_SIZE(arg) != kEntries) {
        PyErr_Format(PyExc_TypeError, "bind() takes a tuple of %d addresses", (int)kEntries);
        return nullptr;
    }
    void* entry[kEntries];
    for (Py_ssize_t k = 0; k < kEntries; ++k) {
        entry[k] = PyLong_AsVoidPtr(PyTuple_GET_ITEM(arg, k));
        if (!entry[k]) {
            if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "bind(): null address");
            return nullptr;
        }
    }
    std::memcpy(&lib, entry, sizeof lib);
    bound = true;
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", bind, METH_O, "addresses of the library's entry points"},
    {"stage", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(stage)), METH_FASTCALL, "one stage"},
    {"table_stage", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(table_stage)), METH_FASTCALL, "one stage behind a table"},
    {"stack", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(stack)), METH_FASTCALL, "a trained stack"},
    {"radix", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(radix)), METH_FASTCALL, "radix levels"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_ncn_torch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

extern "C" __attribute__((visibility("default"))) const char* ncn_torch_id() { return NCN_TORCH_ID_TEXT; }
extern "C" __attribute__((visibility("default"))) const char* ncn_torch_for() { return NCN_TORCH_FOR_TEXT; }

PyMODINIT_FUNC PyInit__ncn_torch() { return PyModule_Create(&module); }
