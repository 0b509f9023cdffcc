// Host side of the layers' calls as one native module (`_host`): operand checks, output and workspace allocation, the
// launches through the C ABI, and the autograd nodes.  What it replaces is Python that runs between the launches: a
// ctypes call with twenty converted arguments per launch group, a Python autograd function per projection (its backward
// takes the interpreter lock on the engine's thread), and a dozen tensor methods per check.  At the sizes of one short
// sequence that was most of a step's time.
//
// Every entry returns None when an operand is not what the kernels take, and while a call is being traced or carries
// forward-mode tangents (neither sees launches made here); the Python caller then runs its own checks, which name what is
// wrong (one place for the error texts), or takes its general path.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>

#include "../../include/ggml_mmq_gfx950.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// ------------------------------------------------------------------------------------------------
struct ReleaseGil {
    PyThreadState* state = PyEval_SaveThread();
    ~ReleaseGil() { PyEval_RestoreThread(state); }
};

void check(int rc) {
    if (rc == 0) return;
    if (rc == -3 || rc == -5 || rc == -6) TORCH_CHECK(false, "ggml_mmq_gfx950 error ", rc, ": ", ggq_last_error());
    TORCH_CHECK_VALUE(false, "ggml_mmq_gfx950 error ", rc, ": ", ggq_last_error());
}

Tensor empty(at::IntArrayRef shape, at::ScalarType type, const Tensor& like) { return at::detail::empty_cuda(shape, type, like.device(), std::nullopt); }
Tensor empty_bytes(int64_t n, const Tensor& like) { return empty({n}, at::kByte, like); }
void* stream_of(const Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
int rank_pad(int64_t r) { return (int)(r + 15) / 16 * 16; }

// What a kernel takes as it is: on the device, of the type, dense, 16-byte aligned.
bool usable(const Tensor& t, at::ScalarType type) {
    return t.defined() && t.is_cuda() && t.scalar_type() == type && t.is_contiguous() && ((uintptr_t)t.data_ptr() & 15) == 0;
}

// A cotangent as the kernels take it: autograd may hand over expanded or strided tensors.
Tensor usable_cotangent(const Tensor& g, const char* what) {
    TORCH_CHECK_TYPE(g.scalar_type() == at::kBFloat16, what, " must have dtype torch.bfloat16, got ", g.scalar_type());
    Tensor c = g.contiguous();
    return ((uintptr_t)c.data_ptr() & 15) ? c.clone() : c;
}

void refuse_higher_order(const char* what) { TORCH_CHECK(!at::GradMode::is_enabled(), what, " does not support higher-order gradients"); }

// Tracing records Python autograd functions, and forward mode has them refuse: those calls are left to the general path.
bool traced_or_forward_mode(std::initializer_list<const Tensor*> ts) {
    if (c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::Tracer)) return true;
    for (const Tensor* t : ts)
        if (t->defined() && t->_fw_grad(0).defined()) return true;
    return false;
}

bool any_requires_grad(std::initializer_list<const Tensor*> ts) {
    if (!at::GradMode::is_enabled()) return false;
    for (const Tensor* t : ts)
        if (t->defined() && t->requires_grad()) return true;
    return false;
}

// ------------------------------------------------------------------------------------------------
// Dense linear over a packed weight, with or without the LoRA term: y [..., n], and x A^T when LoRA is on.
Tensor linear_forward(const Tensor& x, const Tensor& payload, const Tensor& a, const Tensor& b, int64_t qt, int64_t n, double scaling, Tensor* xa_out) {
    const int64_t k = x.size(-1), m = k ? x.numel() / k : 0;
    c10::SmallVector<int64_t, 5> shape(x.sizes().begin(), x.sizes().end());
    shape.back() = n;
    Tensor y = empty(shape, at::kBFloat16, x);
    if (!a.defined()) {
        if (m) {
            Tensor ws = empty_bytes(ggq_lora_workspace_bytes(m, 0, 1, n, k, 0), x);
            check(ggq_lora_mmq_forward(x.data_ptr(), payload.data_ptr(), (int)qt, m, n, k, nullptr, nullptr, 0, 0.f, nullptr, y.data_ptr(), ws.data_ptr(), ws.numel(), stream_of(x)));
        }
        return y;
    }
    const int64_t r = a.size(0);
    Tensor xa = empty({m, rank_pad(r)}, at::kBFloat16, x);
    if (m) {
        Tensor ws = empty_bytes(ggq_lora_workspace_bytes(m, 0, 1, n, k, (int)r), x);
        check(ggq_lora_mmq_forward(x.data_ptr(), payload.data_ptr(), (int)qt, m, n, k, a.data_ptr(), b.data_ptr(), (int)r, (float)scaling, xa.data_ptr(),
                                   y.data_ptr(), ws.data_ptr(), ws.numel(), stream_of(x)));
    }
    if (xa_out) *xa_out = xa;
    return y;
}

// (An autograd node takes an absent tensor as an empty optional, not as an undefined tensor.)
using Maybe = std::optional<Tensor>;
Maybe maybe(const Tensor& t) { return t.defined() ? Maybe(t) : Maybe(); }

struct Linear : torch::autograd::Function<Linear> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& payload, const Maybe& a_in, const Maybe& b_in, int64_t qt, int64_t n, double scaling) {
        const Tensor a = a_in.value_or(Tensor()), b = b_in.value_or(Tensor());
        Tensor xa;
        Tensor y = linear_forward(x, payload, a, b, qt, n, scaling, &xa);
        if (a.defined()) ctx->save_for_backward({payload, x, xa, a, b});
        else ctx->save_for_backward({payload});
        ctx->saved_data["qt"] = qt, ctx->saved_data["k"] = x.size(-1), ctx->saved_data["scaling"] = scaling;
        return y;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        refuse_higher_order("packed MMQ linear");
        const variable_list saved = ctx->get_saved_variables();
        const bool lora = saved.size() > 1;
        const Tensor& payload = saved[0];
        const int qt = (int)ctx->saved_data["qt"].toInt();
        const int64_t k = ctx->saved_data["k"].toInt();
        const Tensor g = usable_cotangent(grads[0], "LoRA linear cotangent");
        const int64_t n = g.size(-1), m = n ? g.numel() / n : 0;
        variable_list out(7);
        c10::SmallVector<int64_t, 5> shape(g.sizes().begin(), g.sizes().end());
        shape.back() = k;
        if (!lora) {
            if (!ctx->needs_input_grad(0)) return out;
            out[0] = empty(shape, at::kBFloat16, g);
            if (m) {
                Tensor ws = empty_bytes(ggq_lora_workspace_bytes(m, 0, 1, n, k, 0), g);
                check(ggq_lora_mmq_backward(g.data_ptr(), payload.data_ptr(), qt, m, n, k, nullptr, nullptr, nullptr, nullptr, 0, 0.f, out[0].data_ptr(), nullptr, nullptr,
                                            ws.data_ptr(), ws.numel(), stream_of(g)));
            }
            return out;
        }
        const Tensor &x = saved[1], &xa = saved[2], &a = saved[3], &b = saved[4];
        const int r = (int)a.size(0);
        Tensor dx = empty(shape, at::kBFloat16, g);
        Tensor da = ctx->needs_input_grad(2) ? empty(a.sizes(), at::kBFloat16, g) : Tensor();
        Tensor db = ctx->needs_input_grad(3) ? empty(b.sizes(), at::kBFloat16, g) : Tensor();
        Tensor ws = empty_bytes(ggq_lora_workspace_bytes(m, 0, 1, n, k, r), g);
        check(ggq_lora_mmq_backward(g.data_ptr(), payload.data_ptr(), qt, m, n, k, x.data_ptr(), xa.data_ptr(), a.data_ptr(), b.data_ptr(), r,
                                    (float)ctx->saved_data["scaling"].toDouble(), dx.data_ptr(), ptr(da), ptr(db), ws.data_ptr(), ws.numel(), stream_of(g)));
        if (ctx->needs_input_grad(0)) out[0] = dx;
        out[2] = da, out[3] = db;
        return out;
    }
};

// ------------------------------------------------------------------------------------------------
// A routed expert FFN: plan, gate/up pair, activation, down projection, combine.
struct ExpertsOptions {
    int64_t qt_gate_up, qt_down;
    double scaling, limit;  // limit 0: no clamp
};

struct ExpertsBuffers {  // what the backward needs beside the inputs
    Tensor plan, gate, up, act, xa_gate_up, xa_down;
};

// Whether some launch of the layer reads row-tile tables built once: Q4_K launches, and the forwards of a few rows per expert (in
// every format; without the plan's tables each of them builds its own, 5 us in front of a launch).
bool shares_tables(int64_t qt_gate_up, int64_t qt_down, int64_t routes, int64_t experts) { return qt_gate_up == 12 || qt_down == 12 || routes <= 10 * experts; }

// Pieces of the one buffer that holds the routing plan, the row-tile tables and the plan's scratch.
struct PlanView {
    int64_t *sorted_ids, *permutation, *inverse, *active_ids;
    int32_t *counts, *ends, *active_ends, *status;
    void *tables, *scratch;
    int64_t tables_bytes, scratch_bytes, bytes;
};
PlanView plan_view(void* base, int64_t tokens, int64_t top_k, int64_t experts, bool with_tables) {
    PlanView v;
    const int64_t routes = tokens * top_k;
    int64_t used = 0;
    auto take = [&](int64_t n) { char* p = (char*)base + used; used += (n + 255) / 256 * 256; return (void*)p; };
    v.permutation = (int64_t*)take(routes * 8), v.inverse = (int64_t*)take(routes * 8), v.sorted_ids = (int64_t*)take(routes * 8);
    v.active_ids = (int64_t*)take(experts * 8);
    v.counts = (int32_t*)take(experts * 4), v.ends = (int32_t*)take(experts * 4), v.active_ends = (int32_t*)take(experts * 4), v.status = (int32_t*)take(8);
    v.tables_bytes = with_tables ? ggq_group_tables_bytes(routes, experts, experts) : 0;
    v.tables = with_tables ? take(v.tables_bytes) : nullptr;
    v.scratch_bytes = ggq_route_plan_workspace_bytes(tokens, (int)top_k, (int)experts);
    v.scratch = take(v.scratch_bytes);
    v.bytes = used;
    return v;
}

Tensor experts_forward(const Tensor& x, const Tensor& ids, const Tensor& weights, const Tensor& gate_w, const Tensor& up_w, const Tensor& down_w,
                       const Tensor& a1, const Tensor& b1, const Tensor& a2, const Tensor& b2, const Tensor& all_experts, const ExpertsOptions& o, ExpertsBuffers& s) {
    const int64_t tokens = ids.size(0), top_k = ids.size(1), routes = tokens * top_k;
    const int64_t experts = gate_w.size(0), inter = gate_w.size(1), hidden = down_w.size(1);
    const bool lora = a1.defined();
    const int64_t r1 = lora ? a1.size(1) : 0, r2 = lora ? a2.size(1) : 0;
    const bool tables = shares_tables(o.qt_gate_up, o.qt_down, routes, experts);
    void* stream = stream_of(x);
    s.plan = empty_bytes(plan_view(nullptr, tokens, top_k, experts, tables).bytes, x);
    const PlanView v = plan_view(s.plan.data_ptr(), tokens, top_k, experts, tables);
    const int64_t* groups = all_experts.const_data_ptr<int64_t>();
    if (tables)
        check(ggq_route_plan_with_tables(ids.data_ptr(), ids.scalar_type() == at::kLong, tokens, (int)top_k, (int)experts, v.sorted_ids, v.permutation, v.inverse,
                                         v.counts, v.ends, v.active_ids, v.active_ends, v.status, v.tables, v.tables_bytes, v.scratch, v.scratch_bytes, stream));
    else
        check(ggq_route_plan(ids.data_ptr(), ids.scalar_type() == at::kLong, tokens, (int)top_k, (int)experts, v.sorted_ids, v.permutation, v.inverse, v.counts,
                             v.ends, v.active_ids, v.active_ends, v.status, v.scratch, v.scratch_bytes, stream));
    s.gate = empty({routes, inter}, at::kBFloat16, x), s.up = empty({routes, inter}, at::kBFloat16, x), s.act = empty({routes, inter}, at::kBFloat16, x);
    if (lora) s.xa_gate_up = empty({routes, rank_pad(r1)}, at::kBFloat16, x), s.xa_down = empty({routes, rank_pad(r2)}, at::kBFloat16, x);
    Tensor y = empty({routes, hidden}, at::kBFloat16, x);
    Tensor out = empty(x.sizes(), at::kBFloat16, x);
    const int64_t ws_bytes = std::max(ggq_lora_workspace_bytes(routes, experts, experts, 2 * inter, hidden, (int)std::max<int64_t>(r1, 1)),
                                      ggq_lora_workspace_bytes(routes, experts, experts, hidden, inter, (int)std::max<int64_t>(r2, 1)));
    Tensor ws = empty_bytes(ws_bytes, x);
    check(ggq_grouped_lora_mmq_forward_indexed(x.data_ptr(), tokens, v.permutation, (int)top_k, gate_w.data_ptr(), up_w.data_ptr(), groups, v.ends, experts,
                                               experts, (int)o.qt_gate_up, routes, inter, hidden, ptr(a1), ptr(b1), (int)r1, (float)o.scaling,
                                               ptr(s.xa_gate_up), s.gate.data_ptr(), s.up.data_ptr(), v.tables, ws.data_ptr(), ws_bytes, stream));
    if (o.limit > 0) check(ggq_swiglu_clamped_forward(s.gate.data_ptr(), s.up.data_ptr(), s.act.data_ptr(), routes * inter, (float)o.limit, stream));
    else check(ggq_swiglu_forward(s.gate.data_ptr(), s.up.data_ptr(), s.act.data_ptr(), routes * inter, stream));
    check(ggq_grouped_lora_mmq_forward(s.act.data_ptr(), down_w.data_ptr(), nullptr, groups, v.ends, experts, experts, (int)o.qt_down, routes, hidden, inter,
                                       ptr(a2), ptr(b2), (int)r2, (float)o.scaling, ptr(s.xa_down), y.data_ptr(), nullptr, v.tables, ws.data_ptr(),
                                       ws_bytes, stream));
    check(ggq_route_combine_forward(y.data_ptr(), weights.data_ptr(), weights.scalar_type() == at::kBFloat16, v.inverse, out.data_ptr(), tokens, (int)top_k,
                                    (int)hidden, stream));
    return out;
}

// The forward of a few routes (sampling): two launches, nothing kept.
bool experts_few_routes(const Tensor& x, const Tensor& ids, const Tensor& weights, const Tensor& gate_w, const Tensor& up_w, const Tensor& down_w, const Tensor& a1,
                        const Tensor& b1, const Tensor& a2, const Tensor& b2, const ExpertsOptions& o, Tensor& out) {
    const int64_t tokens = ids.size(0), top_k = ids.size(1), inter = gate_w.size(1), hidden = down_w.size(1);
    if (!ggq_experts_few_routes_takes((int)o.qt_gate_up, (int)o.qt_down, tokens, (int)top_k, hidden, inter)) return false;
    Tensor act = empty({tokens * top_k, inter}, at::kBFloat16, x);
    out = empty(x.sizes(), at::kBFloat16, x);
    check(ggq_experts_few_routes_forward(x.data_ptr(), ids.data_ptr(), ids.scalar_type() == at::kLong, weights.data_ptr(), weights.scalar_type() == at::kBFloat16,
                                         tokens, (int)top_k, gate_w.size(0), hidden, inter, (int)o.qt_gate_up, (int)o.qt_down, gate_w.data_ptr(), up_w.data_ptr(),
                                         down_w.data_ptr(), ptr(a1), ptr(b1), a1.defined() ? (int)a1.size(1) : 0, ptr(a2), ptr(b2), a2.defined() ? (int)a2.size(1) : 0,
                                         (float)o.scaling, (float)o.limit, act.data_ptr(), out.data_ptr(), stream_of(x)));
    return true;
}

struct Experts : torch::autograd::Function<Experts> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& ids, const Tensor& weights, const Tensor& gate_w, const Tensor& up_w,
                          const Tensor& down_w, const Maybe& a1_in, const Maybe& b1_in, const Maybe& a2_in, const Maybe& b2_in, const Tensor& all_experts,
                          int64_t qt_gate_up, int64_t qt_down, double scaling, double limit) {
        const Tensor a1 = a1_in.value_or(Tensor()), b1 = b1_in.value_or(Tensor()), a2 = a2_in.value_or(Tensor()), b2 = b2_in.value_or(Tensor());
        ExpertsBuffers s;
        Tensor out = experts_forward(x, ids, weights, gate_w, up_w, down_w, a1, b1, a2, b2, all_experts, {qt_gate_up, qt_down, scaling, limit}, s);
        variable_list keep = {x, weights, gate_w, up_w, down_w, all_experts, s.plan, s.gate, s.up, s.act};
        if (a1.defined()) keep.insert(keep.end(), {s.xa_gate_up, s.xa_down, a1, b1, a2, b2});
        ctx->save_for_backward(std::move(keep));
        ctx->saved_data["qt_gate_up"] = qt_gate_up, ctx->saved_data["qt_down"] = qt_down;
        ctx->saved_data["scaling"] = scaling, ctx->saved_data["limit"] = limit;
        return out;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        refuse_higher_order("packed grouped MMQ");
        const variable_list s = ctx->get_saved_variables();
        const Tensor &x = s[0], &weights = s[1], &gate_w = s[2], &up_w = s[3], &down_w = s[4], &all_experts = s[5], &plan = s[6], &gate = s[7], &up = s[8], &act = s[9];
        const bool lora = s.size() > 10;
        const Tensor xa1 = lora ? s[10] : Tensor(), xa2 = lora ? s[11] : Tensor(), a1 = lora ? s[12] : Tensor(), b1 = lora ? s[13] : Tensor(),
                     a2 = lora ? s[14] : Tensor(), b2 = lora ? s[15] : Tensor();
        const int qt1 = (int)ctx->saved_data["qt_gate_up"].toInt(), qt2 = (int)ctx->saved_data["qt_down"].toInt();
        const float scaling = (float)ctx->saved_data["scaling"].toDouble(), limit = (float)ctx->saved_data["limit"].toDouble();
        const int64_t tokens = weights.size(0), top_k = weights.size(1), routes = tokens * top_k;
        const int64_t experts = gate_w.size(0), inter = gate_w.size(1), hidden = down_w.size(1);
        const int r1 = lora ? (int)a1.size(1) : 0, r2 = lora ? (int)a2.size(1) : 0, w_bf16 = weights.scalar_type() == at::kBFloat16;
        const Tensor g = usable_cotangent(grads[0], "combined output cotangent");
        void* stream = stream_of(g);
        const PlanView v = plan_view(plan.data_ptr(), tokens, top_k, experts, shares_tables(qt1, qt2, routes, experts));
        const int64_t* groups = all_experts.const_data_ptr<int64_t>();
        variable_list out(15);
        if (ctx->needs_input_grad(2)) out[2] = empty(weights.sizes(), weights.scalar_type(), g);
        if (lora) {
            if (ctx->needs_input_grad(6)) out[6] = empty(a1.sizes(), at::kBFloat16, g);
            if (ctx->needs_input_grad(7)) out[7] = empty(b1.sizes(), at::kBFloat16, g);
            if (ctx->needs_input_grad(8)) out[8] = empty(a2.sizes(), at::kBFloat16, g);
            if (ctx->needs_input_grad(9)) out[9] = empty(b2.sizes(), at::kBFloat16, g);
        }
        const int64_t ws_bytes = std::max(ggq_lora_workspace_bytes(routes, experts, experts, 2 * inter, hidden, std::max(r1, 1)),
                                          ggq_lora_workspace_bytes(routes, experts, experts, hidden, inter, std::max(r2, 1)));
        Tensor ws = empty_bytes(ws_bytes, g);
        // down projection: the cotangent rows are the tokens' rows, read through the permutation; their routing weight is
        // applied in the activation's backward, which also forms the weights' gradient
        Tensor d_act = empty({routes, inter}, at::kBFloat16, g);
        check(ggq_grouped_lora_mmq_backward_routed_output(g.data_ptr(), tokens, v.permutation, (int)top_k, weights.data_ptr(), w_bf16, down_w.data_ptr(), groups,
                                                          v.ends, experts, experts, qt2, routes, hidden, inter, act.data_ptr(), ptr(xa2), ptr(a2), ptr(b2), r2,
                                                          scaling, d_act.data_ptr(), ptr(out[8]), ptr(out[9]), v.tables, ws.data_ptr(), ws_bytes, stream));
        Tensor d_gate = empty({routes, inter}, at::kBFloat16, g), d_up = empty({routes, inter}, at::kBFloat16, g);
        check(ggq_swiglu_backward_routed(gate.data_ptr(), up.data_ptr(), d_act.data_ptr(), weights.data_ptr(), w_bf16, v.permutation, d_gate.data_ptr(),
                                         d_up.data_ptr(), ptr(out[2]), routes, (int)inter, limit, stream));
        if (!ctx->needs_input_grad(0) && !out[6].defined() && !out[7].defined()) return out;
        Tensor d_rows = empty({routes, hidden}, at::kBFloat16, g);
        check(ggq_grouped_lora_mmq_backward_indexed(d_gate.data_ptr(), d_up.data_ptr(), gate_w.data_ptr(), up_w.data_ptr(), groups, v.ends, experts, experts, qt1,
                                                    routes, inter, hidden, x.data_ptr(), tokens, v.permutation, (int)top_k, ptr(xa1), ptr(a1), ptr(b1), r1,
                                                    scaling, d_rows.data_ptr(), ptr(out[6]), ptr(out[7]), v.tables, ws.data_ptr(), ws_bytes, stream));
        if (ctx->needs_input_grad(0)) {
            out[0] = empty(x.sizes(), at::kBFloat16, g);
            check(ggq_route_gather_backward(d_rows.data_ptr(), v.inverse, out[0].data_ptr(), tokens, (int)top_k, (int)hidden, stream));
        }
        return out;
    }
};

// ------------------------------------------------------------------------------------------------
// Router logits, selection and softmax weights without autograd.
void router_forward(const Tensor& weight, const Tensor& flat, int64_t top_k, Tensor& logits, Tensor& scores, Tensor& indices) {
    if (flat.size(0) <= 8 && usable(flat, at::kBFloat16) && usable(weight, at::kBFloat16) && flat.size(0) > 0 && flat.size(1) % 8 == 0) {
        logits = empty({flat.size(0), weight.size(0)}, at::kBFloat16, flat);
        check(ggq_router_logits(flat.data_ptr(), weight.data_ptr(), flat.size(0), weight.size(0), flat.size(1), logits.data_ptr(), stream_of(flat)));
    } else {
        at::NoGradGuard no_grad;
        logits = at::linear(flat, weight);
    }
    const int64_t tokens = logits.size(0), experts = logits.size(1);
    indices = empty({tokens, top_k}, at::kLong, logits);
    scores = empty({tokens, top_k}, logits.scalar_type(), logits);
    check(ggq_router_topk(logits.data_ptr(), logits.scalar_type() == at::kBFloat16, tokens, (int)experts, (int)top_k, nullptr, 0, indices.data_ptr<int64_t>(),
                          scores.data_ptr(), 1, 1.0f, stream_of(logits)));
}

// ------------------------------------------------------------------------------------------------
// Arguments
Tensor arg_tensor(PyObject* o) { return THPVariable_Check(o) ? THPVariable_Unpack(o) : Tensor(); }
int64_t arg_int(PyObject* o) {
    const long long v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) throw python_error();
    return v;
}
double arg_double(PyObject* o) {
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) throw python_error();
    return v;
}
void arg_count(Py_ssize_t got, Py_ssize_t want, const char* name) { TORCH_CHECK_TYPE(got == want, name, " takes ", want, " arguments, got ", got); }

bool usable_weight(const Tensor& w, int64_t dims, int64_t qt, int64_t k) {
    return usable(w, at::kByte) && w.dim() == dims && !w.requires_grad() && k > 0 && k % 64 == 0 && ggq_row_bytes((int)qt, k) == w.size(-1);
}

// linear(x, payload, quant_type, out_features, lora_A | None, lora_B | None, scaling) -> y | None
PyObject* host_linear(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    arg_count(nargs, 7, "linear");
    const Tensor x = arg_tensor(args[0]), payload = arg_tensor(args[1]), a = arg_tensor(args[4]), b = arg_tensor(args[5]);
    const int64_t qt = arg_int(args[2]), n = arg_int(args[3]);
    const double scaling = arg_double(args[6]);
    if (traced_or_forward_mode({&x, &a, &b})) Py_RETURN_NONE;
    if (!usable(x, at::kBFloat16) || x.dim() < 1 || !usable_weight(payload, 2, qt, x.size(-1)) || payload.size(0) != n || x.device() != payload.device()) Py_RETURN_NONE;
    if (a.defined() != b.defined()) Py_RETURN_NONE;
    if (a.defined() && (!usable(a, at::kBFloat16) || !usable(b, at::kBFloat16) || a.dim() != 2 || b.dim() != 2 || a.size(1) != x.size(-1) || b.size(0) != n ||
                        b.size(1) != a.size(0) || a.device() != x.device() || b.device() != x.device()))
        Py_RETURN_NONE;
    Tensor y;
    {
        ReleaseGil nogil;
        y = any_requires_grad({&x, &a, &b}) ? Linear::apply(x, payload, maybe(a), maybe(b), qt, n, scaling) : linear_forward(x, payload, a, b, qt, n, scaling, nullptr);
    }
    return THPVariable_Wrap(y);
    END_HANDLE_TH_ERRORS
}

// experts(hidden, ids, weights, gate, up, down, A | None, B | None, A_down | None, B_down | None, all_experts, quant_gate_up, quant_down, scaling, limit)
//   -> out | None
PyObject* host_experts(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    arg_count(nargs, 15, "experts");
    const Tensor x = arg_tensor(args[0]), ids = arg_tensor(args[1]), weights = arg_tensor(args[2]), gate = arg_tensor(args[3]), up = arg_tensor(args[4]),
                 down = arg_tensor(args[5]), a1 = arg_tensor(args[6]), b1 = arg_tensor(args[7]), a2 = arg_tensor(args[8]), b2 = arg_tensor(args[9]),
                 all_experts = arg_tensor(args[10]);
    const int64_t qt1 = arg_int(args[11]), qt2 = arg_int(args[12]);
    const double scaling = arg_double(args[13]), limit = arg_double(args[14]);
    if (traced_or_forward_mode({&x, &weights, &a1, &b1, &a2, &b2})) Py_RETURN_NONE;
    if (!usable(x, at::kBFloat16) || x.dim() < 2 || x.size(-1) % 8 || x.size(-1) == 0) Py_RETURN_NONE;
    const int64_t hidden = x.size(-1), tokens = x.numel() / hidden;
    if (!ids.defined() || !ids.is_cuda() || (ids.scalar_type() != at::kLong && ids.scalar_type() != at::kInt) || !ids.is_contiguous() || ids.dim() != 2 ||
        ids.size(0) != tokens || tokens <= 0 || ids.size(1) < 1 || ids.size(1) > 16 || ((uintptr_t)ids.data_ptr() & 15))
        Py_RETURN_NONE;
    if (!weights.defined() || !weights.is_cuda() || (weights.scalar_type() != at::kFloat && weights.scalar_type() != at::kBFloat16) || !weights.is_contiguous() ||
        weights.sizes() != ids.sizes())
        Py_RETURN_NONE;
    if (!usable_weight(gate, 3, qt1, hidden) || !usable_weight(up, 3, qt1, hidden) || gate.sizes() != up.sizes()) Py_RETURN_NONE;
    const int64_t experts = gate.size(0), inter = gate.size(1);
    if (!usable_weight(down, 3, qt2, inter) || down.size(0) != experts || down.size(1) != hidden) Py_RETURN_NONE;
    if (!usable(all_experts, at::kLong) || all_experts.numel() != experts) Py_RETURN_NONE;
    for (const Tensor* t : {&ids, &weights, &gate, &up, &down, &all_experts})
        if (t->device() != x.device()) Py_RETURN_NONE;
    if (a1.defined() != b1.defined() || a1.defined() != a2.defined() || a1.defined() != b2.defined()) Py_RETURN_NONE;
    if (a1.defined()) {
        for (const Tensor* t : {&a1, &b1, &a2, &b2})
            if (!usable(*t, at::kBFloat16) || t->dim() != 3 || t->size(0) != experts || t->device() != x.device()) Py_RETURN_NONE;
        if (a1.size(2) != hidden || b1.size(1) != 2 * inter || b1.size(2) != a1.size(1) || a2.size(2) != inter || b2.size(1) != hidden || b2.size(2) != a2.size(1)) Py_RETURN_NONE;
    }
    // the launches read the token rows through the permutation with 32-bit offsets; a larger matrix takes the general path
    if (!ggq_grouped_forward_reads_indexed_rows((int)qt1, tokens * ids.size(1), experts, tokens, hidden)) Py_RETURN_NONE;
    Tensor y;
    {
        ReleaseGil nogil;
        if (any_requires_grad({&x, &weights, &a1, &b1, &a2, &b2})) {
            y = Experts::apply(x, ids, weights, gate, up, down, maybe(a1), maybe(b1), maybe(a2), maybe(b2), all_experts, qt1, qt2, scaling, limit);
        } else if (ExpertsBuffers s; !experts_few_routes(x, ids, weights, gate, up, down, a1, b1, a2, b2, {qt1, qt2, scaling, limit}, y)) {
            y = experts_forward(x, ids, weights, gate, up, down, a1, b1, a2, b2, all_experts, {qt1, qt2, scaling, limit}, s);
        }
    }
    return THPVariable_Wrap(y);
    END_HANDLE_TH_ERRORS
}

// router(weight, hidden, top_k) -> (logits, scores, indices) | None, for callers that nothing differentiates through
PyObject* host_router(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    arg_count(nargs, 3, "router");
    const Tensor weight = arg_tensor(args[0]), hidden = arg_tensor(args[1]);
    const int64_t top_k = arg_int(args[2]);
    if (!weight.defined() || !hidden.defined() || !weight.is_cuda() || hidden.device() != weight.device() || weight.dim() != 2 || hidden.dim() != 2 ||
        weight.scalar_type() != hidden.scalar_type() || (weight.scalar_type() != at::kBFloat16 && weight.scalar_type() != at::kFloat) ||
        hidden.size(1) != weight.size(1) || any_requires_grad({&weight, &hidden}) || traced_or_forward_mode({&weight, &hidden}))
        Py_RETURN_NONE;
    const int64_t experts = weight.size(0);
    if (experts > 256 || experts % 4 || top_k < 1 || top_k > std::min<int64_t>(8, experts)) Py_RETURN_NONE;
    Tensor logits, scores, indices;
    {
        ReleaseGil nogil;
        router_forward(weight, hidden, top_k, logits, scores, indices);
    }
    PyObject* out = PyTuple_New(3);
    if (!out) throw python_error();
    PyTuple_SET_ITEM(out, 0, THPVariable_Wrap(logits));
    PyTuple_SET_ITEM(out, 1, THPVariable_Wrap(scores));
    PyTuple_SET_ITEM(out, 2, THPVariable_Wrap(indices));
    return out;
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"linear", (PyCFunction)(void (*)(void))host_linear, METH_FASTCALL, "packed linear with an optional LoRA term, differentiable"},
    {"experts", (PyCFunction)(void (*)(void))host_experts, METH_FASTCALL, "routed packed expert FFN, differentiable"},
    {"router", (PyCFunction)(void (*)(void))host_router, METH_FASTCALL, "router logits, selected experts and their softmax weights"},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) { return PyModule_Create(&module_def); }
