// The package's autograd functions in C++ over the C ABI of librwkv6_amd.so: argument preparation,
// allocation and the launches of a forward or a backward, without the Python interpreter between
// them (a backward node here runs without taking its lock).  The kernels take 5-40 us each at the
// sizes of a small model or a short prompt, and a Python autograd function with its ctypes call
// cost 40-80 us a direction.
//
// Every function keeps no state between calls; tensors whose values it needs again go through
// save_for_backward (version checks, saved-tensor hooks and checkpointing apply; LayerNorm's
// backward works on its own copy of a parameter wider than bf16 and keeps the parameters beside it
// for their types and for a second derivative), kernels run on the current stream of the tensors'
// device, and a call from forward-mode differentiation or a function transform is refused.
//
// Mathematics and reference lines: wkv.py, timemix.py, channelmix.py and modules.py, whose
// functions check their arguments and call these.
#include <torch/extension.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/TracerMode.h>
#include <ATen/autocast_mode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>

#include <cstring>
#include <optional>
#include <vector>

#include "../../include/rwkv6_amd.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;
using OptTensor = std::optional<Tensor>;

PyObject* g_error = nullptr;            // the package's Rwkv6Error

void check(int status, const char* what) {
    if (status == RWKV6_OK) return;
    const std::string msg = std::string(what) + ": " + rwkv6_strerror(status);
    if (status == RWKV6_ERR_UNSUPPORTED) C10_THROW_ERROR(NotImplementedError, msg);
    if (status == RWKV6_ERR_INVALID_ARG || status == RWKV6_ERR_ALIGNMENT) C10_THROW_ERROR(ValueError, msg);
    const std::string full = msg + " (status " + std::to_string(status) + ")";
    if (!g_error) throw std::runtime_error(full);
    // a backward node runs without the interpreter lock; the exception keeps its Python type on the way
    // through the autograd engine's threads
    py::gil_scoped_acquire gil;
    PyErr_SetString(g_error, full.c_str());
    python_error e;
    e.persist();
    throw e;
}

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
float* fptr(const Tensor& t) { return static_cast<float*>(ptr(t)); }

// dense and 16-byte aligned, as the kernels read tensors
Tensor dense(const Tensor& t) {
    Tensor c = t.contiguous();
    return reinterpret_cast<uintptr_t>(c.data_ptr()) % 16 ? c.clone() : c;
}
Tensor to_bf16(const Tensor& t) { return dense(t.scalar_type() == at::kBFloat16 ? t : t.to(at::kBFloat16)); }
Tensor to_f32(const Tensor& t) { return dense(t.scalar_type() == at::kFloat ? t : t.to(at::kFloat)); }
Tensor cast(const Tensor& t, at::ScalarType dt) { return t.scalar_type() == dt ? t : t.to(dt); }

// A parameter: bf16 as it is, anything else as fp32.
struct Param {
    Tensor t;
    int dt;
};
Param param(const Tensor& t) {
    return t.scalar_type() == at::kBFloat16 ? Param{dense(t), RWKV6_BF16} : Param{to_f32(t), RWKV6_F32};
}
at::ScalarType param_type(int dt) { return dt == RWKV6_BF16 ? at::kBFloat16 : at::kFloat; }
Tensor empty(at::IntArrayRef s, at::ScalarType dt, const Tensor& like) {
    return at::empty(s, like.options().dtype(dt));
}
Tensor bytes(size_t n, const Tensor& like) { return empty({(int64_t)n}, at::kByte, like); }

int64_t bits(double d) {
    int64_t i;
    std::memcpy(&i, &d, sizeof i);
    return i;
}
double unbits(int64_t i) {
    double d;
    std::memcpy(&d, &i, sizeof d);
    return d;
}
int64_t code(const Tensor& t) { return static_cast<int64_t>(t.scalar_type()); }
at::ScalarType type(int64_t c) { return static_cast<at::ScalarType>(c); }
void put(AutogradContext* ctx, std::vector<int64_t> v) { ctx->saved_data["m"] = std::move(v); }
std::vector<int64_t> meta(AutogradContext* ctx) { return ctx->saved_data["m"].toIntVector(); }

// ---------------------------------------------------------------------------------------
// WKV6, head-first (r, k, v, w [B,H,T,64]) and sequence-first (r, k, v, decay [T,B,H*64])
// ---------------------------------------------------------------------------------------
struct Wkv6 : torch::autograd::Function<Wkv6> {
    static variable_list forward(AutogradContext* ctx, const Tensor& r, const Tensor& k, const Tensor& v,
                                 const Tensor& w, const Tensor& u, const OptTensor& h0, double scale,
                                 int64_t heads, bool final_state, bool grad) {
        const bool seq = heads > 0;
        const int64_t B = r.size(seq ? 1 : 0), H = seq ? heads : r.size(1), T = r.size(seq ? 0 : 2), K = 64;
        const Tensor rb = to_bf16(r), kb = to_bf16(k), vb = to_bf16(v), wb = to_bf16(w);
        const Param ua = param(u);
        const bool state = h0.has_value() && h0->defined();
        const Tensor h0f = state ? to_f32(*h0) : Tensor();
        const Tensor saved = grad ? bytes(rwkv6_wkv_saved_bytes(B, H, T, K, K), rb) : Tensor();
        const Tensor work = bytes(rwkv6_wkv_workspace_bytes(B, H, T, K, K, 0), rb);
        Tensor o = empty({B, H, T, K}, at::kBFloat16, rb);
        const Tensor hT = final_state ? empty({B, H, K, K}, at::kFloat, rb) : Tensor();
        if (grad) {
            auto fn = seq ? rwkv6_wkv_fwd_seqfirst : rwkv6_wkv_fwd;
            check(fn(ptr(rb), ptr(kb), ptr(vb), ptr(wb), ptr(ua.t), ua.dt, fptr(h0f), ptr(o), fptr(hT), ptr(saved),
                     ptr(work), B, H, T, K, K, (float)scale, stream_of(rb)),
                  seq ? "rwkv6_wkv_fwd_seqfirst" : "rwkv6_wkv_fwd");
            ctx->set_materialize_grads(false);
            ctx->save_for_backward({rb, kb, vb, wb, ua.t, saved});
            put(ctx, {B, H, T, heads, bits(scale), ua.dt, state, code(r), code(k), code(v), code(w), code(u),
                      state ? code(*h0) : 0});
        } else {
            check(rwkv6_wkv_infer(ptr(rb), ptr(kb), ptr(vb), ptr(wb), ptr(ua.t), ua.dt, fptr(h0f), ptr(o), fptr(hT),
                                  ptr(work), seq, B, H, T, K, K, (float)scale, stream_of(rb)),
                  "rwkv6_wkv_infer");
        }
        if (!seq) o = cast(o, r.scalar_type());
        if (final_state) return {o, hT};
        return {o};
    }
    static variable_list backward(AutogradContext* ctx, variable_list g) {
        const auto s = ctx->get_saved_variables();
        const auto m = meta(ctx);
        const Tensor &rb = s[0], &kb = s[1], &vb = s[2], &wb = s[3], &ua = s[4], &saved = s[5];
        const int64_t B = m[0], H = m[1], T = m[2], K = 64;
        const bool seq = m[3] > 0, state = m[6];
        // an output no loss uses has no gradient: zeros for o, nothing for the final state
        const Tensor dob = g[0].defined() ? to_bf16(g[0]) : at::zeros({B, H, T, K}, rb.options());
        const Tensor dht = g.size() > 1 && g[1].defined() ? to_f32(g[1]) : Tensor();
        const Tensor dr = at::empty_like(rb), dk = at::empty_like(kb), dv = at::empty_like(vb), dw = at::empty_like(wb);
        const Tensor du = empty({H, K}, ua.scalar_type(), ua);
        const Tensor dh0 = state && ctx->needs_input_grad(5) ? empty({B, H, K, K}, at::kFloat, rb) : Tensor();
        const Tensor work = bytes(rwkv6_wkv_workspace_bytes(B, H, T, K, K, 1), rb);
        auto fn = seq ? rwkv6_wkv_bwd_seqfirst : rwkv6_wkv_bwd;
        check(fn(ptr(rb), ptr(kb), ptr(vb), ptr(wb), ptr(ua), (int)m[5], ptr(dob), fptr(dht), ptr(saved), ptr(dr),
                 ptr(dk), ptr(dv), ptr(dw), ptr(du), fptr(dh0), ptr(work), B, H, T, K, K, (float)unbits(m[4]),
                 stream_of(rb)),
              seq ? "rwkv6_wkv_bwd_seqfirst" : "rwkv6_wkv_bwd");
        return {cast(dr, type(m[7])), cast(dk, type(m[8])), cast(dv, type(m[9])), cast(dw, type(m[10])),
                cast(du, type(m[11])), dh0.defined() ? cast(dh0, type(m[12])) : dh0, Tensor(), Tensor(), Tensor(), Tensor()};
    }
};

bool wkv_type(const Tensor& t) {
    return t.is_cuda() && (t.scalar_type() == at::kBFloat16 || t.scalar_type() == at::kFloat || t.scalar_type() == at::kHalf);
}

// The functions are opaque to torch.func (vmap, grad, jvp, ...), as a Python autograd function
// without setup_context is: refused, instead of run on wrapped tensors.
void no_transforms() {
    TORCH_CHECK(!c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode),
                "the RWKV-6 kernels' autograd functions do not support torch.func transforms");
}

// A forward without the interpreter lock, as torch's own operators run: a launch that waits for room
// in the queue, or an allocation that synchronises, does not stop the program's other threads.
template <class F>
auto unlocked(F&& f) {
    py::gil_scoped_release nogil;
    return f();
}

// whether a backward can follow (the condition under which torch records the function)
bool recorded(std::initializer_list<const Tensor*> ts, const OptTensor& h0) {
    if (!at::GradMode::is_enabled()) return false;
    for (const Tensor* t : ts)
        if (t->requires_grad()) return true;
    return h0 && h0->requires_grad();
}

// None when an argument does not fit: the caller's own checks then say which and raise.
py::object wkv6(const Tensor& r, const Tensor& k, const Tensor& v, const Tensor& w, const Tensor& u,
                const OptTensor& h0, double scale, bool final_state) {
    for (const Tensor* t : {&r, &k, &v, &w, &u})
        if (!wkv_type(*t) || t->device() != r.device()) return py::none();
    if (r.dim() != 4 || r.size(3) != 64 || k.sizes() != r.sizes() || w.sizes() != r.sizes() || v.sizes() != r.sizes())
        return py::none();
    if (u.dim() != 2 || u.size(0) != r.size(1) || u.size(1) != 64) return py::none();
    if (h0 && (h0->device() != r.device() || h0->sizes() != at::IntArrayRef({r.size(0), r.size(1), 64, 64})))
        return py::none();
    no_transforms();
    const variable_list out = unlocked([&] {
        return Wkv6::apply(r, k, v, w, u, h0, scale, (int64_t)0, final_state, recorded({&r, &k, &v, &w, &u}, h0));
    });
    if (final_state) return py::make_tuple(out[0], out[1]);
    return py::make_tuple(out[0], py::none());
}

py::tuple wkv6_seqfirst(const Tensor& r, const Tensor& k, const Tensor& v, const Tensor& decay, const Tensor& u,
                        const OptTensor& h0, double scale, int64_t heads, bool final_state) {
    no_transforms();
    const variable_list out = unlocked([&] {
        return Wkv6::apply(r, k, v, decay, u, h0, scale, heads, final_state, recorded({&r, &k, &v, &decay, &u}, h0));
    });
    if (final_state) return py::make_tuple(out[0], out[1]);
    return py::make_tuple(out[0], py::none());
}

// ---------------------------------------------------------------------------------------
// The time mix's bottlenecks: maa given, the token shift's (5 mixes); else the decay's
// ---------------------------------------------------------------------------------------
struct Weights {
    Tensor down, up;
    int dt;
};
// both weights in one dtype code: a pair of fp32 ones as they are, anything else as bf16
Weights weights(const Tensor& down, const Tensor& up) {
    if (down.scalar_type() == at::kFloat && up.scalar_type() == at::kFloat) return {dense(down), dense(up), RWKV6_F32};
    return {to_bf16(down), to_bf16(up), RWKV6_BF16};
}
// a parameter gradient's buffer: bf16 for a bf16 parameter, fp32 for any other
Tensor grad_like(const Tensor& t) {
    return empty(t.sizes(), t.scalar_type() == at::kBFloat16 ? at::kBFloat16 : at::kFloat, t);
}
int grad_code(const Tensor& t) { return t.scalar_type() == at::kBFloat16 ? RWKV6_BF16 : RWKV6_F32; }

struct Bottleneck : torch::autograd::Function<Bottleneck> {
    static variable_list forward(AutogradContext* ctx, const Tensor& xi, const OptTensor& maa, const Tensor& w_down,
                                 const Tensor& w_up, const Tensor& bias) {
        const Tensor x = dense(xi);
        const bool lerp = maa.has_value();
        const int64_t T = x.size(0), B = x.size(1), C = x.size(2), E = w_down.size(1), R = w_down.size(2);
        const Weights w = weights(w_down, w_up);
        const Param m = lerp ? param(*maa) : Param{Tensor(), 0}, b = param(bias);
        void* s = stream_of(x);
        const Tensor neck = empty({T * B, E * R}, at::kBFloat16, x);
        variable_list out;
        void* po[5] = {};
        for (int64_t e = 0; e < E; ++e) {
            out.push_back(at::empty_like(x));
            po[e] = ptr(out.back());
        }
        check(rwkv6_lora_down_fwd(ptr(x), ptr(m.t), m.dt, ptr(w.down), w.dt, ptr(neck), T, B, C, E, R, s),
              "rwkv6_lora_down_fwd");
        check(rwkv6_lora_up_fwd(lerp ? ptr(x) : nullptr, ptr(neck), ptr(w.up), w.dt, ptr(b.t), b.dt, po, T, B, C, E, R, s),
              "rwkv6_lora_up_fwd");
        ctx->set_materialize_grads(false);
        ctx->save_for_backward({x, lerp ? *maa : Tensor(), w_down, w_up, bias, neck});
        return out;
    }
    static variable_list backward(AutogradContext* ctx, variable_list g) {
        const auto s = ctx->get_saved_variables();
        const Tensor &x = s[0], &maa = s[1], &w_down = s[2], &w_up = s[3], &bias = s[4], &neck = s[5];
        const bool lerp = maa.defined();
        const int64_t T = x.size(0), B = x.size(1), C = x.size(2), E = w_down.size(1), R = w_down.size(2);
        const Weights w = weights(w_down, w_up);
        const Param m = lerp ? param(maa) : Param{Tensor(), 0}, b = param(bias);
        variable_list d;
        const void* pd[5] = {};
        for (int64_t e = 0; e < E; ++e) {
            d.push_back(g[e].defined() ? to_bf16(g[e]) : at::zeros_like(x));
            pd[e] = ptr(d.back());
        }
        const Tensor dx = at::empty_like(x), d_maa = lerp ? grad_like(maa) : Tensor();
        const Tensor d_down = grad_like(w_down), d_up = grad_like(w_up), d_bias = grad_like(bias);
        const Tensor ws = bytes(rwkv6_lora_bwd_workspace_bytes(T, B, C, E, R), x);
        check(rwkv6_lora_bwd(ptr(x), ptr(m.t), m.dt, pd, ptr(neck), ptr(w.down), ptr(w.up), w.dt, ptr(b.t), b.dt,
                             ptr(dx), ptr(d_maa), ptr(d_down), grad_code(w_down), ptr(d_up), grad_code(w_up),
                             ptr(d_bias), ptr(ws), T, B, C, E, R, stream_of(x)),
              "rwkv6_lora_bwd");
        return {dx, lerp ? cast(d_maa, maa.scalar_type()) : d_maa, cast(d_down, w_down.scalar_type()),
                cast(d_up, w_up.scalar_type()), cast(d_bias, bias.scalar_type())};
    }
};

// Whether the end-to-end kernels take this call (rank and expansion, sizes, parameters of the
// expected sizes on x's device); the caller has checked x ([T,B,C] bf16 on the GPU).
bool fits(const Tensor& x, const Tensor* maa, const Tensor& w_down, const Tensor& w_up, const Tensor& bias) {
    if (w_down.dim() != 3 || w_up.dim() != 3) return false;
    const int64_t T = x.size(0), B = x.size(1), C = x.size(2), E = w_down.size(1), R = w_down.size(2);
    if ((E > 1) != (maa != nullptr) || rwkv6_lora_bwd_workspace_bytes(T, B, C, E, R) == 0) return false;
    if (w_down.size(0) != C || w_up.sizes() != at::IntArrayRef({E, R, C}) || bias.numel() != E * C) return false;
    for (const Tensor* t : {&w_down, &w_up, &bias})
        if (t->device() != x.device()) return false;
    return !maa || (maa->numel() == C && maa->device() == x.device());
}

// None when the kernels do not take the call: the caller runs the general path.
py::object token_shift_mix(const Tensor& x, const Tensor& maa, const Tensor& w_down, const Tensor& w_up,
                           const Tensor& bias) {
    if (!fits(x, &maa, w_down, w_up, bias)) return py::none();
    no_transforms();
    const variable_list o = unlocked([&] { return Bottleneck::apply(x, OptTensor(maa), w_down, w_up, bias); });
    return py::make_tuple(o[0], o[1], o[2], o[3], o[4]);
}
py::object decay_lora(const Tensor& x, const Tensor& w_down, const Tensor& w_up, const Tensor& bias) {
    if (!fits(x, nullptr, w_down, w_up, bias)) return py::none();
    no_transforms();
    return py::cast(unlocked([&] { return Bottleneck::apply(x, OptTensor(), w_down, w_up, bias)[0]; }));
}

// ---------------------------------------------------------------------------------------
// GroupNorm over heads of 64 channels, times silu(g_pre) when there is one
// ---------------------------------------------------------------------------------------
struct GroupNormGate : torch::autograd::Function<GroupNormGate> {
    struct Dims {
        int64_t T, B, H;
    };
    static Dims dims(const Tensor& o, bool head_first) {
        return head_first ? Dims{o.size(2), o.size(0), o.size(1)} : Dims{o.size(0), o.size(1), o.size(2) / 64};
    }
    static std::pair<Param, Param> affine(const Tensor& gamma, const Tensor& beta) {
        Param ga = param(gamma), be = param(beta);
        if (be.dt != ga.dt) be = {dense(be.t.to(ga.t.scalar_type())), ga.dt};
        return {ga, be};
    }
    static Tensor forward(AutogradContext* ctx, const Tensor& oi, const OptTensor& gi, const Tensor& gamma,
                          const Tensor& beta, double eps, bool head_first) {
        const Dims n = dims(oi, head_first);
        const Tensor o = dense(oi), g = gi ? dense(*gi) : Tensor();
        const auto [ga, be] = affine(gamma, beta);
        const Tensor y = empty({n.T, n.B, n.H * 64}, at::kBFloat16, o);
        const Tensor mean = empty({n.T * n.B * n.H}, at::kFloat, o), rstd = at::empty_like(mean);
        check(rwkv6_gn_gate_fwd(ptr(o), head_first, ptr(g), ptr(ga.t), ptr(be.t), ga.dt, (float)eps, ptr(y), fptr(mean),
                                fptr(rstd), n.T, n.B, n.H, 64, stream_of(o)),
              "rwkv6_gn_gate_fwd");
        ctx->save_for_backward({o, g, gamma, beta, mean, rstd});
        put(ctx, {head_first});
        return y;
    }
    static variable_list backward(AutogradContext* ctx, variable_list gr) {
        const auto s = ctx->get_saved_variables();
        const bool head_first = meta(ctx)[0];
        const Tensor &o = s[0], &g = s[1], &gamma = s[2], &beta = s[3];
        const Dims n = dims(o, head_first);
        const auto [ga, be] = affine(gamma, beta);
        const Tensor dy = to_bf16(gr[0]), d_o = at::empty_like(o), d_g = g.defined() ? at::empty_like(g) : Tensor();
        const Tensor dgamma = empty({n.H * 64}, ga.t.scalar_type(), o), dbeta = at::empty_like(dgamma);
        const Tensor ws = bytes(rwkv6_gn_gate_bwd_workspace_bytes(n.T, n.B, n.H, 64), o);
        check(rwkv6_gn_gate_bwd(ptr(o), head_first, ptr(g), ptr(ga.t), ptr(be.t), ga.dt, fptr(s[4]), fptr(s[5]), ptr(dy),
                                ptr(d_o), ptr(d_g), ptr(dgamma), ptr(dbeta), ptr(ws), n.T, n.B, n.H, 64, stream_of(o)),
              "rwkv6_gn_gate_bwd");
        return {d_o, d_g, cast(dgamma, gamma.scalar_type()), cast(dbeta, beta.scalar_type()), Tensor(), Tensor()};
    }
};
Tensor group_norm_gate(const Tensor& o, const OptTensor& g, const Tensor& gamma, const Tensor& beta, double eps,
                       bool head_first) {
    no_transforms();
    return unlocked([&] { return GroupNormGate::apply(o, g, gamma, beta, eps, head_first); });
}

// ---------------------------------------------------------------------------------------
// LayerNorm over the last dimension
// ---------------------------------------------------------------------------------------
struct LayerNorm : torch::autograd::Function<LayerNorm> {
    static Tensor forward(AutogradContext* ctx, const Tensor& xi, const Tensor& gamma, const Tensor& beta, double eps,
                          bool grad) {
        const Tensor x = dense(xi);
        const int64_t C = x.size(-1), N = x.numel() / C;
        Param ga = param(gamma), be = param(beta);
        if (ga.dt != be.dt) ga = {to_f32(gamma), RWKV6_F32}, be = {to_f32(beta), RWKV6_F32};
        const Tensor y = at::empty_like(x), mean = empty({N}, at::kFloat, x), rstd = at::empty_like(mean);
        // A bf16 gamma is saved itself.  Of any other the backward uses the values of this call, from
        // the kernel's copy, so that an update of the parameter in between is not an error.
        const Tensor copy = grad && gamma.scalar_type() != at::kBFloat16 ? empty({C}, at::kFloat, x) : Tensor();
        check(rwkv6_layer_norm_fwd(ptr(x), ptr(ga.t), ptr(be.t), ga.dt, (float)eps, ptr(y), fptr(mean), fptr(rstd),
                                   fptr(copy), N, C, stream_of(x)),
              "rwkv6_layer_norm_fwd");
        if (grad) {
            // the input itself: a dense copy made here has no history for a second derivative
            ctx->save_for_backward({xi, copy.defined() ? copy : gamma, mean, rstd});
            if (copy.defined()) ctx->saved_data["gamma"] = gamma;
            ctx->saved_data["beta"] = beta;
        }
        return y;
    }
    static variable_list backward(AutogradContext* ctx, variable_list gr) {
        const auto s = ctx->get_saved_variables();
        const Tensor x = dense(s[0]), &mean = s[2], &rstd = s[3];
        const bool own = ctx->saved_data.count("gamma") == 0;       // gamma is the saved tensor itself
        const Tensor gamma = own ? s[1] : ctx->saved_data["gamma"].toTensor(), beta = ctx->saved_data["beta"].toTensor();
        const bool ng = ctx->needs_input_grad(1), nb = ctx->needs_input_grad(2);
        const int64_t C = x.size(-1), N = x.numel() / C;
        if (at::GradMode::is_enabled()) {
            // a backward that is differentiated itself: torch's differentiable form, on the values used
            const Tensor g = own ? gamma : gamma + (s[1].to(gamma.scalar_type()) - gamma).detach();
            std::vector<int64_t> st(x.sizes().begin(), x.sizes().end());
            st.back() = 1;
            const auto [dx, dg, db] = at::native_layer_norm_backward(gr[0], x, {C}, mean.view(st), rstd.view(st),
                                                                     g.to(x.scalar_type()), beta.to(x.scalar_type()),
                                                                     {true, ng, nb});
            return {dx, ng ? cast(dg, gamma.scalar_type()) : Tensor(), nb ? cast(db, beta.scalar_type()) : Tensor(), Tensor(), Tensor()};
        }
        const Param ga = param(s[1]);
        const Tensor dy = to_bf16(gr[0]), dx = at::empty_like(x);
        const int dt = grad_code(gamma) == grad_code(beta) ? grad_code(gamma) : RWKV6_F32;
        const bool sums = ng || nb;
        const Tensor dg = sums ? empty({C}, param_type(dt), x) : Tensor(), db = sums ? at::empty_like(dg) : Tensor();
        const Tensor ws = sums ? bytes(rwkv6_layer_norm_bwd_workspace_bytes(N, C), x) : Tensor();
        check(rwkv6_layer_norm_bwd(ptr(x), ptr(ga.t), ga.dt, fptr(mean), fptr(rstd), ptr(dy), ptr(dx), ptr(dg), ptr(db), dt,
                                   ptr(ws), N, C, stream_of(x)),
              "rwkv6_layer_norm_bwd");
        return {dx, ng ? cast(dg, gamma.scalar_type()) : Tensor(), nb ? cast(db, beta.scalar_type()) : Tensor(), Tensor(), Tensor()};
    }
};
// Whether an operator on these tensors is a plain call of its kernel: no autocast, transform,
// tracing, forward-mode derivative or mode that wants to see it.
bool plain(std::initializer_list<const Tensor*> ts) {
    if (at::autocast::is_autocast_enabled(at::kCUDA) || c10::impl::dispatch_mode_enabled() ||
        at::impl::torch_function_mode_enabled() || at::tracer::impl::is_dispatch_enabled() ||
        c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode))
        return false;
    for (const Tensor* t : ts)
        if (t->key_set().has(c10::DispatchKey::Python) || t->_fw_grad(0).defined()) return false;
    return true;
}
// None when the kernels do not take the call: the caller runs torch's.
py::object layer_norm(const Tensor& x, const OptTensor& gamma, const OptTensor& beta, double eps) {
    if (!gamma || !beta || x.dim() < 1 || x.numel() == 0 || x.layout() != at::kStrided) return py::none();
    const int64_t C = x.size(-1);
    if (rwkv6_layer_norm_bwd_workspace_bytes(x.numel() / C, C) == 0) return py::none();
    for (const Tensor* t : {&*gamma, &*beta})
        if (t->sizes() != at::IntArrayRef({C}) || t->device() != x.device() ||
            (t->scalar_type() != at::kBFloat16 && t->scalar_type() != at::kFloat && t->scalar_type() != at::kHalf))
            return py::none();
    if (!plain({&x, &*gamma, &*beta})) return py::none();
    return py::cast(unlocked([&] { return LayerNorm::apply(x, *gamma, *beta, eps, recorded({&x, &*gamma}, beta)); }));
}

// ---------------------------------------------------------------------------------------
// channel mix
// ---------------------------------------------------------------------------------------
struct CmixLerp : torch::autograd::Function<CmixLerp> {
    static variable_list forward(AutogradContext* ctx, const Tensor& xi, const Tensor& mix) {
        const Tensor x = dense(xi);
        const Param m = param(mix);
        const Tensor a = at::empty_like(x), b = at::empty_like(x);
        void* po[2] = {ptr(a), ptr(b)};
        check(rwkv6_cmix_lerp_fwd(ptr(x), ptr(m.t), m.dt, po, x.size(0), x.size(1), x.size(2), stream_of(x)),
              "rwkv6_cmix_lerp_fwd");
        ctx->set_materialize_grads(false);
        ctx->save_for_backward({x, m.t});
        put(ctx, {m.dt, code(mix)});
        return {a, b};
    }
    static variable_list backward(AutogradContext* ctx, variable_list g) {
        const auto s = ctx->get_saved_variables();
        const auto m = meta(ctx);
        const Tensor& x = s[0];
        const int64_t T = x.size(0), B = x.size(1), C = x.size(2);
        Tensor d[2];
        const void* pd[2];
        for (int e = 0; e < 2; ++e) {
            d[e] = g[e].defined() ? to_bf16(g[e]) : at::zeros_like(x);
            pd[e] = ptr(d[e]);
        }
        const Tensor dx = at::empty_like(x), d_mix = empty({2, C}, s[1].scalar_type(), x);
        const Tensor ws = bytes(rwkv6_cmix_lerp_bwd_workspace_bytes(T, B, C), x);
        check(rwkv6_cmix_lerp_bwd(ptr(x), ptr(s[1]), (int)m[0], pd, ptr(dx), ptr(d_mix), ptr(ws), T, B, C, stream_of(x)),
              "rwkv6_cmix_lerp_bwd");
        return {dx, cast(d_mix, type(m[1]))};
    }
};
py::tuple cmix_lerp(const Tensor& x, const Tensor& mix) {
    no_transforms();
    const variable_list o = unlocked([&] { return CmixLerp::apply(x, mix); });
    return py::make_tuple(o[0], o[1]);
}

struct ReluSq : torch::autograd::Function<ReluSq> {
    static Tensor forward(AutogradContext* ctx, const Tensor& ui) {
        const Tensor up = dense(ui), h = at::empty_like(up);
        check(rwkv6_relu_sq_fwd(ptr(up), ptr(h), up.numel(), stream_of(up)), "rwkv6_relu_sq_fwd");
        ctx->save_for_backward({up});
        return h;
    }
    static variable_list backward(AutogradContext* ctx, variable_list g) {
        const Tensor up = ctx->get_saved_variables()[0], dh = to_bf16(g[0]), d = at::empty_like(up);
        check(rwkv6_relu_sq_bwd(ptr(up), ptr(dh), ptr(d), up.numel(), stream_of(up)), "rwkv6_relu_sq_bwd");
        return {d};
    }
};
Tensor relu_sq(const Tensor& up) {
    no_transforms();
    return unlocked([&] { return ReluSq::apply(up); });
}

struct SigmoidGate : torch::autograd::Function<SigmoidGate> {
    static Tensor forward(AutogradContext* ctx, const Tensor& oi, const Tensor& gi) {
        const Tensor o = dense(oi), g = dense(gi), y = at::empty_like(o);
        check(rwkv6_sigmoid_gate_fwd(ptr(o), ptr(g), ptr(y), o.numel(), stream_of(o)), "rwkv6_sigmoid_gate_fwd");
        ctx->save_for_backward({o, g});
        return y;
    }
    static variable_list backward(AutogradContext* ctx, variable_list gr) {
        const auto s = ctx->get_saved_variables();
        const Tensor &o = s[0], &g = s[1];
        const Tensor dy = to_bf16(gr[0]), d_o = at::empty_like(o), d_g = at::empty_like(g);
        check(rwkv6_sigmoid_gate_bwd(ptr(o), ptr(g), ptr(dy), ptr(d_o), ptr(d_g), o.numel(), stream_of(o)),
              "rwkv6_sigmoid_gate_bwd");
        return {d_o, d_g};
    }
};
Tensor sigmoid_gate(const Tensor& out, const Tensor& gate_pre) {
    no_transforms();
    return unlocked([&] { return SigmoidGate::apply(out, gate_pre); });
}

// ---------------------------------------------------------------------------------------
// y = x W^T with the weight gradient split over the tokens
// ---------------------------------------------------------------------------------------

// part [S, ...] fp32 summed over S in order, in `dt` (bf16 directly, else fp32 and a cast)
Tensor sum_partials(const Tensor& part, at::ScalarType dt) {
    const bool bf = dt == at::kBFloat16;
    const Tensor out = empty(part.sizes().slice(1), bf ? at::kBFloat16 : at::kFloat, part);
    check(rwkv6_sum_partials(fptr(part), part.size(0), out.numel(), bf ? RWKV6_BF16 : RWKV6_F32, ptr(out), stream_of(part)),
          "rwkv6_sum_partials");
    return cast(out, dt);
}

// dW = dy^T x for dy [N, O], x [N, I] (N = tokens), fp32-accumulated.  A projection's weight
// gradient has a small output (O x I, e.g. 2048 x 2048 = 64 tiles of 256 x 256) and a long
// reduction (16 K tokens): one GEMM occupies a quarter of the 256 CUs.  The tokens are split into s
// chunks that run as one batched GEMM with fp32 outputs, summed in a fixed order, where that is
// faster than the s partial sums cost: s doubles up to 4 while the tiles of all chunks are below
// the CU count and a chunk keeps 4096 tokens (2560 for an output of a few tiles, which leaves more
// CUs idle).  Measured on MI355X, us for s = 1, 2, 4: 2048 x 2048 of 16384 tokens 163, 140, 136, of
// 8192 tokens 102, 88, 91, of 4096 tokens 44, 49, 56; 7168 x 2048 of 8192 tokens 297, 258, 302, of
// 4096 tokens 140, 168, 206; 1024 x 1024 of 8192 tokens 55, 39, 36.  One chunk writes dt directly (a
// parameter wider than bf16 gets the fp32 accumulator).
Tensor splitk_wgrad(const Tensor& dy, const Tensor& x, at::ScalarType dt) {
    const int64_t N = dy.size(0), O = dy.size(1), I = x.size(1), tiles = (O + 255) / 256 * ((I + 255) / 256);
    const int64_t chunk = tiles > 32 ? 4096 : 2560;
    int64_t s = 1;
    while (s < 4 && tiles * s < 256 && N % (2 * s) == 0 && N / (2 * s) >= chunk) s *= 2;
    if (s == 1 && (!dy.is_cuda() || dt == dy.scalar_type() || dy.scalar_type() != at::kBFloat16 || N == 0))
        return cast(at::mm(dy.t(), x), dt);
    TORCH_CHECK_TYPE(dy.is_cuda(), "split weight gradients run on the GPU");
    // A backward that is differentiated itself: bmm with an output type and the summing kernel have no
    // derivative.  One product in fp32 for a parameter wider than bf16 (exact products, as the batched
    // one's), else in the operands' type.
    if (at::GradMode::is_enabled()) {
        const bool wide = dt != dy.scalar_type() && dy.scalar_type() == at::kBFloat16;
        return cast(wide ? at::mm(dy.t().to(at::kFloat), x.to(at::kFloat)) : at::mm(dy.t(), x), dt);
    }
    const Tensor part = at::bmm(dy.view({s, N / s, O}).transpose(1, 2), x.view({s, N / s, I}), at::kFloat);
    return s == 1 ? cast(part.view({O, I}), dt) : sum_partials(part, dt);
}

// Whether y = x W^T runs on the kernel that rounds an fp32 W inside instead of a cast and the library's
// product: up to 2^30 multiplications (1024 tokens x 1024 x 1024: 12.1 us against 13.7; 1536: 16.5
// against 14.5), 2048 inputs (a longer chain of steps: 1024 x 3584 of 64 tokens 18.5 and 20.1 us, of
// 777 33 and 24) and 2^21 elements of x (more of them through 64-token tiles cost what the cast saved:
// 65536 tokens x 128 x 128 17.0 against 13.3, 4096 x 512 x 512 11.5 against 12.5).
bool small_f32(const Tensor& x, const Tensor& w) {
    if (!x.is_cuda() || x.device() != w.device() || x.scalar_type() != at::kBFloat16 || w.scalar_type() != at::kFloat ||
        w.dim() != 2 || x.dim() < 1 || x.size(-1) != w.size(1) || x.layout() != at::kStrided || w.layout() != at::kStrided)
        return false;
    const int64_t O = w.size(0), I = w.size(1);
    if (x.numel() == 0 || O == 0 || O % 4 || I % 8 || I > 2048) return false;
    return x.numel() <= (1 << 21) && x.numel() <= (int64_t(1) << 30) / O && plain({&x, &w});
}

struct Linear : torch::autograd::Function<Linear> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w, bool small, bool grad) {
        if (small) {
            const Tensor xd = dense(x), wd = dense(w);
            std::vector<int64_t> size(x.sizes().begin(), x.sizes().end());
            size.back() = w.size(0);
            const Tensor y = empty(size, at::kBFloat16, x), wc = grad ? empty(w.sizes(), at::kBFloat16, x) : Tensor();
            check(rwkv6_linear_f32(ptr(xd), fptr(wd), ptr(y), ptr(wc), xd.numel() / w.size(1), w.size(0), w.size(1),
                                   stream_of(x)),
                  "rwkv6_linear_f32");
            if (grad) {
                ctx->save_for_backward({x, wc});
                put(ctx, {code(w)});
            }
            return y;
        }
        const Tensor wc = cast(w, x.scalar_type());
        ctx->save_for_backward({x, wc});
        put(ctx, {code(w)});
        return at::linear(x, wc);
    }
    static variable_list backward(AutogradContext* ctx, variable_list g) {
        const auto s = ctx->get_saved_variables();
        const Tensor &x = s[0], &wc = s[1];
        const Tensor dy = g[0].reshape({-1, g[0].size(-1)}).contiguous();
        Tensor dx, dw;
        if (ctx->needs_input_grad(0)) dx = at::mm(dy, wc).view(x.sizes());
        if (ctx->needs_input_grad(1))
            dw = splitk_wgrad(dy, x.reshape({-1, x.size(-1)}).contiguous(), type(meta(ctx)[0]));
        return {dx, dw, Tensor(), Tensor()};
    }
};
Tensor linear(const Tensor& x, const Tensor& w) {
    no_transforms();
    return unlocked([&] { return Linear::apply(x, w, small_f32(x, w), recorded({&x, &w}, OptTensor())); });
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    m.attr("ABI_VERSION") = RWKV6_ABI_VERSION;
    // a status as the functions here raise it, from a thread that does not hold the interpreter lock
    m.def("check", [](int status, const std::string& what) {
        py::gil_scoped_release nogil;
        check(status, what.c_str());
    });
    m.def("set_error", [](py::object cls) { g_error = cls.release().ptr(); });
    m.def("wkv6", torch::wrap_pybind_function(wkv6));
    m.def("wkv6_seqfirst", torch::wrap_pybind_function(wkv6_seqfirst));
    m.def("token_shift_mix", torch::wrap_pybind_function(token_shift_mix));
    m.def("decay_lora", torch::wrap_pybind_function(decay_lora));
    m.def("group_norm_gate", torch::wrap_pybind_function(group_norm_gate));
    m.def("layer_norm", torch::wrap_pybind_function(layer_norm));
    m.def("cmix_lerp", torch::wrap_pybind_function(cmix_lerp));
    m.def("relu_sq", torch::wrap_pybind_function(relu_sq));
    m.def("sigmoid_gate", torch::wrap_pybind_function(sigmoid_gate));
    m.def("linear", torch::wrap_pybind_function(linear));
}
