// The operator's autograd functions as native torch nodes (Python module theseus._native).
//
// theseus/wkv7.py's _WKV and theseus/gdn.py's _GDN do the same through Python: contiguous
// inputs, the checks of kernels/wkv7_state.cpp:10-15, outputs and workspace from torch's
// allocator, one C-ABI call on the current stream.  For few tokens that host work is the
// call: a forward+backward through the Python functions takes 225 us of host time (B=1, T=64,
// H=2, bf16), a good part of it the engine's device thread taking the interpreter lock for
// the backward; here it takes 49 us.  Python keeps its functions for what these do not cover
// (functorch transforms, tensor subclasses).
#include <torch/extension.h>

#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>

#include <cstdlib>
#include <cstring>

#include "../../include/theseus_gdn_ex.h"
#include "../../include/theseus_wkv7.h"

namespace py = pybind11;
using torch::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

namespace {

void raise_status(int st, const char* who) {
    TORCH_CHECK(st == 0, who, ": ", theseus_wkv7_error_string(st));
}
hipStream_t stream_of(const Tensor& t) {
    return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream();
}
Tensor scratch(size_t bytes, const Tensor& like) {
    return bytes ? at::empty({(int64_t)bytes}, like.options().dtype(torch::kUInt8)) : Tensor();
}
void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
float* fptr(const Tensor& t) { return static_cast<float*>(ptr(t)); }

// check() of kernels/wkv7_state.cpp:10-15, the same messages
void check(const Tensor& r, std::initializer_list<Tensor> xs) {
    TORCH_CHECK(r.is_cuda() && r.is_contiguous() && r.dim() == 4, "expected contiguous CUDA [B,T,H,N]");
    TORCH_CHECK(r.size(1) > 0 && r.size(3) >= 2 && r.size(3) <= 128, "invalid T or head size (2..128)");
    TORCH_CHECK(r.scalar_type() == torch::kBFloat16 || r.scalar_type() == torch::kFloat32, "expected BF16 or FP32");
    for (const Tensor& x : xs)
        TORCH_CHECK(x.device() == r.device() && x.sizes() == r.sizes() && x.scalar_type() == r.scalar_type() &&
                        x.is_contiguous(),
                    "input mismatch");
}
struct Dims {
    int B, T, H, N, dt;
    explicit Dims(const Tensor& r)
        : B((int)r.size(0)), T((int)r.size(1)), H((int)r.size(2)), N((int)r.size(3)),
          dt(r.scalar_type() == torch::kBFloat16 ? THESEUS_WKV7_BF16 : THESEUS_WKV7_FP32) {}
    std::vector<int64_t> saved() const { return {B, H, (int64_t)theseus_wkv7_checkpoint_count(T), N, N}; }
    int family() const { return theseus_wkv7_kernel_family(B, T, H, N, dt); }
};
bool env_is_1(const char* name) {
    const char* e = std::getenv(name);
    return e && std::strcmp(e, "1") == 0;
}
// Extension._warn_fallback: a warning (or, THESEUS_WKV7_STRICT=1, an error) when a call runs
// on the step-serial kernels without having asked for them.  The warning names the caller of
// theseus.wkv7.wkv7 (three frames up: this function, wkv7, the caller).
void warn_fallback(const Dims& d, int family) {
    if (family != THESEUS_WKV7_FAMILY_FP32 && family != THESEUS_WKV7_FAMILY_HEAD_SIZE &&
        family != THESEUS_WKV7_FAMILY_SIZE)
        return;
    py::gil_scoped_acquire gil;
    py::module_::import("theseus.wkv7").attr("extension")().attr("_warn_fallback")(d.B, d.T, d.H, d.N, d.dt, 3);
}
// THESEUS_WKV7_CHECK_WAITS=1 (Extension._check_waits)
void check_waits() {
    if (!env_is_1("THESEUS_WKV7_CHECK_WAITS")) return;
    unsigned int n = 0;
    raise_status(theseus_wkv7_wait_timeouts(&n, 1), "theseus_wkv7");
    TORCH_CHECK(n == 0, "theseus_wkv7: ", n,
                " bounded wait(s) timed out in the chunked kernels; the outputs hold NaN where they depended on them");
}

struct Fwd {
    Tensor y, end, saved;
};
Fwd wkv7_forward(const std::array<Tensor, 6>& x, const Tensor& s0, bool save) {
    const auto& [r, w, k, v, a, b] = x;
    check(r, {w, k, v, a, b});
    const Dims d(r);
    TORCH_CHECK(s0.device() == r.device() && s0.scalar_type() == torch::kFloat32 && s0.is_contiguous(),
                "s0 must be contiguous CUDA FP32");
    TORCH_CHECK(s0.sizes() == at::IntArrayRef({d.B, d.H, d.N, d.N}), "invalid s0 shape");
    c10::OptionalDeviceGuard guard(r.device());
    Fwd o{at::empty_like(r), at::empty_like(s0), Tensor()};
    if (save) o.saved = at::empty(d.saved(), s0.options());
    if (d.T > 1 || save) warn_fallback(d, d.family());
    const size_t need = theseus_wkv7_forward_best_workspace_size(d.B, d.T, d.H, d.N, d.dt, save);
    const Tensor ws = scratch(need, r);
    raise_status(theseus_wkv7_forward(d.B, d.T, d.H, d.N, d.dt, ptr(r), ptr(w), ptr(k), ptr(v), ptr(a), ptr(b), fptr(s0),
                                      ptr(o.y), fptr(o.end), fptr(o.saved), ptr(ws), need, stream_of(r)),
                 "theseus_wkv7");
    check_waits();
    return o;
}

Tensor float_rows(const Tensor& t) { return t.to(torch::kFloat32).contiguous(); }

struct Wkv7 : torch::autograd::Function<Wkv7> {
    static variable_list forward(AutogradContext* ctx, const Tensor& r, const Tensor& w, const Tensor& k, const Tensor& v,
                                 const Tensor& a, const Tensor& b, const Tensor& state) {
        ctx->set_materialize_grads(false);
        const std::array<Tensor, 6> x{r.contiguous(), w.contiguous(), k.contiguous(),
                                      v.contiguous(), a.contiguous(), b.contiguous()};
        const Fwd o = wkv7_forward(x, float_rows(state), true);
        ctx->save_for_backward({x[0], x[1], x[2], x[3], x[4], x[5], o.saved});
        // the saved states' order is the chunked kernels' (family 0) or [value][key]
        ctx->saved_data["tiled"] = Dims(x[0]).family() == THESEUS_WKV7_FAMILY_CHUNKED;
        return {o.y, o.end};
    }
    static variable_list backward(AutogradContext* ctx, variable_list g) {
        const variable_list s = ctx->get_saved_variables();
        const Tensor &r = s[0], &saved = s[6];
        const Tensor dy = g[0].defined() ? g[0].to(r.scalar_type()).contiguous() : at::zeros_like(r);
        const Tensor dend = g[1].defined() ? float_rows(g[1]) : Tensor();
        check(r, {s[1], s[2], s[3], s[4], s[5], dy});
        const Dims d(r);
        const int family = d.family();
        TORCH_CHECK(ctx->saved_data["tiled"].toBool() == (family == THESEUS_WKV7_FAMILY_CHUNKED),
                    "saved states were written by the other kernel family (their order differs); run the backward with "
                    "the forward's THESEUS_WKV7_FAMILY");
        TORCH_CHECK(saved.device() == r.device() && saved.scalar_type() == torch::kFloat32 && saved.is_contiguous() &&
                        saved.sizes() == at::IntArrayRef(d.saved()),
                    "invalid history");
        TORCH_CHECK(!dend.defined() ||
                        (dend.device() == r.device() && dend.sizes() == at::IntArrayRef({d.B, d.H, d.N, d.N})),
                    "invalid dend");
        c10::OptionalDeviceGuard guard(r.device());
        variable_list o(7);
        for (int i = 0; i < 6; i++) o[i] = at::empty_like(r);
        o[6] = at::empty({d.B, d.H, d.N, d.N}, saved.options());
        // (the forward of these sizes has warned, and the engine's thread has no caller to name)
        if (env_is_1("THESEUS_WKV7_STRICT")) warn_fallback(d, family);
        const size_t need = theseus_wkv7_backward_workspace_size(d.B, d.T, d.H, d.N, d.dt);
        const Tensor ws = scratch(need, r);
        raise_status(theseus_wkv7_backward(d.B, d.T, d.H, d.N, d.dt, ptr(r), ptr(s[1]), ptr(s[2]), ptr(s[3]), ptr(s[4]),
                                           ptr(s[5]), fptr(saved), ptr(dy), fptr(dend), ptr(o[0]), ptr(o[1]), ptr(o[2]),
                                           ptr(o[3]), ptr(o[4]), ptr(o[5]), fptr(o[6]), ptr(ws), need, stream_of(r)),
                     "theseus_wkv7");
        check_waits();
        return o;
    }
};

std::pair<Tensor, Tensor> wkv7(const Tensor& r, const Tensor& w, const Tensor& k, const Tensor& v, const Tensor& a,
                               const Tensor& b, const Tensor& state) {
    py::gil_scoped_release free;
    bool grad = false;
    if (at::GradMode::is_enabled())
        for (const Tensor* t : {&r, &w, &k, &v, &a, &b, &state}) grad = grad || t->requires_grad();
    if (grad) {
        const variable_list o = Wkv7::apply(r, w, k, v, a, b, state);
        return {o[0], o[1]};
    }
    const std::array<Tensor, 6> x{r.contiguous(), w.contiguous(), k.contiguous(),
                                  v.contiguous(), a.contiguous(), b.contiguous()};
    const Fwd o = wkv7_forward(x, float_rows(state), false);
    return {o.y, o.end};
}

// Extension._gdn_check
void gdn_check(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& g, const Tensor& beta, const Tensor& s0) {
    TORCH_CHECK(q.scalar_type() == torch::kBFloat16 || q.scalar_type() == torch::kFloat32,
                "theseus_gdn: expected bfloat16 or float32 q, k, v");
    for (const Tensor* x : {&q, &k, &v})
        TORCH_CHECK(x->is_cuda() && x->scalar_type() == q.scalar_type() && x->is_contiguous() && x->dim() == 4 &&
                        x->sizes() == q.sizes() && x->device() == q.device(),
                    "theseus_gdn: expected contiguous CUDA q, k, v [B,T,H,N] of one dtype");
    for (const Tensor* x : {&g, &beta})
        TORCH_CHECK(x->device() == q.device() && x->scalar_type() == torch::kFloat32 && x->is_contiguous() &&
                        x->sizes() == q.sizes().slice(0, 3),
                    "theseus_gdn: expected contiguous float32 g, beta [B,T,H]");
    TORCH_CHECK(!s0.defined() || (s0.device() == q.device() && s0.scalar_type() == torch::kFloat32 && s0.is_contiguous() &&
                                  s0.sizes() == at::IntArrayRef({q.size(0), q.size(2), q.size(3), q.size(3)})),
                "theseus_gdn: expected contiguous float32 state [B,H,N,N]");
}

struct Gdn : torch::autograd::Function<Gdn> {
    static variable_list forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& g,
                                 const Tensor& beta, const Tensor& s0, bool qk_l2norm) {
        ctx->set_materialize_grads(false);
        gdn_check(q, k, v, g, beta, s0);
        const Dims d(q);
        c10::OptionalDeviceGuard guard(q.device());
        const Tensor o = at::empty_like(q), sT = at::empty_like(s0), saved = at::empty(d.saved(), s0.options());
        const size_t need = theseus_gdn_forward_best_workspace_size(d.B, d.T, d.H, d.N, 1);
        const Tensor ws = scratch(need, q);
        raise_status(theseus_gdn_forward_train_ex(d.B, d.T, d.H, d.N, d.dt, qk_l2norm, ptr(q), ptr(k), ptr(v), fptr(g),
                                                  fptr(beta), fptr(s0), ptr(o), fptr(sT), fptr(saved), ptr(ws), need,
                                                  stream_of(q)),
                     "theseus_wkv7");
        ctx->save_for_backward({q, k, v, g, beta, saved});
        ctx->saved_data["qk_l2norm"] = qk_l2norm;
        return {o, sT};
    }
    static variable_list backward(AutogradContext* ctx, variable_list gr) {
        const variable_list s = ctx->get_saved_variables();
        const Tensor &q = s[0], &k = s[1], &v = s[2], &g = s[3], &beta = s[4], &saved = s[5];
        const Tensor dout = gr[0].defined() ? gr[0].to(q.scalar_type()).contiguous() : at::zeros_like(q);
        const Tensor dsT = gr[1].defined() ? float_rows(gr[1]) : Tensor();
        gdn_check(q, k, v, g, beta, dsT);
        const Dims d(q);
        TORCH_CHECK(dout.sizes() == q.sizes() && dout.device() == q.device(),
                    "theseus_gdn: expected a contiguous output gradient like q");
        TORCH_CHECK(saved.scalar_type() == torch::kFloat32 && saved.is_contiguous() && saved.device() == q.device() &&
                        saved.sizes() == at::IntArrayRef(d.saved()),
                    "theseus_gdn: invalid saved states");
        c10::OptionalDeviceGuard guard(q.device());
        variable_list o{at::empty_like(q), at::empty_like(q), at::empty_like(q), at::empty_like(g), at::empty_like(beta),
                        at::empty({d.B, d.H, d.N, d.N}, saved.options())};
        const size_t need = theseus_gdn_backward_workspace_size(d.B, d.T, d.H, d.N);
        const Tensor ws = scratch(need, q);
        raise_status(theseus_gdn_backward_ex(d.B, d.T, d.H, d.N, d.dt, ctx->saved_data["qk_l2norm"].toBool(), ptr(q),
                                             ptr(k), ptr(v), fptr(g), fptr(beta), fptr(saved), ptr(dout), fptr(dsT),
                                             ptr(o[0]), ptr(o[1]), ptr(o[2]), fptr(o[3]), fptr(o[4]), fptr(o[5]), ptr(ws),
                                             need, stream_of(q)),
                     "theseus_wkv7");
        o.emplace_back();  // (qk_l2norm)
        return o;
    }
};

std::pair<Tensor, Tensor> gdn(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& g, const Tensor& beta,
                              const Tensor& s0, bool qk_l2norm) {
    py::gil_scoped_release free;
    const variable_list o = Gdn::apply(q, k, v, g, beta, s0, qk_l2norm);
    return {o[0], o[1]};
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    m.def("wkv7", &wkv7, "(y, end state) of the recurrence, differentiable");
    m.def("gdn", &gdn, "(o, end state) of the gated delta rule with gradients, differentiable", py::arg("q"),
          py::arg("k"), py::arg("v"), py::arg("g"), py::arg("beta"), py::arg("s0"), py::arg("qk_l2norm") = false);
}
