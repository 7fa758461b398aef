// The host path of the operators in C++: argument checks, output and scratch allocation, the parameter structs of the C ABI
// and the autograd nodes.  Python only names the operators (mamba2/*.py).
//
// An eager call at the sizes of a short prompt or a decode step is bound by the host: the ctypes form of this code (attribute
// access on ~40 struct fields, view and stream objects, one Python autograd node per operator) took 25-60 us per operator,
// several times the kernels' own time.
//
// The library is not linked: its entry points come from the ctypes loader (bind()), so that both sides always use the
// build that _lib.load() opened.  Scratch comes from the caching allocator per call: it is ordered by the stream it was
// allocated on, so calls from several threads and streams never share it.
#include <torch/extension.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <ATen/hip/tunable/Tunable.h>
#include <c10/core/DeviceGuard.h>

#include <initializer_list>
#include <map>
#include <string>

#include "../../include/mamba2_hip.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// ----------------------------------------------------------------------------------------------- the library
#define M2_BOUND(F) \
    F(m2_last_error) F(m2_conv1d_fwd) F(m2_conv1d_prefill) F(m2_conv1d_bwd_workspace_bytes) F(m2_conv1d_bwd) F(m2_conv1d_bwd_partial) F(m2_ssd_chunk_states_bytes) \
    F(m2_ssd_fwd_workspace_bytes) F(m2_ssd_fwd_check) F(m2_ssd_fwd) F(m2_ssd_bwd_workspace_bytes) F(m2_ssd_bwd) F(m2_decode_workspace_bytes) \
    F(m2_decode_step) F(m2_decode_step_static) F(m2_core_norm_fwd_check) F(m2_rmsnorm_gated_fwd) F(m2_rmsnorm_gated_bwd_workspace_bytes) \
    F(m2_rmsnorm_gated_bwd) F(m2_core_norm_fwd) F(m2_core_norm_bwd_partial) F(m2_add_rmsnorm) F(m2_linear_small_fits) F(m2_linear_small) F(m2_decode_rows) F(m2_embed_rows) F(m2_decode_layer) F(m2_mixer_params) F(m2_param_sums) \
    F(m2_product_pays) F(m2_product_workspace_bytes) F(m2_product) \
    F(m2_product_pair_pays) F(m2_product_pair_workspace_bytes) F(m2_product_pair)
struct Lib {
#define M2_FIELD(name) decltype(&::name) name = nullptr;
    M2_BOUND(M2_FIELD)
#undef M2_FIELD
} lib;

std::vector<std::string> bound_names() {
#define M2_NAME(name) #name,
    return {M2_BOUND(M2_NAME)};
#undef M2_NAME
}

void bind(const std::map<std::string, uintptr_t>& addresses) {
#define M2_SET(name) lib.name = reinterpret_cast<decltype(lib.name)>(addresses.at(#name));
    M2_BOUND(M2_SET)
#undef M2_SET
}

void check(int rc, const char* what) {
    if (rc == M2_OK) return;
    const bool bad_argument = rc == M2_ERR_SHAPE || rc == M2_ERR_DTYPE || rc == M2_ERR_ALIGN || rc == M2_ERR_NULL;
    TORCH_CHECK_VALUE(!bad_argument, what, ": ", lib.m2_last_error(), " (code ", rc, ")");
    TORCH_CHECK(false, what, ": ", lib.m2_last_error(), " (code ", rc, ")");
}

// ----------------------------------------------------------------------------------------------- small helpers
// all on the one GPU whose stream the kernels go to
void require_gpu(std::initializer_list<const Tensor*> tensors) {
    const Tensor* first = nullptr;
    for (const Tensor* t : tensors) {
        if (!t || !t->defined()) continue;
        TORCH_CHECK(t->is_cuda(), "mamba2 HIP kernels need tensors on a GPU device (got ", t->device().str(), "); there is no CPU path");
        if (!first) first = t;
        TORCH_CHECK(t->device() == first->device(), "expected all tensors on one device, got ", first->device().str(), " and ", t->device().str());
    }
}

int dtype_code(const Tensor& t) {
    if (t.scalar_type() == at::kFloat) return M2_F32;
    if (t.scalar_type() == at::kBFloat16) return M2_BF16;
    TORCH_CHECK_VALUE(false, "unsupported dtype ", t.scalar_type(), ": the HIP kernels take float32 or bfloat16");
}

const Tensor& or_none(const OptTensor& t) {
    static const Tensor none;
    return t ? *t : none;
}

template <typename T = void> T* ptr(const Tensor& t) { return t.defined() ? static_cast<T*>(t.data_ptr()) : nullptr; }
char* at_column(const Tensor& t, int64_t column) { return static_cast<char*>(t.data_ptr()) + column * t.element_size(); }

// The body of an operator: autograd off, the tensors' device current, its stream at hand.
struct Scope {
    at::AutoDispatchBelowADInplaceOrView no_autograd;
    c10::OptionalDeviceGuard guard;
    void* stream;
    explicit Scope(const Tensor& t) : guard(t.device()) {
        stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream();
    }
};

// fp32 contiguous values of a parameter-like tensor (the tensor itself when it already is)
Tensor f32(const Tensor& t) { return t.defined() ? t.to(at::kFloat).contiguous() : t; }

Tensor scratch(size_t bytes, const Tensor& like) {
    return at::empty({static_cast<int64_t>(bytes)}, like.options().dtype(at::kByte));
}
// Several pieces of one scratch allocation, each on a 256-byte boundary: sizes first, then the pieces in the same order.
struct Pieces {
    size_t total = 0, used = 0;
    Tensor held;
    static size_t rounded(size_t bytes) { return (bytes + 255) / 256 * 256; }
    void want(size_t bytes) { total += rounded(bytes); }
    void allocate(const Tensor& like) { held = scratch(total, like); }
    void* take(size_t bytes) {
        TORCH_INTERNAL_ASSERT(used + rounded(bytes) <= total);
        char* at = static_cast<char*>(held.data_ptr()) + used;
        used += rounded(bytes);
        return at;
    }
};
Tensor empty_f32(at::IntArrayRef shape, const Tensor& like) { return at::empty(shape, like.options().dtype(at::kFloat)); }

// ----------------------------------------------------------------------------------------------- conv1d
struct Blc { int64_t b, l, c, sb, sl, sc; };
Blc blc(const Tensor& t, bool channels_last) {
    const int L = channels_last ? 1 : 2, C = channels_last ? 2 : 1;
    return {t.size(0), t.size(L), t.size(C), t.stride(0), t.stride(L), t.stride(C)};
}

void check_conv(const Tensor& input, const Tensor& weight, const Tensor& bias, bool channels_last) {
    TORCH_CHECK_VALUE(input.dim() == 3 && weight.dim() == 3 && weight.size(1) == 1, "expected input (B, C, L) or (B, L, C) and weight (C, 1, k)");
    TORCH_CHECK_VALUE(!bias.defined() || (bias.dim() == 1 && bias.size(0) == weight.size(0) && bias.scalar_type() == weight.scalar_type()),
                      "bias must have shape (C,) and the dtype of weight");
    require_gpu({&input, &weight, &bias});
    const int64_t channels = input.size(channels_last ? 2 : 1);
    TORCH_CHECK_VALUE(weight.size(0) == channels, "weight has ", weight.size(0), " channels, input has ", channels);
}

// x, y / dy and dx are given as (pointer, strides): columns of packed buffers need no view objects
struct Strided { void* p; int64_t sb, sl, sc; };
m2_conv1d_params conv_params(const Strided& x, const Tensor& w, const Tensor& bias, const Strided& y, int64_t b, int64_t l, int64_t c,
                             int dtype, int activation) {
    m2_conv1d_params p{};
    p.x = x.p; p.w = ptr(w); p.bias = ptr(bias);
    p.batch = b; p.seqlen = l; p.channels = c; p.k = static_cast<int32_t>(w.size(-1));
    p.x_stride_b = x.sb; p.x_stride_l = x.sl; p.x_stride_c = x.sc;
    p.y_stride_b = y.sb; p.y_stride_l = y.sl; p.y_stride_c = y.sc;
    p.dtype = dtype; p.param_dtype = dtype_code(w); p.activation = activation;
    return p;
}

Tensor conv1d_forward(const Tensor& input, const Tensor& weight, const OptTensor& bias_, int64_t activation, bool channels_last, const OptTensor& out) {
    const Tensor& bias = or_none(bias_);
    check_conv(input, weight, bias, channels_last);
    Scope scope(input);
    const Tensor w = weight.contiguous(), bi = bias.defined() ? bias.contiguous() : bias;
    Tensor y = out ? *out : at::empty(input.sizes(), input.options());
    const Blc xi = blc(input, channels_last), yi = blc(y, channels_last);
    m2_conv1d_params p = conv_params({ptr(input), xi.sb, xi.sl, xi.sc}, w, bi, {ptr(y), yi.sb, yi.sl, yi.sc}, xi.b, xi.l, xi.c,
                                     dtype_code(input), static_cast<int>(activation));
    p.y = ptr(y);
    check(lib.m2_conv1d_fwd(&p, scope.stream), "m2_conv1d_fwd");
    return y;
}

// Partial rows of a parameter's gradient, to be summed by a later launch (count == 0: there are none)
struct Partials { const float* rows = nullptr; int64_t count = 0; };

// the launch shared by the operator and the fused core; returns (dw, db).  later: where partials go that the caller will have summed;
// they lie in ws, of as many bytes as the library asks for
std::pair<Tensor, Tensor> launch_conv_bwd(const Strided& x, const Tensor& weight, const Tensor& bias, const Strided& dy, const Strided& dx,
                                          int64_t b, int64_t l, int64_t c, const Tensor& like, int activation, void* stream, Partials* later = nullptr,
                                          void* ws = nullptr) {
    const Tensor w = weight.contiguous(), bi = bias.defined() ? bias.contiguous() : bias;
    Tensor dw = at::empty(w.sizes(), w.options()), db = bi.defined() ? at::empty(bi.sizes(), bi.options()) : Tensor();
    m2_conv1d_params p = conv_params(x, w, bi, dy, b, l, c, dtype_code(like), activation);
    p.dy = dy.p; p.dx = dx.p; p.dw = ptr(dw); p.db = ptr(db);
    p.dx_stride_b = dx.sb; p.dx_stride_l = dx.sl; p.dx_stride_c = dx.sc;
    p.workspace_bytes = lib.m2_conv1d_bwd_workspace_bytes(b, l, c, p.k);
    Tensor own;
    if (!ws) { own = scratch(p.workspace_bytes, like); ws = ptr(own); }
    p.workspace = ws;
    if (later) {
        check(lib.m2_conv1d_bwd_partial(&p, &later->count, stream), "m2_conv1d_bwd");
        later->rows = static_cast<const float*>(ws);
    } else check(lib.m2_conv1d_bwd(&p, stream), "m2_conv1d_bwd");
    return {dw, db};
}

std::tuple<Tensor, Tensor, Tensor> conv1d_backward(const Tensor& input, const Tensor& weight, const OptTensor& bias_, const Tensor& d_output,
                                                   int64_t activation, bool channels_last, const OptTensor& out_dx) {
    const Tensor& bias = or_none(bias_);
    check_conv(input, weight, bias, channels_last);
    require_gpu({&d_output});
    Scope scope(input);
    const Tensor dy = d_output.to(input.scalar_type());
    Tensor dx = out_dx ? *out_dx : at::empty(input.sizes(), input.options());
    const Blc xi = blc(input, channels_last), gi = blc(dy, channels_last), di = blc(dx, channels_last);
    auto [dw, db] = launch_conv_bwd({ptr(input), xi.sb, xi.sl, xi.sc}, weight, bias, {ptr(dy), gi.sb, gi.sl, gi.sc}, {ptr(dx), di.sb, di.sl, di.sc},
                                    xi.b, xi.l, xi.c, input, static_cast<int>(activation), scope.stream);
    return {dx, dw, db};
}

// conv1d_grouped.py:265-292: forward(input, weight, bias, activation), backward -> (dinput, dweight, dbias)
struct ConvFn : torch::autograd::Function<ConvFn> {
    static Tensor forward(AutogradContext* ctx, const Tensor& input, const Tensor& weight, const OptTensor& bias, int64_t activation, bool channels_last) {
        ctx->save_for_backward({input, weight, or_none(bias)});
        ctx->saved_data["activation"] = activation;
        ctx->saved_data["channels_last"] = channels_last;
        return conv1d_forward(input, weight, bias, activation, channels_last, std::nullopt);
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const variable_list s = ctx->get_saved_variables();
        auto [dx, dw, db] = conv1d_backward(s[0], s[1], s[2].defined() ? OptTensor(s[2]) : std::nullopt, grads[0],
                                            ctx->saved_data["activation"].toInt(), ctx->saved_data["channels_last"].toBool(), std::nullopt);
        return {dx, dw, db, Tensor(), Tensor()};
    }
};
Tensor conv1d(const Tensor& input, const Tensor& weight, const OptTensor& bias, int64_t activation, bool channels_last) {
    check_conv(input, weight, or_none(bias), channels_last);
    return ConvFn::apply(input, weight, bias, activation, channels_last);
}

// ----------------------------------------------------------------------------------------------- SSD scan
void check_inner(const char* name, const Tensor& t) {
    TORCH_CHECK_VALUE(t.stride(-1) == 1 || t.size(-1) <= 1, name, ": innermost dimension must be contiguous (stride ", t.stride(-1), ")");
}

void check_ssd(const Tensor& dt, const Tensor& A, const Tensor& X, const Tensor& B, const Tensor& C, const Tensor& D, const Tensor& S0, const Tensor& dt_bias) {
    TORCH_CHECK_VALUE(X.dim() == 4 && B.dim() == 4 && C.dim() == 4 && dt.dim() == 3, "expected dt (b,l,h), X (b,l,h,p), B/C (b,l,g,n)");
    const int64_t b = X.size(0), l = X.size(1), h = X.size(2);
    TORCH_CHECK_VALUE(dt.size(0) == b && dt.size(1) == l && dt.size(2) == h, "dt shape ", dt.sizes(), " != (", b, ", ", l, ", ", h, ")");
    TORCH_CHECK_VALUE(B.sizes() == C.sizes() && B.size(0) == b && B.size(1) == l, "B ", B.sizes(), " / C ", C.sizes(), " do not match X ", X.sizes());
    TORCH_CHECK_VALUE(B.size(2) > 0 && h % B.size(2) == 0, "n_heads ", h, " not divisible by n_groups ", B.size(2));
    TORCH_CHECK_VALUE(A.dim() == 1 && A.size(0) == h && (!D.defined() || (D.dim() == 1 && D.size(0) == h)), "A and D must have shape (n_heads,)");
    TORCH_CHECK_VALUE(B.scalar_type() == X.scalar_type() && C.scalar_type() == X.scalar_type(), "X, B and C must share one dtype");
    TORCH_CHECK_VALUE(dt.scalar_type() == X.scalar_type() || dt.scalar_type() == at::kFloat, "dt must be float32 or have the dtype of X");
    check_inner("X", X); check_inner("B", B); check_inner("C", C); check_inner("dt", dt);
    TORCH_CHECK_VALUE(!S0.defined() || (S0.dim() == 4 && S0.size(0) == b && S0.size(1) == h && S0.size(2) == X.size(3) && S0.size(3) == B.size(3)),
                      "initial_state must have shape (b, h, p, n)");
    TORCH_CHECK_VALUE(!dt_bias.defined() || (dt_bias.dim() == 1 && dt_bias.size(0) == h), "dt_bias must have shape (n_heads,)");
    require_gpu({&dt, &A, &X, &B, &C, &D, &S0, &dt_bias});
}

// A, D, dt_bias: fp32 contiguous (or undefined)
m2_ssd_params ssd_params(const Tensor& dt, const Tensor& A, const Tensor& X, const Tensor& B, const Tensor& C, const Tensor& D, const Tensor& dt_bias) {
    m2_ssd_params p{};
    p.x = ptr(X); p.dt = ptr(dt); p.A = ptr<float>(A); p.B = ptr(B); p.C = ptr(C); p.D = ptr<float>(D); p.dt_bias = ptr<float>(dt_bias);
    p.batch = X.size(0); p.seqlen = X.size(1); p.nheads = X.size(2); p.headdim = X.size(3); p.dstate = B.size(3); p.ngroups = B.size(2);
    p.x_stride_b = X.stride(0); p.x_stride_l = X.stride(1); p.x_stride_h = X.stride(2);
    p.dt_stride_b = dt.stride(0); p.dt_stride_l = dt.stride(1);
    p.B_stride_b = B.stride(0); p.B_stride_l = B.stride(1); p.B_stride_g = B.stride(2);
    p.C_stride_b = C.stride(0); p.C_stride_l = C.stride(1); p.C_stride_g = C.stride(2);
    p.dtype = dtype_code(X); p.dt_dtype = dtype_code(dt);
    return p;
}

Tensor alloc_chunk_states(const Tensor& dt, const Tensor& A, const Tensor& X, const Tensor& B, const Tensor& C) {
    const m2_ssd_params p = ssd_params(dt, A, X, B, C, Tensor(), Tensor());
    return scratch(lib.m2_ssd_chunk_states_bytes(&p), X);
}

void* chunk_states_ptr(const m2_ssd_params& p, const Tensor& states) {
    if (!states.defined()) return nullptr;
    const size_t need = lib.m2_ssd_chunk_states_bytes(&p);
    TORCH_CHECK_VALUE(states.is_contiguous() && static_cast<size_t>(states.numel() * states.element_size()) == need,
                      "chunk_states must be a contiguous buffer of ", need, " bytes (see alloc_chunk_states)");
    return ptr(states);
}

void launch_ssd_fwd(m2_ssd_params& p, const Tensor& like, void* stream) {
    p.workspace_bytes = lib.m2_ssd_fwd_workspace_bytes(&p);
    const Tensor ws = scratch(p.workspace_bytes, like);
    p.workspace = ptr(ws);
    check(lib.m2_ssd_fwd(&p, stream), "m2_ssd_fwd");
}
void launch_ssd_bwd(m2_ssd_params& p, const Tensor& like, void* stream) {
    const Tensor ws = scratch(p.workspace_bytes = lib.m2_ssd_bwd_workspace_bytes(&p), like);
    p.workspace = ptr(ws);
    check(lib.m2_ssd_bwd(&p, stream), "m2_ssd_bwd");
}

std::tuple<Tensor, Tensor> ssd_forward(const Tensor& dt, const Tensor& A, const Tensor& X, const Tensor& B, const Tensor& C, const OptTensor& D_,
                                       const OptTensor& S0_, bool want_final_state, const OptTensor& states, const OptTensor& dt_bias_) {
    check_ssd(dt, A, X, B, C, or_none(D_), or_none(S0_), or_none(dt_bias_));
    Scope scope(X);
    const Tensor A32 = f32(A), D32 = f32(or_none(D_)), S0 = f32(or_none(S0_)), bias = f32(or_none(dt_bias_));
    Tensor Y = at::empty(X.sizes(), X.options());
    Tensor S = want_final_state ? empty_f32({X.size(0), X.size(2), X.size(3), B.size(3)}, X) : Tensor();
    m2_ssd_params p = ssd_params(dt, A32, X, B, C, D32, bias);
    p.initial_state = ptr<float>(S0); p.final_state = ptr<float>(S); p.y = ptr(Y);
    p.chunk_states = chunk_states_ptr(p, or_none(states));
    p.y_stride_b = Y.stride(0); p.y_stride_l = Y.stride(1); p.y_stride_h = Y.stride(2);
    launch_ssd_fwd(p, X, scope.stream);
    return {Y, S};
}

struct SsdGrads { Tensor ddt, dA, dX, dB, dC, dD, dS0, d_bias; };
SsdGrads ssd_backward_impl(const Tensor& dt, const Tensor& A, const Tensor& X, const Tensor& B, const Tensor& C, const Tensor& D, const Tensor& dY_,
                           const Tensor& S0_, const Tensor& dSf_, bool want_dinitial, const Tensor& out_dX, const Tensor& out_dB,
                           const Tensor& out_dC, const Tensor& states, const Tensor& dt_bias, const Tensor& out_ddt) {
    check_ssd(dt, A, X, B, C, D, S0_, dt_bias);
    require_gpu({&dY_, &dSf_});
    Scope scope(X);
    const int64_t b = X.size(0), l = X.size(1), h = X.size(2), hd = X.size(3), g = B.size(2), n = B.size(3);
    const Tensor A32 = f32(A), D32 = f32(D), S0 = f32(S0_), dSf = f32(dSf_), bias = f32(dt_bias);
    // rows of dy are read as 16-byte vectors where they lie
    Tensor dY = dY_;
    if (dY.scalar_type() != X.scalar_type()) dY = dY.to(X.scalar_type());
    const int64_t es = dY.element_size();
    if (dY.stride(-1) != 1 || (dY.stride(0) * es) % 16 || (dY.stride(1) * es) % 16 || (dY.stride(2) * es) % 16 ||
        reinterpret_cast<uintptr_t>(dY.data_ptr()) % 16)
        dY = dY.clone(at::MemoryFormat::Contiguous);
    TORCH_CHECK_VALUE(!out_ddt.defined() || (out_ddt.sizes() == dt.sizes() && out_ddt.scalar_type() == dt.scalar_type() && out_ddt.stride(-1) == 1),
                      "out_ddt must have the shape and dtype of dt, heads contiguous");
    SsdGrads r;
    r.ddt = out_ddt.defined() ? out_ddt : at::empty({b, l, h}, dt.options());
    r.dX = out_dX.defined() ? out_dX : at::empty({b, l, h, hd}, X.options());
    r.dB = out_dB.defined() ? out_dB : at::empty({b, l, g, n}, B.options());
    r.dC = out_dC.defined() ? out_dC : at::empty({b, l, g, n}, C.options());
    // the per-head gradients share one allocation
    const Tensor heads = empty_f32({3, h}, X);
    r.dA = heads.select(0, 0);
    if (D.defined()) r.dD = heads.select(0, 1);
    if (dt_bias.defined()) r.d_bias = heads.select(0, 2);
    if (want_dinitial) r.dS0 = empty_f32({b, h, hd, n}, X);
    m2_ssd_params p = ssd_params(dt, A32, X, B, C, D32, bias);
    p.initial_state = ptr<float>(S0); p.dy = ptr(dY); p.d_final_state = ptr<float>(dSf);
    p.chunk_states = chunk_states_ptr(p, states);
    p.dx = ptr(r.dX); p.ddt = ptr(r.ddt); p.dA = ptr<float>(r.dA); p.dB = ptr(r.dB); p.dC = ptr(r.dC); p.dD = ptr<float>(r.dD);
    p.d_initial_state = ptr<float>(r.dS0); p.d_dt_bias = ptr<float>(r.d_bias);
    p.dy_stride_b = dY.stride(0); p.dy_stride_l = dY.stride(1); p.dy_stride_h = dY.stride(2);
    p.dx_stride_b = r.dX.stride(0); p.dx_stride_l = r.dX.stride(1); p.dx_stride_h = r.dX.stride(2);
    p.ddt_stride_b = r.ddt.stride(0); p.ddt_stride_l = r.ddt.stride(1);
    p.dB_stride_b = r.dB.stride(0); p.dB_stride_l = r.dB.stride(1); p.dB_stride_g = r.dB.stride(2);
    p.dC_stride_b = r.dC.stride(0); p.dC_stride_l = r.dC.stride(1); p.dC_stride_g = r.dC.stride(2);
    launch_ssd_bwd(p, X, scope.stream);
    return r;
}

py::object ssd_backward(const Tensor& dt, const Tensor& A, const Tensor& X, const Tensor& B, const Tensor& C, const OptTensor& D, const Tensor& dY,
                        const OptTensor& S0, const OptTensor& dSf, bool want_dinitial, const OptTensor& out_dX, const OptTensor& out_dB,
                        const OptTensor& out_dC, const OptTensor& states, const OptTensor& dt_bias, const OptTensor& out_ddt) {
    const SsdGrads r = ssd_backward_impl(dt, A, X, B, C, or_none(D), dY, or_none(S0), or_none(dSf), want_dinitial, or_none(out_dX), or_none(out_dB),
                                         or_none(out_dC), or_none(states), or_none(dt_bias), or_none(out_ddt));
    if (dt_bias) return py::make_tuple(r.ddt, r.dA, r.dX, r.dB, r.dC, r.dD, r.dS0, r.d_bias);
    return py::make_tuple(r.ddt, r.dA, r.dX, r.dB, r.dC, r.dD, r.dS0);
}

// mamba2_kernel.py:488-519: forward(dt, A, X, B, C, D) -> Y, backward -> (ddt, dA, dX, dB, dC, dD), with the initial and the
// final state as extensions.  The chunk states are kept for the backward when one can follow.
struct SsdFn : torch::autograd::Function<SsdFn> {
    static variable_list forward(AutogradContext* ctx, const Tensor& dt, const Tensor& A, const Tensor& X, const Tensor& B, const Tensor& C,
                                 const OptTensor& D, const OptTensor& S0, bool return_final_state, bool keep_states) {
        OptTensor states;
        if (keep_states && X.numel() > 0) states = alloc_chunk_states(dt, A, X, B, C);
        auto [Y, S] = ssd_forward(dt, A, X, B, C, D, S0, return_final_state, states, std::nullopt);
        ctx->save_for_backward({dt, A, X, B, C, or_none(D), or_none(S0), or_none(states)});
        ctx->set_materialize_grads(false);
        if (return_final_state) return {Y, S};
        return {Y};
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const variable_list s = ctx->get_saved_variables();
        const Tensor &dt = s[0], &A = s[1], &X = s[2], &D = s[5], &S0 = s[6];
        const Tensor dSf = grads.size() > 1 ? grads[1] : Tensor();
        variable_list out(9);
        if (!grads[0].defined() && !dSf.defined()) return out;
        const Tensor dY = grads[0].defined() ? grads[0] : at::zeros(X.sizes(), X.options());
        const SsdGrads r = ssd_backward_impl(dt, A, X, s[3], s[4], D, dY, S0, dSf, S0.defined() && ctx->needs_input_grad(S0.defined() && D.defined() ? 6 : 5),
                                             Tensor(), Tensor(), Tensor(), s[7], Tensor(), Tensor());
        out[0] = r.ddt; out[1] = r.dA.to(A.scalar_type()); out[2] = r.dX; out[3] = r.dB; out[4] = r.dC;
        if (D.defined()) out[5] = r.dD.to(D.scalar_type());
        out[6] = r.dS0;
        return out;
    }
};
py::object mamba2_kernel(const Tensor& dt, const Tensor& A, const Tensor& X, const Tensor& B, const Tensor& C, const OptTensor& D, const OptTensor& S0,
                         bool return_final_state, bool save_states) {
    check_ssd(dt, A, X, B, C, or_none(D), or_none(S0), Tensor());
    bool needs = false;
    if (at::GradMode::is_enabled())
        for (const Tensor* t : {&dt, &A, &X, &B, &C, &or_none(D), &or_none(S0)}) needs |= t->defined() && t->requires_grad();
    const variable_list r = SsdFn::apply(dt, A, X, B, C, D, S0, return_final_state, save_states && needs);
    if (return_final_state) return py::make_tuple(r[0], r[1]);
    return py::cast(r[0]);
}

// ----------------------------------------------------------------------------------------------- gated RMSNorm
// (rows, channels, row stride) of a (..., channels) tensor whose leading dimensions collapse to one stride
struct Rows { int64_t rows, channels, stride; };
Rows rows2d(const Tensor& t, const char* name) {
    const int64_t ch = t.size(-1);
    TORCH_CHECK_VALUE(t.stride(-1) == 1 || ch <= 1, name, ": innermost dimension must be contiguous");
    if (t.dim() == 1) return {1, ch, ch};
    const int64_t sr = t.stride(-2);
    int64_t expect = sr;
    for (int64_t k = t.dim() - 2; k >= 0; --k) {
        TORCH_CHECK_VALUE(t.size(k) == 1 || t.stride(k) == expect, name, ": rows are not evenly strided (shape ", t.sizes(), ", strides ", t.strides(), ")");
        expect *= t.size(k);
    }
    return {ch ? t.numel() / ch : 0, ch, sr};
}
// rows that can be read as 16-byte vectors where they lie; others are copied once
bool vec_ok(const Tensor& t) {
    const Rows r = rows2d(t, "tensor");
    return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0 && (r.stride * t.element_size()) % 16 == 0;
}
Tensor aligned(const Tensor& t) { return vec_ok(t) ? t : t.clone(at::MemoryFormat::Contiguous); }

m2_rmsnorm_params norm_params(const Tensor& x, const Tensor& z, const Tensor& w32, int64_t n_groups, double eps) {
    m2_rmsnorm_params p{};
    const Rows xr = rows2d(x, "x");
    p.x = ptr(x); p.x_stride_row = xr.stride;
    if (z.defined()) { p.z = ptr(z); p.z_stride_row = rows2d(z, "z").stride; }
    p.rows = xr.rows; p.channels = xr.channels; p.n_groups = static_cast<int32_t>(n_groups);
    p.dtype = dtype_code(x); p.eps = static_cast<float>(eps); p.weight = ptr<float>(w32);
    return p;
}
void check_norm(const Tensor& x, const Tensor& z) {
    TORCH_CHECK_VALUE(!z.defined() || (z.sizes() == x.sizes() && z.scalar_type() == x.scalar_type()), "rmsnorm_gated: z must have the shape and dtype of x");
}

Tensor rmsnorm_forward(const Tensor& x_, const OptTensor& z_, const Tensor& weight, int64_t n_groups, double eps, at::ScalarType out_dtype) {
    require_gpu({&x_, &or_none(z_), &weight});
    Scope scope(x_);
    check_norm(x_, or_none(z_));
    TORCH_CHECK_VALUE(out_dtype == at::kFloat || out_dtype == x_.scalar_type(), "rmsnorm_gated: out_dtype must be float32 or the dtype of x");
    const Tensor x = aligned(x_), z = z_ ? aligned(*z_) : Tensor(), w32 = f32(weight);      // rows that the kernel does not read where they lie: copied
    m2_rmsnorm_params p = norm_params(x, z, w32, n_groups, eps);
    const Tensor out = at::empty(x.sizes(), x.options().dtype(out_dtype));
    p.out = ptr(out); p.out_stride_row = x.size(-1); p.out_f32 = out_dtype == at::kFloat;
    check(lib.m2_rmsnorm_gated_fwd(&p, scope.stream), "m2_rmsnorm_gated_fwd");
    return out;
}

// the gradient of a norm's output as its kernel reads it
Tensor norm_rows(const Tensor& d_out, at::ScalarType dtype) {
    Tensor g = d_out.to(dtype);
    if (g.stride(-1) != 1 || !vec_ok(g)) g = g.clone(at::MemoryFormat::Contiguous);
    return g;
}

std::tuple<Tensor, Tensor, Tensor> rmsnorm_backward(const Tensor& x_, const OptTensor& z_, const Tensor& weight, const Tensor& d_out, int64_t n_groups,
                                                    double eps, const OptTensor& out_dz) {
    require_gpu({&x_, &or_none(z_), &weight, &d_out});
    check_norm(x_, or_none(z_));
    Scope scope(x_);
    const Tensor g = norm_rows(d_out, x_.scalar_type());
    const Tensor x = aligned(x_), z = z_ ? aligned(*z_) : Tensor(), w32 = f32(weight);
    m2_rmsnorm_params p = norm_params(x, z, w32, n_groups, eps);
    p.d_out = ptr(g); p.d_out_stride_row = rows2d(g, "d_out").stride;
    Tensor dx = at::empty(x.sizes(), x.options()), dz;
    p.dx = ptr(dx); p.dx_stride_row = x.size(-1);
    if (z.defined()) {
        TORCH_CHECK_VALUE(!out_dz || (out_dz->scalar_type() == x.scalar_type() && out_dz->sizes() == x.sizes()),
                          "rmsnorm_gated_bwd: out_dz must have the shape and dtype of x");
        dz = out_dz && vec_ok(*out_dz) ? *out_dz : at::empty(x.sizes(), x.options());
        p.dz = ptr(dz); p.dz_stride_row = rows2d(dz, "out_dz").stride;
    }
    Tensor dw = empty_f32({x.size(-1)}, x);
    p.d_weight = ptr<float>(dw);
    p.workspace_bytes = lib.m2_rmsnorm_gated_bwd_workspace_bytes(p.rows, p.channels, p.n_groups, p.dtype);
    const Tensor ws = scratch(p.workspace_bytes, x);
    p.workspace = ptr(ws);
    check(lib.m2_rmsnorm_gated_bwd(&p, scope.stream), "m2_rmsnorm_gated_bwd");
    if (z.defined() && out_dz && !dz.is_same(*out_dz)) {
        out_dz->copy_(dz);
        dz = *out_dz;
    }
    return {dx, dw, dz};
}

struct NormFn : torch::autograd::Function<NormFn> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x, const OptTensor& z, const Tensor& weight, int64_t n_groups, double eps, at::ScalarType out_dtype) {
        ctx->save_for_backward({x, or_none(z), weight});
        ctx->saved_data["n_groups"] = n_groups;
        ctx->saved_data["eps"] = eps;
        return rmsnorm_forward(x, z, weight, n_groups, eps, out_dtype);
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const variable_list s = ctx->get_saved_variables();
        auto [dx, dw, dz] = rmsnorm_backward(s[0], s[1].defined() ? OptTensor(s[1]) : std::nullopt, s[2], grads[0], ctx->saved_data["n_groups"].toInt(),
                                             ctx->saved_data["eps"].toDouble(), std::nullopt);
        return {dx, dz, dw.to(s[2].scalar_type()), Tensor(), Tensor(), Tensor()};
    }
};
Tensor rmsnorm(const Tensor& x, const OptTensor& z, const Tensor& weight, int64_t n_groups, double eps, at::ScalarType out_dtype) {
    return NormFn::apply(x, z, weight, n_groups, eps, out_dtype);
}

Tensor add_rmsnorm(const Tensor& residual, const OptTensor& delta_, const Tensor& w32, double eps, at::ScalarType out_dtype) {
    require_gpu({&residual, &or_none(delta_), &w32});
    TORCH_CHECK_VALUE(residual.scalar_type() == at::kFloat && residual.is_contiguous(), "add_rmsnorm_: the residual stream must be contiguous float32");
    Tensor delta = or_none(delta_);
    TORCH_CHECK_VALUE(!delta.defined() || (delta.sizes() == residual.sizes() && delta.scalar_type() == out_dtype),
                      "add_rmsnorm_: delta must have the residual's shape and the output dtype");
    Scope scope(residual);
    const Rows r = rows2d(residual, "residual");
    if (delta.defined() && delta.stride(-1) != 1) delta = delta.contiguous();
    Tensor out = at::empty(residual.sizes(), residual.options().dtype(out_dtype));
    check(lib.m2_add_rmsnorm(ptr<float>(residual), r.stride, ptr(delta), delta.defined() ? rows2d(delta, "delta").stride : 0, ptr<float>(w32), ptr(out),
                             r.channels, r.rows, r.channels, static_cast<float>(eps), dtype_code(out), scope.stream), "m2_add_rmsnorm");
    return out;
}

// ----------------------------------------------------------------------------------------------- fused mixer core
constexpr double kNormEps = 1e-5;      // fixed in the reference's fused kernel (fused_kernel.py:254)

// Heads of a core of d channels.  The scan writes whole heads only: channels past the last one would stay as they were allocated.
int64_t core_heads(int64_t g, int64_t n, int64_t d, int64_t p) {
    TORCH_CHECK_VALUE(p > 0 && d >= 0 && d % p == 0, "intermediate_size ", d, " is not a multiple of head_dim ", p);
    const int64_t h = d / p;
    TORCH_CHECK_VALUE(g > 0 && h % g == 0, "n_heads ", h, " not divisible by n_groups ", g);
    TORCH_CHECK_VALUE(n > 0, "ssm_state_size ", n, " must be positive");
    return h;
}

// [z | xBC | dt] columns of the packed projection output; the kernels read them where they lie
struct Packed {
    Tensor zx;
    int64_t b, l, h, g, n, d, p, conv, sb, sl;
    Packed(const Tensor& t, int64_t g_, int64_t n_, int64_t d_, int64_t p_) : g(g_), n(n_), d(d_), p(p_) {
        TORCH_CHECK_VALUE(t.dim() == 3, "zxBCdt must be (b, l, width)");
        h = core_heads(g, n, d, p); conv = d + 2 * g * n;
        TORCH_CHECK_VALUE(t.size(2) == d + conv + h, "zxBCdt width ", t.size(2), " != 2*d_inner + 2*g*n + h = ", d + conv + h);
        const bool even = t.stride(2) == 1 && (t.size(0) <= 1 || t.stride(0) == t.size(1) * t.stride(1));
        zx = even ? t : t.contiguous();
        // One token per sequence: contiguous() looks at no stride of a dimension of size one and returns a transposed time-first buffer,
        // say, as it is.  Its rows are a width apart, and so is "the next token" to whoever takes the token stride for that of the rows.
        if (!even && t.size(1) == 1) zx = zx.as_strided(zx.sizes(), {zx.size(2), zx.size(2), 1});
        b = zx.size(0); l = zx.size(1); sb = zx.stride(0); sl = zx.stride(1);
    }
    Strided xBC() const { return {at_column(zx, d), sb, sl, 1}; }
};

// The per-head and per-channel parameters in fp32, contiguous.  As pointers: the whole layer holds them in one buffer, and a view of
// a part of it costs the host more than a launch's arguments.
struct CoreParams { const float *A, *D, *dt_bias, *norm_w; };
CoreParams core_params(const Tensor& A, const Tensor& D, const Tensor& dt_bias, const Tensor& norm_w) {
    return {ptr<float>(A), ptr<float>(D), ptr<float>(dt_bias), ptr<float>(norm_w)};
}

// the norm's parameters: the scan's output, gated by z, per group.  z is read where it lies, on whatever element a row of the packed
// projection starts (a copy into aligned rows in front of the forward and of the backward was a tenth of a core with an odd number of
// heads: 22 of 222 us for a prompt of 13115 tokens with 13 heads of 128).
m2_rmsnorm_params core_norm_params(const Packed& k, const CoreParams& w, const void* scan_out) {
    m2_rmsnorm_params p{};
    p.x = scan_out; p.x_stride_row = k.d; p.z = ptr(k.zx); p.z_stride_row = k.sl;
    p.rows = k.b * k.l; p.channels = k.d; p.n_groups = static_cast<int32_t>(k.g);
    p.dtype = dtype_code(k.zx); p.eps = static_cast<float>(kNormEps); p.weight = w.norm_w;
    return p;
}

// the scan's parameters with x, B and C as columns of the packed conv output
m2_ssd_params core_ssd_params(const Packed& k, const Tensor& conv_out, const CoreParams& w) {
    m2_ssd_params p{};
    const int64_t sb = conv_out.stride(0), sl = conv_out.stride(1);
    p.x = ptr(conv_out); p.B = at_column(conv_out, k.d); p.C = at_column(conv_out, k.d + k.g * k.n); p.dt = at_column(k.zx, k.d + k.conv);
    p.A = w.A; p.D = w.D; p.dt_bias = w.dt_bias;
    p.batch = k.b; p.seqlen = k.l; p.nheads = k.h; p.headdim = k.p; p.dstate = k.n; p.ngroups = k.g;
    p.x_stride_b = p.B_stride_b = p.C_stride_b = sb;
    p.x_stride_l = p.B_stride_l = p.C_stride_l = sl;
    p.x_stride_h = k.p; p.B_stride_g = p.C_stride_g = k.n;
    p.dt_stride_b = k.sb; p.dt_stride_l = k.sl;
    p.dtype = p.dt_dtype = dtype_code(conv_out);
    return p;
}

void check_core(const Packed& k, const Tensor& A, const Tensor& D, const Tensor& conv_w, const Tensor& conv_b, const Tensor& dt_bias, const Tensor& norm_w) {
    require_gpu({&k.zx, &A, &D, &conv_w, &conv_b, &dt_bias, &norm_w});
    TORCH_CHECK_VALUE(A.dim() == 1 && A.size(0) == k.h && (!D.defined() || (D.dim() == 1 && D.size(0) == k.h)), "A and D must have shape (n_heads,)");
    TORCH_CHECK_VALUE(dt_bias.dim() == 1 && dt_bias.size(0) == k.h, "dt_bias must have shape (n_heads,)");
    TORCH_CHECK_VALUE(norm_w.dim() == 1 && norm_w.size(0) == k.d, "norm_weight must have shape (d_inner,)");
    TORCH_CHECK_VALUE(conv_w.dim() == 3 && conv_w.size(0) == k.conv && conv_w.size(1) == 1, "conv1d_weight must be (", k.conv, ", 1, k)");
    TORCH_CHECK_VALUE(!conv_b.defined() || (conv_b.dim() == 1 && conv_b.size(0) == k.conv && conv_b.scalar_type() == conv_w.scalar_type()),
                      "bias must have shape (C,) and the dtype of weight");
}

struct CoreOut { Tensor norm_out, conv_out, scan_out, states; };
// want_norm false: only what the backward needs (conv output, scan output, chunk states).
CoreOut core_forward(const Packed& k, const CoreParams& params, const Tensor& conv_w, const Tensor& conv_b, bool keep_states, bool want_norm, void* stream) {
    CoreOut r;
    r.conv_out = at::empty({k.b, k.l, k.conv}, k.zx.options());
    const Tensor w = conv_w.contiguous(), bi = conv_b.defined() ? conv_b.contiguous() : conv_b;
    m2_conv1d_params c = conv_params(k.xBC(), w, bi, {ptr(r.conv_out), k.l * k.conv, k.conv, 1}, k.b, k.l, k.conv, dtype_code(k.zx), M2_ACT_SILU);
    c.y = ptr(r.conv_out);
    check(lib.m2_conv1d_fwd(&c, stream), "m2_conv1d_fwd");
    m2_ssd_params p = core_ssd_params(k, r.conv_out, params);
    if (keep_states && k.zx.numel() > 0) {
        r.states = scratch(lib.m2_ssd_chunk_states_bytes(&p), k.zx);
        p.chunk_states = ptr(r.states);
    }
    r.scan_out = at::empty({k.b, k.l, k.d}, k.zx.options());
    p.y = ptr(r.scan_out); p.y_stride_b = k.l * k.d; p.y_stride_l = k.d; p.y_stride_h = k.p;
    launch_ssd_fwd(p, k.zx, stream);
    if (want_norm) {
        m2_rmsnorm_params q = core_norm_params(k, params, ptr(r.scan_out));
        r.norm_out = at::empty({k.b, k.l, k.d}, k.zx.options());
        q.out = ptr(r.norm_out); q.out_stride_row = k.d;
        check(lib.m2_core_norm_fwd(&q, stream), "m2_core_norm_fwd");
    }
    return r;
}

// types that the kernels for the small parameters read and write
bool casts(const Tensor& t) { return t.scalar_type() == at::kFloat || t.scalar_type() == at::kBFloat16; }

struct CoreGrads {
    Tensor zx, heads, conv_w, conv_b, norm_w;      // heads: rows of A, dt_bias and D, unless they went into head_grads
    Tensor head(int64_t row, const Tensor& param) const { return heads.select(0, row).to(param.scalar_type()); }
};
// The packed gradient has rows of whole 128-byte cache lines (10576 columns of bf16 are 165.25 lines, and every wave-wide
// access to a column slice of such a buffer straddles two lines in three rows out of four); its consumers take a leading
// dimension.
// The sums of the norm weight's and the conv's partials run in one launch at the end, the former into norm_param's type; with
// head_grads (of A_log, D and dt_bias, in their types) it also leaves those.
CoreGrads core_backward(const Packed& k, const Tensor& d_out_, const CoreParams& w, const Tensor& conv_w, const Tensor& conv_b, const Tensor& conv_out,
                        const Tensor& scan_out, const Tensor& states, const Tensor& norm_param, const variable_list& head_grads, void* stream) {
    CoreGrads r;
    Partials norm_sums, conv_rows;
    const int64_t width = k.zx.size(2), per_line = 128 / k.zx.element_size(), pitch = (width + per_line - 1) / per_line * per_line;
    r.zx = at::empty({k.b, k.l, pitch}, k.zx.options());
    if (pitch != width) r.zx = r.zx.narrow(2, 0, width);
    char* const d_zx = static_cast<char*>(r.zx.data_ptr());
    const Tensor d_out = norm_rows(d_out_, k.zx.scalar_type());
    const bool to_heads = !head_grads.empty();
    require_gpu({&d_out, &scan_out, &conv_out});
    TORCH_CHECK_VALUE(scan_out.dim() == 3 && scan_out.size(0) == k.b && scan_out.size(1) == k.l && scan_out.size(2) == k.d &&
                          scan_out.scalar_type() == k.zx.scalar_type(), "scan_out must be (b, l, d_inner) in the dtype of zxBCdt");
    const Tensor scanned = aligned(scan_out);
    m2_rmsnorm_params q = core_norm_params(k, w, ptr(scanned));
    q.x_stride_row = rows2d(scanned, "scan_out").stride;
    m2_ssd_params p = core_ssd_params(k, conv_out, w);
    p.chunk_states = chunk_states_ptr(p, states);
    p.dy_stride_b = k.l * k.d; p.dy_stride_l = k.d; p.dy_stride_h = k.p;
    p.dx_stride_b = p.dB_stride_b = p.dC_stride_b = k.l * k.conv;
    p.dx_stride_l = p.dB_stride_l = p.dC_stride_l = k.conv;
    p.dx_stride_h = k.p; p.dB_stride_g = p.dC_stride_g = k.n;
    p.ddt_stride_b = k.l * pitch; p.ddt_stride_l = pitch;
    const size_t es = k.zx.element_size(), d_scan_bytes = static_cast<size_t>(k.b * k.l * k.d) * es, d_conv_bytes = static_cast<size_t>(k.b * k.l * k.conv) * es,
                 heads_bytes = to_heads ? static_cast<size_t>(3 * k.h) * 4 : 0, conv_bytes = lib.m2_conv1d_bwd_workspace_bytes(k.b, k.l, k.conv, conv_w.size(2));
    q.workspace_bytes = lib.m2_rmsnorm_gated_bwd_workspace_bytes(q.rows, q.channels, q.n_groups, q.dtype);
    p.workspace_bytes = lib.m2_ssd_bwd_workspace_bytes(&p);
    Pieces pieces;      // everything that does not leave this function, in one allocation
    for (const size_t bytes : {d_scan_bytes, d_conv_bytes, heads_bytes, conv_bytes, q.workspace_bytes, p.workspace_bytes}) pieces.want(bytes);
    pieces.allocate(k.zx);
    void* const d_scan = pieces.take(d_scan_bytes);
    char* const d_conv = static_cast<char*>(pieces.take(d_conv_bytes));
    if (!to_heads) r.heads = empty_f32({3, k.h}, k.zx);
    float* const heads = to_heads ? static_cast<float*>(pieces.take(heads_bytes)) : ptr<float>(r.heads);
    void* const conv_ws = pieces.take(conv_bytes);
    // norm: dz into its columns of r.zx
    q.d_out = ptr(d_out); q.d_out_stride_row = rows2d(d_out, "d_out").stride;
    q.dx = d_scan; q.dx_stride_row = k.d; q.dz = d_zx; q.dz_stride_row = pitch;
    q.workspace = pieces.take(q.workspace_bytes);
    check(lib.m2_core_norm_bwd_partial(&q, &norm_sums.count, stream), "m2_core_norm_bwd");
    norm_sums.rows = static_cast<const float*>(q.workspace);
    // the scan's gradients leave as one packed [dx | dB | dC] buffer, that of the raw dt in its columns of r.zx
    p.dy = d_scan; p.dx = d_conv; p.dB = d_conv + k.d * es; p.dC = d_conv + (k.d + k.g * k.n) * es; p.ddt = d_zx + (k.d + k.conv) * es;
    p.dA = heads; p.d_dt_bias = heads + k.h; p.dD = w.D ? heads + 2 * k.h : nullptr;
    p.workspace = pieces.take(p.workspace_bytes);
    check(lib.m2_ssd_bwd(&p, stream), "m2_ssd_bwd");
    std::tie(r.conv_w, r.conv_b) = launch_conv_bwd(k.xBC(), conv_w, conv_b, {d_conv, k.l * k.conv, k.conv, 1}, {d_zx + k.d * es, k.l * pitch, pitch, 1}, k.b, k.l,
                                                   k.conv, k.zx, M2_ACT_SILU, stream, &conv_rows, conv_ws);
    r.norm_w = at::empty({k.d}, casts(norm_param) ? norm_param.options() : norm_param.options().dtype(at::kFloat));
    auto head = [&](size_t i) { return to_heads && head_grads[i].defined() ? ptr(head_grads[i]) : nullptr; };
    auto head_type = [&](size_t i) { return to_heads && head_grads[i].defined() ? dtype_code(head_grads[i]) : M2_F32; };
    check(lib.m2_param_sums(norm_sums.rows, norm_sums.count, k.d, ptr(r.norm_w), dtype_code(r.norm_w), conv_rows.rows, conv_rows.count, k.conv,
                            ptr(r.conv_w), ptr(r.conv_b), dtype_code(r.conv_w), to_heads ? k.h : 0, w.A, p.dA, p.dD, p.d_dt_bias, head(0), head_type(0), head(1), head_type(1), head(2), head_type(2), stream),
          "m2_param_sums");
    return r;
}

py::tuple forward_parts(const Tensor& zx, const Tensor& A, const OptTensor& D, const Tensor& conv_w, const OptTensor& conv_b, const Tensor& dt_bias,
                        const Tensor& norm_w, int64_t g, int64_t n, int64_t d, int64_t hd, bool keep_states) {
    Scope scope(zx);
    const Packed k(zx, g, n, d, hd);
    check_core(k, A, or_none(D), conv_w, or_none(conv_b), dt_bias, norm_w);
    const Tensor A32 = f32(A), D32 = f32(or_none(D)), bias = f32(dt_bias), norm32 = f32(norm_w);
    const CoreOut r = core_forward(k, core_params(A32, D32, bias, norm32), conv_w, or_none(conv_b), keep_states, true, scope.stream);
    return py::make_tuple(r.norm_out, r.conv_out, r.scan_out, r.states);
}
py::tuple backward_parts(const Tensor& d_out, const Tensor& zx, const Tensor& A, const OptTensor& D, const Tensor& conv_w, const OptTensor& conv_b,
                         const Tensor& dt_bias, const Tensor& norm_w, const Tensor& conv_out, const Tensor& scan_out, const OptTensor& states,
                         int64_t g, int64_t n, int64_t d, int64_t hd) {
    Scope scope(zx);
    const Packed k(zx, g, n, d, hd);
    check_core(k, A, or_none(D), conv_w, or_none(conv_b), dt_bias, norm_w);
    const Tensor A32 = f32(A), D32 = f32(or_none(D)), bias = f32(dt_bias), norm32 = f32(norm_w);
    const CoreGrads r = core_backward(k, d_out, core_params(A32, D32, bias, norm32), conv_w, or_none(conv_b), conv_out, scan_out, or_none(states), norm_w, {},
                                      scope.stream);
    return py::make_tuple(r.zx, r.head(0, A), D ? r.head(2, *D) : Tensor(), r.conv_w, r.conv_b, r.head(1, dt_bias),
                          r.norm_w.to(norm_w.scalar_type()));
}

// fused_kernel.py:423-487.  caching: the conv output, scan output and chunk states are kept; otherwise only the inputs are,
// and the backward recomputes those three (not the norm, which it does not need).
struct CoreFn : torch::autograd::Function<CoreFn> {
    static Tensor forward(AutogradContext* ctx, const Tensor& zx, const Tensor& A, const OptTensor& D, const Tensor& conv_w, const OptTensor& conv_b,
                          const Tensor& dt_bias, const Tensor& norm_w, int64_t g, int64_t n, int64_t d, int64_t hd, bool keep) {
        Scope scope(zx);
        const Packed k(zx, g, n, d, hd);
        check_core(k, A, or_none(D), conv_w, or_none(conv_b), dt_bias, norm_w);
        const Tensor A32 = f32(A), D32 = f32(or_none(D)), bias = f32(dt_bias), norm32 = f32(norm_w);
        const CoreOut r = core_forward(k, core_params(A32, D32, bias, norm32), conv_w, or_none(conv_b), keep, true, scope.stream);
        variable_list saved = {zx, A, or_none(D), conv_w, or_none(conv_b), dt_bias, norm_w};
        if (keep) { saved.push_back(r.conv_out); saved.push_back(r.scan_out); saved.push_back(r.states); }
        ctx->save_for_backward(std::move(saved));
        ctx->saved_data["dims"] = std::vector<int64_t>{g, n, d, hd};
        return r.norm_out;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const variable_list s = ctx->get_saved_variables();
        const std::vector<int64_t> dims = ctx->saved_data["dims"].toIntVector();
        Scope scope(s[0]);
        const Packed k(s[0], dims[0], dims[1], dims[2], dims[3]);
        const Tensor A = f32(s[1]), D = f32(s[2]), dt_bias = f32(s[5]), norm_w = f32(s[6]);
        const CoreParams params = core_params(A, D, dt_bias, norm_w);
        CoreOut f;
        if (s.size() > 7) { f.conv_out = s[7]; f.scan_out = s[8]; f.states = s[9]; }
        else f = core_forward(k, params, s[3], s[4], true, false, scope.stream);
        const CoreGrads r = core_backward(k, grads[0], params, s[3], s[4], f.conv_out, f.scan_out, f.states, s[6], {}, scope.stream);
        variable_list out(12);
        out[0] = r.zx; out[1] = r.head(0, s[1]);
        if (s[2].defined()) out[2] = r.head(2, s[2]);
        out[3] = r.conv_w; out[4] = r.conv_b; out[5] = r.head(1, s[5]); out[6] = r.norm_w.to(s[6].scalar_type());
        return out;
    }
};
Tensor fused_core(const Tensor& zx, const Tensor& A, const OptTensor& D, const Tensor& conv_w, const OptTensor& conv_b, const Tensor& dt_bias,
                  const Tensor& norm_w, int64_t g, int64_t n, int64_t d, int64_t hd, bool caching) {
    core_heads(g, n, d, hd);
    require_gpu({&zx});
    bool keep = caching && at::GradMode::is_enabled();
    return CoreFn::apply(zx, A, D, conv_w, conv_b, dt_bias, norm_w, g, n, d, hd, keep);
}

// ----------------------------------------------------------------------------------------------- whole mixer layer
// mamba2_mixer.py:213-240: in_proj -> core -> out_proj as one node, the products on few tokens by the kernel for them and the
// large ones by the library that torch uses, the small parameters cast (and A = -exp(A_log) formed) by one kernel and their
// gradients cast back by one.

// A program that has torch's TunableOp on wants the general library's solutions timed and the best one taken: its products go there.
// At 128 rows of a 2560-channel layer the best ones beat this library's kernel, which beats the library's default choice (64-layer
// step, replayed: 11.18 to 11.29 ms with the kernel; 10.98 to 11.13 with the chosen solutions in five of seven graphs and 11.28 in
// two, by what the tuner's own timing preferred; 11.8 with the default ones).  Asking costs 2 ns.
bool library_is_tuned() { return at::cuda::tunable::getTuningContext()->IsTunableOpEnabled(); }

m2_product_params product_params(const Tensor& a, bool a_k, const Tensor& b, bool b_k) {
    m2_product_params p{};
    p.M = a.size(a_k ? 0 : 1); p.K = a.size(a_k ? 1 : 0); p.N = b.size(b_k ? 0 : 1);
    p.a = ptr(a); p.b = ptr(b); p.lda = a.stride(0); p.ldb = b.stride(0); p.ldo = p.N; p.a_k = a_k; p.b_k = b_k;
    return p;
}
// an operand as the kernels read it
bool product_rows(const Tensor& t) {
    return t.scalar_type() == at::kBFloat16 && t.stride(1) == 1 && t.stride(0) % 8 == 0 && t.stride(0) >= t.size(1) &&
           t.size(0) * t.stride(0) < (int64_t{1} << 31) && reinterpret_cast<uintptr_t>(ptr(t)) % 16 == 0;
}

// out (M, N) = A B (+ bias): `a` is A or, if !a_k, A^T (K, M); `b` is B^T (N, K) or, if !b_k, B
Tensor product(const Tensor& a, bool a_k, const Tensor& b, bool b_k, const Tensor& bias, void* stream) {
    m2_product_params p = product_params(a, a_k, b, b_k);
    const bool plain_bias = !bias.defined() || (bias.scalar_type() == at::kBFloat16 && bias.is_contiguous() && bias.dim() == 1 && bias.size(0) == p.N);
    if (!plain_bias || !product_rows(a) || !product_rows(b) || b.size(b_k ? 1 : 0) != p.K || !lib.m2_product_pays(p.M, p.N, p.K, a_k, b_k) || library_is_tuned()) {
        const Tensor at_ = a_k ? a : a.t(), bt = b_k ? b.t() : b;
        return bias.defined() ? at::addmm(bias, at_, bt) : at::mm(at_, bt);
    }
    const Tensor out = at::empty({p.M, p.N}, a.options());
    p.workspace_bytes = lib.m2_product_workspace_bytes(p.M, p.N, p.K);
    const Tensor ws = p.workspace_bytes ? at::empty({static_cast<int64_t>(p.workspace_bytes)}, a.options().dtype(at::kByte)) : Tensor();
    p.bias = ptr(bias); p.out = ptr(out); p.workspace = ptr(ws);
    check(lib.m2_product(&p, stream), "m2_product");
    return out;
}

// What a linear layer's backward needs of its products, (dy W, dy^T x) or only one of them: in one launch where that pays.
std::pair<Tensor, Tensor> linear_grads(const Tensor& dy, const Tensor& w, const Tensor& x, bool want_x, bool want_w, void* stream) {
    if (want_x && want_w && product_rows(dy) && product_rows(w) && product_rows(x) && !library_is_tuned()) {
        m2_product_params px = product_params(dy, true, w, false), pw = product_params(dy, false, x, false);
        if (w.size(0) == px.K && x.size(0) == pw.K && lib.m2_product_pair_pays(&px, &pw)) {
            const Tensor dx = at::empty({px.M, px.N}, dy.options()), dw = at::empty({pw.M, pw.N}, dy.options());
            px.workspace_bytes = lib.m2_product_pair_workspace_bytes(&px, &pw);
            const Tensor ws = px.workspace_bytes ? at::empty({static_cast<int64_t>(px.workspace_bytes)}, dy.options().dtype(at::kByte)) : Tensor();
            px.out = ptr(dx); pw.out = ptr(dw); px.workspace = ptr(ws);
            check(lib.m2_product_pair(&px, &pw, stream), "m2_product_pair");
            return {dx, dw};
        }
    }
    return {want_x ? product(dy, true, w, false, Tensor(), stream) : Tensor(), want_w ? product(dy, false, x, false, Tensor(), stream) : Tensor()};
}
Tensor project(const Tensor& x, const Tensor& w, const Tensor& bias, void* stream) { return product(x, true, w, true, bias, stream); }

// a linear layer outside autograd
Tensor linear(const Tensor& x, const Tensor& w, const OptTensor& bias) {
    require_gpu({&x, &w, &or_none(bias)});
    TORCH_CHECK_VALUE(x.dim() >= 1 && w.dim() == 2 && x.size(-1) == w.size(1), "linear: x (..., in) and weight (out, in) are required");
    Scope scope(x);
    std::vector<int64_t> shape = x.sizes().vec();
    shape.back() = w.size(0);
    return project(x.reshape({-1, w.size(1)}), w, or_none(bias), scope.stream).view(shape);
}

// a small parameter as the casting kernel reads it; types that it does not take come as fp32
Tensor small_param(const Tensor& t) { return (casts(t) ? t : t.to(at::kFloat)).contiguous(); }

struct MixerFn : torch::autograd::Function<MixerFn> {
    enum { kHidden, kInW, kALog, kD, kDtBias, kConvW, kNormW, kOutW, kConvB, kInB, kOutB, kSmall, kZx, kNormOut, kConvOut, kScanOut, kStates };
    // the casting kernel leaves A, D and dt_bias (a value per head each) and the norm's weight one behind the other
    static CoreParams params_in(const Tensor& small, int64_t h) {
        const float* at = ptr<float>(small);
        return {at, at + h, at + 2 * h, at + 3 * h};
    }
    static Tensor forward(AutogradContext* ctx, const Tensor& hidden, const Tensor& in_w, const Tensor& A_log, const Tensor& D, const Tensor& dt_bias,
                          const Tensor& conv_w, const Tensor& norm_w, const Tensor& out_w, const OptTensor& conv_b, const OptTensor& in_b,
                          const OptTensor& out_b, int64_t g, int64_t n, int64_t d, int64_t hd, bool differentiable, bool recompute) {
        Scope scope(hidden);
        const int64_t b = hidden.size(0), l = hidden.size(1), h = core_heads(g, n, d, hd);
        const Tensor x = hidden.reshape({b * l, hidden.size(2)});
        const Tensor zx = project(x, in_w, or_none(in_b), scope.stream).view({b, l, in_w.size(0)});
        const Packed k(zx, g, n, d, hd);
        check_core(k, A_log, D, conv_w, or_none(conv_b), dt_bias, norm_w);
        const Tensor small = empty_f32({3 * h + d}, zx);
        const Tensor a = small_param(A_log), dd = small_param(D), tb = small_param(dt_bias), nw = small_param(norm_w);
        check(lib.m2_mixer_params(ptr(a), dtype_code(a), ptr(dd), dtype_code(dd), ptr(tb), dtype_code(tb), ptr(nw), dtype_code(nw), ptr<float>(small),
                                  h, d, scope.stream), "m2_mixer_params");
        const CoreOut r = core_forward(k, params_in(small, h), conv_w, or_none(conv_b), differentiable && !recompute, true, scope.stream);
        const Tensor y = r.norm_out.view({b * l, d});
        if (differentiable) {
            variable_list saved = {hidden, in_w, A_log, D, dt_bias, conv_w, norm_w, out_w, or_none(conv_b), or_none(in_b), or_none(out_b), small, zx, y};
            if (!recompute) { saved.push_back(r.conv_out); saved.push_back(r.scan_out); saved.push_back(r.states); }
            ctx->save_for_backward(std::move(saved));
            ctx->saved_data["dims"] = std::vector<int64_t>{g, n, d, hd};
        }
        return project(y, out_w, or_none(out_b), scope.stream).view({b, l, out_w.size(0)});
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const variable_list s = ctx->get_saved_variables();
        const std::vector<int64_t> dims = ctx->saved_data["dims"].toIntVector();
        const Tensor& zx = s[kZx];
        Scope scope(zx);
        const Packed k(zx, dims[0], dims[1], dims[2], dims[3]);
        const int64_t rows = k.b * k.l;
        const Tensor& small = s[kSmall];
        const CoreParams params = params_in(small, k.h);
        variable_list out(17);
        const Tensor dy = grads[0].reshape({rows, s[kOutW].size(0)});
        Tensor d_core;
        std::tie(d_core, out[kOutW]) = linear_grads(dy, s[kOutW], s[kNormOut], true, ctx->needs_input_grad(kOutW), scope.stream);
        d_core = d_core.view({k.b, k.l, k.d});
        if (s[kOutB].defined()) out[kOutB] = dy.sum(0);
        CoreOut f;
        if (s.size() > kConvOut) { f.conv_out = s[kConvOut]; f.scan_out = s[kScanOut]; f.states = s[kStates]; }
        else f = core_forward(k, params, s[kConvW], s[kConvB], true, false, scope.stream);
        for (const int i : {kALog, kD, kDtBias}) out[i] = at::empty(s[i].sizes(), casts(s[i]) ? s[i].options() : s[i].options().dtype(at::kFloat));
        const CoreGrads r = core_backward(k, d_core, params, s[kConvW], s[kConvB], f.conv_out, f.scan_out, f.states, s[kNormW],
                                          {out[kALog], out[kD], out[kDtBias]}, scope.stream);
        out[kNormW] = r.norm_w.view(s[kNormW].sizes());
        for (const int i : {kALog, kD, kDtBias, kNormW})
            if (!casts(s[i])) out[i] = out[i].to(s[i].scalar_type());
        out[kConvW] = r.conv_w; out[kConvB] = r.conv_b;
        const Tensor d_zx = r.zx.view({rows, zx.size(2)});
        std::tie(out[kHidden], out[kInW]) = linear_grads(d_zx, s[kInW], s[kHidden].reshape({rows, s[kHidden].size(2)}), ctx->needs_input_grad(kHidden),
                                                         ctx->needs_input_grad(kInW), scope.stream);
        if (out[kHidden].defined()) out[kHidden] = out[kHidden].view(s[kHidden].sizes());
        if (s[kInB].defined()) out[kInB] = d_zx.sum(0);
        return out;
    }
};
Tensor mixer(const Tensor& hidden, const Tensor& in_w, const Tensor& A_log, const Tensor& D, const Tensor& dt_bias, const Tensor& conv_w, const Tensor& norm_w,
             const Tensor& out_w, const OptTensor& conv_b, const OptTensor& in_b, const OptTensor& out_b, int64_t g, int64_t n, int64_t d, int64_t hd,
             bool recompute) {
    core_heads(g, n, d, hd);
    require_gpu({&hidden, &in_w, &out_w, &or_none(in_b), &or_none(out_b)});
    TORCH_CHECK_VALUE(hidden.dim() == 3, "hidden_states must be (batch, seqlen, hidden_size)");
    bool differentiable = false;
    if (at::GradMode::is_enabled())
        for (const Tensor* t : {&hidden, &in_w, &A_log, &D, &dt_bias, &conv_w, &norm_w, &out_w, &or_none(conv_b), &or_none(in_b), &or_none(out_b)})
            differentiable |= t->defined() && t->requires_grad();
    return MixerFn::apply(hidden, in_w, A_log, D, dt_bias, conv_w, norm_w, out_w, conv_b, in_b, out_b, g, n, d, hd, differentiable, recompute);
}

// Inference forward that hands the sequence over to the decode step: final SSM state and last W conv inputs into the cache.
Tensor fused_prefill(const Tensor& zx, const Tensor& A, const OptTensor& D, const Tensor& conv_w, const OptTensor& conv_b_, const Tensor& dt_bias,
                     const Tensor& norm_w, int64_t g, int64_t n, int64_t d, int64_t hd, const Tensor& conv_state, const Tensor& ssm_state, bool continuing) {
    core_heads(g, n, d, hd);
    require_gpu({&zx, &conv_state, &ssm_state});
    Scope scope(zx);
    const Packed k(zx, g, n, d, hd);
    const Tensor& conv_b = or_none(conv_b_);
    check_core(k, A, or_none(D), conv_w, conv_b, dt_bias, norm_w);
    const int64_t taps = conv_w.size(2);
    TORCH_CHECK_VALUE(conv_state.dim() == 3 && conv_state.size(0) == k.b && conv_state.size(1) == k.conv && conv_state.size(2) >= taps - 1,
                      "conv_state must be (b, conv_dim, W >= k-1), got ", conv_state.sizes());
    TORCH_CHECK_VALUE(ssm_state.dim() == 4 && ssm_state.size(0) == k.b && ssm_state.size(1) == k.h && ssm_state.size(2) == hd && ssm_state.size(3) == n &&
                          ssm_state.scalar_type() == at::kFloat, "ssm_state must be (b, h, p, n) float32");
    if (k.l == 0) return at::empty({k.b, 0, d}, zx.options());
    // the kernels work in the caller's cache tensors where those are contiguous and of the kernels' types
    const bool own_conv = conv_state.is_contiguous() && conv_state.scalar_type() == zx.scalar_type(), own_ssm = ssm_state.is_contiguous();
    const Tensor cs = own_conv ? conv_state : conv_state.to(zx.options(), false, true).contiguous(), S = own_ssm ? ssm_state : ssm_state.contiguous();
    const Tensor w = conv_w.contiguous(), bi = conv_b.defined() ? conv_b.contiguous() : conv_b;
    const Tensor conv_out = at::empty({k.b, k.l, k.conv}, zx.options());
    m2_conv1d_params c = conv_params(k.xBC(), w, bi, {ptr(conv_out), k.l * k.conv, k.conv, 1}, k.b, k.l, k.conv, dtype_code(k.zx), M2_ACT_SILU);
    c.y = ptr(conv_out);
    // The conv moves the cache on, so everything behind it is allocated and checked first: a call that is refused leaves the cache
    // as it was.
    const Tensor A32 = f32(A), D32 = f32(or_none(D)), bias = f32(dt_bias), norm32 = f32(norm_w);
    const CoreParams params = core_params(A32, D32, bias, norm32);
    m2_ssd_params p = core_ssd_params(k, conv_out, params);
    const Tensor y = at::empty({k.b, k.l, d}, zx.options());
    p.initial_state = continuing ? ptr<float>(S) : nullptr; p.final_state = ptr<float>(S);
    p.y = ptr(y); p.y_stride_b = k.l * d; p.y_stride_l = d; p.y_stride_h = hd;
    p.workspace_bytes = lib.m2_ssd_fwd_workspace_bytes(&p);
    const Tensor ws = scratch(p.workspace_bytes, zx);
    p.workspace = ptr(ws);
    check(lib.m2_ssd_fwd_check(&p), "m2_ssd_fwd");
    const Tensor out = at::empty({k.b, k.l, d}, zx.options());
    m2_rmsnorm_params q = core_norm_params(k, params, ptr(y));
    q.out = ptr(out); q.out_stride_row = d;
    check(lib.m2_core_norm_fwd_check(&q), "m2_core_norm_fwd");
    check(lib.m2_conv1d_prefill(&c, ptr(cs), static_cast<int32_t>(cs.size(2)), continuing, scope.stream), "m2_conv1d_prefill");
    check(lib.m2_ssd_fwd(&p, scope.stream), "m2_ssd_fwd");
    if (!own_conv) conv_state.copy_(cs);
    if (!own_ssm) ssm_state.copy_(S);
    check(lib.m2_core_norm_fwd(&q, scope.stream), "m2_core_norm_fwd");
    return out;
}

// ----------------------------------------------------------------------------------------------- decode step
void check_conv_bias(const Tensor& conv_w, const Tensor& conv_b, int64_t channels) {
    TORCH_CHECK_VALUE(!conv_b.defined() || (conv_b.numel() == channels && conv_b.scalar_type() == conv_w.scalar_type()),
                      "the conv bias must have ", channels, " values in the dtype of the conv weight");
}

std::tuple<Tensor, Tensor, Tensor> decode_step(const Tensor& xBC, const Tensor& conv_state, const Tensor& conv_w, const OptTensor& conv_b_, const Tensor& S,
                                               const Tensor& dt, const Tensor& A_, const OptTensor& D_, int64_t g, int64_t activation,
                                               const OptTensor& dt_bias_, const OptTensor& out, bool static_scratch) {
    const Tensor &conv_b = or_none(conv_b_), &dt_bias = or_none(dt_bias_);
    TORCH_CHECK_VALUE(S.dim() == 4 && xBC.dim() == 3 && conv_state.dim() == 3 && dt.dim() == 3, "expected xBC (b,1,Cx), conv_state (b,Cx,W), S (b,h,p,n), dt (b,1,h)");
    const int64_t b = S.size(0), h = S.size(1), p_ = S.size(2), n = S.size(3), d = h * p_, cx = xBC.size(2);
    TORCH_CHECK_VALUE(S.scalar_type() == at::kFloat, "the SSM state must be float32");
    TORCH_CHECK_VALUE(conv_state.scalar_type() == xBC.scalar_type() && dt.scalar_type() == xBC.scalar_type(), "xBC, conv_state and dt must share one dtype");
    TORCH_CHECK_VALUE(S.is_contiguous() && conv_state.is_contiguous(), "S and conv_state must be contiguous (they are updated in place)");
    TORCH_CHECK_VALUE(xBC.stride(2) == 1 && dt.stride(2) == 1, "xBC and dt must be contiguous in their last dimension");
    require_gpu({&xBC, &conv_state, &conv_w, &conv_b, &S, &dt, &A_, &or_none(D_), &dt_bias});
    TORCH_CHECK_VALUE(!dt_bias.defined() || (dt_bias.dim() == 1 && dt_bias.size(0) == h), "dt_bias must have shape (n_heads,)");
    TORCH_CHECK_VALUE(!out || (out->dim() == 3 && out->size(0) == b && out->size(1) == 1 && out->size(2) == d && out->scalar_type() == xBC.scalar_type() &&
                               out->stride(2) == 1 && out->device() == xBC.device()),
                      "out must be (batch, 1, n_heads * d_head) in the dtype of xBC, on its device");
    Scope scope(xBC);
    const Tensor w = conv_w.contiguous(), bi = conv_b.defined() ? conv_b.contiguous() : conv_b;
    const Tensor A = f32(A_), D = f32(or_none(D_)), bias = f32(dt_bias);
    Tensor Y = out ? *out : at::empty({b, 1, d}, xBC.options());
    m2_decode_params p{};
    p.xBC = ptr(xBC); p.conv_state = ptr(conv_state); p.conv_w = ptr(w); p.conv_b = ptr(bi);
    p.S = ptr<float>(S); p.dt = ptr(dt); p.A = ptr<float>(A); p.D = ptr<float>(D); p.y = ptr(Y); p.dt_bias = ptr<float>(bias);
    p.batch = b; p.nheads = h; p.headdim = p_; p.dstate = n; p.ngroups = g;
    p.k = static_cast<int32_t>(w.size(-1)); p.W = static_cast<int32_t>(conv_state.size(2));
    check_conv_bias(w, bi, cx);
    TORCH_CHECK_VALUE(A.numel() == h && (!D.defined() || D.numel() == h), "A and D must have shape (n_heads,)");
    TORCH_CHECK_VALUE(w.numel() == cx * p.k && conv_state.size(0) == b && conv_state.size(1) == cx, "conv weight and state must have ", cx, " channels");
    p.xBC_stride_b = xBC.stride(0); p.dt_stride_b = dt.stride(0); p.y_stride_b = Y.stride(0);
    p.dtype = dtype_code(xBC); p.param_dtype = dtype_code(w); p.activation = static_cast<int32_t>(activation);
    if (static_scratch) {
        check(lib.m2_decode_step_static(&p, scope.stream), "m2_decode_step_static");
    } else {
        p.workspace_bytes = lib.m2_decode_workspace_bytes(b, h, p_, n, g);
        const Tensor ws = scratch(p.workspace_bytes, xBC);
        p.workspace = ptr(ws);
        check(lib.m2_decode_step(&p, scope.stream), "m2_decode_step");
    }
    return {Y, conv_state, S};
}

// ----------------------------------------------------------------------------------------------- decode step of a layer
// mamba2_mixer.py:243-282, and with a residual stream the block around it (modeling_mamba2.py:133-140): in place on the layer's
// states and on the stream.
struct StepArgs {
    const Tensor &in_w, &in_b, &conv_w, &conv_b, &A, &D, &dt_bias, &norm_w, &out_w, &out_b, &conv_state, &ssm_state;
    int64_t g, norm_groups;
    double eps;
};

// The fp32 residual rows of a model's step between two of its layers: either `delta` is still to be added (separate kernels),
// or `x` holds the rows times the next norm's weight and `sq` their sums of squares (chained kernels), or neither.
struct ResidualStream {
    Tensor rows, delta, x, sq;
    Tensor first;                  // embedding rows that `rows` is yet to be set to, or
    Tensor table, ids;             // the embedding and the rows of it that will be these
};

bool starts_at(const Tensor& t, size_t bytes) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % bytes == 0; }

// the small product's kernel copies 16 bytes at a time (a view into a flat buffer of parameters may start anywhere)
bool linear_takes(const Tensor& w, const Tensor& bias) {
    return w.scalar_type() == at::kBFloat16 && w.is_contiguous() && starts_at(w, 16) &&
           (!bias.defined() || (bias.is_contiguous() && bias.scalar_type() == at::kBFloat16 && bias.dim() == 1 && bias.size(0) == w.size(0)));
}

// rows as that kernel reads them: 16-byte pieces at 32-bit byte offsets from the first row; others are copied once
Tensor linear_input(const Tensor& x) {
    const bool fits = x.stride(1) == 1 && starts_at(x, 16) && x.stride(0) % 8 == 0 && x.stride(0) < (int64_t{1} << 26);
    return fits ? x : x.clone(at::MemoryFormat::Contiguous);
}

m2_linear_params linear_params(const Tensor& w, const Tensor& bias, int64_t rows) {
    m2_linear_params p{};
    p.w = ptr(w); p.bias = ptr(bias); p.M = rows; p.N = w.size(0); p.K = w.size(1); p.groups = 1;
    return p;
}

// out = x w^T + bias for a few bf16 rows; the library's product where the kernel does not take the shape
Tensor linear_rows(const Tensor& x, const Tensor& w, const Tensor& bias, void* stream) {
    m2_linear_params p = linear_params(w, bias, x.size(0));
    if (x.scalar_type() != at::kBFloat16 || !linear_takes(w, bias) || !lib.m2_linear_small_fits(p.M, p.N, p.K, 1)) return project(x, w, bias, stream);
    const Tensor xr = linear_input(x);
    Tensor out = at::empty({p.M, p.N}, x.options());
    p.x = ptr(xr); p.x_stride_row = xr.stride(0); p.out = ptr(out); p.out_stride_row = p.N;
    check(lib.m2_linear_small(&p, stream), "m2_linear_small");
    return out;
}

// a tensor of the stream's width, on its device; how many rows the stream has
const Tensor& stream_anchor(const ResidualStream& r) { return r.first.defined() ? r.first : r.ids.defined() ? r.table : r.rows; }
int64_t stream_count(const ResidualStream& r) { return r.ids.defined() ? r.ids.numel() : stream_anchor(r).size(0); }

// the stream's rows out of the embedding; norm_w: that norm's x and sq of them too
void embed_rows(ResidualStream& r, const Tensor& norm_w) {
    Scope scope(r.table);
    r.rows = at::empty({r.ids.numel(), r.table.size(1)}, r.table.options().dtype(at::kFloat));
    if (norm_w.defined()) {
        r.x = at::empty(r.rows.sizes(), r.rows.options().dtype(at::kBFloat16));
        r.sq = at::empty({r.rows.size(0), 1}, r.rows.options());
    }
    check(lib.m2_embed_rows(ptr(r.table), dtype_code(r.table), r.table.size(0), r.ids.data_ptr<int64_t>(), ptr<float>(r.rows), ptr<float>(norm_w), ptr(r.x),
                            ptr<float>(r.sq), r.rows.size(0), r.rows.size(1), scope.stream), "m2_embed_rows");
    r.table = r.ids = Tensor();
}

// the stream's rows, set from the embedding if they are not yet
const Tensor& stream_rows(ResidualStream& r) {
    if (r.ids.defined()) embed_rows(r, Tensor());
    if (r.first.defined()) {
        r.rows = r.first.to(at::kFloat, /*non_blocking=*/false, /*copy=*/true, at::MemoryFormat::Contiguous);
        r.first = Tensor();
    }
    return r.rows;
}

// The stream's rows, everything added, after a norm, in out_dtype: one kernel, or where what is left to add is of another type (a
// head or a layer of its own precision behind it) that sum first.
Tensor stream_add_norm(ResidualStream& r, const Tensor& norm_w, double eps, at::ScalarType out_dtype) {
    const Tensor& rows = stream_rows(r);
    if (r.delta.defined() && r.delta.scalar_type() != out_dtype) {
        rows.add_(r.delta);
        r.delta = Tensor();
    }
    const Tensor w = starts_at(norm_w, 16) ? norm_w : norm_w.clone();
    const Tensor out = add_rmsnorm(rows, r.delta.defined() ? OptTensor(r.delta) : std::nullopt, w, eps, out_dtype);
    r.delta = r.x = r.sq = Tensor();
    return out;
}

// x and sq of the stream for a norm weight
void stream_heads(ResidualStream& r, const Tensor& norm_w, void* stream) {
    if (r.x.defined()) return;
    if (r.ids.defined()) return embed_rows(r, norm_w);
    const bool set = r.first.defined();
    const Tensor src = set ? r.first.contiguous() : (r.delta.defined() ? r.delta.contiguous() : Tensor());
    if (set) r.rows = at::empty(src.sizes(), src.options().dtype(at::kFloat));
    r.x = at::empty(r.rows.sizes(), r.rows.options().dtype(at::kBFloat16));
    r.sq = at::empty({r.rows.size(0), 1}, r.rows.options());
    check(lib.m2_decode_rows(ptr<float>(r.rows), ptr(src), src.defined() ? dtype_code(src) : M2_F32, set, ptr<float>(norm_w), ptr(r.x), ptr<float>(r.sq), r.rows.size(0),
                             r.rows.size(1), stream), "m2_decode_rows");
    r.first = r.delta = Tensor();
}

void set_rows(m2_linear_params& p, const Tensor& x, const Tensor& sq, double eps) {
    p.x = ptr(x); p.x_stride_row = x.stride(0); p.sq = ptr<float>(sq); p.nsq = sq.defined() ? sq.size(1) : 0; p.eps = static_cast<float>(eps);
}

// hidden: (b, hidden) rows -> the layer's output rows.  With a stream instead, the block: its norm, the layer, and the sum in the
// stream; next_norm: the weight of the norm that will read it, if that is known.
Tensor step_rows(const Tensor& hidden, ResidualStream* r, const Tensor& block_norm, double block_eps, const Tensor& next_norm, const StepArgs& a, void* stream) {
    const int64_t b = a.ssm_state.size(0), h = a.ssm_state.size(1), hd = a.ssm_state.size(2), n = a.ssm_state.size(3), d = h * hd;
    const at::TensorOptions act = a.in_w.options();
    const at::ScalarType act_type = a.in_w.scalar_type();
    m2_linear_params in = linear_params(a.in_w, a.in_b, b), out = linear_params(a.out_w, a.out_b, b);
    const bool fused = linear_takes(a.in_w, a.in_b) && linear_takes(a.out_w, a.out_b) && (r || hidden.scalar_type() == at::kBFloat16) &&
                       lib.m2_linear_small_fits(in.M, in.N, in.K, 1) && lib.m2_linear_small_fits(out.M, out.N, out.K, static_cast<int32_t>(a.norm_groups)) &&
                       (hd == 64 || hd == 128) && (n == 64 || n == 128) && a.conv_w.size(-1) == 4 && h % a.norm_groups == 0;
    if (!fused) {
        const Tensor rows = r ? stream_add_norm(*r, block_norm, block_eps, act_type) : hidden;
        const Tensor packed = linear_rows(rows, a.in_w, a.in_b, stream).unsqueeze(1);
        const int64_t cx = d + 2 * a.g * n;
        const Tensor y = std::get<0>(decode_step(packed.narrow(2, d, cx), a.conv_state, a.conv_w, a.conv_b.defined() ? OptTensor(a.conv_b) : std::nullopt,
                                                 a.ssm_state, packed.narrow(2, d + cx, h), a.A, a.D, a.g, M2_ACT_SILU, a.dt_bias, std::nullopt, false));
        const Tensor normed = rmsnorm_forward(y.view({b, d}), packed.select(1, 0).narrow(1, 0, d), a.norm_w, a.norm_groups, a.eps, act_type);
        const Tensor o = linear_rows(normed, a.out_w, a.out_b, stream);
        if (r) r->delta = o;
        return o;
    }
    const Tensor zx = at::empty({b, a.in_w.size(0)}, act);
    const Tensor conv_c = a.conv_w.contiguous(), conv_b = a.conv_b.defined() ? a.conv_b.contiguous() : a.conv_b;
    const Tensor conv_w = starts_at(conv_c, 4 * conv_c.element_size()) ? conv_c : conv_c.clone();      // a channel's four taps in one load
    const Tensor mid = at::empty({b * (d * 2 + h * 4)}, act.dtype(at::kByte));          // gated rows (bf16), then the head sums (fp32)
    const Tensor x = r ? Tensor() : linear_input(hidden);
    Tensor result, next_x, next_sq;
    if (r) {
        stream_heads(*r, block_norm, stream);
        set_rows(in, r->x, r->sq, block_eps);
        out.out = ptr(r->rows); out.out_kind = 2;
        if (next_norm.defined()) {
            next_x = at::empty({b, out.N}, act);
            next_sq = at::empty({b, (out.N + 15) / 16}, r->rows.options());
            out.next_weight = ptr<float>(next_norm); out.next_x = ptr(next_x); out.next_sq = ptr<float>(next_sq);
        }
    } else {
        set_rows(in, x, Tensor(), 0.0);
        result = at::empty({b, out.N}, act);
        out.out = ptr(result);
    }
    in.out = ptr(zx); in.out_stride_row = in.N;
    out.x = ptr(mid); out.x_stride_row = d; out.sq = reinterpret_cast<float*>(at_column(mid, b * d * 2)); out.nsq = h;
    out.groups = static_cast<int32_t>(a.norm_groups); out.eps = static_cast<float>(a.eps); out.out_stride_row = out.N;
    m2_decode_params p{};
    p.conv_state = ptr(a.conv_state); p.conv_w = ptr(conv_w); p.conv_b = ptr(conv_b); p.S = ptr<float>(a.ssm_state);
    p.A = ptr<float>(a.A); p.D = ptr<float>(a.D); p.dt_bias = ptr<float>(a.dt_bias);
    p.batch = b; p.nheads = h; p.headdim = hd; p.dstate = n; p.ngroups = a.g; p.k = 4; p.W = static_cast<int32_t>(a.conv_state.size(2));
    p.dtype = M2_BF16; p.param_dtype = dtype_code(conv_w); p.activation = M2_ACT_SILU;
    check(lib.m2_decode_layer(&in, &p, ptr<float>(a.norm_w), &out, stream), "m2_decode_layer");
    if (r) { r->x = next_x; r->sq = next_sq; }
    return result;
}

void check_fp32(std::initializer_list<const Tensor*> tensors, const char* what) {
    for (const Tensor* t : tensors)
        TORCH_CHECK_VALUE(!t->defined() || (t->scalar_type() == at::kFloat && t->is_contiguous()), what, " must be contiguous float32");
}

// A, D, dt_bias, norm weights: fp32 (the caller keeps them).  Either hidden (b, 1, hidden) -> output, or a stream with the norms.
Tensor mixer_step(const OptTensor& hidden_, ResidualStream* r, const OptTensor& block_norm_, double block_eps, const OptTensor& next_norm_, const Tensor& in_w,
                  const OptTensor& in_b, const Tensor& conv_w, const OptTensor& conv_b, const Tensor& A, const Tensor& D, const Tensor& dt_bias, const Tensor& norm_w,
                  double eps, int64_t norm_groups, const Tensor& out_w, const OptTensor& out_b, const Tensor& conv_state, const Tensor& ssm_state, int64_t g) {
    const Tensor &hidden = or_none(hidden_), &block_norm = or_none(block_norm_), &next_norm = or_none(next_norm_);
    const Tensor& x = r ? stream_anchor(*r) : hidden;
    TORCH_CHECK_VALUE(x.defined() && (r ? x.dim() == 2 : x.dim() == 3 && x.size(1) == 1), "hidden_states must be (batch, 1, hidden_size)");
    const int64_t b = r ? stream_count(*r) : x.size(0), width = x.size(-1);
    require_gpu({&x, &in_w, &or_none(in_b), &conv_w, &or_none(conv_b), &A, &D, &dt_bias, &norm_w, &block_norm, &next_norm, &out_w, &or_none(out_b),
                 &conv_state, &ssm_state});
    TORCH_CHECK_VALUE(ssm_state.dim() == 4 && ssm_state.size(0) == b && ssm_state.scalar_type() == at::kFloat && ssm_state.is_contiguous(),
                      "the SSM state must be float32 (batch, heads, headdim, state), contiguous");
    const int64_t h = ssm_state.size(1), d = h * ssm_state.size(2), cx = d + 2 * g * ssm_state.size(3);
    TORCH_CHECK_VALUE(conv_state.dim() == 3 && conv_state.size(0) == b && conv_state.size(1) == cx && conv_state.size(2) >= conv_w.size(-1) - 1 &&
                          conv_state.scalar_type() == in_w.scalar_type() && conv_state.is_contiguous(),
                      "the conv state must be (batch, ", cx, ", W >= k-1), contiguous, in the dtype of the projections");
    TORCH_CHECK_VALUE(in_w.dim() == 2 && in_w.size(0) == d + cx + h && in_w.size(1) == width && out_w.dim() == 2 && out_w.size(1) == d,
                      "the projections do not match the states");
    TORCH_CHECK_VALUE(g > 0 && h % g == 0 && conv_w.numel() == cx * conv_w.size(-1) && A.numel() == h && D.numel() == h && dt_bias.numel() == h && norm_w.numel() == d,
                      "parameter shapes do not match the states");
    check_conv_bias(conv_w, or_none(conv_b), cx);
    check_fp32({&A, &D, &dt_bias, &norm_w, &block_norm, &next_norm}, "A, D, dt_bias and the norm weights");
    TORCH_CHECK_VALUE(!r || (block_norm.defined() && block_norm.numel() == width && out_w.size(0) == width && (!next_norm.defined() || next_norm.numel() == width)),
                      "the norm weights must have the width of the residual stream");
    Scope scope(x);
    const StepArgs a{in_w, or_none(in_b), conv_w, or_none(conv_b), A, D, dt_bias, norm_w, out_w, or_none(out_b), conv_state, ssm_state, g, norm_groups, eps};
    if (r) {
        step_rows(Tensor(), r, block_norm, block_eps, next_norm, a, scope.stream);
        return Tensor();
    }
    return step_rows(hidden.reshape({b, width}), nullptr, Tensor(), 0.0, Tensor(), a, scope.stream).view({b, 1, out_w.size(0)});
}

ResidualStream residual_stream(const Tensor& embedded) {
    require_gpu({&embedded});
    const bool read = embedded.scalar_type() == at::kFloat || embedded.scalar_type() == at::kBFloat16;      // as the kernels read it
    ResidualStream r;
    r.first = (read ? embedded : embedded.to(at::kFloat)).reshape({-1, embedded.size(-1)});
    return r;
}

// A model's stream at its embedding, which the stream's first kernel reads itself where the table lies as it takes it.
ResidualStream embedded_stream(const Tensor& table, const Tensor& ids) {
    require_gpu({&table, &ids});
    const bool reads = (table.scalar_type() == at::kFloat || table.scalar_type() == at::kBFloat16) && table.dim() == 2 && table.is_contiguous() &&
                       table.size(1) > 0 && ids.scalar_type() == at::kLong && ids.numel() <= INT32_MAX;
    if (!reads) return residual_stream(at::embedding(table, ids));
    ResidualStream r;
    r.table = table;
    r.ids = ids.reshape({-1}).contiguous();
    return r;
}

// the stream's rows as they are, everything added
Tensor stream_sum(ResidualStream& r) {
    const Tensor any = stream_anchor(r);
    Scope scope(any);
    const Tensor& rows = stream_rows(r);
    if (r.delta.defined()) { rows.add_(r.delta); r.delta = Tensor(); }
    return rows;
}

// the stream's rows after its last norm, in out_dtype
Tensor stream_norm(ResidualStream& r, const Tensor& norm_w, double eps, at::ScalarType out_dtype) {
    check_fp32({&norm_w}, "the norm weight");
    Scope scope(norm_w);
    return stream_add_norm(r, norm_w, eps, out_dtype);
}

// fp32 product of the normalised rows: norm_f and the LM head (modeling_mamba2.py:350, 489-490)
Tensor stream_norm_linear(ResidualStream& r, const Tensor& norm_w, double eps, const Tensor& w, const OptTensor& bias_) {
    const Tensor& bias = or_none(bias_);
    require_gpu({&norm_w, &w, &bias});
    check_fp32({&norm_w}, "the norm weight");
    const Tensor any = stream_anchor(r);
    require_gpu({&any, &w});
    TORCH_CHECK_VALUE(w.dim() == 2 && any.size(1) == w.size(1) && norm_w.numel() == w.size(1), "the norm weight and the product must have the width of the residual stream");
    Scope scope(w);
    m2_linear_params p = linear_params(w, bias, stream_count(r));
    if (!linear_takes(w, bias) || !lib.m2_linear_small_fits(p.M, p.N, p.K, 1)) {
        const at::ScalarType normed = w.scalar_type() == at::kBFloat16 ? at::kBFloat16 : at::kFloat;      // the norm's output types
        return linear_rows(stream_add_norm(r, norm_w, eps, normed).to(w.scalar_type()), w, bias, scope.stream).to(at::kFloat);
    }
    stream_heads(r, norm_w, scope.stream);
    const Tensor out = at::empty({p.M, p.N}, r.rows.options());
    set_rows(p, r.x, r.sq, eps);
    p.out = ptr(out); p.out_stride_row = p.N; p.out_kind = 1;
    check(lib.m2_linear_small(&p, scope.stream), "m2_linear_small");
    return out;
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    py::class_<ResidualStream>(m, "ResidualStream");
    m.def("bound_names", &bound_names);
    m.def("bind", &bind);
    m.def("conv1d_forward", &conv1d_forward);
    m.def("conv1d_backward", &conv1d_backward);
    m.def("conv1d", &conv1d);
    m.def("alloc_chunk_states", &alloc_chunk_states);
    m.def("ssd_forward", &ssd_forward);
    m.def("ssd_backward", &ssd_backward);
    m.def("mamba2_kernel", &mamba2_kernel);
    m.def("rmsnorm_forward", &rmsnorm_forward);
    m.def("rmsnorm_backward", &rmsnorm_backward);
    m.def("rmsnorm", &rmsnorm);
    m.def("add_rmsnorm", &add_rmsnorm);
    m.def("forward_parts", &forward_parts);
    m.def("backward_parts", &backward_parts);
    m.def("fused_core", &fused_core);
    m.def("mixer", &mixer);
    m.def("fused_prefill", &fused_prefill);
    m.def("mixer_step", &mixer_step);
    m.def("residual_stream", &residual_stream);
    m.def("embedded_stream", &embedded_stream);
    m.def("stream_sum", &stream_sum);
    m.def("stream_norm", &stream_norm);
    m.def("linear", &linear);
    m.def("stream_norm_linear", &stream_norm_linear);
    m.def("decode_step", &decode_step);
}
