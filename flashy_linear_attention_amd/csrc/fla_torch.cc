// The operators' host path between PyTorch and the C ABI (fla.h), natively: argument tests, output and
// workspace allocation, the call, and the autograd node whose backward runs without the interpreter.
//
// A small problem is bound by this path, not by its kernels (forward + backward of B 1, H 2, N 256,
// D 64: 5 + 7 us of kernels).  With the same steps in Python (torch.autograd.Function, ctypes) the pair
// took 55 us on one host and 113 us on a slower one, of which most is interpreter work on two threads that
// hand the interpreter lock to each other.
//
// Every entry point returns None where a call is not the plain case (tensor types and shapes that
// the operator refuses or converts, wrapped tensors, forward-mode tangents, torch.jit.trace, a status other
// than FLA_OK): the Python class then runs its own forward, which raises what there is to raise.
#include <Python.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/types.h>
#include <ATen/autocast_mode.h>
#include <torch/custom_class.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#include <tuple>
#include <utility>
#include <vector>

#include "fla.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::variable_list;

struct Refused : std::runtime_error {  // the library returned a status: the Python path reports it
    explicit Refused(int status) : std::runtime_error(fla_strerror(status)) {}
};

void must(int status) {
    if (status != FLA_OK) throw Refused(status);
}

int dtype_code(at::ScalarType t) {
    return t == at::kBFloat16 ? FLA_DTYPE_BF16 : t == at::kHalf ? FLA_DTYPE_F16 : -1;
}

// Calls in flight on a device: its guard, the current stream and uninitialised tensors on it.
struct Call {
    c10::DeviceGuard guard;
    at::TensorOptions like;
    void *stream;
    int64_t b, h, n, dqk, dv;
    int dtype;
    Call(const Tensor &q, const Tensor &v)
        : guard(q.device()), like(q.options().requires_grad(false)),
          stream(c10::hip::getCurrentHIPStream(q.device().index()).stream()), b(q.size(0)), h(q.size(1)), n(q.size(2)),
          dqk(q.size(3)), dv(v.size(3)), dtype(dtype_code(q.scalar_type())) {}
    Tensor rows(int64_t width) const { return at::empty({b, h, n, width}, like); }
    Tensor row_floats() const { return at::empty({b, h, n}, like.dtype(at::kFloat)); }
    bool grads_f32(bool plain, bool state) const { return fla_linear_attn_chunked_grads_f32(b, h, n, dqk, dv, plain, state) != 0; }
    // (a quadratic product of widths off the eights: the workspace of fla_linear_attn_copies_fwd / _bwd, 0 where those are not taken)
    int64_t copies(bool backward) const {
        if (dqk % 8 == 0 && dv % 8 == 0) return 0;
        return fla_linear_attn_operator_prefers_copies(b, h, n, dqk, dv, backward) ? fla_linear_attn_copies_bytes(b, h, n, dqk, dv, backward) : 0;
    }
    Tensor bytes(int64_t count) const { return count ? at::empty({count}, like.dtype(at::kByte)) : Tensor(); }
};

void *ptr(const Tensor &t) { return t.defined() ? t.data_ptr() : nullptr; }
const int64_t *str(const Tensor &t) { return t.strides().data(); }
int64_t size_of(const Tensor &t) { return t.defined() ? t.numel() : 0; }

// (the innermost dimension dense: what the library asks of every operand)
Tensor dense(const Tensor &t) { return t.stride(3) != 1 && t.size(3) > 1 ? t.contiguous() : t; }

// Whether the walks' tile loads take a tensor's rows as they are (others go product by product)
bool rows_for_walks(const Tensor &t) {
    if (t.stride(3) != 1) return true;  // (dense() copies it)
    for (int i = 0; i < 3; ++i)
        if (t.stride(i) % 8 != 0) return false;
    return (uintptr_t)t.data_ptr() % 16 == 0 && t.stride(2) >= t.size(3) && t.size(2) * t.stride(2) < (int64_t(1) << 28);
}

// ---- tests of a call's tensors

bool plain(const Tensor &t) {
    using K = c10::DispatchKey;
    static const c10::DispatchKeySet odd({K::Python, K::PythonTLSSnapshot, K::FuncTorchBatched, K::FuncTorchGradWrapper,
                                          K::Functionalize, K::Conjugate, K::Negative, K::ZeroTensor});
    // (a forward-mode tangent: the operators have no formula for it, and the Python class says so)
    return t.defined() && t.is_cuda() && t.layout() == at::kStrided && t.dim() == 4 && !t.key_set().has_any(odd) &&
           !t._fw_grad(/*level=*/0).defined();
}

// q, k: (B, H, N, D_qk), v: (B, H, N, D_v), one device; `cast`: autocast turns any floating type into bf16
bool agree(const Tensor &q, const Tensor &k, const Tensor &v, bool cast) {
    if (!plain(q) || !plain(k) || !plain(v) || k.device() != q.device() || v.device() != q.device()) return false;
    if (q.sizes() != k.sizes() || v.size(0) != q.size(0) || v.size(1) != q.size(1) || v.size(2) != q.size(2)) return false;
    if (q.size(3) < 1 || v.size(3) < 1 || q.numel() == 0) return false;
    auto castable = [](at::ScalarType t) { return t == at::kFloat || t == at::kBFloat16 || t == at::kHalf; };
    if (cast) return castable(q.scalar_type()) && castable(k.scalar_type()) && castable(v.scalar_type());
    return dtype_code(q.scalar_type()) >= 0 && k.scalar_type() == q.scalar_type() && v.scalar_type() == q.scalar_type();
}

// Operands as the kernels take them.  `cast` (autocast): in bf16, the fp32 ones in one launch; `widened` remembers which
// came in fp32, so that their gradients leave in fp32 from one launch too (the engine would convert them one by one).
struct Casts {
    Tensor q, k, v;
    int64_t widened = 0;
    Casts(const Tensor &q_, const Tensor &k_, const Tensor &v_, bool cast) : q(q_), k(k_), v(v_) {
        if (!cast) return;
        at::AutoDispatchBelowADInplaceOrView below;
        Tensor *all[3] = {&q, &k, &v}, out[3];
        const void *src[3];
        void *dst[3];
        int64_t count[3];
        int n = 0;
        for (int i = 0; i < 3; ++i) {
            const Tensor &t = *all[i];
            if (t.scalar_type() == at::kFloat) widened |= 1 << i;
            if (t.scalar_type() == at::kFloat && t.is_non_overlapping_and_dense() && (uintptr_t)t.data_ptr() % 16 == 0) {
                out[i] = at::empty_strided(t.sizes(), t.strides(), t.options().dtype(at::kBFloat16));
                src[n] = t.data_ptr(), dst[n] = out[i].data_ptr(), count[n++] = t.numel();
            } else {
                out[i] = t.to(at::kBFloat16);
            }
        }
        if (n) {
            const c10::DeviceGuard guard(q.device());
            must(fla_convert(src, dst, count, n, 0, FLA_DTYPE_BF16, c10::hip::getCurrentHIPStream(q.device().index()).stream()));
        }
        q = out[0], k = out[1], v = out[2];
    }
};

// A chunk-wise backward: allocates the gradients and makes `call(dq, dk, dv, dtype)`.  For inputs that all came in fp32
// (`widened` == 7) the gradients are stored in fp32 where the library's kernels can do so; `sizes`: they can for these sizes (what is
// refused then is an operand's alignment, and asked for again in 16 bits.  To find out by a refusal for every shape cost the shapes
// without such a kernel 2 us of the host, three allocations and a call: B 1 H 2 N 100 D 64 51.5 -> 53.9 us).
template <typename Backward>
variable_list chunked_gradients(const Call &c, int64_t widened, bool sizes, Backward &&call) {
    for (bool wide = widened == 7 && sizes && c.dtype == FLA_DTYPE_BF16;; wide = false) {
        const at::TensorOptions as = wide ? c.like.dtype(at::kFloat) : c.like;
        const Tensor dq = at::empty({c.b, c.h, c.n, c.dqk}, as), dk = at::empty({c.b, c.h, c.n, c.dqk}, as),
                     dv = at::empty({c.b, c.h, c.n, c.dv}, as);
        const int status = call(dq, dk, dv, c.dtype | (wide ? FLA_GRADS_F32 : 0));
        if (wide && status == FLA_ERR_UNSUPPORTED) continue;
        must(status);
        return {dq, dk, dv};
    }
}

// gradients of the inputs that came in fp32, in fp32
void widen(variable_list &g, int64_t which) {
    if (!which || g[0].scalar_type() == at::kFloat) return;  // (already: FLA_GRADS_F32)
    at::AutoDispatchBelowADInplaceOrView below;
    const void *src[3];
    void *dst[3];
    int64_t count[3];
    int n = 0;
    const c10::DeviceGuard guard(g[0].device());
    variable_list out = g;
    for (int i = 0; i < 3; ++i)
        if (which >> i & 1) {
            out[i] = at::empty(g[i].sizes(), g[i].options().dtype(at::kFloat));
            src[n] = g[i].data_ptr(), dst[n] = out[i].data_ptr(), count[n++] = g[i].numel();
        }
    must(fla_convert(src, dst, count, n, 1, dtype_code(g[0].scalar_type()),
                     c10::hip::getCurrentHIPStream(g[0].device().index()).stream()));
    g = std::move(out);
}

bool wants_grad(const Tensor &q, const Tensor &k, const Tensor &v) {
    return at::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() || v.requires_grad());
}

// ---- tril(Q K^T) V

// (kChosen: chunk-wise because the shape says so, with the quadratic evaluation's causality of dQ; kWalks: and, an fp16 pair, by the walks,
// which alone keep the quadratic evaluation's range)
enum Evaluation { kEqual = 0, kSmallV = 1, kChunked = 2, kChosen = 3, kWalks = 4 };

std::tuple<Tensor, Tensor> product_fwd(const Tensor &q_, const Tensor &k_, const Tensor &v_, int ev, bool want_state) {
    at::AutoDispatchBelowADInplaceOrView below;
    const Tensor q = dense(q_), k = dense(k_), v = dense(v_);
    const Call c(q, v);
    Tensor o = c.rows(c.dv), state;
    if (const int64_t bytes = ev == kEqual || ev == kSmallV ? c.copies(false) : 0) {
        const Tensor work = c.bytes(bytes);
        must(fla_linear_attn_copies_fwd(ptr(q), ptr(k), ptr(v), ptr(o), c.b, c.h, c.n, c.dqk, c.dv, str(q), str(k), str(v), str(o),
                                        c.dtype, ptr(work), bytes, c.stream));
    } else if (ev == kEqual) {
        must(fla_linear_attn_fwd(ptr(q), ptr(k), ptr(v), ptr(o), c.b, c.h, c.n, c.dqk, str(q), str(k), str(v), str(o), c.dtype,
                                 c.stream));
    } else if (ev == kSmallV) {
        must(fla_linear_attn_smallv_fwd(ptr(q), ptr(k), ptr(v), ptr(o), c.b, c.h, c.n, c.dqk, c.dv, str(q), str(k), str(v),
                                        str(o), c.dtype, c.stream));
    } else {
        if (want_state) state = c.bytes(fla_linear_attn_chunked_state_bytes(c.b, c.h, c.n, c.dqk, c.dv));
        const Tensor work = c.bytes(fla_linear_attn_chunked_fwd_workspace_bytes(c.b, c.h, c.n, c.dqk, c.dv, state.defined()));
        int32_t valid = 0;
        must(fla_linear_attn_chunked_fwd(ptr(q), ptr(k), ptr(v), ptr(o), c.b, c.h, c.n, c.dqk, c.dv, str(q), str(k), str(v),
                                         str(o), c.dtype, ptr(state), &valid, ptr(work), size_of(work), c.stream));
        if (!valid) state = Tensor();
    }
    return {o, state};
}

variable_list product_bwd(const Tensor &go_, const Tensor &q_, const Tensor &k_, const Tensor &v_, const Tensor &state, int ev,
                          int64_t widened) {
    at::AutoDispatchBelowADInplaceOrView below;
    // (kWalks: a gradient whose rows their loads do not take is copied; other calls, widths off the eights among them, go as they come)
    auto rows = [&](const Tensor &t) {
        const Tensor d = dense(t);
        return ev != kWalks || rows_for_walks(d) ? d : d.clone(at::MemoryFormat::Contiguous);
    };
    const Tensor go = rows(go_), q = rows(q_), k = rows(k_), v = rows(v_);
    const Call c(q, v);
    if (ev == kChunked || ev == kChosen || ev == kWalks) {
        const Tensor work = c.bytes(fla_linear_attn_chunked_workspace_bytes(c.b, c.h, c.n, c.dqk, c.dv));
        return chunked_gradients(c, widened, c.grads_f32(true, state.defined()), [&](const Tensor &dq, const Tensor &dk, const Tensor &dv, int dtype) {
            return (ev == kChunked ? fla_linear_attn_chunked_bwd : fla_linear_attn_chunked_bwd_causal)(
                ptr(go), ptr(q), ptr(k), ptr(v), ptr(dq), ptr(dk), ptr(dv), c.b, c.h, c.n, c.dqk, c.dv, str(go), str(q), str(k),
                str(v), str(dq), str(dk), str(dv), dtype, ptr(state), ptr(work), size_of(work), c.stream);
        });
    }
    Tensor dq = c.rows(c.dqk), dk = c.rows(c.dqk), dv = c.rows(c.dv);
    if (const int64_t bytes = c.copies(true)) {
        const Tensor work = c.bytes(bytes);
        must(fla_linear_attn_copies_bwd(ptr(go), ptr(q), ptr(k), ptr(v), ptr(dq), ptr(dk), ptr(dv), c.b, c.h, c.n, c.dqk, c.dv, str(go),
                                        str(q), str(k), str(v), str(dq), str(dk), str(dv), c.dtype, ptr(work), bytes, c.stream));
    } else if (ev == kEqual) {
        must(fla_linear_attn_bwd(ptr(go), ptr(q), ptr(k), ptr(v), ptr(dq), ptr(dk), ptr(dv), c.b, c.h, c.n, c.dqk, str(go),
                                 str(q), str(k), str(v), str(dq), str(dk), str(dv), c.dtype, c.stream));
    } else {
        must(fla_linear_attn_smallv_bwd(ptr(go), ptr(q), ptr(k), ptr(v), ptr(dq), ptr(dk), ptr(dv), c.b, c.h, c.n, c.dqk, c.dv,
                                        str(go), str(q), str(k), str(v), str(dq), str(dk), str(dv), c.dtype, c.stream));
    }
    return {dq, dk, dv};
}

// Operands that a node does not keep: backward is refused all the same once one of them was written to in place
struct Unkept : torch::CustomClassHolder {
    std::vector<std::pair<c10::VariableVersion, uint32_t>> seen;
    void add(const Tensor &t) {
        const c10::VariableVersion &version = t.unsafeGetTensorImpl()->version_counter();
        if (version.enabled()) seen.emplace_back(version, version.current_version());
    }
    void check() const {
        for (const auto &[version, then] : seen)
            TORCH_CHECK(version.current_version() == then, "one of the variables needed for gradient computation has been "
                        "modified by an inplace operation: it is at version ", version.current_version(),
                        "; expected version ", then, " instead");
    }
};

struct Product : Function<Product> {
    static Tensor forward(AutogradContext *ctx, const Tensor &q_, const Tensor &k_, const Tensor &v_, int64_t ev, bool cast) {
        const Casts in(q_, k_, v_, cast);
        const Tensor &q = in.q, &k = in.k, &v = in.v;
        ctx->saved_data["widened"] = in.widened;
        auto [o, state] = product_fwd(q, k, v, (int)ev, true);
        ctx->saved_data["ev"] = ev;
        variable_list s = {q, k, v};
        if (state.defined()) {
            // (copies with aligned rows in the state buffer are what backward reads: kept in place of the operands)
            int64_t at[3], pitch[3];
            const int64_t b = q.size(0), h = q.size(1), n = q.size(2);
            if (fla_linear_attn_chunked_state_operands(b, h, n, q.size(3), v.size(3), at, pitch)) {
                at::AutoDispatchBelowADInplaceOrView below;
                auto unkept = c10::make_intrusive<Unkept>();
                for (int i = 0; i < 3; ++i)
                    if (at[i] >= 0) {
                        unkept->add(s[i]);
                        s[i] = state.narrow(0, at[i], 2 * b * h * n * pitch[i]).view(q.scalar_type()).view({b, h, n, pitch[i]})
                                   .narrow(3, 0, s[i].size(3));
                    }
                ctx->saved_data["unkept"] = c10::IValue::make_capsule(std::move(unkept));
            }
            s.push_back(state);
        }
        ctx->save_for_backward(std::move(s));
        return o;
    }
    static variable_list backward(AutogradContext *ctx, variable_list go) {
        const variable_list s = ctx->get_saved_variables();
        if (const auto unkept = ctx->saved_data.find("unkept"); unkept != ctx->saved_data.end())
            c10::static_intrusive_pointer_cast<Unkept>(unkept->second.toCapsule())->check();
        const int64_t widened = ctx->saved_data["widened"].toInt();
        variable_list g =
            product_bwd(go[0], s[0], s[1], s[2], s.size() > 3 ? s[3] : Tensor(), (int)ctx->saved_data["ev"].toInt(), widened);
        widen(g, widened);
        g.resize(5);
        return g;
    }
};

// ---- the normalised operator, without and with a feature map; the feature map alone

struct Options {
    int fmap;  // 0: none
    bool normalise;
    int chunked;  // 0, 1 or FLA_CHUNKED_PRODUCTS
    double eps;
    int64_t code() const { return fmap | (normalise ? 16 : 0) | chunked << 5; }
    static Options of(int64_t code) { return {(int)(code & 15), (code & 16) != 0, (int)(code >> 5), 0.0}; }
};

struct MappedResult {
    Tensor o, q, k, denom, state;  // q, k: phi(xq), phi(xk) with a feature map
};

MappedResult mapped_fwd(const Tensor &q_, const Tensor &k_, const Tensor &v_, const Options &opt, bool want_state) {
    at::AutoDispatchBelowADInplaceOrView below;
    const Tensor q = dense(q_), k = dense(k_), v = dense(v_);
    const Call c(q, v);
    MappedResult r;
    r.o = c.rows(c.dv);
    if (opt.fmap) r.q = c.rows(c.dqk), r.k = c.rows(c.dqk);
    if (want_state && opt.chunked) r.state = c.bytes(fla_linear_attn_chunked_state_bytes(c.b, c.h, c.n, c.dqk, c.dv));
    int32_t valid = 0;
    if (opt.normalise) {
        r.denom = c.row_floats();
        const Tensor work = c.bytes(fla_normalised_workspace_bytes(c.b, c.h, c.n, c.dqk, c.dv, opt.chunked));
        if (opt.fmap)
            must(fla_feature_attn_normalised_fwd(ptr(q), ptr(k), ptr(v), ptr(r.o), ptr(r.q), ptr(r.k), r.denom.data_ptr<float>(),
                                                 c.b, c.h, c.n, c.dqk, c.dv, str(q), str(k), str(v), str(r.o), str(r.q),
                                                 str(r.k), opt.fmap, (float)opt.eps, c.dtype, opt.chunked, ptr(r.state), &valid,
                                                 ptr(work), size_of(work), c.stream));
        else
            must(fla_linear_attn_normalised_fwd(ptr(q), ptr(k), ptr(v), ptr(r.o), r.denom.data_ptr<float>(), c.b, c.h, c.n,
                                                c.dqk, c.dv, str(q), str(k), str(v), str(r.o), (float)opt.eps, c.dtype,
                                                opt.chunked, ptr(r.state), &valid, ptr(work), size_of(work), c.stream));
    } else {
        const Tensor work = c.bytes(fla_linear_attn_chunked_workspace_bytes(c.b, c.h, c.n, c.dqk, c.dv));
        must(fla_feature_attn_fwd(ptr(q), ptr(k), ptr(v), ptr(r.o), ptr(r.q), ptr(r.k), c.b, c.h, c.n, c.dqk, c.dv, str(q),
                                  str(k), str(v), str(r.o), str(r.q), str(r.k), opt.fmap, c.dtype, ptr(r.state), &valid,
                                  ptr(work), size_of(work), c.stream));
    }
    if (!valid) r.state = Tensor();
    return r;
}

variable_list mapped_bwd(const Tensor &go_, const Tensor &q_, const Tensor &k_, const Tensor &v_, const Tensor &o,
                         const Tensor &denom, const Tensor &state, const Options &opt, int64_t widened) {
    at::AutoDispatchBelowADInplaceOrView below;
    const Tensor go = dense(go_), q = dense(q_), k = dense(k_), v = dense(v_);
    const Call c(q, v);
    const float *n = opt.normalise ? denom.data_ptr<float>() : nullptr;
    const Tensor work = c.bytes(opt.normalise ? fla_normalised_workspace_bytes(c.b, c.h, c.n, c.dqk, c.dv, opt.chunked)
                                              : fla_linear_attn_chunked_workspace_bytes(c.b, c.h, c.n, c.dqk, c.dv));
    return chunked_gradients(c, widened, (opt.chunked == 1 || !opt.normalise) && c.grads_f32(false, state.defined()),
                             [&](const Tensor &dq, const Tensor &dk, const Tensor &dv, int dtype) {
        if (!opt.normalise)
            return fla_feature_attn_bwd(ptr(go), ptr(q), ptr(k), ptr(v), ptr(dq), ptr(dk), ptr(dv), c.b, c.h, c.n, c.dqk, c.dv,
                                        str(go), str(q), str(k), str(v), str(dq), str(dk), str(dv), opt.fmap, dtype, ptr(state),
                                        ptr(work), size_of(work), c.stream);
        if (opt.fmap)
            return fla_feature_attn_normalised_bwd(ptr(go), ptr(q), ptr(k), ptr(v), ptr(o), n, ptr(dq), ptr(dk), ptr(dv), c.b, c.h,
                                                   c.n, c.dqk, c.dv, str(go), str(q), str(k), str(v), str(o), str(dq), str(dk),
                                                   str(dv), opt.fmap, dtype, opt.chunked, ptr(state), ptr(work), size_of(work),
                                                   c.stream);
        return fla_linear_attn_normalised_bwd(ptr(go), ptr(q), ptr(k), ptr(v), ptr(o), n, ptr(dq), ptr(dk), ptr(dv), c.b, c.h, c.n,
                                              c.dqk, c.dv, str(go), str(q), str(k), str(v), str(o), str(dq), str(dk), str(dv),
                                              dtype, opt.chunked, ptr(state), ptr(work), size_of(work), c.stream);
    });
}

struct Mapped : Function<Mapped> {
    static Tensor forward(AutogradContext *ctx, const Tensor &q_, const Tensor &k_, const Tensor &v_, int64_t code, double eps,
                          bool cast) {
        Options opt = Options::of(code);
        opt.eps = eps;
        const Casts in(q_, k_, v_, cast);
        const Tensor &q = in.q, &k = in.k, &v = in.v;
        ctx->saved_data["widened"] = in.widened;
        MappedResult r = mapped_fwd(q, k, v, opt, true);
        ctx->saved_data["opt"] = code;
        variable_list s = {opt.fmap ? r.q : q, opt.fmap ? r.k : k, v};
        if (opt.normalise) s.push_back(r.o), s.push_back(r.denom);
        if (r.state.defined()) s.push_back(r.state);
        ctx->save_for_backward(std::move(s));
        return r.o;
    }
    static variable_list backward(AutogradContext *ctx, variable_list go) {
        const Options opt = Options::of(ctx->saved_data["opt"].toInt());
        const variable_list s = ctx->get_saved_variables();
        const size_t base = opt.normalise ? 5 : 3;
        const int64_t widened = ctx->saved_data["widened"].toInt();
        variable_list g = mapped_bwd(go[0], s[0], s[1], s[2], opt.normalise ? s[3] : Tensor(), opt.normalise ? s[4] : Tensor(),
                                     s.size() > base ? s[base] : Tensor(), opt, widened);
        widen(g, widened);
        g.resize(6);
        return g;
    }
};

// ---- the polynomial score map

struct Poly {
    float c[3];
    bool normalise;
    float eps;
};

struct PolyResult {
    Tensor o, denom, state;  // state: of the chunk-wise evaluation, for its backward
};

PolyResult poly_fwd(const Tensor &q_, const Tensor &k_, const Tensor &v_, const Poly &p, bool want_state) {
    at::AutoDispatchBelowADInplaceOrView below;
    const Tensor q = dense(q_), k = dense(k_), v = dense(v_);
    const Call c(q, v);
    PolyResult r;
    r.o = c.rows(c.dv);
    if (p.normalise) r.denom = c.row_floats();
    float *n = static_cast<float *>(ptr(r.denom));
    if (fla_poly_attn_operator_prefers_chunked(c.b, c.h, c.n, c.dqk, c.dv, c.dtype, want_state, p.normalise)) {
        if (want_state) r.state = c.bytes(fla_poly_attn_chunked_state_bytes(c.b, c.h, c.n, c.dqk, c.dv));
        const Tensor work = c.bytes(fla_poly_attn_chunked_fwd_workspace_bytes(c.b, c.h, c.n, c.dqk, c.dv));
        must(fla_poly_attn_chunked_fwd(ptr(q), ptr(k), ptr(v), ptr(r.o), n, c.b, c.h, c.n, c.dqk, c.dv, str(q), str(k), str(v),
                                       str(r.o), p.c, p.eps, c.dtype, ptr(r.state), ptr(work), size_of(work), c.stream));
    } else {
        must(fla_poly_attn_fwd(ptr(q), ptr(k), ptr(v), ptr(r.o), n, c.b, c.h, c.n, c.dqk, c.dv, str(q), str(k), str(v), str(r.o),
                               p.c, p.eps, c.dtype, c.stream));
    }
    return r;
}

variable_list poly_bwd(const Tensor &go_, const Tensor &q_, const Tensor &k_, const Tensor &v_, const Tensor &o,
                       const Tensor &denom, const Tensor &state, const Poly &p, int64_t widened) {
    at::AutoDispatchBelowADInplaceOrView below;
    const Tensor go = dense(go_), q = dense(q_), k = dense(k_), v = dense(v_);
    const Call c(q, v);
    const float *n = static_cast<const float *>(ptr(denom));
    const int64_t *os = o.defined() ? str(o) : nullptr;
    if (state.defined()) {
        const Tensor work = c.bytes(fla_poly_attn_chunked_workspace_bytes(c.b, c.h, c.n, c.dqk, c.dv));
        return chunked_gradients(c, widened, true, [&](const Tensor &dq, const Tensor &dk, const Tensor &dv, int dtype) {
            return fla_poly_attn_chunked_bwd(ptr(go), ptr(q), ptr(k), ptr(v), ptr(o), n, ptr(dq), ptr(dk), ptr(dv), c.b, c.h, c.n,
                                             c.dqk, c.dv, str(go), str(q), str(k), str(v), os, str(dq), str(dk), str(dv), p.c,
                                             dtype, ptr(state), ptr(work), size_of(work), c.stream);
        });
    }
    Tensor dq = c.rows(c.dqk), dk = c.rows(c.dqk), dv = c.rows(c.dv);
    const Tensor work = c.bytes(fla_poly_attn_workspace_bytes(c.b, c.h, c.n, c.dqk, c.dv));
    must(fla_poly_attn_bwd(ptr(go), ptr(q), ptr(k), ptr(v), ptr(o), n, ptr(dq), ptr(dk), ptr(dv), c.b, c.h, c.n, c.dqk, c.dv,
                           str(go), str(q), str(k), str(v), os, str(dq), str(dk), str(dv), p.c, c.dtype, ptr(work),
                           size_of(work), c.stream));
    return {dq, dk, dv};
}

struct Polynomial : Function<Polynomial> {
    static Tensor forward(AutogradContext *ctx, const Tensor &q_, const Tensor &k_, const Tensor &v_, double c0, double c1,
                          double c2, bool normalise, double eps, bool cast) {
        const Casts in(q_, k_, v_, cast);
        const Tensor &q = in.q, &k = in.k, &v = in.v;
        ctx->saved_data["widened"] = in.widened;
        PolyResult r = poly_fwd(q, k, v, Poly{{(float)c0, (float)c1, (float)c2}, normalise, (float)eps}, true);
        ctx->saved_data["c0"] = c0, ctx->saved_data["c1"] = c1, ctx->saved_data["c2"] = c2, ctx->saved_data["n"] = normalise;
        variable_list s = {q, k, v};
        if (normalise) s.push_back(r.o), s.push_back(r.denom);
        if (r.state.defined()) s.push_back(r.state);
        ctx->save_for_backward(std::move(s));
        return r.o;
    }
    static variable_list backward(AutogradContext *ctx, variable_list go) {
        const variable_list s = ctx->get_saved_variables();
        const bool normalise = ctx->saved_data["n"].toBool();
        const size_t base = normalise ? 5 : 3;
        auto c = [&](const char *key) { return (float)ctx->saved_data[key].toDouble(); };
        const int64_t widened = ctx->saved_data["widened"].toInt();
        variable_list g = poly_bwd(go[0], s[0], s[1], s[2], normalise ? s[3] : Tensor(), normalise ? s[4] : Tensor(),
                                   s.size() > base ? s[base] : Tensor(), Poly{{c("c0"), c("c1"), c("c2")}, normalise, 0.f}, widened);
        widen(g, widened);
        g.resize(9);
        return g;
    }
};

// ---- Python entry points: each takes q, k, v and plain numbers, and returns a tensor or None

struct Operands {
    Tensor q, k, v;
    bool cast = false, ok = false;
};

Operands operands(PyObject *const *args) {
    Operands a;
    // (torch.jit.trace records the Python Function as a whole; of the calls made here it would see the allocations alone)
    if (torch::jit::tracer::isTracing()) return a;
    if (!THPVariable_Check(args[0]) || !THPVariable_Check(args[1]) || !THPVariable_Check(args[2])) return a;
    a.q = THPVariable_Unpack(args[0]), a.k = THPVariable_Unpack(args[1]), a.v = THPVariable_Unpack(args[2]);
    a.cast = at::autocast::is_autocast_enabled(at::kCUDA);
    a.ok = agree(a.q, a.k, a.v, a.cast);
    return a;
}

template <typename Run>
PyObject *released(Run &&run) {  // (allocation and launches without the interpreter lock)
    Tensor out;
    {
        PyThreadState *ts = PyEval_SaveThread();
        try {
            out = run();
        } catch (const Refused &) {  // (out stays undefined)
        } catch (...) {
            PyEval_RestoreThread(ts);
            throw;
        }
        PyEval_RestoreThread(ts);
    }
    if (!out.defined()) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(out));
}

bool pow2(int64_t x) { return (x & (x - 1)) == 0; }
int64_t next_pow2(int64_t x) {
    int64_t p = 1;
    while (p < x) p <<= 1;
    return p;
}

// product(kind, q, k, v): kind 0 LinearAttention, 1 LinearAttentionSmallVHD, 2 LinearAttentionAuto, 3 LinearAttentionChunked
PyObject *py_product(PyObject *, PyObject *const *args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 4) Py_RETURN_NONE;
    const long kind = PyLong_AsLong(args[0]);
    const Operands a = operands(args + 1);
    if (!a.ok) Py_RETURN_NONE;
    const int64_t rows = a.q.size(2), dqk = a.q.size(3), dv = a.v.size(3);
    if (dqk > 256 || dv > 256) Py_RETURN_NONE;
    const bool bf16 = a.cast || a.q.scalar_type() == at::kBFloat16, equal = dqk == dv;
    const bool grad = wants_grad(a.q, a.k, a.v);
    auto prefers = [&] {
        return fla_linear_attn_operator_prefers_chunked(a.q.size(0), a.q.size(1), rows, dqk, dv, grad) != 0;
    };
    // (fp16: auto.py, chunked_keeps_range; with gradients from rows that the walks take, which scale their states in both directions)
    const bool range = bf16 || (!grad ? dqk <= 128 && dv <= 128 && dqk % 8 == 0 && dv % 8 == 0 && rows > 256
                                      : fla_linear_attn_f16_pair_prefers_chunked(a.q.size(0), a.q.size(1), rows, dqk, dv) &&
                                            rows_for_walks(a.q) && rows_for_walks(a.k) && rows_for_walks(a.v));
    // (a v above 128 columns: chunk-wise where every sum is rounded once, beside a q / k above 128 too)
    const bool once = dv <= 128 || (dqk > 128 && dqk % 8 == 0 && dv % 8 == 0);
    const int chosen = !bf16 && grad && range ? kWalks : kChosen;
    int ev = equal ? kEqual : kSmallV;
    if (kind == 0) {  // (the shapes its forward takes, and its choice: linear_attn.py)
        if (!equal || rows % (dqk > 128 ? 32 : 64) != 0) Py_RETURN_NONE;
        if (range && once && prefers()) ev = chosen;
    } else if (kind == 1) {  // (linear_attn_smallv_hd.py)
        if (!pow2(dv) || dv > next_pow2(dqk) || rows % 64 != 0) Py_RETURN_NONE;
        ev = range && once && prefers() ? chosen : kSmallV;
    } else if (kind == 2) {  // (auto.py)
        if (rows % 64 != 0 || (!equal && (dv > dqk || !pow2(dv))) || (range && prefers())) ev = chosen;
    } else {
        ev = kChunked;
    }
    return released([&]() -> Tensor {
        if (wants_grad(a.q, a.k, a.v)) return Product::apply(a.q, a.k, a.v, (int64_t)ev, a.cast);
        const Casts in(a.q, a.k, a.v, a.cast);
        return std::get<0>(product_fwd(in.q, in.k, in.v, ev, false));
    });
    END_HANDLE_TH_ERRORS
}

// mapped(q, k, v, feature map code, normalise, eps, chunked)
PyObject *py_mapped(PyObject *, PyObject *const *args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 7) Py_RETURN_NONE;
    const Operands a = operands(args);
    if (!a.ok || a.q.size(3) > 256 || a.v.size(3) > 256) Py_RETURN_NONE;
    Options opt;
    opt.fmap = (int)PyLong_AsLong(args[3]);
    opt.normalise = PyObject_IsTrue(args[4]) == 1, opt.eps = PyFloat_AsDouble(args[5]), opt.chunked = PyObject_IsTrue(args[6]) == 1 ? 1 : 0;
    if (PyErr_Occurred()) {  // (not numbers: the Python path says so)
        PyErr_Clear();
        Py_RETURN_NONE;
    }
    if (!opt.fmap && opt.normalise && !opt.chunked) {  // (normalised.py)
        const int dtype = a.cast ? FLA_DTYPE_BF16 : dtype_code(a.q.scalar_type());
        const bool grad = wants_grad(a.q, a.k, a.v);
        const int prefers = (grad ? fla_normalised_prefers_chunked : fla_normalised_forward_prefers_chunked)(
            a.q.size(0), a.q.size(1), a.q.size(2), a.q.size(3), a.v.size(3), dtype);
        opt.chunked = !prefers ? 0 : grad ? FLA_CHUNKED_PRODUCTS : 1;
    }
    return released([&]() -> Tensor {
        if (wants_grad(a.q, a.k, a.v)) return Mapped::apply(a.q, a.k, a.v, opt.code(), opt.eps, a.cast);
        const Casts in(a.q, a.k, a.v, a.cast);
        return mapped_fwd(in.q, in.k, in.v, opt, false).o;
    });
    END_HANDLE_TH_ERRORS
}

// polynomial(xq, xk, v, c0, c1, c2, normalise, eps)
PyObject *py_polynomial(PyObject *, PyObject *const *args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 8) Py_RETURN_NONE;
    const Operands a = operands(args);
    if (!a.ok || a.q.size(3) > 32 || a.q.size(3) % 8 != 0 || a.v.size(3) > 128 || a.v.size(3) % 8 != 0) Py_RETURN_NONE;
    double c[3];
    for (int i = 0; i < 3; ++i) c[i] = PyFloat_AsDouble(args[3 + i]);
    const bool normalise = PyObject_IsTrue(args[6]) == 1;
    const double eps = PyFloat_AsDouble(args[7]);
    if (PyErr_Occurred()) {
        PyErr_Clear();
        Py_RETURN_NONE;
    }
    return released([&]() -> Tensor {
        if (wants_grad(a.q, a.k, a.v)) return Polynomial::apply(a.q, a.k, a.v, c[0], c[1], c[2], normalise, eps, a.cast);
        const Casts in(a.q, a.k, a.v, a.cast);
        return poly_fwd(in.q, in.k, in.v,
                        Poly{{(float)c[0], (float)c[1], (float)c[2]}, normalise, (float)eps}, false).o;
    });
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"product", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_product)), METH_FASTCALL, nullptr},
    {"mapped", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_mapped)), METH_FASTCALL, nullptr},
    {"polynomial", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_polynomial)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fla_torch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fla_torch() { return PyModule_Create(&module); }
