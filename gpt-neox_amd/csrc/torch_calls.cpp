// The calls that a training or generation step makes most, from Python into the kernels without a detour:
// allocation, launch and autograd bookkeeping in native code.  A call of a few microseconds on the GPU used
// to spend 40 to 140 us of the host's time in Python autograd Functions and ctypes.
//
// Every function serves the plain form of its call and returns None for any other -- unusual layouts, types,
// devices, and everything that has to be refused --, for which the Python modules keep their general path with its
// checks and messages.  The kernels are those of include/neox_fused.h.  Nothing is kept between calls: what a
// backward pass needs is saved through autograd, under its version checks and saved-tensor hooks.
#include <torch/extension.h>
#include <torch/version.h>

#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#include <optional>
#include <stdexcept>
#include <string>
#include <tuple>

#include "../../include/neox_fused.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

void check(int status) {
    if (status == NEOX_OK) return;
    const char* message = neox_fused_last_error();
    throw std::runtime_error(*message ? message : neox_fused_strerror(status));
}

bool half_type(const Tensor& t) { return t.scalar_type() == at::kHalf || t.scalar_type() == at::kBFloat16; }
int32_t code(const Tensor& t) {
    switch (t.scalar_type()) {
        case at::kHalf: return NEOX_F16;
        case at::kBFloat16: return NEOX_BF16;
        case at::kFloat: return NEOX_F32;
        default: throw std::runtime_error("Only fp16 and bf16 are supported");
    }
}
void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
bool fits_int32(int64_t n) { return n >= 0 && n <= INT32_MAX; }
bool records(const Tensor& t) { return at::GradMode::is_enabled() && t.requires_grad(); }
// a tensor whose memory this code may look at
bool on_gpu(const Tensor& t) { return t.defined() && t.is_cuda() && t.layout() == at::kStrided && !t.is_neg() && !t.is_conj(); }
// ... and that a call may be served for: one with a forward-mode tangent goes to the Python autograd Functions,
// which refuse it (a result computed here would have lost the tangent)
bool plain(const Tensor& t) { return on_gpu(t) && !t._fw_grad(/*level=*/0).defined(); }

// ---- softmax ---------------------------------------------------------------------------------------
enum Kind : int64_t { kCausal = -1, kMasked = -2 };  // a window width otherwise

struct SoftmaxCall {
    double scale;
    int64_t kind;
    const Tensor* mask;    // kMasked
    const Tensor* slopes;  // kCausal, optional
    double p;              // kCausal: attention dropout, 0 = none
    int64_t seed, offset;
};

// probabilities, and the dropped ones (undefined without dropout); x is contiguous [b, np, sq, sk]
std::tuple<Tensor, Tensor> softmax_forward(const Tensor& x, const SoftmaxCall& c) {
    const c10::DeviceGuard guard(x.device());
    const auto b = (int32_t)x.size(0), np = (int32_t)x.size(1), sq = (int32_t)x.size(2), sk = (int32_t)x.size(3);
    Tensor y = at::empty_like(x), dropped;
    const auto scale = (float)c.scale;
    const void* in = x.const_data_ptr();
    void *out = y.mutable_data_ptr(), *stream = stream_of(x);
    const float* slopes = c.slopes ? static_cast<const float*>(c.slopes->const_data_ptr()) : nullptr;
    if (c.kind == kMasked) {
        check(neox_masked_softmax_fwd(out, in, static_cast<const uint8_t*>(c.mask->const_data_ptr()), scale, b, np, sq, sk,
                                      (int32_t)c.mask->size(0), code(x), stream));
    } else if (c.kind >= 0) {
        check(neox_sliding_window_softmax_fwd(out, in, scale, (int64_t)b * np, sq, sk, (int32_t)c.kind, code(x), stream));
    } else if (c.p != 0) {
        dropped = at::empty_like(x);
        check(neox_causal_softmax_dropout_fwd(dropped.mutable_data_ptr(), out, in, slopes, nullptr, 0, scale, (float)c.p,
                                              (uint64_t)c.seed, (uint64_t)c.offset, nullptr, b, np, sq, sk, code(x), stream));
    } else if (slopes) {
        check(neox_causal_softmax_alibi_fwd(out, in, slopes, scale, b, np, sq, sk, code(x), stream));
    } else {
        check(neox_causal_softmax_fwd(out, in, scale, (int64_t)b * np, sq, sk, code(x), stream));
    }
    return {y, dropped};
}

class Softmax : public torch::autograd::Function<Softmax> {
public:
    static Tensor forward(AutogradContext* ctx, const Tensor& x, const SoftmaxCall& c) {
        auto [y, dropped] = softmax_forward(x, c);
        ctx->save_for_backward({y});
        ctx->saved_data["scale"] = c.scale;
        ctx->saved_data["kind"] = c.kind;
        if (c.p != 0) {
            ctx->saved_data["p"] = c.p;
            ctx->saved_data["seed"] = c.seed;
            ctx->saved_data["offset"] = c.offset;
        }
        return dropped.defined() ? dropped : y;
    }

    // d(input), written into the incoming gradient when that is contiguous
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const Tensor y = ctx->get_saved_variables()[0].contiguous();
        const Tensor g = grads[0].contiguous();
        if (g.sizes() != y.sizes() || g.scalar_type() != y.scalar_type() || g.device() != y.device() || !on_gpu(g))
            throw std::runtime_error("output_grads and softmax_results must have the same dtype and shape");
        const c10::DeviceGuard guard(g.device());
        const auto scale = (float)ctx->saved_data["scale"].toDouble();
        const int64_t kind = ctx->saved_data["kind"].toInt();
        const int64_t batches = g.size(0) * g.size(1);
        const auto sq = (int32_t)g.size(2), sk = (int32_t)g.size(3);
        void *dx = g.mutable_data_ptr(), *stream = stream_of(g);
        const void* probs = y.const_data_ptr();
        const auto p = ctx->saved_data.find("p");
        if (kind == kMasked) {
            check(neox_masked_softmax_bwd(dx, dx, probs, scale, batches * sq, sk, code(g), stream));
        } else if (kind >= 0) {
            check(neox_sliding_window_softmax_bwd(dx, dx, probs, scale, batches, sq, sk, (int32_t)kind, code(g), stream));
        } else if (p != ctx->saved_data.end()) {
            check(neox_causal_softmax_dropout_bwd(dx, dx, probs, scale, (float)p->second.toDouble(),
                                                  (uint64_t)ctx->saved_data["seed"].toInt(),
                                                  (uint64_t)ctx->saved_data["offset"].toInt(), nullptr, batches, sq, sk,
                                                  code(g), stream));
        } else {
            check(neox_causal_softmax_bwd(dx, dx, probs, scale, batches, sq, sk, code(g), stream));
        }
        return {g, Tensor()};
    }
};

bool plain_scores(const Tensor& x) {
    return plain(x) && half_type(x) && x.dim() == 4 && x.numel() > 0 && x.is_contiguous() && fits_int32(x.size(0)) &&
           fits_int32(x.size(1)) && fits_int32(x.size(2)) && fits_int32(x.size(3));
}

Tensor run_softmax(const Tensor& x, const SoftmaxCall& c) {
    if (records(x)) return Softmax::apply(x, c);
    auto [y, dropped] = softmax_forward(x, c);
    return dropped.defined() ? dropped : y;
}

// whether causal_softmax serves these scores (and slopes): asked before random numbers are drawn for it
bool causal_takes(const Tensor& x, const std::optional<Tensor>& slopes) {
    return plain_scores(x) && (!slopes || (plain(*slopes) && slopes->device() == x.device() && slopes->scalar_type() == at::kFloat &&
                                           slopes->numel() == x.size(1) && slopes->is_contiguous() && !slopes->requires_grad()));
}

// causal (window < 0) or sliding-window scores [b, np, sq, sk]; slopes: fp32 [np]; p, seed, offset: dropout
std::optional<Tensor> causal_softmax(const Tensor& x, double scale, int64_t window, const std::optional<Tensor>& slopes,
                                     double p, uint64_t seed, uint64_t offset) {
    if (!causal_takes(x, slopes)) return std::nullopt;
    if (window >= 0 && (slopes || p != 0 || !fits_int32(window))) return std::nullopt;
    return run_softmax(x, {scale, window >= 0 ? window : (int64_t)kCausal, nullptr, slopes ? &*slopes : nullptr, p, (int64_t)seed,
                           (int64_t)offset});
}

// scores [b, np, sq, sk] under a mask tensor [1 or b, 1, sq, sk]
std::optional<Tensor> masked_softmax(const Tensor& x, const Tensor& mask, double scale) {
    if (!plain_scores(x) || !on_gpu(mask) || mask.device() != x.device() || mask.dim() != 4 || !mask.is_contiguous() ||
        (mask.scalar_type() != at::kBool && mask.scalar_type() != at::kByte) ||
        (mask.size(0) != 1 && mask.size(0) != x.size(0)) || mask.size(1) != 1 || mask.size(2) != x.size(2) ||
        mask.size(3) != x.size(3))
        return std::nullopt;
    return run_softmax(x, {scale, kMasked, &mask, nullptr, 0, 0, 0});
}

// ---- rotary embedding ------------------------------------------------------------------------------
struct Tables {
    Tensor cos, sin;  // rows of d_rot values; sin undefined: cos holds angles
    int64_t d_rot, offset;
};

void rope_launch(const Tensor& out_q, const Tensor* out_k, const Tensor& q, const Tensor* k, const Tables& t, int64_t d,
                 bool backward) {
    const c10::DeviceGuard guard(q.device());
    auto strides = [](const Tensor& x) { return x.strides().data(); };
    const int64_t row = t.cos.size(0) > 1 ? t.cos.stride(0) : t.d_rot;
    const auto s = (int32_t)q.size(0), b = (int32_t)q.size(1), hq = (int32_t)q.size(2), hk = k ? (int32_t)k->size(2) : 0;
    void* oq = out_q.mutable_data_ptr();
    void* ok = k ? out_k->mutable_data_ptr() : nullptr;
    const void* kp = k ? k->const_data_ptr() : nullptr;
    const int64_t *ks = k ? strides(*k) : nullptr, *oks = k ? strides(*out_k) : nullptr;
    if (!t.sin.defined()) {
        check(neox_rope_apply_freqs(oq, ok, q.const_data_ptr(), kp, static_cast<const float*>(t.cos.const_data_ptr()), s, b,
                                    hq, hk, (int32_t)t.d_rot, (int32_t)d, strides(q), ks, strides(out_q), oks, row,
                                    (int32_t)t.offset, code(q), backward, stream_of(q)));
    } else {
        check(neox_rope_apply(oq, ok, q.const_data_ptr(), kp, t.cos.const_data_ptr(), t.sin.const_data_ptr(), s, b, hq, hk,
                              (int32_t)t.d_rot, (int32_t)d, strides(q), ks, strides(out_q), oks, row, (int32_t)t.offset,
                              code(q), code(t.cos), backward, stream_of(q)));
    }
}

void save_tables(AutogradContext* ctx, const Tables& t) {
    if (t.sin.defined()) ctx->save_for_backward({t.cos, t.sin});
    else ctx->save_for_backward({t.cos});
    ctx->saved_data["d_rot"] = t.d_rot;
    ctx->saved_data["offset"] = t.offset;
}
// The saved tables, for a gradient g [s, ..]: a saved-tensor hook may have given back another tensor than the forward
// pass left with it, so everything the kernel takes for granted is looked at again.
Tables saved_tables(AutogradContext* ctx, const Tensor& g) {
    variable_list v = ctx->get_saved_variables();
    const int64_t d_rot = ctx->saved_data["d_rot"].toInt(), offset = ctx->saved_data["offset"].toInt();
    for (Tensor& t : v) {
        if (!on_gpu(t) || t.device() != g.device())
            throw std::runtime_error("the saved cos/sin tables or angles must be on the device of the gradient");
        if (t.dim() != 4 || t.size(1) != 1 || t.size(2) != 1 || t.size(3) != d_rot || t.size(0) < offset + g.size(0))
            throw std::runtime_error("the saved cos/sin tables or angles have another shape than in the forward pass");
        if (t.scalar_type() != v[0].scalar_type() ||
            (t.scalar_type() != at::kFloat && (v.size() == 1 || t.scalar_type() != g.scalar_type())))
            throw std::runtime_error("the saved cos/sin tables must be float32 or have the dtype of the gradient, angles float32");
        t = t.contiguous();
    }
    return {v[0], v.size() > 1 ? v[1] : Tensor(), d_rot, offset};
}
Tensor dense_last(const Tensor& t) { return t.stride(-1) == 1 ? t : t.contiguous(); }

// q and k rotated into new tensors, one launch
std::tuple<Tensor, Tensor> rotary_pair(const Tensor& q, const Tensor& k, const Tables& t, bool backward) {
    Tensor oq = at::empty(q.sizes(), q.options()), ok = at::empty(k.sizes(), k.options());
    rope_launch(oq, &ok, q, &k, t, t.d_rot, backward);
    return {oq, ok};
}

class Rotary : public torch::autograd::Function<Rotary> {
public:
    static variable_list forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tables& t) {
        save_tables(ctx, t);
        auto [oq, ok] = rotary_pair(q, k, t, false);
        return {oq, ok};
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        auto [dq, dk] = rotary_pair(dense_last(grads[0]), dense_last(grads[1]), saved_tables(ctx, grads[0]), true);
        return {dq, dk, Tensor()};
    }
};

// one tensor's whole heads; transposed: the memory of the result is [b, s, h, d]
Tensor rope_whole(const Tensor& x, const Tables& t, bool transposed, bool backward) {
    Tensor out = transposed ? at::empty({x.size(1), x.size(0), x.size(2), x.size(3)}, x.options()).transpose(0, 1)
                            : at::empty(x.sizes(), x.options());
    rope_launch(out, nullptr, x, nullptr, t, x.size(3), backward);
    return out;
}

class Rope : public torch::autograd::Function<Rope> {
public:
    static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tables& t, bool transposed) {
        save_tables(ctx, t);
        ctx->saved_data["transposed"] = transposed;
        return rope_whole(x, t, transposed, false);
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        return {rope_whole(dense_last(grads[0]), saved_tables(ctx, grads[0]), ctx->saved_data["transposed"].toBool(), true), Tensor(),
                Tensor()};
    }
};

// strides that count from the tensor's first element upwards, and extents the kernels count in 32 bits
bool plain_heads(const Tensor& x) {
    return plain(x) && half_type(x) && x.dim() == 4 && x.numel() > 0 && x.stride(3) == 1 && fits_int32(x.size(0)) &&
           fits_int32(x.size(1)) && fits_int32(x.size(2)) && fits_int32(x.size(3));
}
// a table [n, 1, 1, d_rot] of dense rows in memory order, with the rows offset .. offset + s
bool plain_table(const Tensor& t, const Tensor& x, int64_t d_rot, int64_t rows) {
    return plain(t) && t.device() == x.device() && t.dim() == 4 && t.size(1) == 1 && t.size(2) == 1 && t.size(3) == d_rot &&
           t.size(0) >= rows && t.is_contiguous() && !t.requires_grad();
}

// q, k [s, b, h, d_rot] -> rotated, or None
std::optional<std::tuple<Tensor, Tensor>> rotary(const Tensor& q, const Tensor& k, const Tensor& cos, const Tensor& sin,
                                                 int64_t offset) {
    if (!plain_heads(q) || !plain_heads(k) || q.scalar_type() != k.scalar_type() || q.device() != k.device() ||
        q.size(0) != k.size(0) || q.size(1) != k.size(1) || q.size(3) != k.size(3) || q.size(3) % 2 != 0 || offset < 0 ||
        !fits_int32(offset + q.size(0)))
        return std::nullopt;
    const int64_t d_rot = q.size(3);
    if (!plain_table(cos, q, d_rot, offset + q.size(0)) || !plain_table(sin, q, d_rot, offset + q.size(0)) ||
        cos.scalar_type() != sin.scalar_type() || cos.size(0) != sin.size(0) ||
        (cos.scalar_type() != at::kFloat && cos.scalar_type() != q.scalar_type()))
        return std::nullopt;
    const Tables t{cos, sin, d_rot, offset};
    if (records(q) || records(k)) {
        variable_list out = Rotary::apply(q, k, t);
        return std::make_tuple(out[0], out[1]);
    }
    return rotary_pair(q, k, t, false);
}

// x [s, b, h, d], rotated over the first dims by angles (sin absent) or by tables [s, 1, 1, d_rot], or None
std::optional<Tensor> rope(const Tensor& x, const Tensor& cos, const std::optional<Tensor>& sin, bool transposed) {
    if (!plain_heads(x) || cos.dim() != 4) return std::nullopt;
    const int64_t d_rot = cos.size(3);
    if (d_rot > x.size(3) || d_rot < 2 || d_rot % 2 != 0 || cos.size(0) != x.size(0) || !plain_table(cos, x, d_rot, x.size(0)))
        return std::nullopt;
    if (sin ? (sin->dim() != 4 || sin->size(0) != x.size(0) || !plain_table(*sin, x, d_rot, x.size(0)) ||
               cos.scalar_type() != sin->scalar_type() ||
               (cos.scalar_type() != at::kFloat && cos.scalar_type() != x.scalar_type()))
            : cos.scalar_type() != at::kFloat)
        return std::nullopt;
    const Tables t{cos, sin ? *sin : Tensor(), d_rot, 0};
    if (records(x)) return Rope::apply(x, t, transposed);
    return rope_whole(x, t, transposed, false);
}

}  // namespace

// The interpreter is not held while a launch waits for room in its queue.  An exception that a saved-tensor hook
// raises (activation checkpointing ends its recomputation with one) comes back as what it is.
PYBIND11_MODULE(neox_torch, m) {
    namespace py = pybind11;
    using torch::wrap_pybind_function_no_gil;
    m.attr("abi_version") = NEOX_FUSED_ABI_VERSION;  // what this was compiled against, for the loader to compare
    m.attr("torch_version") = TORCH_VERSION;
    m.def("causal_softmax", wrap_pybind_function_no_gil(causal_softmax), py::arg("x"), py::arg("scale"), py::arg("window") = -1,
          py::arg("slopes") = std::optional<Tensor>(), py::arg("p") = 0.0, py::arg("seed") = 0, py::arg("offset") = 0);
    m.def("causal_takes", wrap_pybind_function_no_gil(causal_takes), py::arg("x"), py::arg("slopes") = std::optional<Tensor>());
    m.def("masked_softmax", wrap_pybind_function_no_gil(masked_softmax), py::arg("x"), py::arg("mask"), py::arg("scale"));
    m.def("rotary", wrap_pybind_function_no_gil(rotary), py::arg("q"), py::arg("k"), py::arg("cos"), py::arg("sin"),
          py::arg("offset"));
    m.def("rope", wrap_pybind_function_no_gil(rope), py::arg("x"), py::arg("cos"), py::arg("sin"), py::arg("transposed"));
}
