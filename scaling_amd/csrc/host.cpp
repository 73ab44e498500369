// Native host path of the package: argument blocks, output allocation, launches and autograd nodes of the layer operations
// in C++, as the Python extension module `mi355_host`.  The kernels stay behind the C ABI of libmi355_layer.so.
//
// Why it exists: a layer step on a few hundred tokens is 40 launches of a few microseconds each, and the Python form of
// these functions took 10 - 40 us of host time per operation (argument blocks built field by field through ctypes, a
// torch.cuda.current_stream() per launch, a Python autograd node per operation whose backward waits for the interpreter).
// Here an operation costs its allocations and launches, and a backward pass runs without the interpreter.
//
// Linear projections run on mi_gemm or on the library product (at::mm); see small_product, long_chain, wide_product and thin for the lines
// between the two.
#include <torch/extension.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/graph_task.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <ATen/SavedTensorHooks.h>
#include <ATen/hip/HIPContext.h>
#include <ATen/autocast_mode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <c10/hip/HIPGuard.h>
#include <hip/hip_runtime_api.h>
#include <algorithm>
#include <optional>
#include <tuple>
#include <vector>
#include "../../include/mi355_layer.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;
using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::variable_list;

// ---- plumbing ----------------------------------------------------------------------------------------------------------
void check(int status, const char* what) {
    if (status != MI_OK)
        throw std::runtime_error(std::string(what) + " failed: " + mi_status_string(status) + " (" + std::to_string(status) + "): " + mi_last_error());
}

void need_gpu(const Tensor& t) {
    if (!t.is_cuda()) throw std::runtime_error("scaling_amd ops take GPU tensors only (got a CPU tensor); there is no CPU path");
    static const int arch = mi_check_device();            // once per process; a failure is reported by every call
    if (arch != MI_OK) check(mi_check_device(), "mi_check_device");
}

int code_of(const Tensor& t) {
    switch (t.scalar_type()) {
        case at::kBFloat16: return MI_BF16;
        case at::kHalf: return MI_F16;
        case at::kFloat: return MI_F32;
        default: throw py::type_error(std::string("dtype ") + c10::toString(t.scalar_type()) + " is not supported by the HIP kernels");
    }
}

// device of the tensors, and that device's current stream
struct Launch {
    c10::hip::HIPGuard guard;
    void* stream;
    explicit Launch(const Tensor& t) : guard(t.device().index()), stream(c10::hip::getCurrentHIPStream(t.device().index()).stream()) {}
};

void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
Tensor opt(const OptTensor& t) { return t.has_value() ? *t : Tensor(); }
Tensor float_buffer(size_t bytes, const Tensor& like) {
    return at::empty({(int64_t)((bytes + 3) / 4)}, like.options().dtype(at::kFloat));
}
// contiguous and on a 16-byte boundary, as the kernels read it
Tensor vectors(const Tensor& t) {
    const Tensor c = t.contiguous();
    return (reinterpret_cast<uintptr_t>(c.data_ptr()) & 15) == 0 ? c : c.clone();
}
// x as rows of its last dimension
int64_t row_count(const Tensor& x) { return x.size(-1) == 0 ? 0 : x.numel() / x.size(-1); }

// Where an operation is a part of a larger node, of AutogradContext what the nodes below use of it: in the forward pass, and in the backward pass.
struct Kept {
    bool keeps = false;                                    // a gradient will come by here
    std::vector<torch::autograd::SavedVariable> saved;
    decltype(AutogradContext::saved_data) saved_data;
    void save_for_backward(const variable_list& tensors) {
        if (!keeps) return;
        saved.reserve(tensors.size());
        for (const Tensor& t : tensors) saved.emplace_back(t, false);
    }
    void set_materialize_grads(bool) {}
    void give_back() { for (auto& t : saved) t.reset_data(); }
};
struct Replayed {
    variable_list saved;
    decltype(AutogradContext::saved_data)& saved_data;
    std::vector<bool> needs;                               // of the operation's tensor inputs
    const variable_list& get_saved_variables() const { return saved; }
    bool needs_input_grad(size_t i) const { return needs[i]; }
};

// ---- norms -------------------------------------------------------------------------------------------------------------
Tensor op_rms_norm_forward(const Tensor& x_, const Tensor& w_, double eps) {
    need_gpu(x_);
    TORCH_CHECK(x_.scalar_type() == w_.scalar_type() && x_.size(-1) == w_.size(0), "rms_norm: x and weight do not match");
    Launch l(x_);
    const Tensor x = x_.contiguous(), w = w_.contiguous();
    Tensor y = at::empty_like(x);
    check(mi_rmsnorm_fwd(ptr(x), ptr(w), ptr(y), nullptr, row_count(x), x.size(-1), (float)eps, code_of(x), l.stream), "mi_rmsnorm_fwd");
    return y;
}

std::tuple<Tensor, Tensor> op_rms_norm_backward(const Tensor& x_, const Tensor& w_, const Tensor& dy_, double eps) {
    need_gpu(x_);
    if (x_.numel() == 0) return {at::empty_like(x_), at::zeros_like(w_)};   // no rows: the weight gradient is a sum over nothing
    Launch l(x_);
    const Tensor x = x_.contiguous(), w = w_.contiguous(), dy = dy_.contiguous();
    Tensor dx = at::empty_like(x), dw = at::empty_like(w);
    const size_t bytes = mi_rmsnorm_bwd_workspace_bytes(row_count(x), x.size(-1));
    Tensor ws = float_buffer(bytes, x);
    check(mi_rmsnorm_bwd(ptr(x), ptr(w), ptr(dy), ptr(dx), ptr(dw), ptr(ws), bytes, row_count(x), x.size(-1), (float)eps, code_of(x), l.stream),
          "mi_rmsnorm_bwd");
    return {dx, dw};
}

struct RmsNorm : Function<RmsNorm> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w, double eps) {
        ctx->save_for_backward({x, w});
        ctx->saved_data["eps"] = eps;
        return op_rms_norm_forward(x, w, eps);
    }
    static variable_list backward(AutogradContext* ctx, variable_list g) {
        const variable_list saved = ctx->get_saved_variables();
        auto [dx, dw] = op_rms_norm_backward(saved[0], saved[1], g[0], ctx->saved_data["eps"].toDouble());
        return {dx, dw, Tensor()};
    }
};

std::tuple<Tensor, Tensor> op_layer_norm_forward(const Tensor& x_, const Tensor& w_, const OptTensor& b_, double eps, bool save_stats) {
    need_gpu(x_);
    TORCH_CHECK(x_.scalar_type() == w_.scalar_type() && x_.size(-1) == w_.size(0), "layer_norm: x and weight do not match");
    Launch l(x_);
    const Tensor x = x_.contiguous(), w = w_.contiguous(), b = b_.has_value() ? b_->contiguous() : Tensor();
    Tensor y = at::empty_like(x), stats;
    const int64_t rows = row_count(x);
    if (save_stats) stats = at::empty({2, rows}, x.options().dtype(at::kFloat));
    float* mean = save_stats ? stats.data_ptr<float>() : nullptr;
    check(mi_layernorm_fwd(ptr(x), ptr(w), ptr(b), ptr(y), mean, mean ? mean + rows : nullptr, rows, x.size(-1), (float)eps, code_of(x), l.stream),
          "mi_layernorm_fwd");
    return {y, stats};
}

std::tuple<Tensor, Tensor, Tensor> op_layer_norm_backward(const Tensor& x_, const Tensor& w_, const Tensor& dy_, double eps, bool need_bias_grad,
                                                       const OptTensor& stats) {
    need_gpu(x_);
    if (x_.numel() == 0) return {at::empty_like(x_), at::zeros_like(w_), need_bias_grad ? at::zeros_like(w_) : Tensor()};
    Launch l(x_);
    const Tensor x = x_.contiguous(), w = w_.contiguous(), dy = dy_.contiguous();
    Tensor dx = at::empty_like(x), dw = at::empty_like(w), db = need_bias_grad ? at::empty_like(w) : Tensor();
    const int64_t rows = row_count(x);
    const float* mean = stats.has_value() && stats->defined() ? stats->data_ptr<float>() : nullptr;
    const size_t bytes = mi_layernorm_bwd_workspace_bytes(rows, x.size(-1));
    Tensor ws = float_buffer(bytes, x);
    check(mi_layernorm_bwd(ptr(x), ptr(w), ptr(dy), mean, mean ? mean + rows : nullptr, ptr(dx), ptr(dw), ptr(db), ptr(ws), bytes, rows, x.size(-1),
                           (float)eps, code_of(x), l.stream),
          "mi_layernorm_bwd");
    return {dx, dw, db};
}

struct LayerNorm : Function<LayerNorm> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w, const OptTensor& b, double eps) {
        auto [y, stats] = op_layer_norm_forward(x, w, b, eps, true);
        ctx->save_for_backward({x, w, stats});
        ctx->saved_data["eps"] = eps;
        ctx->saved_data["bias"] = b.has_value();
        return y;
    }
    static variable_list backward(AutogradContext* ctx, variable_list g) {
        const variable_list saved = ctx->get_saved_variables();
        auto [dx, dw, db] = op_layer_norm_backward(saved[0], saved[1], g[0], ctx->saved_data["eps"].toDouble(), ctx->saved_data["bias"].toBool(), saved[2]);
        return {dx, dw, db, Tensor()};
    }
};

// A norm together with the residual stream it branches off: sum = x + residual (x itself without a residual), y = norm(sum).  Both
// outputs are differentiable; the gradient that reaches `sum` directly is added inside the norm's backward kernel.
struct AddNorm : Function<AddNorm> {
    template <class Context> static variable_list run(Context* ctx, const Tensor& x_, const OptTensor& residual_, const Tensor& w_, const OptTensor& b_, double eps,
                                                      bool layer_norm) {
        need_gpu(x_);
        TORCH_CHECK(x_.scalar_type() == w_.scalar_type() && x_.dim() >= 1 && x_.size(-1) == w_.size(0), "norm: x and weight do not match");
        TORCH_CHECK(!residual_.has_value() || (residual_->sizes() == x_.sizes() && residual_->scalar_type() == x_.scalar_type()),
                    "norm: x and residual do not match");
        Launch l(x_);
        const Tensor x = residual_.has_value() ? vectors(x_) : x_.contiguous(), w = w_.contiguous(), b = b_.has_value() ? b_->contiguous() : Tensor();
        const Tensor residual = residual_.has_value() ? vectors(*residual_) : Tensor();
        const int64_t rows = row_count(x), hidden = x.size(-1);
        const Tensor sum = residual.defined() ? at::empty_like(x) : x_;
        Tensor y = at::empty_like(x), stats;
        if (layer_norm) {
            stats = at::empty({2, rows}, x.options().dtype(at::kFloat));
            float *mean = stats.data_ptr<float>(), *rstd = mean + rows;
            if (residual.defined())
                check(mi_add_layernorm_fwd(ptr(x), ptr(residual), ptr(w), ptr(b), ptr(sum), ptr(y), mean, rstd, rows, hidden, (float)eps, code_of(x), l.stream),
                      "mi_add_layernorm_fwd");
            else
                check(mi_layernorm_fwd(ptr(x), ptr(w), ptr(b), ptr(y), mean, rstd, rows, hidden, (float)eps, code_of(x), l.stream), "mi_layernorm_fwd");
        } else if (residual.defined()) {
            check(mi_add_rmsnorm_fwd(ptr(x), ptr(residual), ptr(w), ptr(sum), ptr(y), rows, hidden, (float)eps, code_of(x), l.stream), "mi_add_rmsnorm_fwd");
        } else {
            check(mi_rmsnorm_fwd(ptr(x), ptr(w), ptr(y), nullptr, rows, hidden, (float)eps, code_of(x), l.stream), "mi_rmsnorm_fwd");
        }
        ctx->set_materialize_grads(false);                 // an output that does not reach the loss costs nothing
        ctx->save_for_backward({sum, w_, stats});
        ctx->saved_data["eps"] = eps;
        ctx->saved_data["layer_norm"] = layer_norm;
        ctx->saved_data["residual"] = residual.defined();
        ctx->saved_data["bias"] = b.defined();
        return {sum, y};
    }
    template <class Context> static variable_list gradients(Context* ctx, const variable_list& g) {
        const variable_list saved = ctx->get_saved_variables();
        const bool layer_norm = ctx->saved_data["layer_norm"].toBool(), bias = ctx->saved_data["bias"].toBool();
        const Tensor& dsum_ = g[0];
        Tensor dx, dw, db;
        if (!g[1].defined()) {                             // the norm does not reach the loss
            dx = dsum_;
        } else if (saved[0].numel() == 0) {
            dx = at::empty_like(saved[0]);
            dw = at::zeros_like(saved[1]);
            if (bias) db = at::zeros_like(saved[1]);
        } else {
            Launch l(saved[0]);
            const Tensor x = saved[0].contiguous(), w = saved[1].contiguous(), dy = g[1].contiguous(), dsum = dsum_.defined() ? vectors(dsum_) : Tensor();
            const int64_t rows = row_count(x), hidden = x.size(-1);
            const float eps = (float)ctx->saved_data["eps"].toDouble();
            dx = at::empty_like(x);
            dw = at::empty_like(w);
            if (layer_norm) {
                const float* mean = saved[2].data_ptr<float>();
                if (bias) db = at::empty_like(w);
                const size_t bytes = mi_layernorm_bwd_workspace_bytes(rows, hidden);
                Tensor ws = float_buffer(bytes, x);
                check(mi_add_layernorm_bwd(ptr(x), ptr(w), ptr(dy), ptr(dsum), mean, mean + rows, ptr(dx), ptr(dw), ptr(db), ptr(ws), bytes, rows, hidden, eps,
                                           code_of(x), l.stream),
                      "mi_add_layernorm_bwd");
            } else {
                const size_t bytes = mi_rmsnorm_bwd_workspace_bytes(rows, hidden);
                Tensor ws = float_buffer(bytes, x);
                check(mi_add_rmsnorm_bwd(ptr(x), ptr(w), ptr(dy), ptr(dsum), ptr(dx), ptr(dw), ptr(ws), bytes, rows, hidden, eps, code_of(x), l.stream),
                      "mi_add_rmsnorm_bwd");
            }
        }
        return {dx, ctx->saved_data["residual"].toBool() ? dx : Tensor(), dw, db, Tensor(), Tensor()};
    }
    static variable_list forward(AutogradContext* ctx, const Tensor& x, const OptTensor& residual, const Tensor& w, const OptTensor& b, double eps, bool layer_norm) {
        return run(ctx, x, residual, w, b, eps, layer_norm);
    }
    static variable_list backward(AutogradContext* ctx, variable_list g) { return gradients(ctx, g); }
};

std::tuple<Tensor, Tensor> op_add_norm(const Tensor& x, const OptTensor& residual, const Tensor& w, const OptTensor& b, double eps, bool layer_norm) {
    const auto out = AddNorm::apply(x, residual, w, b, eps, layer_norm);
    return {out[0], out[1]};
}

// ---- activations -------------------------------------------------------------------------------------------------------
Tensor op_gelu_forward(const Tensor& x_) {
    need_gpu(x_);
    Launch l(x_);
    const Tensor x = x_.contiguous();
    Tensor y = at::empty_like(x);
    check(mi_gelu_fwd(ptr(x), ptr(y), x.numel(), code_of(x), l.stream), "mi_gelu_fwd");
    return y;
}

Tensor op_gelu_backward(const Tensor& x_, const Tensor& dy_) {
    need_gpu(x_);
    Launch l(x_);
    const Tensor x = x_.contiguous(), dy = dy_.contiguous();
    Tensor dx = at::empty_like(x);
    check(mi_gelu_bwd(ptr(x), ptr(dy), ptr(dx), x.numel(), code_of(x), l.stream), "mi_gelu_bwd");
    return dx;
}

struct Gelu : Function<Gelu> {
    template <class Context> static Tensor run(Context* ctx, const Tensor& x) {
        ctx->save_for_backward({x});
        return op_gelu_forward(x);
    }
    template <class Context> static variable_list gradients(Context* ctx, const variable_list& g) { return {op_gelu_backward(ctx->get_saved_variables()[0], g[0])}; }
    static Tensor forward(AutogradContext* ctx, const Tensor& x) { return run(ctx, x); }
    static variable_list backward(AutogradContext* ctx, variable_list g) { return gradients(ctx, g); }
};

Tensor op_swiglu_forward(const Tensor& a_, const Tensor& gate_) {
    need_gpu(a_);
    need_gpu(gate_);
    TORCH_CHECK(a_.sizes() == gate_.sizes() && a_.scalar_type() == gate_.scalar_type(), "swiglu: a and gate do not match");
    Launch l(a_);
    const Tensor a = a_.contiguous(), gate = gate_.contiguous();
    Tensor out = at::empty_like(a);
    check(mi_swiglu_fwd(ptr(a), ptr(gate), ptr(out), a.numel(), code_of(a), l.stream), "mi_swiglu_fwd");
    return out;
}

std::tuple<Tensor, Tensor> op_swiglu_backward(const Tensor& a_, const Tensor& gate_, const Tensor& dout_) {
    need_gpu(a_);
    Launch l(a_);
    const Tensor a = a_.contiguous(), gate = gate_.contiguous(), dout = dout_.contiguous();
    Tensor da = at::empty_like(a), dg = at::empty_like(a);
    check(mi_swiglu_bwd(ptr(a), ptr(gate), ptr(dout), ptr(da), ptr(dg), a.numel(), code_of(a), l.stream), "mi_swiglu_bwd");
    return {da, dg};
}

struct SwiGlu : Function<SwiGlu> {
    template <class Context> static Tensor run(Context* ctx, const Tensor& a, const Tensor& gate) {
        ctx->save_for_backward({a, gate});
        return op_swiglu_forward(a, gate);
    }
    template <class Context> static variable_list gradients(Context* ctx, const variable_list& g) {
        const variable_list saved = ctx->get_saved_variables();
        auto [da, dg] = op_swiglu_backward(saved[0], saved[1], g[0]);
        return {da, dg};
    }
    static Tensor forward(AutogradContext* ctx, const Tensor& a, const Tensor& gate) { return run(ctx, a, gate); }
    static variable_list backward(AutogradContext* ctx, variable_list g) { return gradients(ctx, g); }
};

// ---- rotary ------------------------------------------------------------------------------------------------------------
// x [tokens, heads, head_dim] with contiguous features; the tables decide the pairing: fp32 [rows, head_dim / 2] with
// `interleaved`, else [rows, rot_dim]
Tensor rotary_launch(const Tensor& x, const Tensor& cos, const Tensor& sin, const OptTensor& ids, int64_t seq_len_for_null_ids, bool inverse,
                     bool interleaved) {
    need_gpu(x);
    TORCH_CHECK(x.dim() == 3 && x.stride(2) == 1 && cos.is_contiguous() && sin.is_contiguous(), "rotary: bad layout");
    Launch l(x);
    Tensor out = at::empty(x.sizes(), x.options());
    const Tensor pos = ids.has_value() && ids->defined() ? ids->contiguous() : Tensor();
    TORCH_CHECK(!pos.defined() || (pos.scalar_type() == at::kLong && pos.numel() == x.size(0)), "rotary: one int64 position id per token");
    if (interleaved)
        check(mi_rotary_complex(ptr(x), ptr(out), (const float*)ptr(cos), (const float*)ptr(sin), (const int64_t*)ptr(pos), x.size(0), (int)x.size(1),
                                (int)x.size(2), x.stride(0), x.stride(1), out.stride(0), out.stride(1), cos.size(0), seq_len_for_null_ids, inverse,
                                code_of(x), l.stream),
              "mi_rotary_complex");
    else
        check(mi_rotary(ptr(x), ptr(out), ptr(cos), ptr(sin), (const int64_t*)ptr(pos), x.size(0), (int)x.size(1), (int)x.size(2), (int)cos.size(1),
                        x.stride(0), x.stride(1), out.stride(0), out.stride(1), cos.size(0), seq_len_for_null_ids, inverse, code_of(x), code_of(cos),
                        l.stream),
              "mi_rotary");
    return out;
}

// The same of two tensors of the same tokens
std::tuple<Tensor, Tensor> rotary_launch_two(const Tensor& q, const Tensor& k, const Tensor& cos, const Tensor& sin, const OptTensor& ids,
                                             int64_t seq_len_for_null_ids, bool inverse, bool interleaved) {
    for (const Tensor* t : {&q, &k}) {
        need_gpu(*t);
        TORCH_CHECK(t->dim() == 3 && t->stride(2) == 1 && t->size(0) == q.size(0) && t->size(2) == q.size(2) && t->scalar_type() == q.scalar_type() &&
                        t->device() == q.device(),
                    "rotary: bad layout");
    }
    TORCH_CHECK(cos.is_contiguous() && sin.is_contiguous(), "rotary: bad layout");
    Launch l(q);
    const Tensor q_out = at::empty(q.sizes(), q.options()), k_out = at::empty(k.sizes(), k.options());
    const Tensor pos = ids.has_value() && ids->defined() ? ids->contiguous() : Tensor();
    TORCH_CHECK(!pos.defined() || (pos.scalar_type() == at::kLong && pos.numel() == q.size(0)), "rotary: one int64 position id per token");
    const auto rows = [](const Tensor& x, const Tensor& out) {
        return mi_rotary_rows{ptr(x), ptr(out), x.stride(0), x.stride(1), out.stride(0), out.stride(1), (int32_t)x.size(1)};
    };
    const mi_rotary_rows both[2] = {rows(q, q_out), rows(k, k_out)};
    check(mi_rotary_two(both, ptr(cos), ptr(sin), (const int64_t*)ptr(pos), q.size(0), (int)q.size(2), interleaved ? (int)q.size(2) : (int)cos.size(1),
                        cos.size(0), seq_len_for_null_ids, inverse, interleaved, code_of(q), code_of(cos), l.stream),
          "mi_rotary_two");
    return {q_out, k_out};
}

struct Rotary : Function<Rotary> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& cos, const Tensor& sin, const OptTensor& ids, int64_t seq_len, bool interleaved) {
        ctx->save_for_backward({cos, sin, opt(ids)});
        ctx->saved_data["seq_len"] = seq_len;
        ctx->saved_data["interleaved"] = interleaved;
        return rotary_launch(x, cos, sin, ids, seq_len, false, interleaved);
    }
    static variable_list backward(AutogradContext* ctx, variable_list g) {
        const variable_list saved = ctx->get_saved_variables();
        const Tensor dout = g[0].stride(-1) == 1 ? g[0] : g[0].contiguous();
        return {rotary_launch(dout, saved[0], saved[1], saved[2], ctx->saved_data["seq_len"].toInt(), true, ctx->saved_data["interleaved"].toBool()),
                Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
    }
};

// q and k of a layer
struct RotaryTwo : Function<RotaryTwo> {
    template <class Context> static variable_list run(Context* ctx, const Tensor& q, const Tensor& k, const Tensor& cos, const Tensor& sin, const OptTensor& ids,
                                                      int64_t seq_len, bool interleaved) {
        ctx->set_materialize_grads(false);
        ctx->save_for_backward({cos, sin, opt(ids)});
        ctx->saved_data["seq_len"] = seq_len;
        ctx->saved_data["interleaved"] = interleaved;
        auto [q_rot, k_rot] = rotary_launch_two(q, k, cos, sin, ids, seq_len, false, interleaved);
        return {q_rot, k_rot};
    }
    template <class Context> static variable_list gradients(Context* ctx, const variable_list& g) {
        const variable_list saved = ctx->get_saved_variables();
        const int64_t seq_len = ctx->saved_data["seq_len"].toInt();
        const bool interleaved = ctx->saved_data["interleaved"].toBool();
        variable_list d(7);
        Tensor in[2];
        for (int i : {0, 1})
            if (g[i].defined()) in[i] = g[i].stride(-1) == 1 ? g[i] : g[i].contiguous();
        if (in[0].defined() && in[1].defined()) {
            std::tie(d[0], d[1]) = rotary_launch_two(in[0], in[1], saved[0], saved[1], saved[2], seq_len, true, interleaved);
        } else {
            for (int i : {0, 1})
                if (in[i].defined()) d[i] = rotary_launch(in[i], saved[0], saved[1], saved[2], seq_len, true, interleaved);
        }
        return d;
    }
    static variable_list forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& cos, const Tensor& sin, const OptTensor& ids, int64_t seq_len,
                                 bool interleaved) {
        return run(ctx, q, k, cos, sin, ids, seq_len, interleaved);
    }
    static variable_list backward(AutogradContext* ctx, variable_list g) { return gradients(ctx, g); }
};

// ---- linear projections ------------------------------------------------------------------------------------------------
// Whether a product of m x n x k multiply-adds goes to mi_gemm.  A library call costs the host 18 us whatever its size (the
// heuristic lookup), mi_gemm 3; on the device the two meet near 3 GFLOP (16-bit: 1024 x 1024 x 1024, forward + both
// gradients 26.7 us here and 28.6 on the library, 2048 x 512 x 2048 53 and 39 us) and 0.75 GFLOP (fp32: 333 x 1000 x 520
// 30.5 and 29.0 us, 1024 x 1024 x 1024 80 and 57; below it the library also picks 256 x 256 blocks for
// 256 x 256 x 256 and takes 63 us per product where mi_gemm takes 6).
bool small_product(const Tensor& t, int64_t m, int64_t n, int64_t k) {
    const int64_t v = t.scalar_type() == at::kFloat ? 4 : 8;
    const double work = 2.0 * (double)m * (double)n * (double)k;
    return n % v == 0 && k % v == 0 && work <= (v == 4 ? 0.75e9 : 3e9);
}
// Forward products of inference (modules in eval mode) over a long contraction stay on the library: mi_gemm walks it in one chain per
// workgroup, the library splits it.  16-bit, 32 rows, us on the device / issued one by one, mi_gemm and library: 2048 -> 2048
// 10.5 / 10.3 and 8.4 / 17.5; 2816 -> 1024 13.1 / 13.0 and 7.3 / 17.6; 4096 -> 4096 20.6 / 20.1 and 13.2 / 18.2; 8192 -> 1024
// 35.0 / 34.7 and 15.0 / 17.9; with the weights from memory, per product of a captured graph: 2816 -> 1024 14.5 and 9.3 - 11.2; 2048 -> 512
// 10.3 and 7.9; 2048 -> 2048 11.8 and 11.0 - 11.7; 1024 -> 2816 7.6 and 11.  Below 3072 a graph loses up to 5 us with mi_gemm, and a
// step that the host issues loses up to 45 with the library (prefill of 175 tokens, 3 layers with 2816 -> 1024: 1.10 and 1.26 ms).  The
// line is the same for a stream that is being captured: what runs once before the capture has to have made the library's
// handles and loaded its kernels.
// A training step, which the host bounds at these sizes, keeps mi_gemm (forward and both gradients,
// issued one by one, with either forward product: 4096 -> 4096 57 and 74, 8192 -> 1024 54 and 76).  Up to MI_ROWS_MAX rows have a
// kernel that splits the contraction.  Whether gradients are wanted does not matter: reentrant checkpointing runs a layer without
// and again with them and counts on the same bits.
// float32 has no kernel for few rows: 8 - 64 rows, us issued one by one, mi_gemm and library: 1024 -> 1024 12.7 and 24.5; 2816 -> 1024 27.5
// and 24.5; 4096 -> 1024 38 and 24.5.
bool long_chain(const Tensor& t, int64_t rows, int64_t k) { return k >= 3072 && (t.scalar_type() == at::kFloat || rows > MI_ROWS_MAX); }
// Larger products of 16-bit types with whole vectors in every direction: blocks of 128 or 256 rows and columns in mi_gemm, all layouts at the rate
// of the library's fastest.  us on the device, mi_gemm and library: 4084 x 1024 -> 4096 forward 34.4 / 30.5, input gradient 34.6 / 40.0,
// weight gradient 32.7 / 37.5; 1024 -> 1024 13.8 / 13.4, 13.7 / 15.0, 22.4 / 33.0; 8192 x 4096 -> 14336 649 / 618, 629 / 693, 660 / 827 (767 + 24
// with x transposed first).  Fewer than 128 rows, or 32 features on either side, fill no block (8192 x 32768 -> 16, forward and gradients, 409 / 442).
//   Training (forward and gradients, here and with the library): 2048 x 1024 -> 1024 33 / 78, 2048 x 4096 -> 4096 177 / 193, 301 x 4096 -> 14336
// 188 / 227; forward products of 100 GFLOP and more stay on the library.
//   Inference keeps the library where its own time exceeds what it costs the host, or nearly: issued one by one (on the device alone) 2048 x 1024 ->
// 1024 12.2 / 19.7 (11.8 / 10.2), 1024 x 1024 -> 4096 13.7 / 19.9 (14.2 / 13.4), 2048 x 1024 -> 4096 26.5 / 21.8, 1024 x 2816 -> 1024 22.5 / 19.8 (22.5 /
// 13.4), 513 x 2048 -> 2048 19.2 / 19.8 (19.7 / 12.3), 4084 x 2048 -> 2048 41 / 35, 301 x 4096 -> 14336 59 / 40.  So does a second round of blocks, beyond
// 512 contraction indices (issued one by one, where the library is 20.2): one round 1078 x 1024 -> 3072 12.8, 2897 x 1536 -> 1024 15.8,
// two 1163 x 1024 -> 4096 22.0, 739 x 800 -> 6912 23.2, 1142 x 640 -> 5632 21.8, 1982 x 552 -> 2544 22.4, 1785 x 512 -> 4224 19.7, 1450 x 384 -> 3072 16.5, three
// 1350 x 384 -> 8192 18.2.  Of several projections, which are a library call each, the average decides.
enum class Pass { kInference, kForward, kBackward };
bool wide_product(const Tensor& t, int64_t rows, int64_t n, int64_t k, Pass pass) {
    const double work = 2.0 * (double)rows * (double)n * (double)k;
    if (pass == Pass::kInference ? k > 1536 || work > 1e10 : pass == Pass::kForward && work >= 1e11) return false;
    if (std::max({rows, n, k}) > 0x7fffffff) return false;
    return t.scalar_type() != at::kFloat && rows >= 128 && n >= 32 && k >= 32 && n % 8 == 0 && k % 8 == 0;
}
// Short contractions into large outputs: a block spends more on its fill and its results than on products, and the library's kernels for whole
// blocks do that part better.  us, mi_gemm and library, forward / input gradient / weight gradient layout:
//   8192 x 8192, k 32  51 30 / 51 32 / 49 32   k 192  65 50 / 65 51 / 61 50   k 320  83 62 / 81 66 / 75 65   k 448  91 78 / 88 80 / 85 80   k 512  89 84 / 88 86 / 85 87
//   4096 x 4096, k 256  29 20 / 19 18 / 18 19        2048 x 4096, k 256  15 18 / 16 18 / 15 19        8192 x 32768, forward, k 96  226 145   k 144  279 240
// Where the library's blocks are not whole, mi_gemm stays: 8192 x 8256, k 256  78 87 / 78 90 / 74 91;  16001 x 3072, k 360  67 67 / 64 66;  4096 x 14920, k 64
// 51 56 / 51 58 / 50 59;  8192 x 32768, forward, k 200  248 250.
bool thin(int64_t m, int64_t n, int64_t k) { return k < 512 && k % 16 == 0 && n % 256 == 0 && (double)m * (double)n >= 33554432.0; }
bool aligned(const Tensor& t) {        // as an operand of mi_gemm: contiguous rows, none on top of another, that start on 16-byte boundaries
    const int64_t v = t.scalar_type() == at::kFloat ? 4 : 8;
    return t.dim() == 2 && t.stride(1) == 1 && t.stride(0) >= t.size(1) && t.stride(0) % v == 0 && (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0;
}
// rows that the large blocks of mi_gemm reach: 128 of them within 2^31 bytes
bool in_reach(const Tensor& t) { return t.stride(0) < (1 << 22); }

void segment(mi_gemm_problem& pr, const Tensor& p, const Tensor& q, int64_t k) {
    mi_gemm_segment& s = pr.segments[pr.n_segments++];
    s.p = ptr(p); s.q = ptr(q); s.ldp = p.stride(0); s.ldq = q.stride(0); s.k = (int32_t)k;
}
mi_gemm_problem problem(const Tensor& c, bool p_kmajor, bool q_kmajor) {
    mi_gemm_problem pr{};
    pr.c = ptr(c); pr.ldc = c.stride(0); pr.m = (int32_t)c.size(0); pr.n = (int32_t)c.size(1);
    pr.p_kmajor = p_kmajor; pr.q_kmajor = q_kmajor;
    return pr;
}

void run_gemm(const mi_gemm_problem* pr, int count, const Tensor& like, const Launch& l) {
    const size_t bytes = mi_gemm_workspace_bytes(pr, count, code_of(like));
    const Tensor ws = bytes > 0 ? float_buffer(bytes, like) : Tensor();
    check(mi_gemm_with_workspace(pr, count, code_of(like), ptr(ws), bytes, l.stream), "mi_gemm");
}

Tensor bias_gradient(const Tensor& dy) {
    if (!aligned(dy) || dy.size(0) == 0) return dy.sum(0);
    const int64_t v = dy.scalar_type() == at::kFloat ? 4 : 8;
    if (dy.size(1) % v != 0) return dy.sum(0);
    Launch l(dy);
    Tensor db = at::empty({dy.size(1)}, dy.options());
    check(mi_column_sum(ptr(dy), dy.stride(0), dy.size(0), dy.size(1), ptr(db), code_of(dy), l.stream), "mi_column_sum");
    return db;
}

// Weight gradients dW = dY^T X contract over the rows of both operands, which is the library's slowest layout for 16-bit types; with one of
// them transposed first it runs a fifth faster, which pays for the transposed copy once the other side is wide.  us, product as it is /
// with X or dY transposed + the copy:
//   8192 x 4096 -> 14340   972 / 732 + 24        8192 x 14340 -> 4096 (dY)   1006 / 766 + 24
//   8192 x 4096 -> 4100    424 / 261 + 24        4096 x 2048 -> 8196          169 / 155 + 7
//   4096 x 2048 -> 32004   474 / 409 + 6         3001 x 8196 -> 2056 (dY)     165 / 140 + 7
// and not where the copy or the product is small: 4084 x 1024 -> 4096 55 / 51 + 5, 2047 x 1024 -> 50257 271 / 256 + 5 (2047 x 2048 -> 50257 471 / 476 + 6).
bool transpose_pays(int64_t rows, int64_t in, int64_t out) {
    return 2.0 * (double)rows * (double)in * (double)out >= 1e11 && std::max(in, out) >= 4096 && std::min(in, out) >= 2048;
}
bool transposable(const Tensor& x) { return x.scalar_type() != at::kFloat && aligned(x) && x.size(1) % 8 == 0 && x.size(0) <= 64 * 65535; }
// x^T as a tensor whose rows are contiguous, on 128-byte boundaries
Tensor transposed(const Tensor& x, const Launch& l) {
    const int64_t rows = x.size(0), ld = (rows + 63) / 64 * 64;
    const Tensor t = at::empty({x.size(1), ld}, x.options());
    check(mi_transpose16(ptr(x), x.stride(0), rows, x.size(1), ptr(t), ld, l.stream), "mi_transpose16");
    return t.narrow(1, 0, rows);
}

// A transform that has to see library calls: torch.func (grad, vmap, jvp), forward-mode AD, torch.jit tracing, a dispatch mode or a
// tensor subclass (fake tensors among them); in a backward pass also batched gradients (torch.autograd.grad with is_grads_batched)
bool transformed(const Tensor& t) {
    return t.unsafeGetTensorImpl()->is_python_dispatch() || t._fw_grad(0).defined() ||
           t.key_set().has_any(c10::DispatchKeySet({c10::DispatchKey::Batched, c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper}));
}
bool transforming() {
    return c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) || c10::impl::TorchDispatchModeTLS::any_modes_set() ||
           torch::jit::tracer::isTracing();
}

// Several projections of one input: y_i = x W_i^T + b_i.  Their input gradient is one sum, their forward products and (for small
// problems) all their gradients are one launch each.
struct Projections : Function<Projections> {
    // params: the n weights, then the biases of those projections whose has_bias is set (an autograd node takes no undefined
    // tensors); bias_at gives the position of projection i's bias in params, -1 without one
    static std::vector<int64_t> bias_at(const std::vector<int64_t>& has_bias) {
        std::vector<int64_t> at(has_bias.size(), -1);
        int64_t next = (int64_t)has_bias.size();
        for (size_t i = 0; i < has_bias.size(); ++i)
            if (has_bias[i]) at[i] = next++;
        return at;
    }
    // residual (one projection only): added to the output
    // need_dx: a gradient of x will be wanted
    template <class Context> static variable_list run(Context* ctx, const Tensor& x, at::TensorList params, const OptTensor& residual,
                                                      const std::vector<int64_t>& has_bias, bool inference, bool need_dx) {
        const int64_t n = (int64_t)has_bias.size(), in = x.size(-1);
        const auto at = bias_at(has_bias);
        const Tensor x2 = x.reshape({-1, in});
        const int64_t rows = x2.size(0);
        variable_list saved, out;
        bool small = !(inference && long_chain(x, rows, in)), wide = true, fit = aligned(x2);
        int64_t blocks = 0;
        for (int64_t i = 0; i < n; ++i) {
            const Tensor& w = params[i];
            blocks += (rows + 127) / 128 * ((w.size(0) + 127) / 128);
            fit = fit && aligned(w);
            small = small && small_product(x, rows, w.size(0), in);
            wide = wide && wide_product(x, rows, w.size(0), in, inference ? Pass::kInference : Pass::kForward) && !thin(rows, w.size(0), in) && in_reach(x2) &&
                   in_reach(w);
        }
        if (inference && in > 512 && blocks > n * at::cuda::getDeviceProperties(x.device().index())->multiProcessorCount) wide = false;
        // What the gradients read and no more, so that the rest may be changed or freed before the backward pass: x (itself: what is
        // differentiated again reaches it) for the weights, the weights for x.  The same for a recomputation inside a backward pass.
        bool any_weight = false;
        for (int64_t i = 0; i < n; ++i) any_weight = any_weight || params[i].requires_grad();
        saved.push_back(any_weight ? x : Tensor());
        for (int64_t i = 0; i < n; ++i) saved.push_back(need_dx ? params[i] : Tensor());
        std::vector<int64_t> shape(x.sizes().begin(), x.sizes().end());
        if (fit && (small || wide)) {
            Launch l(x);
            mi_gemm_problem pr[MI_GEMM_MAX_PROBLEMS];
            for (int64_t i = 0; i < n; ++i) {
                shape.back() = params[i].size(0);
                out.push_back(at::empty(shape, x.options()));
                pr[i] = problem(out.back().view({rows, shape.back()}), false, false);
                segment(pr[i], x2, params[i], in);
                if (at[i] >= 0) pr[i].bias = ptr(params[at[i]]);
            }
            Tensor add;
            if (residual.has_value()) {
                add = vectors(*residual);
                pr[0].add = ptr(add);
                pr[0].ldadd = pr[0].n;
            }
            run_gemm(pr, (int)n, x, l);
        } else {
            for (int64_t i = 0; i < n; ++i) {
                shape.back() = params[i].size(0);
                const Tensor wt = params[i].t();
                // not a view of the product: a caller may change the output in place
                out.push_back(at::_unsafe_view(at[i] >= 0 ? at::addmm(params[at[i]], x2, wt) : at::mm(x2, wt), shape));
            }
            if (residual.has_value()) out[0].add_(*residual);
        }
        ctx->set_materialize_grads(false);
        ctx->save_for_backward(saved);
        ctx->saved_data["x_shape"] = x.sizes().vec();
        ctx->saved_data["residual"] = residual.has_value();
        ctx->saved_data["has_bias"] = has_bias;
        return out;
    }
    template <class Context> static variable_list gradients(Context* ctx, const variable_list& g) {
        const variable_list saved = ctx->get_saved_variables();
        const auto x_shape = ctx->saved_data["x_shape"].toIntVector();
        const int64_t n = (int64_t)g.size(), in = x_shape.back();
        int64_t rows = 1;
        for (size_t i = 0; i + 1 < x_shape.size(); ++i) rows *= x_shape[i];
        const Tensor x = saved[0].defined() ? saved[0].reshape({rows, in}) : Tensor();     // undefined: no weight takes a gradient
        // a graph of this pass is wanted, or a transform watches it: library products, out of place
        bool again = at::GradMode::is_enabled() || transforming();
        for (const Tensor& t : saved) again = again || (t.defined() && transformed(t));
        for (const Tensor& t : g) again = again || (t.defined() && transformed(t));
        const auto has_bias = ctx->saved_data["has_bias"].toIntVector();
        const auto at = bias_at(has_bias);                 // tensor input 1 + at[i] of the node
        const bool need_dx = ctx->needs_input_grad(0);
        const auto need_weight = [&](int64_t i) { return ctx->needs_input_grad(1 + i); };
        const auto need_bias = [&](int64_t i) { return at[i] >= 0 && ctx->needs_input_grad(1 + at[i]); };
        std::vector<Tensor> dy(n), dw(n), db(n);
        bool small = true, wide = true, fit = !again && rows > 0 && (!x.defined() || aligned(x));
        for (int64_t i = 0; i < n; ++i) {
            if (!g[i].defined()) continue;                 // this projection does not reach the loss
            dy[i] = g[i].reshape({rows, g[i].size(-1)});
            if (!again && !aligned(dy[i])) dy[i] = dy[i].contiguous();
            fit = fit && aligned(dy[i]);
            small = small && small_product(dy[i], rows, dy[i].size(1), in);
            wide = wide && wide_product(dy[i], rows, dy[i].size(1), in, Pass::kBackward) && in_reach(dy[i]) && (!x.defined() || in_reach(x)) &&
                   (!need_dx || in_reach(saved[1 + i]));
            // the forward product may have been the library's, and saved-tensor hooks may bring the weight back in another layout
            if (need_dx) fit = fit && aligned(saved[1 + i]);
        }
        Tensor dx, any;                                    // any: a gradient, for device and type
        for (int64_t i = 0; i < n && !any.defined(); ++i) any = dy[i];
        if (!any.defined()) return variable_list(n + at.size() - std::count(at.begin(), at.end(), -1) + 4);
        Launch l(any);
        int64_t sum_out = 0;
        for (const Tensor& t : dy) sum_out += t.defined() ? t.size(1) : 0;
        const auto mine = [&](int64_t m, int64_t k) { return fit && (small || (wide && !thin(m, in, k))); };
        mi_gemm_problem pr[MI_GEMM_MAX_PROBLEMS];
        int count = 0;
        if (need_dx && mine(rows, sum_out)) {
            dx = at::empty({rows, in}, any.options());
            mi_gemm_problem p = problem(dx, false, true);
            for (int64_t i = 0; i < n; ++i)
                if (dy[i].defined()) segment(p, dy[i], saved[1 + i], dy[i].size(1));
            pr[count++] = p;
        }
        int64_t out = 0;                                   // of the weight gradients that the library makes
        for (int64_t i = 0; i < n; ++i) {
            if (!dy[i].defined() || !need_weight(i)) continue;
            if (!mine(dy[i].size(1), rows)) {
                out += dy[i].size(1);
                continue;
            }
            dw[i] = at::empty({dy[i].size(1), in}, any.options());
            mi_gemm_problem p = problem(dw[i], true, true);
            segment(p, dy[i], x, rows);
            if (need_bias(i)) {
                db[i] = at::empty({dy[i].size(1)}, any.options());
                p.p_sum = ptr(db[i]);
            }
            pr[count++] = p;
        }
        if (count > 0) run_gemm(pr, count, any, l);
        Tensor xt, dyt;                                    // the smaller of the two operands, where that pays
        if (!again && out > 0 && transpose_pays(rows, in, out)) {
            if (in <= out && transposable(x)) xt = transposed(x, l);
            else if (n == 1 && transposable(dy[0])) dyt = transposed(dy[0], l);
        }
        const bool library_dx = need_dx && !dx.defined();
        for (int64_t i = 0; i < n; ++i) {
            if (!dy[i].defined()) continue;
            if (library_dx) {
                const Tensor& w = saved[1 + i];
                if (!dx.defined()) dx = at::mm(dy[i], w);
                else if (again) dx = dx + at::mm(dy[i], w);
                else dx.addmm_(dy[i], w);                  // summed inside the product
            }
            if (need_weight(i) && !dw[i].defined()) dw[i] = dyt.defined() ? at::mm(dyt, x) : at::mm(dy[i].t(), xt.defined() ? xt.t() : x);
            if (need_bias(i) && !db[i].defined()) db[i] = again ? dy[i].sum(0) : bias_gradient(dy[i]);
        }
        variable_list grads{dx.defined() ? dx.view(x_shape) : Tensor()};
        for (int64_t i = 0; i < n; ++i) grads.push_back(dw[i]);
        for (int64_t i = 0; i < n; ++i)
            if (at[i] >= 0) grads.push_back(db[i]);
        grads.push_back(g[0]);                             // residual (ignored without one)
        if (!ctx->saved_data["residual"].toBool()) grads.back() = Tensor();
        grads.resize(grads.size() + 2);                    // has_bias, inference
        return grads;
    }
    static variable_list forward(AutogradContext* ctx, const Tensor& x, at::TensorList params, const OptTensor& residual, const std::vector<int64_t>& has_bias,
                                 bool inference) {
        return run(ctx, x, params, residual, has_bias, inference, x.requires_grad());
    }
    static variable_list backward(AutogradContext* ctx, variable_list g) { return gradients(ctx, g); }
};

// The plain library call where the native nodes do not apply: autocast chooses the dtype, CPU tensors have no kernel, and operands that
// do not fit each other in shape, type or device are the library's to broadcast or refuse.
bool plain_linear(const Tensor& x, const Tensor& w, const OptTensor& b) {
    if (!x.is_cuda() || x.numel() == 0 || w.numel() == 0 || w.dim() != 2 || w.size(1) != x.size(-1) || w.scalar_type() != x.scalar_type() ||
        w.device() != x.device() || (x.scalar_type() != at::kBFloat16 && x.scalar_type() != at::kHalf && x.scalar_type() != at::kFloat))
        return true;
    if (b.has_value() && (b->dim() != 1 || b->size(0) != w.size(0) || b->stride(0) != 1 || b->scalar_type() != x.scalar_type() || b->device() != x.device()))
        return true;
    return at::autocast::is_autocast_enabled(at::kCUDA) || transforming() || transformed(x) || transformed(w) || (b.has_value() && transformed(*b));
}

std::vector<Tensor> op_projections(const Tensor& x, const std::vector<Tensor>& weights, const std::vector<OptTensor>& biases, bool inference) {
    TORCH_CHECK(weights.size() == biases.size() && weights.size() >= 1 && weights.size() <= 3, "projections: one to three weights");
    bool plain = false;
    for (size_t i = 0; i < weights.size(); ++i) plain = plain || plain_linear(x, weights[i], biases[i]);
    if (plain) {
        std::vector<Tensor> out;
        for (size_t i = 0; i < weights.size(); ++i) out.push_back(at::linear(x, weights[i], biases[i]));
        return out;
    }
    variable_list params(weights.begin(), weights.end());
    std::vector<int64_t> has_bias;
    for (const OptTensor& b : biases) {
        has_bias.push_back(b.has_value());
        if (b.has_value()) params.push_back(*b);
    }
    return Projections::apply(x, at::TensorList(params), OptTensor(), has_bias, inference);
}

Tensor op_linear(const Tensor& x, const Tensor& w, const OptTensor& b, const OptTensor& residual, bool inference) {
    const auto residual_fits = [&] {
        return residual->scalar_type() == x.scalar_type() && residual->device() == x.device() && residual->dim() == x.dim() &&
               residual->size(-1) == w.size(0) && residual->sizes().slice(0, x.dim() - 1) == x.sizes().slice(0, x.dim() - 1) && !transformed(*residual);
    };
    const bool plain = plain_linear(x, w, b);
    if (plain || (residual.has_value() && !residual_fits())) {
        const Tensor y = plain ? at::linear(x, w, b) : op_linear(x, w, b, std::nullopt, inference);
        return residual.has_value() ? y + *residual : y;
    }
    variable_list params{w};
    if (b.has_value()) params.push_back(*b);
    return Projections::apply(x, at::TensorList(params), residual, std::vector<int64_t>{b.has_value()}, inference)[0];
}

// ---- attention core ----------------------------------------------------------------------------------------------------
struct AttnOptions {
    bool causal = true;
    double scale = 1.0, dropout_p = 0.0;
    uint64_t seed = 0;
    int flags = 0;
    bool interleaved = false;
    Tensor cos, sin, pos_q, pos_k;      // undefined: no rotary; pos_k undefined (forward): k arrives rotated
};

void fill_args(mi_attn_args& a, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o, const Tensor& lse, const Tensor& cu_q,
               const Tensor& cu_k, const AttnOptions& opts, void* stream) {
    a = mi_attn_args{};
    a.flags = opts.flags;
    a.q = ptr(q); a.k = ptr(k); a.v = ptr(v); a.o = ptr(o); a.lse = (float*)ptr(lse);
    a.cu_seqlens_q = (const int32_t*)ptr(cu_q); a.cu_seqlens_k = (const int32_t*)ptr(cu_k);
    a.n_docs = (int32_t)cu_q.numel() - 1;
    a.causal = opts.causal;
    a.total_q = q.size(0); a.total_k = k.size(0);
    a.n_q_heads = (int32_t)q.size(1); a.n_kv_heads = (int32_t)k.size(1); a.head_dim = (int32_t)q.size(2);
    a.dtype = code_of(q);
    a.q_stride_token = q.stride(0); a.q_stride_head = q.stride(1);
    a.k_stride_token = k.stride(0); a.k_stride_head = k.stride(1);
    a.v_stride_token = v.stride(0); a.v_stride_head = v.stride(1);
    a.o_stride_token = o.stride(0); a.o_stride_head = o.stride(1);
    a.softmax_scale = (float)opts.scale;
    if (opts.cos.defined()) {
        a.rotary_cos = ptr(opts.cos); a.rotary_sin = ptr(opts.sin);
        a.position_ids_q = (const int64_t*)ptr(opts.pos_q); a.position_ids_k = (const int64_t*)ptr(opts.pos_k);
        a.rotary_table_rows = opts.cos.size(0);
        a.rotary_interleaved = opts.interleaved;
    }
    if (opts.dropout_p > 0.0) { a.dropout_p = (float)opts.dropout_p; a.dropout_seed = opts.seed; }
    a.stream = stream;
}

void check_qkv(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& cu_q, const Tensor& cu_k) {
    need_gpu(q); need_gpu(k); need_gpu(v); need_gpu(cu_q);
    for (const Tensor* t : {&q, &k, &v})
        TORCH_CHECK(t->dim() == 3 && t->stride(2) == 1, "q/k/v must be [tokens, heads, head_dim] with contiguous features");
    TORCH_CHECK(k.sizes() == v.sizes() && q.size(2) == k.size(2) && q.scalar_type() == k.scalar_type() && q.scalar_type() == v.scalar_type(),
                "attention: q, k and v do not match");
    TORCH_CHECK(cu_q.scalar_type() == at::kInt && cu_q.is_contiguous() && cu_q.numel() >= 1, "attention: int32 cumulative sequence lengths");
    TORCH_CHECK(!cu_k.defined() || (cu_k.scalar_type() == at::kInt && cu_k.is_contiguous() && cu_k.numel() == cu_q.numel()),
                "attention: int32 cumulative key lengths, as many as for the queries");
}

std::tuple<Tensor, Tensor> attn_forward(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& cu_q, const Tensor& cu_k,
                                        const AttnOptions& opts, const Tensor& q_rot) {
    Launch l(q);
    Tensor o = at::empty({q.size(0), q.size(1), q.size(2)}, q.options());
    Tensor lse = at::empty({q.size(1), q.size(0)}, q.options().dtype(at::kFloat));
    mi_attn_args a;
    fill_args(a, q, k, v, o, lse, cu_q, cu_k, opts, l.stream);
    a.q_rot_out = ptr(q_rot);
    check(mi_attn_fwd(&a), "mi_attn_fwd");
    return {o, lse};
}

// Whether the allocator has so many bytes without giving its cache back first: in a free block of the cache, or on the device within the process's
// share.  (Nothing asks the device while a graph is captured, and not every allocator answers.)
bool has_room(size_t bytes, const Tensor& like) {
    namespace allocator = c10::hip::HIPCachingAllocator;
    const auto device = like.device().index();
    try {
        size_t block = 1, free = 0, total = 0;             // not 0, which would ask the device for a first guess
        allocator::cacheInfo(device, &block);
        if (block >= bytes || c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None) return true;
        if (hipMemGetInfo(&free, &total) != hipSuccess) return true;
        const double share = allocator::getMemoryFraction(device) * (double)total - (double)allocator::getDeviceStats(device).reserved_bytes[0].current;
        return std::min((double)free, share) >= (double)bytes;
    } catch (const c10::Error&) {
        return true;
    }
}

// dq must have the strides of q; `ws` may be undefined
void attn_backward(const Tensor& d_o_, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o, const Tensor& lse, const Tensor& cu_q,
                   const Tensor& cu_k, const AttnOptions& opts, const Tensor& dq, const Tensor& dk, const Tensor& dv, Tensor ws) {
    Launch l(q);
    TORCH_CHECK(dq.strides() == q.strides(), "attention backward: dq needs the layout of q");
    Tensor d_o = d_o_;
    if (d_o.strides() != o.strides()) d_o = at::empty_strided(o.sizes(), o.strides(), o.options()).copy_(d_o_);
    mi_attn_bwd_args b{};
    fill_args(b.fwd, q, k, v, o, lse, cu_q, cu_k, opts, l.stream);
    if (!ws.defined()) {
        const size_t least = std::max<size_t>(16, mi_attn_bwd_workspace_bytes_kv(q.size(0), k.size(0), (int)q.size(1), (int)k.size(1), (int)q.size(2)));
        size_t best = std::max(least, mi_attn_bwd_workspace_bytes_for(&b.fwd));
        if (best > least && !has_room(best, q)) best = least;
        try {
            ws = float_buffer(best, q);
        } catch (const c10::OutOfMemoryError&) {           // does with less, as it did
            if (best == least) throw;
            ws = float_buffer(least, q);
        }
    }
    b.d_o = ptr(d_o); b.dq = ptr(dq); b.dk = ptr(dk); b.dv = ptr(dv);
    b.dk_stride_token = dk.stride(0); b.dk_stride_head = dk.stride(1);
    b.dv_stride_token = dv.stride(0); b.dv_stride_head = dv.stride(1);
    b.workspace = ptr(ws);
    b.workspace_bytes = (size_t)ws.numel() * 4;
    check(mi_attn_bwd(&b), "mi_attn_bwd");
}

AttnOptions options(bool causal, double scale, int flags, double dropout_p, uint64_t seed, const OptTensor& cos, const OptTensor& sin,
                    const OptTensor& pos_q, const OptTensor& pos_k, bool interleaved) {
    AttnOptions o;
    o.causal = causal; o.scale = scale; o.flags = flags; o.dropout_p = dropout_p; o.seed = seed; o.interleaved = interleaved;
    o.cos = opt(cos); o.sin = opt(sin); o.pos_q = opt(pos_q); o.pos_k = opt(pos_k);
    return o;
}

std::tuple<Tensor, Tensor, Tensor> op_attention_forward(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& cu_q, const OptTensor& cu_k,
                                                     bool causal, double scale, int flags, double dropout_p, uint64_t seed, const OptTensor& cos,
                                                     const OptTensor& sin, const OptTensor& pos_q, const OptTensor& pos_k, bool interleaved,
                                                     bool return_rotated_q) {
    check_qkv(q, k, v, cu_q, opt(cu_k));
    Tensor q_rot;
    if (return_rotated_q) q_rot = at::empty_strided(q.sizes(), q.strides(), q.options());
    auto [o, lse] = attn_forward(q, k, v, cu_q, opt(cu_k), options(causal, scale, flags, dropout_p, seed, cos, sin, pos_q, pos_k, interleaved), q_rot);
    return {o, lse, q_rot};
}

std::tuple<Tensor, Tensor, Tensor> op_attention_backward(const Tensor& d_o, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o,
                                                      const Tensor& lse, const Tensor& cu_q, const OptTensor& cu_k, bool causal, double scale, int flags,
                                                      double dropout_p, uint64_t seed, const OptTensor& cos, const OptTensor& sin, const OptTensor& pos_q,
                                                      const OptTensor& pos_k, bool interleaved, const OptTensor& dq_, const OptTensor& dk_,
                                                      const OptTensor& dv_, const OptTensor& ws) {
    check_qkv(q, k, v, cu_q, opt(cu_k));
    const Tensor dq = dq_.has_value() ? *dq_ : at::empty_strided(q.sizes(), q.strides(), q.options());
    const Tensor dk = dk_.has_value() ? *dk_ : at::empty(k.sizes(), k.options());
    const Tensor dv = dv_.has_value() ? *dv_ : at::empty(v.sizes(), v.options());
    attn_backward(d_o, q, k, v, o, lse, cu_q, opt(cu_k), options(causal, scale, flags, dropout_p, seed, cos, sin, pos_q, pos_k, interleaved), dq, dk, dv, opt(ws));
    return {dq, dk, dv};
}

// What the autograd node of the attention core keeps beside its tensors
template <class Context> void keep_options(Context* ctx, const AttnOptions& o) {
    ctx->saved_data["causal"] = o.causal;
    ctx->saved_data["scale"] = o.scale;
    ctx->saved_data["dropout_p"] = o.dropout_p;
    ctx->saved_data["seed"] = (int64_t)o.seed;
    ctx->saved_data["flags"] = (int64_t)o.flags;
    ctx->saved_data["interleaved"] = o.interleaved;
}
template <class Context> AttnOptions kept_options(Context* ctx) {
    AttnOptions o;
    o.causal = ctx->saved_data["causal"].toBool();
    o.scale = ctx->saved_data["scale"].toDouble();
    o.dropout_p = ctx->saved_data["dropout_p"].toDouble();
    o.seed = (uint64_t)ctx->saved_data["seed"].toInt();
    o.flags = (int)ctx->saved_data["flags"].toInt();
    o.interleaved = ctx->saved_data["interleaved"].toBool();
    return o;
}

// Forward of either node; with rotary, k is rotated once by the stand-alone kernel and q while the attention kernel loads it, and
// the rotated tensors are what the backward kernels stream, so they are kept instead of q and k.
template <class Context> Tensor attention_node_forward(Context* ctx, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& cu_q, const Tensor& cu_k,
                                                       const AttnOptions& opts, bool need_grad) {
    check_qkv(q, k, v, cu_q, cu_k);
    keep_options(ctx, opts);
    if (!opts.cos.defined()) {
        auto [o, lse] = attn_forward(q, k, v, cu_q, cu_k, opts, Tensor());
        ctx->save_for_backward({q, k, v, o, lse, cu_q, cu_k, Tensor(), Tensor(), Tensor(), Tensor()});
        return o;
    }
    const Tensor k_rot = rotary_launch(k, opts.cos, opts.sin, opts.pos_k, 0, false, opts.interleaved);
    AttnOptions f = opts;
    f.pos_k = Tensor();
    // nothing to differentiate: the rotated q is not written out
    const Tensor q_rot = need_grad ? at::empty_strided(q.sizes(), q.strides(), q.options()) : Tensor();
    auto [o, lse] = attn_forward(q, k_rot, v, cu_q, cu_k, f, q_rot);
    if (need_grad) ctx->save_for_backward({q_rot, k_rot, v, o, lse, cu_q, cu_k, opts.cos, opts.sin, opts.pos_q, opts.pos_k});
    return o;
}

struct Attention : Function<Attention> {
    static Tensor forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& cu_q, const OptTensor& cu_k,
                          const AttnOptions* opts, bool need_grad) {
        return attention_node_forward(ctx, q, k, v, cu_q, opt(cu_k), *opts, need_grad);
    }
    template <class Context> static variable_list gradients(Context* ctx, const variable_list& g) {
        const variable_list s = ctx->get_saved_variables();         // read once: saved-tensor hooks unpack on access
        AttnOptions opts = kept_options(ctx);
        opts.cos = s[7]; opts.sin = s[8]; opts.pos_q = s[9]; opts.pos_k = s[10];
        const Tensor &q = s[0], &k = s[1], &v = s[2];
        const Tensor dq = at::empty_strided(q.sizes(), q.strides(), q.options()), dk = at::empty(k.sizes(), k.options()), dv = at::empty(v.sizes(), v.options());
        attn_backward(g[0], q, k, v, s[3], s[4], s[5], s[6], opts, dq, dk, dv, Tensor());
        return {dq, dk, dv, Tensor(), Tensor(), Tensor(), Tensor()};
    }
    static variable_list backward(AutogradContext* ctx, variable_list g) { return gradients(ctx, g); }
};

Tensor op_attention(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& cu_q, const OptTensor& cu_k, bool causal, double scale,
                 double dropout_p, uint64_t seed, const OptTensor& cos, const OptTensor& sin, const OptTensor& pos_q, const OptTensor& pos_k,
                 bool interleaved, bool precise) {
    const AttnOptions o = options(causal, scale, precise ? MI_ATTN_SPLIT_P : 0, dropout_p, seed, cos, sin, pos_q, pos_k, interleaved);
    const bool need_grad = at::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() || v.requires_grad());
    return Attention::apply(q, k, v, cu_q, cu_k, &o, need_grad);
}

// The same on one projection output qkv [tokens, heads, 3 d] (per head q, then k, then v): the gradient is written into one tensor of
// that layout by the kernels themselves.  (As three slices of qkv, each gradient would be padded with zeros to the
// size of qkv and the three summed: eight passes over a tensor of that size.)
struct AttentionQkv : Function<AttentionQkv> {
    template <class Context> static Tensor run(Context* ctx, const Tensor& qkv, const Tensor& cu_q, const OptTensor& cu_k, const AttnOptions& opts, bool need_grad) {
        const int64_t d = qkv.size(2) / 3;
        return attention_node_forward(ctx, qkv.narrow(2, 0, d), qkv.narrow(2, d, d), qkv.narrow(2, 2 * d, d), cu_q, opt(cu_k), opts, need_grad);
    }
    static Tensor forward(AutogradContext* ctx, const Tensor& qkv, const Tensor& cu_q, const OptTensor& cu_k, const AttnOptions* opts, bool need_grad) {
        return run(ctx, qkv, cu_q, cu_k, *opts, need_grad);
    }
    template <class Context> static variable_list gradients(Context* ctx, const variable_list& g) {
        const variable_list s = ctx->get_saved_variables();
        AttnOptions opts = kept_options(ctx);
        opts.cos = s[7]; opts.sin = s[8]; opts.pos_q = s[9]; opts.pos_k = s[10];
        const int64_t d = s[0].size(2);
        const Tensor dqkv = at::empty({s[0].size(0), s[0].size(1), 3 * d}, s[0].options()), dq = dqkv.narrow(2, 0, d);
        // saved-tensor hooks (activations kept on the host) may bring q back with rows of its own instead of a slice of qkv's
        const Tensor q = s[0].strides() == dq.strides() ? s[0] : at::empty_strided(dq.sizes(), dq.strides(), dq.options()).copy_(s[0]);
        attn_backward(g[0], q, s[1], s[2], s[3], s[4], s[5], s[6], opts, dq, dqkv.narrow(2, d, d), dqkv.narrow(2, 2 * d, d), Tensor());
        return {dqkv, Tensor(), Tensor(), Tensor(), Tensor()};
    }
    static variable_list backward(AutogradContext* ctx, variable_list g) { return gradients(ctx, g); }
};

Tensor op_attention_qkv(const Tensor& qkv, const Tensor& cu_q, const OptTensor& cu_k, bool causal, double scale, double dropout_p, uint64_t seed,
                        const OptTensor& cos, const OptTensor& sin, const OptTensor& pos_q, const OptTensor& pos_k, bool interleaved) {
    TORCH_CHECK(qkv.dim() == 3 && qkv.is_contiguous() && qkv.size(2) % 3 == 0, "qkv must be contiguous [tokens, heads, 3 head_dim]");
    const AttnOptions o = options(causal, scale, 0, dropout_p, seed, cos, sin, pos_q, pos_k, interleaved);
    return AttentionQkv::apply(qkv, cu_q, cu_k, &o, at::GradMode::is_enabled() && qkv.requires_grad());
}

// ---- a layer in one call -----------------------------------------------------------------------------------------------
// The kernels take the tables' bytes for what `interleaved` and the type of the rows say: float32 [rows, head_dim / 2], or [rows, head_dim] of x's type where
// the attention kernel rotates (whole), or any part of a head, of x's type or float32.
void check_tables(const Tensor& x, int64_t head_dim, const OptTensor& cos, const OptTensor& sin, bool interleaved, bool whole) {
    const auto fits = [&](at::ScalarType type, int64_t width) { return cos->scalar_type() == type && cos->size(1) == width; };
    TORCH_CHECK(cos.has_value() && sin.has_value() && cos->dim() == 2 && cos->sizes() == sin->sizes() && cos->scalar_type() == sin->scalar_type() &&
                    cos->device() == x.device() && sin->device() == x.device() && cos->is_contiguous() && sin->is_contiguous() &&
                    (interleaved ? fits(at::kFloat, head_dim / 2)
                     : whole     ? fits(x.scalar_type(), head_dim)
                                 : cos->size(1) <= head_dim && (cos->scalar_type() == x.scalar_type() || cos->scalar_type() == at::kFloat)),
                "rotary: tables have to fit the type and the features of the rows");
}

// Attention over the rows of a prefill [batch * seq, heads, head_dim] (inference), which leaves rotated k and v in the caches
// [batch, max_ctx, KV heads, head_dim] and raises ctx_len to seq: two launches, or with q_first one more that rotates q in front of the attention kernel.
Tensor prefill_attention(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& cu, const Tensor& pos, const Tensor& cos, const Tensor& sin,
                         bool interleaved, double scale, int64_t batch, const Tensor& k_cache, const Tensor& v_cache, const Tensor& ctx_len, bool q_first) {
    check_qkv(q, k, v, cu, Tensor());
    TORCH_CHECK(batch > 0 && k.size(0) % batch == 0 && k.size(0) == q.size(0) && k_cache.dim() == 4 && k_cache.sizes() == v_cache.sizes() &&
                    k_cache.strides() == v_cache.strides() && k_cache.stride(3) == 1 && k_cache.size(0) == batch && k_cache.size(2) == k.size(1) &&
                    k_cache.size(3) == k.size(2) && k_cache.scalar_type() == k.scalar_type() && v_cache.scalar_type() == k.scalar_type() &&
                    ctx_len.scalar_type() == at::kInt && ctx_len.is_contiguous() && ctx_len.numel() == batch && pos.scalar_type() == at::kLong &&
                    pos.is_contiguous() && pos.numel() == k.size(0),
                "prefill attention: caches, lengths and position ids have to fit the rows");
    check_tables(k, k.size(2), cos, sin, interleaved, true);
    for (const Tensor* t : {&k_cache, &v_cache, &ctx_len, &pos}) need_gpu(*t);
    Launch l(q);
    const Tensor k_rot = at::empty(k.sizes(), k.options());
    mi_fill_cache_args a{};
    a.k = ptr(k); a.v = ptr(v); a.k_rot = ptr(k_rot); a.k_cache = ptr(k_cache); a.v_cache = ptr(v_cache); a.ctx_len = static_cast<int32_t*>(ptr(ctx_len));
    a.rotary_cos = ptr(cos); a.rotary_sin = ptr(sin); a.position_ids = static_cast<const int64_t*>(ptr(pos)); a.table_rows = cos.size(0);
    a.k_stride_token = k.stride(0); a.k_stride_head = k.stride(1); a.v_stride_token = v.stride(0); a.v_stride_head = v.stride(1);
    a.cache_stride_batch = k_cache.stride(0); a.cache_stride_token = k_cache.stride(1); a.cache_stride_head = k_cache.stride(2);
    a.batch = (int32_t)batch; a.seq = (int32_t)(k.size(0) / batch); a.max_ctx = (int32_t)k_cache.size(1); a.n_kv_heads = (int32_t)k.size(1);
    a.head_dim = (int32_t)k.size(2); a.dtype = code_of(k); a.rotary_interleaved = interleaved; a.stream = l.stream;
    check(mi_fill_cache(&a), "mi_fill_cache");
    if (q_first) {
        const Tensor q_rot = rotary_launch(q, cos, sin, pos, 0, false, interleaved);
        const auto plain = options(true, scale, 0, 0.0, 0, std::nullopt, std::nullopt, std::nullopt, std::nullopt, false);
        return std::get<0>(attn_forward(q_rot, k_rot, v, cu, Tensor(), plain, Tensor()));
    }
    return std::get<0>(attn_forward(q, k_rot, v, cu, Tensor(), options(true, scale, 0, 0.0, 0, cos, sin, pos, std::nullopt, interleaved), Tensor()));
}

Tensor op_prefill_attention(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& cu, const Tensor& pos, const Tensor& cos, const Tensor& sin,
                            bool interleaved, double scale, int64_t batch, const Tensor& k_cache, const Tensor& v_cache, const Tensor& ctx_len) {
    return prefill_attention(q, k, v, cu, pos, cos, sin, interleaved, scale, batch, k_cache, v_cache, ctx_len, false);
}

// A pre-norm layer on x [batch, seq, hidden]: the same operations, one after the other, as the modules of the layer issue them; what it saves is the way
// through those modules (half of a small layer's forward pass).
struct LayerCall : torch::CustomClassHolder {
    Tensor x, cu;
    OptTensor pos, cos, sin;
    std::vector<OptTensor> norms;                          // [weight, bias (RMSNorm: none)] of either norm
    double eps1, eps2, scale;
    bool layer_norm1, layer_norm2, in_one, causal, interleaved, inference;
    std::vector<Tensor> qkv_w, rest_w;                     // qkv: one weight, per head q, k, v (in_one) or the rows of q, of k and of v; or three
    std::vector<OptTensor> qkv_b, rest_b;                  // rest: dense, and in, (gate,) out of the MLP
    int64_t nq, nkv, d;
    int rotary;                                            // 0 none, 1 inside the attention core, 2 in front of it
    std::vector<Tensor> caches;                            // [k, v, ctx_len] of a prefill (rotary 1, inference) or empty
    enum Part { kNorm1, kQkv, kRotary, kAttention, kDense, kNorm2, kIn, kActivation, kOut, kParts };
    bool split() const { return !in_one || rotary == 2; }  // q, k and v reach the attention core as three
};
// Of a layer that is one node, with what its gradients need: as in nodes of their own, each part looks at its tensors when its turn comes (whether they were
// changed in place), gives them back then, and keeps none where no gradient comes by.
struct LayerKept : LayerCall {
    Kept parts[kParts];
    torch::autograd::SavedVariable input;                  // x, and versions of the rest: what a graph of the gradients is made from
    std::vector<uint32_t> versions;
    void give_back() {
        for (Kept& part : parts) part.give_back();
        input.reset_data();
    }
};

// The operations of a layer, each with a node of its own
struct Apart {
    const LayerCall& c;
    std::tuple<Tensor, Tensor> norm(LayerCall::Part, const Tensor& x, const OptTensor& residual, const Tensor& w, const OptTensor& b, double eps, bool layer_norm) {
        return op_add_norm(x, residual, w, b, eps, layer_norm);
    }
    std::vector<Tensor> projections(LayerCall::Part, const Tensor& x, const std::vector<Tensor>& w, const std::vector<OptTensor>& b, const OptTensor& residual) {
        if (w.size() > 1) return op_projections(x, w, b, c.inference);
        return {op_linear(x, w[0], b[0], residual, c.inference)};
    }
    variable_list rotary(const Tensor& q, const Tensor& k, int64_t s) { return RotaryTwo::apply(q, k, *c.cos, *c.sin, c.pos, s, c.interleaved); }
    Tensor attention(const Tensor& q, const Tensor& k, const Tensor& v, const AttnOptions& o) {
        return Attention::apply(q, k, v, c.cu, OptTensor(), &o, at::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() || v.requires_grad()));
    }
    Tensor attention_qkv(const Tensor& qkv, const AttnOptions& o) {
        return AttentionQkv::apply(qkv, c.cu, OptTensor(), &o, at::GradMode::is_enabled() && qkv.requires_grad());
    }
    Tensor gelu(const Tensor& x) { return Gelu::apply(x); }
    Tensor swiglu(const Tensor& a, const Tensor& gate) { return SwiGlu::apply(a, gate); }
};

// The same with no node of their own: what the gradients need stays in the call.  `grad`: something up to here takes a gradient
struct Together {
    LayerKept& c;
    bool recorded, grad;
    Together(LayerKept& call, bool recorded_) : c(call), recorded(recorded_), grad(recorded_ && call.x.requires_grad()) {}
    void reaches(const Tensor& p) { grad = grad || (recorded && p.requires_grad()); }
    Kept* kept(LayerCall::Part p) {
        c.parts[p].keeps = grad;
        return &c.parts[p];
    }
    std::tuple<Tensor, Tensor> norm(LayerCall::Part p, const Tensor& x, const OptTensor& residual, const Tensor& w, const OptTensor& b, double eps, bool layer_norm) {
        reaches(w);
        if (b.has_value()) reaches(*b);
        auto out = AddNorm::run(kept(p), x, residual, w, b, eps, layer_norm);
        return {out[0], out[1]};
    }
    std::vector<Tensor> projections(LayerCall::Part p, const Tensor& x, const std::vector<Tensor>& w, const std::vector<OptTensor>& b, const OptTensor& residual) {
        variable_list params(w.begin(), w.end());
        std::vector<int64_t> has_bias;
        for (const OptTensor& t : b) {
            has_bias.push_back(t.has_value());
            if (t.has_value()) params.push_back(*t);
        }
        const bool need_dx = grad;
        for (const Tensor& t : params) reaches(t);
        return Projections::run(kept(p), x, params, residual, has_bias, c.inference, need_dx);
    }
    variable_list rotary(const Tensor& q, const Tensor& k, int64_t s) {
        return RotaryTwo::run(kept(LayerCall::kRotary), q, k, *c.cos, *c.sin, c.pos, s, c.interleaved);
    }
    Tensor attention(const Tensor& q, const Tensor& k, const Tensor& v, const AttnOptions& o) {
        return attention_node_forward(kept(LayerCall::kAttention), q, k, v, c.cu, Tensor(), o, grad);
    }
    Tensor attention_qkv(const Tensor& qkv, const AttnOptions& o) { return AttentionQkv::run(kept(LayerCall::kAttention), qkv, c.cu, OptTensor(), o, grad); }
    Tensor gelu(const Tensor& x) { return Gelu::run(kept(LayerCall::kActivation), x); }
    Tensor swiglu(const Tensor& a, const Tensor& gate) { return SwiGlu::run(kept(LayerCall::kActivation), a, gate); }
};

template <class Operations> Tensor layer_forward(const LayerCall& c, Operations ops) {
    const int64_t b = c.x.size(0), s = c.x.size(1), tokens = b * s, nq = c.nq, nkv = c.nkv, d = c.d;
    auto [h, n] = ops.norm(LayerCall::kNorm1, c.x, std::nullopt, *c.norms[0], c.norms[1], c.eps1, c.layer_norm1);
    const auto into = ops.projections(LayerCall::kQkv, n, c.qkv_w, c.qkv_b, std::nullopt);
    const bool fused = c.rotary == 1;
    const auto rotated = [&] {
        return options(c.causal, c.scale, 0, 0.0, 0, fused ? c.cos : OptTensor(), fused ? c.sin : OptTensor(), fused ? c.pos : OptTensor(),
                       fused ? c.pos : OptTensor(), c.interleaved);
    };
    Tensor ctx;
    if (!c.split()) {
        ctx = ops.attention_qkv(into[0].view({tokens, nq, 3 * d}), rotated());
    } else {
        Tensor q, k, v;
        if (c.in_one) {
            const Tensor qkv = into[0].view({tokens, nq, 3 * d});
            q = qkv.narrow(2, 0, d); k = qkv.narrow(2, d, d); v = qkv.narrow(2, 2 * d, d);
        } else if (into.size() == 1) {
            const Tensor qkv = into[0].view({tokens, nq + 2 * nkv, d});
            q = qkv.narrow(1, 0, nq); k = qkv.narrow(1, nq, nkv); v = qkv.narrow(1, nq + nkv, nkv);
        } else {
            q = into[0].view({tokens, nq, d}); k = into[1].view({tokens, nkv, d}); v = into[2].view({tokens, nkv, d});
        }
        if (!c.caches.empty()) {
            // float16: the stand-alone kernel rounds some sums of q otherwise than the attention kernel does on its loads, and the modules take that kernel
            ctx = prefill_attention(q, k, v, c.cu, *c.pos, *c.cos, *c.sin, c.interleaved, c.scale, b, c.caches[0], c.caches[1], c.caches[2],
                                    q.scalar_type() == at::kHalf);
        } else {
            if (c.rotary == 2) {
                const auto both = ops.rotary(q, k, s);
                q = both[0];
                k = both[1];
            }
            ctx = ops.attention(q, k, v, rotated());
        }
    }
    const Tensor a = ops.projections(LayerCall::kDense, ctx.view({b, s, nq * d}), {c.rest_w[0]}, {c.rest_b[0]}, std::nullopt)[0];
    std::tie(h, n) = ops.norm(LayerCall::kNorm2, a, h, *c.norms[2], c.norms[3], c.eps2, c.layer_norm2);
    Tensor act;
    if (c.rest_w.size() == 4) {
        const auto out = ops.projections(LayerCall::kIn, n, {c.rest_w[1], c.rest_w[2]}, {c.rest_b[1], c.rest_b[2]}, std::nullopt);
        act = ops.swiglu(out[0], out[1]);
    } else {
        act = ops.gelu(ops.projections(LayerCall::kIn, n, {c.rest_w[1]}, {c.rest_b[1]}, std::nullopt)[0]);
    }
    return ops.projections(LayerCall::kOut, act, {c.rest_w.back()}, {c.rest_b.back()}, h)[0];
}

constexpr int64_t kOneNode = 1 << 19;                      // elements of x

// The layer as one autograd node.  Inputs: x and the parameters in the order of `parameters`.
struct Layer : Function<Layer> {
    template <class Call, class F> static void parameters(Call& c, F f) {
        const auto all = [&](auto& w, auto& b, size_t first, size_t last) {
            for (size_t i = first; i < last; ++i) f(w[i]);
            for (size_t i = first; i < last; ++i)
                if (b[i].has_value()) f(*b[i]);
        };
        const size_t out = c.rest_w.size() - 1;
        for (int i : {0, 1}) if (c.norms[i].has_value()) f(*c.norms[i]);
        all(c.qkv_w, c.qkv_b, 0, c.qkv_w.size());
        all(c.rest_w, c.rest_b, 0, 1);
        for (int i : {2, 3}) if (c.norms[i].has_value()) f(*c.norms[i]);
        all(c.rest_w, c.rest_b, 1, out);
        all(c.rest_w, c.rest_b, out, out + 1);
    }
    static std::vector<uint32_t> versions(const LayerCall& c) {
        std::vector<uint32_t> v;
        const auto add = [&](const Tensor& t) {
            if (t.defined() && !t.is_inference()) v.push_back(t._version());
        };
        parameters(c, add);
        add(c.cu);
        if (c.rotary != 0)
            for (const OptTensor* t : {&c.pos, &c.cos, &c.sin}) add(opt(*t));
        return v;
    }
    static Tensor forward(AutogradContext* ctx, at::TensorList, const c10::intrusive_ptr<LayerKept>& c) {
        const Tensor y = layer_forward(*c, Together(*c, true));
        c->input = torch::autograd::SavedVariable(c->x, false);
        c->x = Tensor();
        c->versions = versions(*c);
        ctx->set_materialize_grads(false);
        ctx->saved_data["call"] = at::IValue::make_capsule(c);
        return y;
    }
    static variable_list backward(AutogradContext* ctx, variable_list g) {
        using Part = LayerCall::Part;
        ctx->get_saved_variables();                        // raises where the graph is used up
        const auto held = ctx->saved_data["call"].toCapsule();
        LayerKept& c = static_cast<LayerKept&>(*held);
        struct UsedUp {                                    // a pass that keeps the graph leaves everything, any other nothing
            LayerKept& c;
            bool kept;
            ~UsedUp() { if (!kept) c.give_back(); }
        } const graph{c, torch::autograd::get_current_graph_task_keep_graph()};
        size_t n_inputs = 1;
        parameters(c, [&](const Tensor&) { ++n_inputs; });
        variable_list grads(n_inputs + 1), inputs;         // of the inputs and the call
        if (!g[0].defined()) return grads;
        if (at::GradMode::is_enabled()) {                  // this pass is to be differentiated again: the graph of many nodes
            // On an alias of each input at each of its places, differentiated with respect to these alone: hooks and retained gradients of the inputs themselves,
            // their other uses and what x was made of belong to the pass that is under way.  An alias leads to where this node's gradient of it goes.
            // The forward pass is gone through again, so what it reads has to be what it was: biases, say, are not among what the node saves.
            TORCH_CHECK(versions(c) == c.versions, "layer: one of the variables needed for gradient computation has been modified by an inplace operation: "
                                                   "a parameter, the lengths, the positions or a rotary table, all of which a graph of the gradients is made from");
            const auto node = torch::autograd::get_current_node();
            const auto alias = [&](const Tensor& t) {
                const Tensor a = t.detach();
                const auto& edge = node->next_edge(inputs.size());
                if (edge.is_valid()) {
                    const auto way = std::make_shared<torch::autograd::Identity>();
                    way->add_next_edge(edge);
                    torch::autograd::set_history(a, way);
                }
                inputs.push_back(a);
                return a;
            };
            LayerCall again = c;
            again.x = alias(c.input.unpack());
            parameters(again, [&](Tensor& p) { p = alias(p); });
            const Tensor y = [&] {                         // in the types of the pass that was, whatever this one is under
                const c10::impl::ExcludeDispatchKeyGuard no_autocast(c10::autocast_dispatch_keyset);
                return layer_forward(again, Apart{again});
            }();
            variable_list wanted;
            for (size_t i = 0; i < inputs.size(); ++i)
                if (ctx->needs_input_grad(i)) wanted.push_back(inputs[i]);
            const variable_list got = torch::autograd::grad({y}, wanted, {g[0]}, true, true, true);
            for (size_t i = 0, next = 0; i < inputs.size(); ++i)
                if (ctx->needs_input_grad(i)) grads[i] = got[next++];
            return grads;
        }
        // Tensor inputs of each operation that takes parameters, whether they need a gradient, and where it goes
        struct Group { size_t first; std::vector<bool> needs; bool any; };
        size_t next = 1;
        const auto group = [&](size_t weights, const OptTensor* b) {
            Group r{next, {}, false};
            size_t n = weights;
            for (size_t i = 0; i < weights; ++i) n += b[i].has_value();
            for (; next < r.first + n; ++next) {
                r.needs.push_back(ctx->needs_input_grad(next));
                r.any = r.any || r.needs.back();
            }
            return r;
        };
        const size_t mlp_in = c.rest_w.size() - 2;
        const Group norm1 = group(1, &c.norms[1]), qkv = group(c.qkv_w.size(), c.qkv_b.data()), dense = group(1, c.rest_b.data()),
                    norm2 = group(1, &c.norms[3]), in = group(mlp_in, c.rest_b.data() + 1), out = group(1, c.rest_b.data() + 1 + mlp_in);
        // Whether a gradient goes on from each operation to what comes before it
        const bool from_qkv = ctx->needs_input_grad(0) || norm1.any, from_dense = from_qkv || qkv.any, from_in = from_dense || dense.any || norm2.any,
                   from_out = from_in || in.any;
        const auto part = [&](Part p) {
            Replayed r{{}, c.parts[p].saved_data, {}};
            for (const auto& t : c.parts[p].saved) r.saved.push_back(t.unpack());
            if (!graph.kept) c.parts[p].give_back();
            return r;
        };
        const auto projections = [&](Part p, const Group& own, bool on, const variable_list& dy) {
            Replayed r = part(p);
            r.needs = own.needs;
            r.needs.insert(r.needs.begin(), on);
            const variable_list d = Projections::gradients(&r, dy);
            std::copy(d.begin() + 1, d.begin() + 1 + own.needs.size(), grads.begin() + own.first);
            return d[0];
        };
        const auto norm = [&](Part p, const Group& own, const Tensor& dsum, const Tensor& dy) {
            Replayed r = part(p);
            const variable_list d = AddNorm::gradients(&r, {dsum, dy});
            std::copy(d.begin() + 2, d.begin() + 2 + own.needs.size(), grads.begin() + own.first);
            return d[0];
        };
        Tensor d = projections(LayerCall::kOut, out, from_out, g);
        if (!from_out) return grads;
        const auto activation = [&](Tensor dy) {
            Replayed r = part(LayerCall::kActivation);
            return mlp_in == 2 ? SwiGlu::gradients(&r, {dy}) : Gelu::gradients(&r, {dy});
        };
        variable_list dmany = activation(std::move(d));
        d = projections(LayerCall::kIn, in, from_in, dmany);
        dmany.clear();
        if (!from_in) return grads;
        const Tensor dh = norm(LayerCall::kNorm2, norm2, g[0], d);
        if (!from_dense && !dense.any) return grads;
        d = projections(LayerCall::kDense, dense, from_dense, {dh});
        if (!from_dense) return grads;
        const int64_t tokens = dh.numel() / dh.size(-1);
        const auto attention = [&](Tensor dctx) {
            Replayed r = part(LayerCall::kAttention);
            const variable_list dout{dctx.view({tokens, c.nq, c.d})};
            variable_list dqkv = c.split() ? Attention::gradients(&r, dout) : AttentionQkv::gradients(&r, dout);
            dqkv.resize(c.split() ? 3 : 1);
            return dqkv;
        };
        dmany = attention(std::move(d));
        if (c.rotary == 2) {
            Replayed rotary = part(LayerCall::kRotary);
            const variable_list two = RotaryTwo::gradients(&rotary, {dmany[0], dmany[1]});
            std::copy(two.begin(), two.begin() + 2, dmany.begin());
        }
        if (c.in_one && c.split()) dmany = {at::cat(dmany, 2)};
        for (Tensor& t : dmany) t = t.reshape({tokens, -1});
        d = projections(LayerCall::kQkv, qkv, from_qkv, dmany);
        dmany.clear();
        if (!from_qkv) return grads;
        grads[0] = norm(LayerCall::kNorm1, norm1, dh, d);
        return grads;
    }
};

// Whether the operations of a layer may run with no dispatch between them: nothing watches them, and every operand is one that their own nodes take to the
// kernels of this package.
bool unwatched(const LayerCall& c) {
    if (at::SavedTensorDefaultHooks::get_hooks().has_value() || at::autocast::is_autocast_enabled(at::kCUDA) || transforming() || transformed(c.x) ||
        c.x.numel() == 0 || !c.x.is_cuda() || (c.cos.has_value() && (c.cos->requires_grad() || c.sin->requires_grad())))
        return false;
    const int64_t hidden = c.x.size(2), inter = c.rest_w.back().dim() == 2 ? c.rest_w.back().size(1) : -1;
    const auto own = [&](const Tensor& t) { return t.is_leaf() && t.scalar_type() == c.x.scalar_type() && t.device() == c.x.device() && !transformed(t); };
    const auto linear = [&](const Tensor& w, const OptTensor& b, int64_t out_features, int64_t in_features) {
        return w.dim() == 2 && w.size(0) == out_features && w.size(1) == in_features && w.numel() > 0 && own(w) &&
               (!b.has_value() || (b->dim() == 1 && b->size(0) == out_features && b->stride(0) == 1 && own(*b)));
    };
    const int64_t q = c.nq * c.d, kv = c.nkv * c.d;
    bool fits = linear(c.rest_w[0], c.rest_b[0], hidden, q) && linear(c.rest_w.back(), c.rest_b.back(), hidden, inter);
    for (size_t i = 1; i + 1 < c.rest_w.size(); ++i) fits = fits && linear(c.rest_w[i], c.rest_b[i], inter, hidden);
    if (c.qkv_w.size() == 3)
        fits = fits && !c.in_one && linear(c.qkv_w[0], c.qkv_b[0], q, hidden) && linear(c.qkv_w[1], c.qkv_b[1], kv, hidden) && linear(c.qkv_w[2], c.qkv_b[2], kv, hidden);
    else
        fits = fits && linear(c.qkv_w[0], c.qkv_b[0], c.in_one ? 3 * q : q + 2 * kv, hidden);
    for (const OptTensor& t : c.norms) fits = fits && (!t.has_value() || (t->dim() == 1 && t->size(0) == hidden && own(*t)));
    return fits;
}

Tensor op_layer(const Tensor& x, const Tensor& cu, const OptTensor& pos, std::vector<OptTensor> norms, double eps1, double eps2, bool layer_norm1,
                bool layer_norm2, std::vector<Tensor> qkv_w, std::vector<OptTensor> qkv_b, bool in_one, std::vector<Tensor> rest_w,
                std::vector<OptTensor> rest_b, int64_t nq, int64_t nkv, int64_t d, bool causal, double scale, int rotary, bool interleaved,
                const OptTensor& cos, const OptTensor& sin, std::vector<Tensor> caches, bool inference) {
    TORCH_CHECK(x.dim() == 3 && norms.size() == 4 && norms[0].has_value() && norms[2].has_value() && (qkv_w.size() == 1 || qkv_w.size() == 3) &&
                    qkv_b.size() == qkv_w.size() && (rest_w.size() == 3 || rest_w.size() == 4) && rest_b.size() == rest_w.size() &&
                    (caches.empty() || caches.size() == 3),
                "layer: bad arguments");
    if (rotary != 0) check_tables(x, d, cos, sin, interleaved, rotary == 1);
    auto c = c10::make_intrusive<LayerKept>();
    c->x = x; c->cu = cu; c->pos = pos; c->cos = cos; c->sin = sin; c->norms = std::move(norms);
    c->eps1 = eps1; c->eps2 = eps2; c->scale = scale; c->layer_norm1 = layer_norm1; c->layer_norm2 = layer_norm2; c->in_one = in_one; c->causal = causal;
    c->interleaved = interleaved; c->inference = inference; c->qkv_w = std::move(qkv_w); c->qkv_b = std::move(qkv_b); c->rest_w = std::move(rest_w);
    c->rest_b = std::move(rest_b); c->nq = nq; c->nkv = nkv; c->d = d; c->rotary = rotary; c->caches = std::move(caches);
    if (!unwatched(*c)) return layer_forward(*c, Apart{*c});
    variable_list inputs{x};
    bool recorded = x.requires_grad();
    Layer::parameters(*c, [&](const Tensor& p) {
        inputs.push_back(p);
        recorded = recorded || p.requires_grad();
    });
    if (!recorded || !at::GradMode::is_enabled()) return layer_forward(*c, Together(*c, false));
    // One node instead of 9 to 14, views included: the engine takes 4 us for a node beside its launches, and a small step waits for the host.  Forward and backward
    // of 256 x 256, float32: 354 us with nodes of their own, 286 so; 512 x 1024, bf16: 430 and 380 (on a slower host); 1000 x 1024, where the device is what a step
    // waits for: 370 and 370.  What the parts keep is given back one by one either way.
    // An inference tensor can be no input of it: the node keeps x, which nodes of their own need not.
    if (x.numel() > kOneNode || x.is_inference() || (c->qkv_w.size() == 1 && !in_one)) return layer_forward(*c, Apart{*c});
    return Layer::apply(at::TensorList(inputs), c);
}

// ---- loss --------------------------------------------------------------------------------------------------------------
// Weighted mean of the cross entropy of logits [rows, vocab], and the accuracy.  The gradient takes the log-sum-exp of the forward
// pass, so it reads the logits once.
struct WeightedCrossEntropy : Function<WeightedCrossEntropy> {
    static variable_list forward(AutogradContext* ctx, const Tensor& logits, const Tensor& targets, const Tensor& weights) {
        Launch l(logits);
        const int64_t n = logits.size(0), vocab = logits.size(1);
        const auto f32 = logits.options().dtype(at::kFloat);
        const Tensor rows = at::empty({2, n}, f32), argmax = at::empty({n}, f32.dtype(at::kInt));
        const Tensor loss = at::empty({}, f32), total = at::empty({}, f32), accuracy = at::empty({}, f32);
        float *losses = rows.data_ptr<float>(), *lse = losses + n;
        check(mi_cross_entropy(ptr(logits), targets.data_ptr<int64_t>(), nullptr, losses, lse, argmax.data_ptr<int32_t>(), nullptr, n, vocab,
                               logits.stride(0), 0, code_of(logits), l.stream),
              "mi_cross_entropy");
        check(mi_loss_reduce(losses, argmax.data_ptr<int32_t>(), targets.data_ptr<int64_t>(), weights.data_ptr<float>(), n, loss.data_ptr<float>(),
                             total.data_ptr<float>(), accuracy.data_ptr<float>(), l.stream),
              "mi_loss_reduce");
        ctx->set_materialize_grads(false);
        ctx->mark_non_differentiable({accuracy});
        ctx->save_for_backward({logits, targets, weights, rows, total});
        return {loss, accuracy};
    }
    static variable_list backward(AutogradContext* ctx, variable_list g) {
        if (!g[0].defined()) return {Tensor(), Tensor(), Tensor()};
        const variable_list saved = ctx->get_saved_variables();
        const Tensor& logits = saved[0];
        Launch l(logits);
        const Tensor dloss = g[0].contiguous(), dlogits = at::empty_like(logits);
        const int64_t n = logits.size(0);
        check(mi_cross_entropy_mean_grad(ptr(logits), saved[1].data_ptr<int64_t>(), saved[3].data_ptr<float>() + n, saved[2].data_ptr<float>(),
                                         dloss.data_ptr<float>(), saved[4].data_ptr<float>(), ptr(dlogits), n, logits.size(1), logits.stride(0),
                                         dlogits.stride(0), code_of(logits), l.stream),
              "mi_cross_entropy_mean_grad");
        return {dlogits, Tensor(), Tensor()};
    }
};

std::tuple<Tensor, Tensor> op_weighted_cross_entropy(const Tensor& logits, const Tensor& targets, const Tensor& weights) {
    need_gpu(logits); need_gpu(targets); need_gpu(weights);
    TORCH_CHECK(logits.dim() == 2 && logits.stride(1) == 1 && targets.scalar_type() == at::kLong && targets.is_contiguous() &&
                    targets.numel() == logits.size(0) && weights.scalar_type() == at::kFloat && weights.is_contiguous() &&
                    weights.numel() == logits.size(0),
                "cross entropy: logits [rows, vocab], one int64 target and one float32 weight per row");
    const auto out = WeightedCrossEntropy::apply(logits, targets, weights);
    return {out[0], out[1]};
}

// LM head and weighted mean loss, chunk by chunk: a chunk's logits become their gradient in place and are folded into dh and dW at
// once, so the gradients exist when the forward pass ends and the backward pass only scales them.
struct LinearCrossEntropy : Function<LinearCrossEntropy> {
    static variable_list forward(AutogradContext* ctx, const Tensor& h, const Tensor& weight, const Tensor& targets, const Tensor& weights, int64_t chunk,
                                 bool need_dh, bool need_dw) {
        Launch l(h);
        const int64_t n = h.size(0), vocab = weight.size(0);
        const auto f32 = h.options().dtype(at::kFloat);
        const Tensor rows = at::empty({3, n}, f32), argmax = at::empty({n}, f32.dtype(at::kInt));
        const Tensor loss = at::empty({}, f32), total = at::empty({}, f32), accuracy = at::empty({}, f32);
        float *losses = rows.data_ptr<float>(), *lse = losses + n, *row_scale = lse + n;
        const bool grad = need_dh || need_dw;
        if (grad) check(mi_loss_row_scale(weights.data_ptr<float>(), n, row_scale, l.stream), "mi_loss_row_scale");
        Tensor dh = need_dh ? at::empty_like(h) : Tensor(), dw;       // dw: one chunk: the product itself; several: their sum in fp32
        // Rows of the logits start on 128-byte boundaries (16-bit types) whatever the vocabulary: the library's three products of
        // 2047 x 50257 x 1024 take 776 us with a stride of 50304 and 846 with 50257, and the loss kernel reads and writes
        // whole vectors.
        const int64_t ld = (vocab + 63) / 64 * 64;
        const Tensor buffer = at::empty({std::min(n, chunk), ld}, h.options()), wt = weight.t();
        for (int64_t r0 = 0; r0 < n; r0 += chunk) {
            const int64_t r = std::min(n - r0, chunk);
            const Tensor hc = h.narrow(0, r0, r);
            Tensor logits = buffer.narrow(0, 0, r).narrow(1, 0, vocab);
            // 2047 x 50257 x 1024, us, mi_gemm and library: logits 216 / 257, dh 161 / 291, dW 197 / 252
            const bool wide = wide_product(h, r, 32, h.size(1), Pass::kBackward) && 2.0 * (double)r * (double)vocab * (double)h.size(1) > 3e9 && aligned(hc) &&
                              aligned(weight) && in_reach(hc) && in_reach(weight) && ld < (1 << 22);
            if (wide && !thin(r, vocab, h.size(1))) {
                mi_gemm_problem p = problem(logits, false, false);
                segment(p, hc, weight, h.size(1));
                run_gemm(&p, 1, h, l);
            } else {
                at::mm_out(logits, hc, wt);
            }
            const int64_t* t = targets.data_ptr<int64_t>() + r0;
            if (grad)
                check(mi_cross_entropy_padded(ptr(logits), t, row_scale + r0, losses + r0, lse + r0, argmax.data_ptr<int32_t>() + r0, r, vocab, ld,
                                              code_of(h), l.stream),
                      "mi_cross_entropy_padded");
            else
                check(mi_cross_entropy(ptr(logits), t, nullptr, losses + r0, nullptr, argmax.data_ptr<int32_t>() + r0, nullptr, r, vocab, ld, 0, code_of(h),
                                       l.stream),
                      "mi_cross_entropy");
            if (need_dh) {
                Tensor out = dh.narrow(0, r0, r);
                // a contraction over a ragged vocabulary reads on to the next whole vector: zeros, where the loss kernel owns the padding
                if (wide && (vocab % 8 == 0 || vocab <= 131072)) {
                    mi_gemm_problem p = problem(out, false, true);
                    segment(p, logits, weight, vocab);
                    run_gemm(&p, 1, h, l);
                } else {
                    at::mm_out(out, logits, weight);
                }
            }
            if (need_dw) {
                Tensor product;
                if (wide && !thin(vocab, h.size(1), r)) {
                    product = at::empty({vocab, h.size(1)}, h.options());
                    mi_gemm_problem p = problem(product, true, true);
                    segment(p, logits, hc, r);
                    run_gemm(&p, 1, h, l);
                } else {
                    const bool turn = transpose_pays(r, h.size(1), vocab) && h.size(1) <= vocab && transposable(hc);
                    product = at::mm(logits.t(), turn ? transposed(hc, l).t() : hc);
                }
                if (n <= chunk) dw = product;
                else if (!dw.defined()) dw = product.to(at::kFloat);
                else dw.add_(product);
            }
        }
        if (need_dw && !dw.defined()) dw = at::zeros_like(weight);    // no rows
        check(mi_loss_reduce(losses, argmax.data_ptr<int32_t>(), targets.data_ptr<int64_t>(), weights.data_ptr<float>(), n, loss.data_ptr<float>(),
                             total.data_ptr<float>(), accuracy.data_ptr<float>(), l.stream),
              "mi_loss_reduce");
        ctx->set_materialize_grads(false);
        ctx->mark_non_differentiable({argmax, accuracy});
        ctx->save_for_backward({dh, dw});
        ctx->saved_data["hooked"] = at::SavedTensorDefaultHooks::get_hooks().has_value();
        ctx->saved_data["dtype"] = (int64_t)weight.scalar_type();
        return {loss, argmax, accuracy};
    }
    static variable_list backward(AutogradContext* ctx, variable_list g) {
        variable_list grads(7);
        if (!g[0].defined()) return grads;
        const variable_list saved = ctx->get_saved_variables();
        // A graph that is used up by this pass hands its gradients over, scaled in place; one that is kept (or differentiated
        // further) keeps them, and what a saved-tensor hook returns belongs to the hook.
        const bool hand_over = !torch::autograd::get_current_graph_task_keep_graph() && !at::GradMode::is_enabled() && !ctx->saved_data["hooked"].toBool();
        const Tensor dloss = g[0].contiguous();
        for (int i = 0; i < 2; ++i) {
            const Tensor& x = saved[i];
            if (!x.defined()) continue;
            if (hand_over && x.is_non_overlapping_and_dense()) {
                Launch l(x);
                check(mi_scale_inplace(ptr(x), x.numel(), dloss.data_ptr<float>(), code_of(x), l.stream), "mi_scale_inplace");
                grads[i] = x;
            } else {
                grads[i] = x * dloss;
            }
        }
        const auto dtype = (at::ScalarType)ctx->saved_data["dtype"].toInt();
        if (grads[1].defined()) grads[1] = grads[1].to(dtype);
        return grads;
    }
};

std::tuple<Tensor, Tensor, Tensor> op_linear_cross_entropy(const Tensor& h, const Tensor& weight, const Tensor& targets, const Tensor& weights, int64_t chunk) {
    need_gpu(h); need_gpu(weight); need_gpu(targets); need_gpu(weights);
    TORCH_CHECK(h.dim() == 2 && h.is_contiguous() && weight.dim() == 2 && h.size(1) == weight.size(1) && h.scalar_type() == weight.scalar_type() &&
                    targets.scalar_type() == at::kLong && targets.is_contiguous() && targets.numel() == h.size(0) &&
                    weights.scalar_type() == at::kFloat && weights.is_contiguous() && weights.numel() == h.size(0) && chunk >= 1,
                "linear cross entropy: h [rows, hidden], weight [vocab, hidden], one int64 target and one float32 weight per row");
    const bool on = at::GradMode::is_enabled();
    const auto out = LinearCrossEntropy::apply(h, weight, targets, weights, chunk, on && h.requires_grad(), on && weight.requires_grad());
    return {out[0], out[1], out[2]};
}

// ---- decode ------------------------------------------------------------------------------------------------------------
void op_decode_attention(const Tensor& q, const Tensor& k_cache, const Tensor& v_cache, const Tensor& ctx_len, const OptTensor& k_new,
                      const OptTensor& v_new, const OptTensor& cos, const OptTensor& sin, const OptTensor& pos, bool interleaved, double scale,
                      const OptTensor& workspace, const OptTensor& tickets, int n_splits, const Tensor& out, bool static_scratch) {
    need_gpu(q); need_gpu(k_cache); need_gpu(v_cache); need_gpu(ctx_len);
    Launch l(q);
    mi_decode_args a{};
    a.q = ptr(q); a.k_cache = ptr(k_cache); a.v_cache = ptr(v_cache); a.o = ptr(out); a.ctx_len = (const int32_t*)ptr(ctx_len);
    a.q_stride_batch = q.stride(0);
    if (k_new.has_value()) {
        a.k_new = ptr(*k_new); a.v_new = ptr(*v_new);
        a.k_new_stride_batch = k_new->stride(0); a.v_new_stride_batch = v_new->stride(0);
    }
    if (cos.has_value()) {
        a.rotary_cos = ptr(*cos); a.rotary_sin = ptr(*sin); a.position_ids = (const int64_t*)ptr(*pos);
        a.rotary_table_rows = cos->size(0);
        a.rotary_interleaved = interleaved;
    }
    a.batch = (int32_t)q.size(0); a.max_ctx = (int32_t)k_cache.size(1); a.n_q_heads = (int32_t)q.size(1); a.n_kv_heads = (int32_t)k_cache.size(2);
    a.head_dim = (int32_t)q.size(2);
    a.dtype = code_of(q);
    a.cache_stride_batch = k_cache.stride(0); a.cache_stride_token = k_cache.stride(1); a.cache_stride_head = k_cache.stride(2);
    a.softmax_scale = (float)scale;
    a.n_splits = n_splits;
    a.stream = l.stream;
    if (static_scratch) {
        check(mi_attn_decode_static(&a), "mi_attn_decode_static");
        return;
    }
    a.workspace = ptr(*workspace);
    a.workspace_bytes = (size_t)workspace->numel() * 4;
    // One launch less where the tickets that came with the workspace are enough.  A graph issues the second one for nothing, and on the device two are level or
    // ahead (us in a graph, one / two launches: 1500 keys, 32 / 8 heads of 128 7.4 / 6.7; 2 x 960, 16 / 16 of 64 6.1 / 5.3; 536, 32 / 8 of 128 6.2 / 6.4).
    const bool merge = tickets.has_value() && tickets->scalar_type() == at::kInt && tickets->is_contiguous() && tickets->device() == out.device() &&
                       tickets->numel() >= (int64_t)a.batch * a.n_q_heads &&
                       c10::hip::currentStreamCaptureStatusMayInitCtx() == c10::hip::CaptureStatus::None;
    if (merge) check(mi_attn_decode_with_tickets(&a, static_cast<int32_t*>(ptr(*tickets)), tickets->numel()), "mi_attn_decode_with_tickets");
    else check(mi_attn_decode(&a), "mi_attn_decode");
}

// ---- a decode step's layer ---------------------------------------------------------------------------------------------
bool rows_weight(const Tensor& w, const Tensor& x, int64_t k) {
    return !transformed(w) && w.dim() == 2 && w.size(0) > 0 && w.size(1) == k && w.scalar_type() == x.scalar_type() && w.device() == x.device() &&
           aligned(w);
}
bool rows_norm(const Tensor& w, const Tensor& x, int64_t k) {
    return !transformed(w) && w.dim() == 1 && w.size(0) == k && w.stride(0) == 1 && w.scalar_type() == x.scalar_type() && w.device() == x.device() &&
           (reinterpret_cast<uintptr_t>(w.data_ptr()) & 15) == 0;
}
bool rows_input(const Tensor& x) {                         // [rows, k]; a transform sees the modules' operations instead
    return !transforming() && !transformed(x) && x.is_cuda() && x.dim() == 2 &&
           (x.scalar_type() == at::kBFloat16 || x.scalar_type() == at::kHalf) && x.size(0) >= 1 && x.size(0) <= MI_ROWS_MAX && x.size(1) > 0 && x.size(1) % 32 == 0 && aligned(x);
}

mi_rows_args rows_args(const Tensor& x, const Tensor& norm, double eps, const Launch& l) {
    mi_rows_args a{};
    a.x = ptr(x); a.norm_weight = ptr(norm); a.ldx = x.stride(0); a.rows = (int32_t)x.size(0); a.k = (int32_t)x.size(1);
    a.eps = (float)eps; a.dtype = code_of(x); a.stream = l.stream;
    return a;
}
void rows_weight(mi_rows_args& a, const Tensor& w, void* out, int64_t ldo) {
    const int i = a.n_weights++;
    a.w[i] = ptr(w); a.ldw[i] = w.stride(0); a.n[i] = (int32_t)w.size(0); a.out[i] = out; a.ldo[i] = ldo;
}

// The norm in front of a product of few rows: inside the product while its workgroups repeat it cheaply, else a launch of its own, after
// which they load the normalised rows.  Inside each of the features / 16 workgroups walks k values of every row, so the line lies at the product of
// the two; from 4096 on the walk outlasts the launch with any number of workgroups.  us, inside / as two launches, 1 row and 16, weights
// from memory, k -> features (x 2: SwiGLU):
//   1024 -> 4096         6.4 / 7.4     7.4 / 9.2          2048 -> 4096       8.6 / 8.8    9.5 / 10.3       4096 -> 1536     11.1 / 10.5   15.1 / 13.4
//   1024 -> 8192        11.1 / 10.6   13.0 / 13.7         2048 -> 6144      13.6 / 12.0  16.4 / 14.5       4096 -> 6144     22.3 / 18.5   29.2 / 23.0
//   1024 -> 12288       15.8 / 14.0   18.5 / 17.8         2048 -> 8192      15.2 / 13.6  17.1 / 15.7       4096 -> 28672    74.8 / 48.6   96.8 / 67.5
//   1024 -> 8192 x 2    11.2 / 12.2   13.1 / 13.7         2048 -> 4096 x 2  12.9 / 13.5  14.2 / 15.0       4096 -> 3072 x 2 17.9 / 17.3   21.9 / 21.3
//   1024 -> 14336 x 2   19.2 / 17.2   22.8 / 20.8         2048 -> 6144 x 2  19.7 / 18.3  23.0 / 21.2       4096 -> 8192 x 2 37.2 / 33.4   46.0 / 41.8
struct RowsNorm {
    Tensor x, weight;
    RowsNorm(const Tensor& x_, const Tensor& weight_, double eps, int64_t features, const Launch& l) : x(x_), weight(weight_) {
        if (x_.size(1) <= 2048 && (features + 15) / 16 * x_.size(1) <= 512 * 1024) return;
        x = x_.is_contiguous() ? at::empty_like(x_) : at::empty(x_.sizes(), x_.options());
        const Tensor in = x_.contiguous();
        check(mi_rmsnorm_fwd(ptr(in), ptr(weight), ptr(x), nullptr, in.size(0), in.size(1), (float)eps, code_of(in), l.stream), "mi_rmsnorm_fwd");
        weight = Tensor();
    }
};

// rms_norm(x) W^T of a few rows [rows, k]; nothing where mi_rows_product does not apply.
OptTensor op_norm_linear_rows(const Tensor& x, const Tensor& norm, double eps, const Tensor& w) {
    if (!rows_input(x) || !rows_norm(norm, x, x.size(1)) || !rows_weight(w, x, x.size(1))) return std::nullopt;
    need_gpu(x);
    Launch l(x);
    const Tensor out = at::empty({x.size(0), w.size(0)}, x.options());
    const RowsNorm in(x, norm, eps, w.size(0), l);
    mi_rows_args a = rows_args(in.x, in.weight, eps, l);
    rows_weight(a, w, ptr(out), out.stride(0));
    check(mi_rows_product(&a), "mi_rows_product");
    return out;
}

// Index of the maximum of each row of x [rows, n]; nothing where mi_argmax does not apply or a transform has to see the operation.
bool argmax_applies(const Tensor& x) {
    return !(transforming() || transformed(x) || !x.is_cuda() || x.dim() != 2 || x.size(0) < 1 || x.size(1) < 1 || x.size(1) > (1 << 30) ||
             (x.size(1) > 1 && x.stride(1) != 1) || (x.scalar_type() != at::kBFloat16 && x.scalar_type() != at::kHalf && x.scalar_type() != at::kFloat));
}
OptTensor op_argmax_rows(const Tensor& x) {
    if (!argmax_applies(x)) return std::nullopt;
    need_gpu(x);
    Launch l(x);
    const Tensor out = at::empty({x.size(0)}, x.options().dtype(at::kLong));
    check(mi_argmax(ptr(x), x.size(0), x.size(1), x.stride(0), out.data_ptr<int64_t>(), code_of(x), l.stream), "mi_argmax");
    return out;
}

// The same and those rows of a table [at least n, hidden] (inference); nothing where mi_argmax_embed does not apply.
std::optional<std::tuple<Tensor, Tensor>> op_argmax_embed(const Tensor& x, const Tensor& table) {
    if (!argmax_applies(x) || transformed(table) || table.scalar_type() != x.scalar_type() || table.device() != x.device() || !aligned(table) ||
        table.size(0) < x.size(1) || table.size(1) < 1 || table.size(1) % (x.scalar_type() == at::kFloat ? 4 : 8) != 0 ||
        (at::GradMode::is_enabled() && table.requires_grad()))
        return std::nullopt;
    need_gpu(x);
    Launch l(x);
    const Tensor index = at::empty({x.size(0)}, x.options().dtype(at::kLong)), out = at::empty({x.size(0), table.size(1)}, table.options());
    check(mi_argmax_embed(ptr(x), x.size(0), x.size(1), x.stride(0), index.data_ptr<int64_t>(), ptr(table), table.size(0), table.stride(0), table.size(1),
                          ptr(out), code_of(x), l.stream),
          "mi_argmax_embed");
    return std::make_tuple(index, out);
}

// One token per sequence through a pre-norm layer (RMSNorm, separate q / k / v, SwiGLU, no biases): five launches, plus the merge of
// the decode attention and the norms in front of wide products.  x [batch, 1, hidden]; raises ctx_len by one and appends to the caches.  Nothing happens, and nothing
// is returned, where a shape, type or alignment does not suit the kernels.
OptTensor op_decode_layer(const Tensor& x, const Tensor& pos, const Tensor& norm1, double eps1, const std::vector<Tensor>& qkv_w, const Tensor& dense,
                          const Tensor& norm2, double eps2, const Tensor& w_in, const Tensor& w_gate, const Tensor& w_out, int64_t head_dim,
                          const Tensor& k_cache, const Tensor& v_cache, const Tensor& ctx_len, const Tensor& cos, const Tensor& sin, bool interleaved,
                          double scale, const Tensor& workspace) {
    if (x.dim() != 3 || x.size(1) != 1 || !x.is_contiguous()) return std::nullopt;
    const Tensor x2 = x.view({x.size(0), x.size(2)});
    const int64_t b = x2.size(0), hidden = x2.size(1);
    if (!rows_input(x2) || !rows_norm(norm1, x, hidden) || !rows_norm(norm2, x, hidden) || qkv_w.size() != 3) return std::nullopt;
    for (const Tensor& w : qkv_w)
        if (!rows_weight(w, x, hidden) || w.size(0) % head_dim != 0) return std::nullopt;
    const int64_t q_rows = qkv_w[0].size(0), kv_rows = qkv_w[1].size(0), inter = w_in.size(0);
    if (qkv_w[2].size(0) != kv_rows || q_rows % 32 != 0 || inter % 32 != 0 || !rows_weight(dense, x, q_rows) || dense.size(0) != hidden ||
        !rows_weight(w_in, x, hidden) || !rows_weight(w_gate, x, hidden) || w_gate.size(0) != inter || !rows_weight(w_out, x, inter) ||
        w_out.size(0) != hidden || pos.scalar_type() != at::kLong || pos.numel() != b || !pos.is_contiguous() || pos.device() != x.device() ||
        k_cache.scalar_type() != x.scalar_type() || k_cache.size(0) != b || k_cache.size(2) * head_dim != kv_rows || k_cache.size(3) != head_dim)
        return std::nullopt;
    need_gpu(x);
    Launch l(x);
    const int64_t width = q_rows + 2 * kv_rows, e = x.element_size();
    const Tensor qkv = at::empty({b, width}, x.options()), ctx = at::empty({b, q_rows}, x.options()), h = at::empty({b, hidden}, x.options()),
                 act = at::empty({b, inter}, x.options()), y = at::empty(x.sizes(), x.options());
    char* base = static_cast<char*>(ptr(qkv));
    const RowsNorm in1(x2, norm1, eps1, width, l);
    mi_rows_args a = rows_args(in1.x, in1.weight, eps1, l);
    a.count_up = static_cast<int32_t*>(ptr(ctx_len));
    rows_weight(a, qkv_w[0], base, width);
    rows_weight(a, qkv_w[1], base + q_rows * e, width);
    rows_weight(a, qkv_w[2], base + (q_rows + kv_rows) * e, width);
    check(mi_rows_product(&a), "mi_rows_product");

    mi_decode_args d{};
    d.q = base; d.k_new = base + q_rows * e; d.v_new = base + (q_rows + kv_rows) * e;
    d.q_stride_batch = d.k_new_stride_batch = d.v_new_stride_batch = width;
    d.k_cache = ptr(k_cache); d.v_cache = ptr(v_cache); d.o = ptr(ctx); d.ctx_len = static_cast<const int32_t*>(ptr(ctx_len));
    d.rotary_cos = ptr(cos); d.rotary_sin = ptr(sin); d.position_ids = static_cast<const int64_t*>(ptr(pos));
    d.rotary_table_rows = cos.size(0); d.rotary_interleaved = interleaved;
    d.batch = (int32_t)b; d.max_ctx = (int32_t)k_cache.size(1); d.n_q_heads = (int32_t)(q_rows / head_dim); d.n_kv_heads = (int32_t)(kv_rows / head_dim);
    d.head_dim = (int32_t)head_dim; d.dtype = code_of(x);
    d.cache_stride_batch = k_cache.stride(0); d.cache_stride_token = k_cache.stride(1); d.cache_stride_head = k_cache.stride(2);
    d.softmax_scale = (float)scale; d.workspace = ptr(workspace); d.workspace_bytes = (size_t)workspace.numel() * 4; d.stream = l.stream;
    check(mi_attn_decode(&d), "mi_attn_decode");

    a = rows_args(ctx, Tensor(), 0.0, l);
    rows_weight(a, dense, ptr(h), hidden);
    a.add[0] = ptr(x2); a.ldadd[0] = hidden;
    check(mi_rows_product(&a), "mi_rows_product");
    const RowsNorm in2(h, norm2, eps2, inter, l);
    a = rows_args(in2.x, in2.weight, eps2, l);
    a.glu = 1;
    rows_weight(a, w_in, ptr(act), inter);
    rows_weight(a, w_gate, nullptr, 0);
    check(mi_rows_product(&a), "mi_rows_product");
    a = rows_args(act, Tensor(), 0.0, l);
    rows_weight(a, w_out, ptr(y), hidden);
    a.add[0] = ptr(h); a.ldadd[0] = hidden;
    check(mi_rows_product(&a), "mi_rows_product");
    return y;
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    // none of these touches Python objects: other interpreter threads run meanwhile
    const auto def = [&](const char* name, auto f) { m.def(name, f, py::call_guard<py::gil_scoped_release>()); };
    def("rms_norm_forward", &op_rms_norm_forward);
    def("rms_norm_backward", &op_rms_norm_backward);
    def("rms_norm", [](const Tensor& x, const Tensor& w, double eps) { return RmsNorm::apply(x, w, eps); });
    def("layer_norm_forward", &op_layer_norm_forward);
    def("layer_norm_backward", &op_layer_norm_backward);
    def("layer_norm", [](const Tensor& x, const Tensor& w, const OptTensor& b, double eps) { return LayerNorm::apply(x, w, b, eps); });
    def("gelu_forward", &op_gelu_forward);
    def("gelu_backward", &op_gelu_backward);
    def("gelu", [](const Tensor& x) { return Gelu::apply(x); });
    def("swiglu_forward", &op_swiglu_forward);
    def("swiglu_backward", &op_swiglu_backward);
    def("swiglu", [](const Tensor& a, const Tensor& g) { return SwiGlu::apply(a, g); });
    def("rotary_launch", &rotary_launch);
    def("rotary", [](const Tensor& x, const Tensor& cos, const Tensor& sin, const OptTensor& ids, int64_t seq_len, bool interleaved) {
        return Rotary::apply(x, cos, sin, ids, seq_len, interleaved);
    });
    def("linear", &op_linear);
    def("projections", &op_projections);
    def("attention_forward", &op_attention_forward);
    def("attention_backward", &op_attention_backward);
    def("attention", &op_attention);
    def("attention_qkv", &op_attention_qkv);
    def("add_norm", &op_add_norm);
    def("layer", &op_layer);
    def("prefill_attention", &op_prefill_attention);
    def("weighted_cross_entropy", &op_weighted_cross_entropy);
    def("linear_cross_entropy", &op_linear_cross_entropy);
    def("decode_attention", &op_decode_attention);
    def("norm_linear_rows", &op_norm_linear_rows);
    def("argmax_rows", &op_argmax_rows);
    def("argmax_embed", &op_argmax_embed);
    def("decode_layer", &op_decode_layer);
}
