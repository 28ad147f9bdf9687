// PyTorch-ROCm C++ extension `ldist_layers`: the layers' host path in native code, over the C ABI of libldist_hip.so.
// What norm_dist.py, mlp.py, harness.py and adamw.py do in Python for tensors they keep the Python route for (CPU
// tensors, other types, hooked sub-modules), done here for float32 GPU tensors: the same entry points in the same order
// with the same results, except that a forward pass at finite p that no gradient follows takes
// ldist_norm_dist_forward_values here and ldist_norm_dist_forward there: the last bits may differ.  A layer's forward is
// one call and one autograd node, and its backward runs without the interpreter; a Python autograd function costs 15 to
// 30 us per call and direction, more than the kernels of a layer of a thousand neurons take.
#include <torch/extension.h>

#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>

#include <climits>
#include <cmath>
#include <string>
#include <tuple>
#include <vector>

#include "inf_forward.hpp"
#include "ldist.h"

namespace {

using torch::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::tensor_list;
using OptTensor = std::optional<Tensor>;

void done(const char* op, int rc) {
    TORCH_CHECK(rc == LDIST_OK, op, " failed: ", ldist_strerror(rc),
                rc == LDIST_ELAUNCH ? " (hipError_t " + std::to_string(ldist_last_hip_error()) + ")" : std::string());
}

void check(const Tensor& t, const char* name, const torch::Device& dev) {
    TORCH_CHECK(t.is_cuda(), name, " must be a CUDA tensor");
    TORCH_CHECK(t.is_contiguous(), name, " must be contiguous");
    TORCH_CHECK(t.scalar_type() == torch::kFloat32, name, " must have dtype torch.float32, got ", t.scalar_type());
    TORCH_CHECK(t.device() == dev, "all tensors must be on the same device");
}

// A saved tensor is what an unpack hook made of it (torch.autograd.graph.saved_tensors_hooks): the kernels read it as it was
// saved, so it has to be that still.  `like`: a tensor of the backward pass that autograd has checked.
void check_saved(const Tensor& t, const char* name, at::ScalarType type, at::IntArrayRef shape, const Tensor& like) {
    TORCH_CHECK(t.is_cuda() && t.device() == like.device(), "saved ", name, " must be a CUDA tensor on the gradient's device");
    TORCH_CHECK(t.is_contiguous(), "saved ", name, " must be contiguous");
    TORCH_CHECK(t.scalar_type() == type && t.sizes() == shape, "saved ", name, " must have the type and shape that it was saved with");
}

// Pins the device of `t` for a scope and knows its current stream.
struct On {
    explicit On(const Tensor& t) : guard(t.device()) {}
    at::hip::OptionalHIPGuardMasqueradingAsCUDA guard;
    ldist_stream_t stream = (ldist_stream_t)at::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream();
};

const float* in(const Tensor& t) { return t.const_data_ptr<float>(); }
const float* in(const OptTensor& t) { return t.has_value() && t->defined() ? t->const_data_ptr<float>() : nullptr; }
float* out(const Tensor& t) { return t.mutable_data_ptr<float>(); }
bool wants_grad(const Tensor& t) { return t.requires_grad(); }
bool wants_grad(const OptTensor& t) { return t.has_value() && t->defined() && t->requires_grad(); }

// ---- the window of a convolution-shaped layer ---------------------------------------------------------------------
struct Window {
    int64_t k, stride, pad, dil;
    bool trivial() const { return k == 1 && stride == 1 && pad == 0; }
    std::pair<int64_t, int64_t> positions(const Tensor& img) const {
        const int64_t span = dil * (k - 1) + 1;
        return {(img.size(2) + 2 * pad - span) / stride + 1, (img.size(3) + 2 * pad - span) / stride + 1};
    }
};
#define WINDOW_ARGS(w) (int)(w).k, (int)(w).k, (int)(w).stride, (int)(w).pad, (int)(w).dil
#define IMAGE_ARGS(img) (int)(img).size(0), (int)(img).size(1), (int)(img).size(2), (int)(img).size(3)
#define GEOMETRY_ARGS(img, co, g, w) (int)(img).size(1), (int)(img).size(2), (int)(img).size(3), (int)(co), (int)(g), WINDOW_ARGS(w)

// ---- what follows the distances: the mean shift of MeanNorm and the bias ---------------------------------------
// `running` undefined: no shift.  Training: y = raw - batch mean, running moves; evaluation: y = raw - running.
struct Shift {
    Tensor running;
    double momentum = 0;
    bool training = false;
    bool batch_mean() const { return training && running.defined(); }
    const float* running_mean() const { return running.defined() ? running.const_data_ptr<float>() : nullptr; }
    // nothing but per-channel constants follow the distances: the forward kernels can apply them on their way out
    bool constant(const OptTensor& bias) const { return !batch_mean() && (running.defined() || (bias.has_value() && bias->defined())); }
};

Tensor mean_shifted(const On& on, const Tensor& x, const Tensor& running, double momentum) {
    Tensor y = torch::empty_like(x);
    done("mean_shift", ldist_mean_shift(in(x), x.size(0), x.size(1), x.numel() / (x.size(0) * x.size(1)), out(y), nullptr,
                                        running.defined() ? out(running) : nullptr, (float)momentum, on.stream));
    return y;
}

void channel_shift(const On& on, const Tensor& x, const float* mean, const float* bias, const Tensor& y) {
    done("channel_shift", ldist_channel_shift(in(x), x.size(0), x.size(1), x.numel() / (x.size(0) * x.size(1)), mean, bias,
                                              out(y), on.stream));
}

// raw (B, CO, L) -> the layer's output; `keep_raw`: the backward needs raw itself, so it is not overwritten.
Tensor shifted(const On& on, const Tensor& raw, const OptTensor& bias, const Shift& s, bool keep_raw) {
    const float* b = in(bias);
    if (s.batch_mean()) {
        Tensor y = mean_shifted(on, raw, s.running, s.momentum);
        if (b) channel_shift(on, y, nullptr, b, y);
        return y;
    }
    if (!b && !s.running.defined()) return raw;
    Tensor y = keep_raw ? torch::empty_like(raw) : raw;
    channel_shift(on, raw, s.running.defined() ? in(s.running) : nullptr, b, y);
    return y;
}

// ---- distances of columns ------------------------------------------------------------------------------------------
// Columns are (B, CI, L), or (B, CI) for a fully connected layer; the results have the same number of dimensions.
struct Sizes {
    int B, CO, CI, HW;
    bool flat;
    std::vector<int64_t> output() const { return flat ? std::vector<int64_t>{B, CO} : std::vector<int64_t>{B, CO, HW}; }
    std::vector<int64_t> input() const { return flat ? std::vector<int64_t>{B, CI} : std::vector<int64_t>{B, CI, HW}; }
};
Sizes sizes_of(const Tensor& x, const Tensor& w, int64_t G) {
    TORCH_CHECK(x.dim() == 2 || x.dim() == 3, "input must be 3-D, or 2-D for a fully connected layer");
    TORCH_CHECK(x.numel() > 0 && w.numel() > 0, "tensors must not be empty");
    TORCH_CHECK(G > 0 && w.numel() / w.size(0) * G == x.size(1), "weight must be (CO, CI/G)");
    return {(int)x.size(0), (int)w.size(0), (int)x.size(1), x.dim() == 3 ? (int)x.size(2) : 1, x.dim() == 2};
}
Tensor sum_per_channel(const Tensor& g) { return g.dim() == 2 ? g.sum(0) : g.sum(at::IntArrayRef{0, 2}); }

// No gradient follows: the argmax that the forward with gradients records has no reader, and p-norm sums may be taken in
// any order.
// The layer's shift and bias included.
Tensor distances(const On& on, const Tensor& x, const Tensor& w, int64_t G, double p, const OptTensor& bias, const Shift& shift) {
    const Sizes s = sizes_of(x, w, G);
    Tensor y = torch::empty(s.output(), x.options());
    if (s.HW == 1 && shift.constant(bias)) {
        const float *mean = shift.running_mean(), *b = in(bias);
        int rc;
        if (std::isinf(p)) {
            rc = ldist_torch::inf_forward_shifted(in(x), in(w), s.B, s.CO, s.CI, (int)G, mean, b, out(y), nullptr, y, on.stream);
            if (rc == LDIST_EUNSUPPORTED) {
                Tensor pos = torch::empty(s.output(), x.options().dtype(torch::kInt32));
                rc = ldist_torch::inf_forward_shifted(in(x), in(w), s.B, s.CO, s.CI, (int)G, mean, b, out(y),
                                                      pos.data_ptr<int32_t>(), y, on.stream);
            }
        } else {
            rc = ldist_norm_dist_forward_values_shifted(in(x), in(w), s.B, s.CO, s.CI, (int)G, mean, b, out(y), (float)p, on.stream);
        }
        if (rc != LDIST_EUNSUPPORTED) {
            done("dist_forward_shifted", rc);
            return y;
        }
    }
    if (std::isinf(p)) {
        const int rc = ldist_torch::inf_forward(in(x), in(w), s.B, s.CO, s.CI, (int)G, s.HW, out(y), nullptr, y, on.stream);
        if (rc != LDIST_EUNSUPPORTED) {
            done("inf_dist_forward_values", rc);
        } else {
            Tensor pos = torch::empty(s.output(), x.options().dtype(torch::kInt32));
            done("inf_dist_forward", ldist_torch::inf_forward(in(x), in(w), s.B, s.CO, s.CI, (int)G, s.HW, out(y),
                                                              pos.data_ptr<int32_t>(), y, on.stream));
        }
    } else {
        done("norm_dist_forward_values", ldist_norm_dist_forward_values(in(x), in(w), s.B, s.CO, s.CI, (int)G, s.HW, out(y),
                                                                        (float)p, on.stream));
    }
    return shifted(on, y, bias, shift, false);
}

// Distances of columns (B, CI, L) with gradients, then the shift: one node.
struct ColumnLayer : public Function<ColumnLayer> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w, const OptTensor& bias, int64_t G, double p,
                          Shift shift) {
        const On on(x);
        const Sizes s = sizes_of(x, w, G);
        const bool inf = std::isinf(p);
        const bool fused = inf && s.HW == 1 && shift.constant(bias);
        Tensor raw = torch::empty(s.output(), x.options());
        if (inf) {
            Tensor pos = torch::empty(s.output(), x.options().dtype(torch::kInt32));
            int32_t* const at = pos.data_ptr<int32_t>();
            done("inf_dist_forward",
                 fused ? ldist_torch::inf_forward_shifted(in(x), in(w), s.B, s.CO, s.CI, (int)G, shift.running_mean(), in(bias),
                                                          out(raw), at, raw, on.stream)
                       : ldist_torch::inf_forward(in(x), in(w), s.B, s.CO, s.CI, (int)G, s.HW, out(raw), at, raw, on.stream));
            ctx->save_for_backward({pos});
        } else {
            done("norm_dist_forward", ldist_norm_dist_forward(in(x), in(w), s.B, s.CO, s.CI, (int)G, s.HW, out(raw), (float)p,
                                                              on.stream));
        }
        Tensor y = fused ? raw : shifted(on, raw, bias, shift, !inf);
        if (!inf) ctx->save_for_backward({x, w, raw});
        ctx->saved_data["w"] = w.sizes().vec();
        ctx->saved_data["sizes"] = std::vector<int64_t>{s.B, s.CO, s.CI, s.HW, s.flat};
        ctx->saved_data["G"] = G;
        ctx->saved_data["p"] = p;
        ctx->saved_data["bias"] = bias.has_value() && bias->defined();
        ctx->saved_data["mean"] = shift.batch_mean();
        return y;
    }
    static tensor_list backward(AutogradContext* ctx, tensor_list grads) {
        const auto saved = ctx->get_saved_variables();   // the argmax at p = infinity, else input, weight, output
        const auto v = ctx->saved_data["sizes"].toIntVector();
        const Sizes s{(int)v[0], (int)v[1], (int)v[2], (int)v[3], v[4] != 0};
        const int64_t G = ctx->saved_data["G"].toInt();
        const double p = ctx->saved_data["p"].toDouble();
        const bool want_x = ctx->needs_input_grad(0), want_w = ctx->needs_input_grad(1);
        const bool want_b = ctx->saved_data["bias"].toBool() && ctx->needs_input_grad(2);
        const auto w_shape = ctx->saved_data["w"].toIntVector();
        Tensor gx, gw, gb;
        Tensor g = grads[0].contiguous();
        const On on(g);
        if (std::isinf(p)) {
            check_saved(saved[0], "argmax", torch::kInt32, s.output(), g);
        } else {
            check_saved(saved[0], "input", torch::kFloat32, s.input(), g);
            check_saved(saved[1], "weight", torch::kFloat32, w_shape, g);
            check_saved(saved[2], "output", torch::kFloat32, s.output(), g);
        }
        if (want_b) gb = sum_per_channel(g);
        if (ctx->saved_data["mean"].toBool()) g = mean_shifted(on, g, Tensor(), 0.0);
        if (want_x) gx = torch::empty(s.input(), g.options());
        if (std::isinf(p)) {
            // the scatter kernels write every element, zeros included: no fill needed here
            const int32_t* pos = saved[0].const_data_ptr<int32_t>();
            if (want_w) gw = torch::empty(w_shape, g.options());
            if (want_x && want_w)
                done("inf_dist_backward", ldist_inf_dist_backward_overwrite(in(g), pos, s.B, s.CO, s.CI, (int)G, s.HW, out(gx),
                                                                            out(gw), on.stream));
            else if (want_x)
                done("inf_dist_backward_input", ldist_inf_dist_backward_input_overwrite(in(g), pos, s.B, s.CO, s.CI, (int)G,
                                                                                        s.HW, out(gx), on.stream));
            else if (want_w)
                done("inf_dist_backward_weight", ldist_inf_dist_backward_weight_overwrite(in(g), pos, s.B, s.CO, s.CI, (int)G,
                                                                                          s.HW, out(gw), on.stream));
        } else {
            const Tensor &x = saved[0], &w = saved[1], &aux = saved[2];
            if (want_w) gw = torch::zeros_like(w);   // the kernels add onto this buffer
            if (at::globalContext().deterministicAlgorithms()) {
                if (want_x || want_w)
                    done("norm_dist_backward_ordered",
                         ldist_norm_dist_backward_ordered(in(g), in(x), in(w), in(aux), s.B, s.CO, s.CI, (int)G, s.HW,
                                                          want_x ? out(gx) : nullptr, want_w ? out(gw) : nullptr, (float)p,
                                                          on.stream));
            } else if (want_x && want_w)
                done("norm_dist_backward", ldist_norm_dist_backward(in(g), in(x), in(w), in(aux), s.B, s.CO, s.CI, (int)G, s.HW,
                                                                    out(gx), out(gw), (float)p, on.stream));
            else if (want_x)
                done("norm_dist_backward_input", ldist_norm_dist_backward_input(in(g), in(x), in(w), in(aux), s.B, s.CO, s.CI,
                                                                                (int)G, s.HW, out(gx), (float)p, on.stream));
            else if (want_w)
                done("norm_dist_backward_weight", ldist_norm_dist_backward_weight(in(g), in(x), in(w), in(aux), s.B, s.CO, s.CI,
                                                                                  (int)G, s.HW, out(gw), (float)p, on.stream));
        }
        return {gx, gw, gb, Tensor(), Tensor(), Tensor()};
    }
};

// ---- patches -----------------------------------------------------------------------------------------------------
Tensor unfolded(const On& on, const Tensor& img, const Window& w) {
    const auto [ho, wo] = w.positions(img);
    Tensor cols = torch::empty({img.size(0), img.size(1) * w.k * w.k, ho * wo}, img.options());
    done("unfold", ldist_unfold(in(img), IMAGE_ARGS(img), WINDOW_ARGS(w), out(cols), on.stream));
    return cols;
}

struct Unfold : public Function<Unfold> {
    static Tensor forward(AutogradContext* ctx, const Tensor& img, Window w) {
        const On on(img);
        ctx->saved_data["shape"] = img.sizes().vec();
        ctx->saved_data["window"] = std::vector<int64_t>{w.k, w.stride, w.pad, w.dil};
        return unfolded(on, img, w);
    }
    static tensor_list backward(AutogradContext* ctx, tensor_list grads) {
        const auto shape = ctx->saved_data["shape"].toIntVector(), v = ctx->saved_data["window"].toIntVector();
        const Window w{v[0], v[1], v[2], v[3]};
        const Tensor g = grads[0].contiguous();
        const On on(g);
        Tensor img = torch::empty(shape, g.options());
        done("fold", ldist_fold(in(g), IMAGE_ARGS(img), WINDOW_ARGS(w), out(img), on.stream));
        return {img, Tensor()};
    }
};

// ---- layers straight from the image -------------------------------------------------------------------------------
// p = infinity.  Forward: the kernel that reads the image where it covers the geometry, else unfold + distances;
// backward: the image gradient directly (scatter and fold fused).
// The layer's shift and bias included.
Tensor inf_image_forward(const On& on, const Tensor& img, const Tensor& w, int64_t G, const Window& win, bool from_image,
                         Tensor* pos, const OptTensor& bias, const Shift& shift) {
    const auto [ho, wo] = win.positions(img);
    const int CO = (int)w.size(0);
    Tensor y = torch::empty({img.size(0), CO, ho * wo}, img.options());
    if (from_image && shift.constant(bias)) {
        if (pos) *pos = torch::empty({img.size(0), CO, ho * wo}, img.options().dtype(torch::kInt32));
        done("inf_dist_conv_forward", ldist_inf_dist_conv_forward_shifted(in(img), in(w), IMAGE_ARGS(img), CO, (int)G,
                                                                          WINDOW_ARGS(win), shift.running_mean(), in(bias), out(y),
                                                                          pos ? pos->data_ptr<int32_t>() : nullptr, on.stream));
        return y;
    }
    if (pos || !from_image) {
        Tensor own = torch::empty({img.size(0), CO, ho * wo}, img.options().dtype(torch::kInt32));
        if (from_image) {
            done("inf_dist_conv_forward", ldist_inf_dist_conv_forward(in(img), in(w), IMAGE_ARGS(img), CO, (int)G,
                                                                      WINDOW_ARGS(win), out(y), own.data_ptr<int32_t>(),
                                                                      on.stream));
        } else {
            const Tensor cols = unfolded(on, img, win);
            done("inf_dist_forward", ldist_inf_dist_forward(in(cols), in(w), (int)img.size(0), CO, (int)cols.size(1), (int)G,
                                                            (int)(ho * wo), out(y), own.data_ptr<int32_t>(), on.stream));
        }
        if (pos) *pos = own;
    } else {
        done("inf_dist_conv_forward_values", ldist_inf_dist_conv_forward_values(in(img), in(w), IMAGE_ARGS(img), CO, (int)G,
                                                                                WINDOW_ARGS(win), out(y), on.stream));
    }
    return shifted(on, y, bias, shift, false);
}

struct InfImageLayer : public Function<InfImageLayer> {
    static Tensor forward(AutogradContext* ctx, const Tensor& img, const Tensor& w, const OptTensor& bias, int64_t G, Window win,
                          bool from_image, Shift shift) {
        const On on(img);
        Tensor pos;
        Tensor y = inf_image_forward(on, img, w, G, win, from_image, &pos, bias, shift);
        ctx->save_for_backward({pos});
        ctx->saved_data["G"] = G;
        ctx->saved_data["img"] = img.sizes().vec();
        ctx->saved_data["w"] = w.sizes().vec();
        ctx->saved_data["window"] = std::vector<int64_t>{win.k, win.stride, win.pad, win.dil};
        ctx->saved_data["bias"] = bias.has_value() && bias->defined();
        ctx->saved_data["mean"] = shift.batch_mean();
        return y;
    }
    static tensor_list backward(AutogradContext* ctx, tensor_list grads) {
        const Tensor pos = ctx->get_saved_variables()[0];
        const auto v = ctx->saved_data["window"].toIntVector();
        const Window win{v[0], v[1], v[2], v[3]};
        const int G = (int)ctx->saved_data["G"].toInt();
        const bool want_b = ctx->saved_data["bias"].toBool() && ctx->needs_input_grad(2);
        Tensor g = grads[0].contiguous();
        const On on(g);
        check_saved(pos, "argmax", torch::kInt32, g.sizes(), g);
        Tensor gi, gw, gb;
        if (want_b) gb = sum_per_channel(g);
        if (ctx->saved_data["mean"].toBool()) g = mean_shifted(on, g, Tensor(), 0.0);
        const int B = (int)g.size(0), CO = (int)g.size(1), L = (int)g.size(2);
        const auto img_shape = ctx->saved_data["img"].toIntVector();
        if (ctx->needs_input_grad(0)) {
            gi = torch::empty(img_shape, g.options());
            done("inf_dist_backward_input_folded",
                 ldist_inf_dist_backward_input_folded(in(g), pos.const_data_ptr<int32_t>(), B, CO, (int)img_shape[1], G,
                                                      (int)img_shape[2], (int)img_shape[3], WINDOW_ARGS(win), out(gi), on.stream));
        }
        if (ctx->needs_input_grad(1)) {
            gw = torch::empty(ctx->saved_data["w"].toIntVector(), g.options());
            done("inf_dist_backward_weight",
                 ldist_inf_dist_backward_weight_overwrite(in(g), pos.const_data_ptr<int32_t>(), B, CO,
                                                          (int)(gw.numel() / CO * G), G, L, out(gw), on.stream));
        }
        return {gi, gw, gb, Tensor(), Tensor(), Tensor(), Tensor()};
    }
};

// Finite p, forward and both gradients from the image.
Tensor norm_image_forward(const On& on, const Tensor& img, const Tensor& w, int64_t G, double p, const Window& win) {
    const auto [ho, wo] = win.positions(img);
    Tensor y = torch::empty({img.size(0), w.size(0), ho * wo}, img.options());
    done("norm_dist_conv_forward", ldist_norm_dist_conv_forward(in(img), in(w), IMAGE_ARGS(img), (int)w.size(0), (int)G,
                                                                WINDOW_ARGS(win), out(y), (float)p, on.stream));
    return y;
}

struct NormImageLayer : public Function<NormImageLayer> {
    static Tensor forward(AutogradContext* ctx, const Tensor& img, const Tensor& w, const OptTensor& bias, int64_t G, double p,
                          Window win, Shift shift) {
        const On on(img);
        Tensor raw = norm_image_forward(on, img, w, G, p, win);
        Tensor y = shifted(on, raw, bias, shift, true);
        ctx->save_for_backward({img, w, raw});
        ctx->saved_data["img"] = img.sizes().vec();
        ctx->saved_data["w"] = w.sizes().vec();
        ctx->saved_data["G"] = G;
        ctx->saved_data["p"] = p;
        ctx->saved_data["window"] = std::vector<int64_t>{win.k, win.stride, win.pad, win.dil};
        ctx->saved_data["bias"] = bias.has_value() && bias->defined();
        ctx->saved_data["mean"] = shift.batch_mean();
        return y;
    }
    static tensor_list backward(AutogradContext* ctx, tensor_list grads) {
        const auto saved = ctx->get_saved_variables();
        const Tensor &img = saved[0], &w = saved[1], &raw = saved[2];
        const auto v = ctx->saved_data["window"].toIntVector();
        const Window win{v[0], v[1], v[2], v[3]};
        const int G = (int)ctx->saved_data["G"].toInt(), CO = (int)ctx->saved_data["w"].toIntVector()[0];
        const float p = (float)ctx->saved_data["p"].toDouble();
        const bool want_x = ctx->needs_input_grad(0), want_w = ctx->needs_input_grad(1);
        const bool want_b = ctx->saved_data["bias"].toBool() && ctx->needs_input_grad(2);
        Tensor g = grads[0].contiguous();
        const On on(g);
        check_saved(img, "input", torch::kFloat32, ctx->saved_data["img"].toIntVector(), g);
        check_saved(w, "weight", torch::kFloat32, ctx->saved_data["w"].toIntVector(), g);
        check_saved(raw, "output", torch::kFloat32, g.sizes(), g);
        Tensor gi, gw, gb;
        if (want_b) gb = sum_per_channel(g);
        if (ctx->saved_data["mean"].toBool()) g = mean_shifted(on, g, Tensor(), 0.0);
        if (want_x) gi = torch::empty_like(img);
        if (want_w) gw = torch::zeros_like(w);   // the kernels add onto this buffer
        if (want_x && want_w)
            done("norm_dist_conv_backward", ldist_norm_dist_conv_backward(in(g), in(img), in(w), in(raw), IMAGE_ARGS(img), CO, G,
                                                                          WINDOW_ARGS(win), out(gi), out(gw), p, on.stream));
        else if (want_x)
            done("norm_dist_conv_backward_input", ldist_norm_dist_conv_backward_input(in(g), in(img), in(w), in(raw),
                                                                                      IMAGE_ARGS(img), CO, G, WINDOW_ARGS(win),
                                                                                      out(gi), p, on.stream));
        else if (want_w)
            done("norm_dist_conv_backward_weight", ldist_norm_dist_conv_backward_weight(in(g), in(img), in(w), in(raw),
                                                                                        IMAGE_ARGS(img), CO, G, WINDOW_ARGS(win),
                                                                                        out(gw), p, on.stream));
        return {gi, gw, gb, Tensor(), Tensor(), Tensor(), Tensor()};
    }
};

// ---- what Python calls -------------------------------------------------------------------------------------------
// Tensors arrive contiguous or are made so where the Python route does the same; p is checked there too.
Tensor norm_dist(const Tensor& x, const Tensor& w, int64_t G, double p) {
    TORCH_CHECK(x.dim() == 3 && w.dim() == 2, "input must be 3-D, weight 2-D");
    check(x, "input", x.device());
    check(w, "weight", x.device());
    if (at::GradMode::is_enabled() && (wants_grad(x) || wants_grad(w)))
        return ColumnLayer::apply(x, w, OptTensor(), G, p, Shift());
    return distances(On(x), x, w, G, p, OptTensor(), Shift());
}

// `w`: a layer's weight with its window, (CO, CI/G, k, k), or the matrix that it is.
// The layer's shift and bias included.
std::tuple<Tensor, Tensor> bounds_of_columns(const Tensor& lower, const Tensor& upper, const Tensor& w, int64_t G,
                                             const OptTensor& bias, const Shift& shift) {
    check(lower, "input_lower", lower.device());
    check(upper, "input_upper", lower.device());
    check(w, "weight", lower.device());
    TORCH_CHECK(lower.sizes() == upper.sizes(), "input_upper must match input_lower");
    const On on(lower);
    const Sizes s = sizes_of(lower, w, G);
    Tensor lo = torch::empty(s.output(), lower.options()), hi = torch::empty_like(lo);
    if (s.HW == 1 && shift.constant(bias)) {
        done("inf_dist_bound_forward",
             ldist_torch::inf_bound_forward_shifted(in(lower), in(upper), in(w), s.B, s.CO, s.CI, (int)G, shift.running_mean(),
                                                    in(bias), out(lo), out(hi), lo, on.stream));
        return {lo, hi};
    }
    done("inf_dist_bound_forward", ldist_torch::inf_bound_forward(in(lower), in(upper), in(w), s.B, s.CO, s.CI, (int)G, s.HW,
                                                                  out(lo), out(hi), lo, on.stream));
    return {shifted(on, lo, bias, shift, false), shifted(on, hi, bias, shift, false)};
}

std::tuple<Tensor, Tensor> inf_dist_bound(const Tensor& lower, const Tensor& upper, const Tensor& w, int64_t G) {
    TORCH_CHECK(lower.dim() == 3 && w.dim() == 2, "input_lower must be 3-D, weight 2-D");
    return bounds_of_columns(lower, upper, w, G, OptTensor(), Shift());
}

Shift make_shift(const OptTensor& running, double momentum, bool training, const torch::Device& dev) {
    Shift s;
    if (running.has_value()) {
        check(*running, "running_mean", dev);
        s.running = *running;
    }
    s.momentum = momentum;
    s.training = training;
    return s;
}

// (B, C, H, W) image as columns for a window that covers one position at a time; (B, C) stays as it is.
Tensor as_columns(const Tensor& t) {
    return t.dim() == 2 ? t.contiguous() : t.reshape({t.size(0), t.size(1), t.size(2) * t.size(3)}).contiguous();
}

// The layer's result in the dimensions of its input.
Tensor as_output(const Tensor& y, const Tensor& x, const Window& win) {
    if (x.dim() == 2) return y;
    const auto [ho, wo] = win.positions(x);
    return y.view({y.size(0), y.size(1), ho, wo});
}

// What the library would refuse, before `positions` divides by the stride.
void check_window(const Window& win) {
    TORCH_CHECK(win.trivial() || (win.k > 0 && win.stride > 0 && win.pad >= 0 && win.dil > 0),
                "the window needs a positive size, stride and dilation, and no negative padding");
}

// The weight of a layer on x (B, CI, H, W) or (B, CI) is (CO, CI/G, k, k): the kernels that read the image take its
// channels from the image and the reduction's length from the window, so both have to agree with what the weight holds.
void check_weight(const Tensor& w, const Tensor& x, int64_t G, const Window& win) {
    check(w, "weight", x.device());
    TORCH_CHECK(x.dim() == 4 || (x.dim() == 2 && win.trivial()), "input must be (B, C, H, W), or (B, C) without a window");
    TORCH_CHECK(G > 0 && w.dim() == 4 && w.size(1) * G == x.size(1) && w.size(2) == win.k && w.size(3) == win.k,
                "weight must be (CO, CI/G, k, k) with as many input channels as the input has");
}

void check_per_channel(const OptTensor& t, const char* name, const Tensor& w) {
    if (!t.has_value()) return;
    check(*t, name, w.device());
    TORCH_CHECK(t->numel() == w.size(0), name, " must hold one value per output channel");
}

// Values of a layer: x (B, CI, H, W) or, fully connected, (B, CI); weight (CO, CI/G, k, k).  Returns (y, whether it came straight from the image).
std::tuple<Tensor, bool> layer(const Tensor& x, const Tensor& weight, const OptTensor& bias, const OptTensor& running,
                               double momentum, bool training, int64_t G, double p, int64_t k, int64_t stride, int64_t pad,
                               int64_t dil, bool finite_p_from_image, int64_t folded_max_row) {
    const Window win{k, stride, pad, dil};
    check_window(win);
    const Tensor w = weight.contiguous();
    check_weight(w, x, G, win);
    check_per_channel(bias, "bias", w);
    check_per_channel(running, "running_mean", w);
    const Shift shift = make_shift(running, momentum, training, x.device());
    const bool inf = std::isinf(p), grad = at::GradMode::is_enabled() && (wants_grad(x) || wants_grad(w) || wants_grad(bias));
    bool from_image = false;
    Tensor y;
    if (!win.trivial()) {
        TORCH_CHECK(x.is_cuda() && x.scalar_type() == torch::kFloat32 && x.device() == w.device(),
                    "all tensors must be float32 on the same device");
        const bool folded = inf && x.size(1) / G * x.size(3) <= folded_max_row;
        if (inf)
            from_image = folded && ldist_inf_dist_conv_forward_supported(GEOMETRY_ARGS(x, w.size(0), G, win));
        else
            from_image = finite_p_from_image && ldist_norm_dist_conv_supported(GEOMETRY_ARGS(x, w.size(0), G, win));
        const Tensor img = x.contiguous();
        if (folded || from_image) {
            if (grad) {
                y = inf ? InfImageLayer::apply(img, w, bias, G, win, from_image, shift)
                        : NormImageLayer::apply(img, w, bias, G, p, win, shift);
            } else {
                const On on(img);
                y = inf ? inf_image_forward(on, img, w, G, win, from_image, nullptr, bias, shift)
                        : shifted(on, norm_image_forward(on, img, w, G, p, win), bias, shift, false);
            }
        } else {
            const Tensor cols = grad && wants_grad(img) ? Unfold::apply(img, win) : unfolded(On(img), img, win);
            if (grad) y = ColumnLayer::apply(cols, w, bias, G, p, shift);
            else { const On on(cols); y = distances(on, cols, w, G, p, bias, shift); }
        }
    } else {
        const Tensor cols = as_columns(x);
        check(cols, "input", w.device());
        if (grad) y = ColumnLayer::apply(cols, w, bias, G, p, shift);
        else { const On on(cols); y = distances(on, cols, w, G, p, bias, shift); }
    }
    return {as_output(y, x, win), from_image};
}

// Interval bounds of a layer in evaluation mode, shifts included: (lower, upper, whether straight from the images).
std::tuple<Tensor, Tensor, bool> layer_bounds(const Tensor& lower, const Tensor& upper, const Tensor& weight, const OptTensor& bias,
                                              const OptTensor& running, int64_t G, int64_t k, int64_t stride, int64_t pad,
                                              int64_t dil) {
    at::NoGradGuard no_grad;
    const Window win{k, stride, pad, dil};
    check_window(win);
    const Tensor w = weight.contiguous();
    check_weight(w, lower, G, win);
    check_per_channel(bias, "bias", w);
    check_per_channel(running, "running_mean", w);
    const Shift shift = make_shift(running, 0.0, false, lower.device());
    const On on(lower);
    Tensor lo, hi;
    bool from_image = false;
    if (!win.trivial() && ldist_inf_dist_bound_conv_forward_supported(GEOMETRY_ARGS(lower, w.size(0), G, win))) {
        from_image = true;
        const Tensor l = lower.contiguous(), u = upper.contiguous();
        check(l, "lower_img", w.device());
        check(u, "upper_img", w.device());
        TORCH_CHECK(l.sizes() == u.sizes(), "lower_img and upper_img must have one shape");
        const auto [ho, wo] = win.positions(l);
        lo = torch::empty({l.size(0), w.size(0), ho * wo}, l.options());
        hi = torch::empty_like(lo);
        done("inf_dist_bound_conv_forward",
             ldist_inf_dist_bound_conv_forward_shifted(in(l), in(u), in(w), IMAGE_ARGS(l), (int)w.size(0), (int)G, WINDOW_ARGS(win),
                                                       shift.running_mean(), in(bias), out(lo), out(hi), on.stream));
    } else if (win.trivial()) {
        std::tie(lo, hi) = bounds_of_columns(as_columns(lower), as_columns(upper), w, G, bias, shift);
    } else {
        const Tensor l = lower.contiguous(), u = upper.contiguous();
        check(l, "lower_img", w.device());
        check(u, "upper_img", w.device());
        std::tie(lo, hi) = bounds_of_columns(unfolded(on, l, win), unfolded(on, u, win), w, G, bias, shift);
    }
    return {as_output(lo, lower, win), as_output(hi, lower, win), from_image};
}

// Whether `layer_value_bounds` has one pass for a wide layer on B rows: one that the lists of outermost values are for.
bool value_bounds_pay(int64_t B, int64_t CO, int64_t CI, int64_t G) {
    int64_t bytes = 0;
    return B <= INT_MAX && ldist_inf_dist_value_bound_workspace((int)B, (int)CO, (int)CI, (int)G, 1, &bytes) == LDIST_OK && bytes > 0;
}

// Values and bounds in one pass, for layers without a window: those with few outputs, and those of `value_bounds_pay`.  And
// whether it was one pass.
std::tuple<Tensor, Tensor, Tensor, bool> layer_value_bounds(const Tensor& x, const Tensor& lower, const Tensor& upper,
                                                            const Tensor& weight, const OptTensor& bias, const OptTensor& running,
                                                            int64_t G) {
    at::NoGradGuard no_grad;
    const Tensor w = weight.contiguous(), cx = as_columns(x), cl = as_columns(lower), cu = as_columns(upper);
    check(cx, "input", w.device());
    check(cl, "input_lower", w.device());
    check(cu, "input_upper", w.device());
    check_weight(w, x, G, Window{1, 1, 0, 1});
    check_per_channel(bias, "bias", w);
    check_per_channel(running, "mean", w);
    TORCH_CHECK(cl.sizes() == cx.sizes() && cu.sizes() == cx.sizes(), "input_lower and input_upper must match input");
    const On on(cx);
    const Sizes s = sizes_of(cx, w, G);
    const Window win{1, 1, 0, 1};
    int64_t bytes = 0;
    done("inf_dist_value_bound_workspace", ldist_inf_dist_value_bound_workspace(s.B, s.CO, s.CI, (int)G, s.HW, &bytes));
    Tensor y = torch::empty(s.output(), cx.options()), lo = torch::empty_like(y), hi = torch::empty_like(y);
    bool together = true;
    if (bytes == 0) {
        done("inf_dist_value_bound_forward",
             ldist_inf_dist_value_bound_forward(in(cx), in(cl), in(cu), in(w), s.B, s.CO, s.CI, (int)G, s.HW, in(running), in(bias),
                                                out(y), out(lo), out(hi), on.stream));
    } else {
        Tensor ws = ldist_torch::scratch(bytes, cx);
        const int rc = !ws.defined() ? LDIST_EUNSUPPORTED
                                     : ldist_inf_dist_value_bound_forward_ws(in(cx), in(cl), in(cu), in(w), s.B, s.CO, s.CI, (int)G,
                                                                             s.HW, in(running), in(bias), out(y), out(lo), out(hi),
                                                                             ws.data_ptr(), ws.numel(), on.stream);
        together = rc != LDIST_EUNSUPPORTED;
        if (!together) {   // no memory for it, or no 128-bit loads: one pass after the other, in the memory that they need by themselves
            ws = y = lo = hi = Tensor();
            const Shift shift = make_shift(running, 0.0, false, cx.device());
            y = distances(on, cx, w, G, INFINITY, bias, shift);
            std::tie(lo, hi) = bounds_of_columns(cl, cu, w, G, bias, shift);
        } else {
            done("inf_dist_value_bound_forward", rc);
        }
    }
    return {as_output(y, x, win), as_output(lo, x, win), as_output(hi, x, win), together};
}

// Certified margins (BoundFinalIdentity) with gradients to both bounds.
struct Margins : public Function<Margins> {
    static Tensor forward(AutogradContext* ctx, const Tensor& lower, const Tensor& upper, const Tensor& targets) {
        const On on(upper);
        // torch's own look-up of the label's lower bound, for what it does with a target that is no class: the kernel below
        // would leave NaN in such a row and go on
        lower.gather(1, targets.view({-1, 1}));
        Tensor m = torch::empty_like(upper);
        done("certified_margins", ldist_certified_margins(in(lower), in(upper), targets.const_data_ptr<int64_t>(),
                                                          (int)upper.size(0), (int)upper.size(1), out(m), on.stream));
        ctx->save_for_backward({targets});
        return m;
    }
    static tensor_list backward(AutogradContext* ctx, tensor_list grads) {
        const Tensor at = ctx->get_saved_variables()[0].view({-1, 1});
        const Tensor gu = grads[0].scatter(1, at, 0.0);       // the target's own margin is the constant 0
        Tensor gl;
        if (ctx->needs_input_grad(0)) gl = torch::zeros_like(gu).scatter_(1, at, gu.sum(1, true).neg_());
        return {gl, ctx->needs_input_grad(1) ? gu : Tensor(), Tensor()};
    }
};

Tensor margins(const Tensor& lower, const Tensor& upper, const Tensor& targets) {
    const Tensor l = lower.contiguous(), u = upper.contiguous(), t = targets.contiguous();
    check(l, "lower", u.device());
    check(u, "upper", u.device());
    TORCH_CHECK(u.dim() == 2 && l.sizes() == u.sizes(), "lower and upper must be (B, classes)");
    TORCH_CHECK(t.device() == u.device() && t.scalar_type() == torch::kInt64 && t.numel() == u.size(0),
                "targets must hold one int64 class per row on the same device");
    return Margins::apply(l, u, t);
}

Tensor pgd_step(const Tensor& adv, const Tensor& grad, const Tensor& centre, double step, double eps, double down, double up) {
    at::NoGradGuard no_grad;
    const Tensor a = adv.contiguous(), g = grad.contiguous(), c = centre.contiguous();
    check(a, "adv", a.device());
    check(g, "grad", a.device());
    check(c, "centre", a.device());
    TORCH_CHECK(g.sizes() == a.sizes() && c.sizes() == a.sizes(), "adv, grad and centre must have one shape");
    const On on(a);
    Tensor next = torch::empty_like(a);
    if (a.numel() > 0)
        done("pgd_step", ldist_pgd_step(in(a), in(g), in(c), a.numel(), (float)step, (float)eps, (float)down, (float)up, out(next),
                                        on.stream));
    return next;
}

// One AdamW step of several parameters: per parameter the p of its module (negative: none), lr, beta1, beta2, eps,
// weight decay and the step count after this one.
void adamw_step(const std::vector<Tensor>& params, const std::vector<Tensor>& grads, const std::vector<Tensor>& exp_avgs,
                const std::vector<Tensor>& exp_avg_sqs, const std::vector<std::tuple<double, double, double, double, double, double, int64_t>>& hyper) {
    TORCH_CHECK(grads.size() == params.size() && exp_avgs.size() == params.size() && exp_avg_sqs.size() == params.size() &&
                hyper.size() == params.size(), "every parameter needs its gradient, moments and hyper-parameters");
    for (size_t i = 0; i < params.size(); i++) {
        const Tensor &w = params[i], &g = grads[i], &m = exp_avgs[i], &v = exp_avg_sqs[i];
        for (const Tensor* t : {&w, &g, &m, &v}) {
            check(*t, "param, grad and moments", w.device());
            TORCH_CHECK(t->sizes() == w.sizes(), "grad and moments must have the shape of param");
        }
        TORCH_CHECK(w.numel() > 0, "param must not be empty");
        const On on(w);
        const int64_t rows = w.dim() > 0 ? w.size(0) : 1;
        const auto& [p, lr, b1, b2, eps, wd, step] = hyper[i];
        done("adamw_lp_step", ldist_adamw_lp_step(out(w), in(g), out(m), out(v), (int)rows, (int)(w.numel() / rows), p, lr, b1, b2,
                                                  eps, wd, (int)step, on.stream));
    }
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    m.doc() = "Native host path of the L_p / L_inf distance layers on MI355X (gfx950)";
    // Without the interpreter lock, which nothing in here needs: threads that each drive a stream run side by side.
    using no_lock = py::call_guard<py::gil_scoped_release>;
    m.def("norm_dist", &norm_dist, no_lock());
    m.def("inf_dist_bound", &inf_dist_bound, no_lock());
    m.def("layer", &layer, no_lock());
    m.def("layer_bounds", &layer_bounds, no_lock());
    m.def("layer_value_bounds", &layer_value_bounds, no_lock());
    m.def("value_bounds_pay", &value_bounds_pay, no_lock());
    m.def("margins", &margins, no_lock());
    m.def("pgd_step", &pgd_step, no_lock());
    m.def("adamw_step", &adamw_step, no_lock());
}
