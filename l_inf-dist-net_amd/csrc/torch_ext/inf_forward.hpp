// The L_inf forward passes on columns, in whichever form the library has for the layer: with scratch memory from torch's
// allocator where it asks for some (given back when the call returns: work that is enqueued later on the stream runs later),
// else the plain entry points.  For both extension modules.
#pragma once
#include <torch/extension.h>

#include "ldist.h"

namespace ldist_torch {

// Undefined for no bytes, and where there is no memory for them: the plain entry points need none.
inline torch::Tensor scratch(int64_t bytes, const torch::Tensor& like) {
    if (bytes == 0) return torch::Tensor();
    try {
        return torch::empty({bytes}, like.options().dtype(torch::kUInt8).requires_grad(false));
    } catch (const c10::OutOfMemoryError&) {
        return torch::Tensor();
    }
}

// Undefined also where the layer has no form with a workspace.
inline torch::Tensor workspace(int B, int CO, int CI, int G, int HW, int what, const torch::Tensor& like) {
    int64_t bytes = 0;
    return ldist_inf_dist_workspace(B, CO, CI, G, HW, what, &bytes) == LDIST_OK ? scratch(bytes, like) : torch::Tensor();
}

// The same with the evaluation-mode shift and bias (either may be null) applied by the forward kernel; fully connected layers.
inline int inf_forward_shifted(const float* x, const float* w, int B, int CO, int CI, int G, const float* mean, const float* bias,
                               float* y, int32_t* pos, const torch::Tensor& like, ldist_stream_t stream) {
    const torch::Tensor ws = workspace(B, CO, CI, G, 1, pos ? LDIST_WITH_POS : LDIST_VALUES_ONLY, like);
    return ldist_inf_dist_forward_shifted(x, w, B, CO, CI, G, mean, bias, y, pos, ws.defined() ? ws.data_ptr() : nullptr,
                                          ws.defined() ? ws.numel() : 0, stream);
}

inline int inf_bound_forward_shifted(const float* lower, const float* upper, const float* w, int B, int CO, int CI, int G,
                                     const float* mean, const float* bias, float* out_lower, float* out_upper,
                                     const torch::Tensor& like, ldist_stream_t stream) {
    const torch::Tensor ws = workspace(B, CO, CI, G, 1, LDIST_BOUNDS, like);
    return ldist_inf_dist_bound_forward_shifted(lower, upper, w, B, CO, CI, G, mean, bias, out_lower, out_upper,
                                                ws.defined() ? ws.data_ptr() : nullptr, ws.defined() ? ws.numel() : 0, stream);
}

// pos == nullptr: values only; LDIST_EUNSUPPORTED where only the form with pos exists.  `like`: a tensor of the call.
inline int inf_forward(const float* x, const float* w, int B, int CO, int CI, int G, int HW, float* y, int32_t* pos,
                       const torch::Tensor& like, ldist_stream_t stream) {
    const torch::Tensor ws = workspace(B, CO, CI, G, HW, pos ? LDIST_WITH_POS : LDIST_VALUES_ONLY, like);
    if (ws.defined()) {
        const int rc = ldist_inf_dist_forward_ws(x, w, B, CO, CI, G, HW, y, pos, ws.data_ptr(), ws.numel(), stream);
        if (rc != LDIST_EUNSUPPORTED) return rc;
    }
    return pos ? ldist_inf_dist_forward(x, w, B, CO, CI, G, HW, y, pos, stream)
               : ldist_inf_dist_forward_values(x, w, B, CO, CI, G, HW, y, stream);
}

inline int inf_bound_forward(const float* lower, const float* upper, const float* w, int B, int CO, int CI, int G, int HW,
                             float* out_lower, float* out_upper, const torch::Tensor& like, ldist_stream_t stream) {
    const torch::Tensor ws = workspace(B, CO, CI, G, HW, LDIST_BOUNDS, like);
    if (ws.defined()) {
        const int rc = ldist_inf_dist_bound_forward_ws(lower, upper, w, B, CO, CI, G, HW, out_lower, out_upper, ws.data_ptr(),
                                                       ws.numel(), stream);
        if (rc != LDIST_EUNSUPPORTED) return rc;
    }
    return ldist_inf_dist_bound_forward(lower, upper, w, B, CO, CI, G, HW, out_lower, out_upper, stream);
}

}  // namespace ldist_torch
