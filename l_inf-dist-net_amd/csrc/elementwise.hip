// The small elementwise operations around the distance layers, one launch each: the evaluation-mode shift of a layer's
// output, the certified margins, and a projected-gradient step.  Each replaces two to six torch kernels that read and
// write tensors of a few megabytes at most, so what they cost is launches (4 to 5 us each on the GPU, as much on the
// host), not bytes.
#include "kernels.hpp"

namespace ldist {

// y[b,c,l] = (x[b,c,l] - mean[c]) + bias[c], in this order and each step rounded as the two torch operations round it;
// either vector may be absent.  y may be x.  One lane per VEC neighbouring values: VEC = 4 needs 16-byte aligned
// tensors and, for L == 1, C % 4 == 0 (four values of one row), for L > 1, L % 4 == 0 (the four values share a channel).
// mean and bias are read a value at a time, from cache: they need no alignment.
template <int VEC, bool ROWS>
__global__ void __launch_bounds__(256)
channel_shift_kernel(const float* __restrict__ mean, const float* __restrict__ bias, const float* x, float* y, int C, int L,
                     unsigned total) {
    for (unsigned i = blockIdx.x * 256u + threadIdx.x; i < total; i += gridDim.x * 256u) {
        const unsigned at = i * VEC;
        float v[VEC], m[VEC], b[VEC];
        if constexpr (VEC == 4) {
            const float4 t = *reinterpret_cast<const float4*>(x + at);
            v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
        } else {
            v[0] = x[at];
        }
        const unsigned c = ROWS ? at % (unsigned)C : at / (unsigned)L % (unsigned)C;
#pragma unroll
        for (int e = 0; e < VEC; e++) {
            m[e] = mean ? mean[ROWS ? c + e : c] : 0.f;
            b[e] = bias ? bias[ROWS ? c + e : c] : 0.f;
        }
#pragma unroll
        for (int e = 0; e < VEC; e++) {
            if (mean) v[e] = v[e] - m[e];
            if (bias) v[e] = v[e] + b[e];
        }
        if constexpr (VEC == 4) *reinterpret_cast<float4*>(y + at) = make_float4(v[0], v[1], v[2], v[3]);
        else y[at] = v[0];
    }
}

static unsigned lanes_grid(unsigned total, int num_cu) {
    const unsigned blocks = (total + 255) / 256, most = 8u * (unsigned)num_cu;
    return blocks < most ? blocks : most;
}

__global__ void __launch_bounds__(256) zero_fill_kernel(float* __restrict__ p, size_t n, bool vec) {
    const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (vec && i + 3 < n) {
        *reinterpret_cast<float4*>(p + i) = make_float4(0.f, 0.f, 0.f, 0.f);
    } else {
        for (size_t j = i; j < n && j < i + 4; j++) p[j] = 0.f;
    }
}

hipError_t zero_fill(float* p, size_t n, hipStream_t stream) {
    hipLaunchKernelGGL(zero_fill_kernel, dim3((unsigned)((n + 1023) / 1024)), dim3(256), 0, stream, p, n, aligned16(p));
    return hipGetLastError();
}

hipError_t channel_shift(const float* x, const float* mean, const float* bias, float* y, int B, int C, int L, int num_cu,
                         hipStream_t stream) {
    const unsigned n = (unsigned)B * C * L;
    const bool vec = aligned16(x) && aligned16(y) && (L == 1 ? C % 4 == 0 : L % 4 == 0);
    const unsigned total = vec ? n / 4 : n;
    const dim3 grid(lanes_grid(total, num_cu)), block(256);
    if (L == 1 && vec) hipLaunchKernelGGL((channel_shift_kernel<4, true>), grid, block, 0, stream, mean, bias, x, y, C, L, total);
    else if (L == 1) hipLaunchKernelGGL((channel_shift_kernel<1, true>), grid, block, 0, stream, mean, bias, x, y, C, L, total);
    else if (vec) hipLaunchKernelGGL((channel_shift_kernel<4, false>), grid, block, 0, stream, mean, bias, x, y, C, L, total);
    else hipLaunchKernelGGL((channel_shift_kernel<1, false>), grid, block, 0, stream, mean, bias, x, y, C, L, total);
    return hipGetLastError();
}

// margins[b,j] = upper[b,j] - lower[b,target_b], 0 at j = target_b.  A target outside [0, J) leaves NaN in its row.
__global__ void __launch_bounds__(256)
certified_margins_kernel(const float* __restrict__ lower, const float* __restrict__ upper, const int64_t* __restrict__ targets,
                         float* __restrict__ margins, int J, unsigned total) {
    const unsigned i = blockIdx.x * 256u + threadIdx.x;
    if (i >= total) return;
    const unsigned b = i / (unsigned)J, j = i % (unsigned)J;
    const int64_t t = targets[b];
    float v = __builtin_nanf("");
    if (t >= 0 && t < J) v = (int64_t)j == t ? 0.f : upper[i] - lower[b * (unsigned)J + (unsigned)t];
    margins[i] = v;
}

hipError_t certified_margins(const float* lower, const float* upper, const int64_t* targets, float* margins, int B, int J,
                             hipStream_t stream) {
    const unsigned total = (unsigned)B * J;
    hipLaunchKernelGGL(certified_margins_kernel, dim3((total + 255) / 256), dim3(256), 0, stream, lower, upper, targets,
                       margins, J, total);
    return hipGetLastError();
}

// x clipped into [lo, hi] as torch.minimum(torch.maximum(x, lo), hi) clips it: a NaN stays one.
__device__ __forceinline__ float box(float x, float lo, float hi) {
    const float a = (x != x || x > lo) ? x : lo;
    return (a != a || a < hi) ? a : hi;
}

// next = box(box(adv + step * sign(grad), centre - eps, centre + eps), down, up), each operation rounded on its own.
__global__ void __launch_bounds__(256)
pgd_step_kernel(const float* __restrict__ adv, const float* __restrict__ grad, const float* __restrict__ centre,
                float* __restrict__ next, unsigned n, float step, float eps, float down, float up) {
    for (unsigned i = blockIdx.x * 256u + threadIdx.x; i < n; i += gridDim.x * 256u) {
        const float g = grad[i], c = centre[i];
        const float s = g > 0.f ? 1.f : g < 0.f ? -1.f : 0.f;   // torch.sign, NaN included: 0
        next[i] = box(box(__fadd_rn(adv[i], __fmul_rn(step, s)), __fsub_rn(c, eps), __fadd_rn(c, eps)), down, up);
    }
}

hipError_t pgd_step(const float* adv, const float* grad, const float* centre, float* next, long long n, float step, float eps,
                    float down, float up, int num_cu, hipStream_t stream) {
    hipLaunchKernelGGL(pgd_step_kernel, dim3(lanes_grid((unsigned)n, num_cu)), dim3(256), 0, stream, adv, grad, centre, next,
                       (unsigned)n, step, eps, down, up);
    return hipGetLastError();
}

}  // namespace ldist
