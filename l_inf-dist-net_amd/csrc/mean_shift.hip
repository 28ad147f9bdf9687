// Per-channel mean shift of a (B, C, L) tensor: y[b,c,l] = x[b,c,l] - mean_c, mean_c the mean of
// x over b and l; optionally moves a running mean.  This is the training-mode
// arithmetic of the reference's MeanNorm (model/norm_dist.py:85-96), which runs it as five
// small torch kernels per layer and direction; the same kernel serves the backward pass
// (gx = gy - mean(gy)).  HBM-bound: a workgroup owns a slab small enough that its second read
// comes from cache, so the tensor is fetched once and written once.
#include <algorithm>

#include "kernels.hpp"
#include "wave_reduce.hpp"

namespace ldist {

constexpr int kMsCols = 32;      // channels per workgroup, L == 1
constexpr int kMsThreads = 256;
constexpr int kMsChanThreads = 1024;   // the channel kernel: one workgroup per channel

__device__ __forceinline__ void move_running_mean(float* running_mean, int c, float mean, float momentum) {
    // (1 - momentum) * running + momentum * mean, rounded after each step as two torch ops would
    const float kept = running_mean[c] * (1.0f - momentum);
    running_mean[c] = kept + momentum * mean;
}

// L == 1: channels are contiguous.  Workgroup = kMsCols channels x all B rows.  A lane owns four
// neighbouring channels (one 128-bit access per row) and the rows ty, ty + 32, ...; eight lanes
// cover a 128-byte row segment.  Sixteen rows per lane are loaded before the first is used, which
// keeps 64 KB in flight per workgroup; up to 512 rows stay in registers for the subtraction, so
// the tensor is read exactly once.  VEC4 needs C % 4 == 0 and 16-byte aligned bases.
template <bool VEC4>
__global__ void __launch_bounds__(kMsThreads)
mean_shift_rows_kernel(const float* __restrict__ x, float* __restrict__ y, float* __restrict__ mean_out,
                       float* __restrict__ running_mean, float momentum, int B, int C) {
    constexpr int TX = kMsCols / 4, RY = kMsThreads / TX, HOLD = 16;   // 8 lanes across, 32 down
    __shared__ float part[RY][kMsCols];
    __shared__ float mean_s[kMsCols];
    const int tx = threadIdx.x % TX, ty = threadIdx.x / TX;
    const int c = blockIdx.x * kMsCols + tx * 4;
    auto load4 = [&](int r) {
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (r < B) {
            const float* p = x + (size_t)r * C + c;
            if constexpr (VEC4) {
                if (c < C) v = *reinterpret_cast<const float4*>(p);
            } else {
                if (c < C) v.x = p[0];
                if (c + 1 < C) v.y = p[1];
                if (c + 2 < C) v.z = p[2];
                if (c + 3 < C) v.w = p[3];
            }
        }
        return v;
    };
    auto store4 = [&](int r, float4 v) {
        if (r >= B) return;
        float* p = y + (size_t)r * C + c;
        if constexpr (VEC4) {
            if (c < C) *reinterpret_cast<float4*>(p) = v;
        } else {
            if (c < C) p[0] = v.x;
            if (c + 1 < C) p[1] = v.y;
            if (c + 2 < C) p[2] = v.z;
            if (c + 3 < C) p[3] = v.w;
        }
    };
    float4 held[HOLD];
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int r0 = 0; r0 < B; r0 += HOLD * RY) {
#pragma unroll
        for (int i = 0; i < HOLD; i++) held[i] = load4(r0 + ty + i * RY);
#pragma unroll
        for (int i = 0; i < HOLD; i++) { s.x += held[i].x; s.y += held[i].y; s.z += held[i].z; s.w += held[i].w; }
    }
    part[ty][tx * 4 + 0] = s.x; part[ty][tx * 4 + 1] = s.y; part[ty][tx * 4 + 2] = s.z; part[ty][tx * 4 + 3] = s.w;
    __syncthreads();
    if (threadIdx.x < kMsCols) {
        float t = 0.f;
#pragma unroll
        for (int q = 0; q < RY; q++) t += part[q][threadIdx.x];
        const float mean = t / (float)B;
        mean_s[threadIdx.x] = mean;
        const int cc = blockIdx.x * kMsCols + threadIdx.x;
        if (cc < C) {
            if (mean_out) mean_out[cc] = mean;
            if (running_mean) move_running_mean(running_mean, cc, mean, momentum);
        }
    }
    __syncthreads();
    const float4 m = make_float4(mean_s[tx * 4], mean_s[tx * 4 + 1], mean_s[tx * 4 + 2], mean_s[tx * 4 + 3]);
    auto shifted = [&](float4 v) { return make_float4(v.x - m.x, v.y - m.y, v.z - m.z, v.w - m.w); };
    if (B <= HOLD * RY) {   // everything is still in registers
#pragma unroll
        for (int i = 0; i < HOLD; i++) store4(ty + i * RY, shifted(held[i]));
    } else {
        for (int r0 = 0; r0 < B; r0 += HOLD * RY) {
#pragma unroll
            for (int i = 0; i < HOLD; i++) held[i] = load4(r0 + ty + i * RY);
#pragma unroll
            for (int i = 0; i < HOLD; i++) store4(r0 + ty + i * RY, shifted(held[i]));
        }
    }
}

// L > 1: for a fixed (b, c) the L values are contiguous.  Workgroup = one channel; lanes run along l
// (128-bit accesses when VEC == 4: L % 4 == 0 and 16-byte aligned bases).  A channel is one workgroup's work, and
// the workgroup is as large as it can be: what limits this kernel is how many loads one CU keeps in flight.
template <int VEC>
__global__ void __launch_bounds__(kMsChanThreads)
mean_shift_channel_kernel(const float* __restrict__ x, float* __restrict__ y, float* __restrict__ mean_out,
                          float* __restrict__ running_mean, float momentum, int B, int C, int L) {
    __shared__ float part[kMsChanThreads / 64];
    __shared__ float mean_s;
    const int c = blockIdx.x;
    const int per_b = L / VEC;                    // vectors per (b, c) run
    const int total = B * per_b;
    // four independent loads in flight per lane: a channel is one workgroup's work, and with one load per trip
    // the workgroup waits out a memory latency per 4 KB (8 KB with 128-bit loads)
    constexpr int UN = 4;
    auto at_of = [&](int i) {
        const int b = i / per_b, q = i - b * per_b;
        return ((size_t)b * C + c) * L + (size_t)q * VEC;
    };
    float s = 0.f;
    for (int i0 = threadIdx.x; i0 < total; i0 += UN * kMsChanThreads) {
        if constexpr (VEC == 4) {
            float4 v[UN];
#pragma unroll
            for (int u = 0; u < UN; u++) {
                const int i = i0 + u * kMsChanThreads;
                v[u] = i < total ? *reinterpret_cast<const float4*>(x + at_of(i)) : make_float4(0.f, 0.f, 0.f, 0.f);
            }
#pragma unroll
            for (int u = 0; u < UN; u++) s += (v[u].x + v[u].y) + (v[u].z + v[u].w);
        } else {
            float v[UN];
#pragma unroll
            for (int u = 0; u < UN; u++) {
                const int i = i0 + u * kMsChanThreads;
                v[u] = i < total ? x[at_of(i)] : 0.f;
            }
#pragma unroll
            for (int u = 0; u < UN; u++) s += v[u];
        }
    }
    s = wave_sum(s);                // lane 63 holds the wave's sum
    if ((threadIdx.x & 63) == 63) part[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        float t = 0.f;
#pragma unroll
        for (int q = 0; q < kMsChanThreads / 64; q++) t += part[q];
        const float mean = t / ((float)B * (float)L);
        mean_s = mean;
        if (mean_out) mean_out[c] = mean;
        if (running_mean) move_running_mean(running_mean, c, mean, momentum);
    }
    __syncthreads();
    const float mean = mean_s;
    for (int i0 = threadIdx.x; i0 < total; i0 += UN * kMsChanThreads) {
        size_t at[UN];
#pragma unroll
        for (int u = 0; u < UN; u++) at[u] = at_of(min(i0 + u * kMsChanThreads, total - 1));
        if constexpr (VEC == 4) {
            float4 v[UN];
#pragma unroll
            for (int u = 0; u < UN; u++) v[u] = *reinterpret_cast<const float4*>(x + at[u]);
#pragma unroll
            for (int u = 0; u < UN; u++)
                if (i0 + u * kMsChanThreads < total)
                    *reinterpret_cast<float4*>(y + at[u]) = make_float4(v[u].x - mean, v[u].y - mean, v[u].z - mean, v[u].w - mean);
        } else {
            float v[UN];
#pragma unroll
            for (int u = 0; u < UN; u++) v[u] = x[at[u]];
#pragma unroll
            for (int u = 0; u < UN; u++)
                if (i0 + u * kMsChanThreads < total) y[at[u]] = v[u] - mean;
        }
    }
}

// The same for channels that are fewer than the CUs and long, in two launches that share a channel out.  The sums are the ones of
// the kernel above, in the same order and so the same bits: a workgroup of the first launch is one of its sixteen waves.  They go
// from one launch to the other through y: every workgroup of the second finds all sixteen in the first places of its own part,
// which it overwrites after reading them, so neither the order of workgroups nor scratch memory matters.  Bound by memory.
constexpr int kMsWaves = kMsChanThreads / 64;
constexpr int kMsPartThreads = 256, kMsPartUnroll = 4;

template <int VEC>
struct ChannelWalk {
    int c, C, L, per_b;
    __device__ __forceinline__ size_t at(int i) const {
        const int b = i / per_b, q = i - b * per_b;
        return ((size_t)b * C + c) * L + (size_t)q * VEC;
    }
};

template <int VEC>
__global__ void __launch_bounds__(64)
mean_shift_sums_kernel(const float* __restrict__ x, float* __restrict__ y, int B, int C, int L, int parts, int len) {
    typedef float V __attribute__((ext_vector_type(VEC)));
    constexpr int UN = 32;   // loads in flight: a lane's work of 32 x 1024 x 1024 values is one such trip
    const int c = blockIdx.x / kMsWaves, wave = blockIdx.x % kMsWaves, lane = threadIdx.x;
    const ChannelWalk<VEC> walk{c, C, L, L / VEC};
    const int total = B * walk.per_b;
    float s = 0.f;
    for (int i0 = wave * 64 + lane; i0 < total; i0 += UN * kMsChanThreads) {
        V v[UN];
#pragma unroll
        for (int u = 0; u < UN; u++) {
            const int i = i0 + u * kMsChanThreads;
            v[u] = i < total ? *reinterpret_cast<const V*>(x + walk.at(i)) : V(0.f);
        }
#pragma unroll
        for (int u = 0; u < UN; u++) {
            if constexpr (VEC == 4) s += (v[u][0] + v[u][1]) + (v[u][2] + v[u][3]);
            else s += v[u][0];
        }
    }
    s = __shfl(wave_sum(s), 63);
    if (lane < parts) y[walk.at(lane * len + wave)] = s;
}

template <int VEC>
__global__ void __launch_bounds__(kMsPartThreads)
mean_shift_part_kernel(const float* __restrict__ x, float* __restrict__ y, float* __restrict__ mean_out,
                       float* __restrict__ running_mean, float momentum, int B, int C, int L, int parts, int len) {
    typedef float V __attribute__((ext_vector_type(VEC)));
    __shared__ float sums[kMsWaves];
    constexpr int UN = kMsPartUnroll;
    const int c = blockIdx.x / parts, part = blockIdx.x - c * parts;
    const ChannelWalk<VEC> walk{c, C, L, L / VEC};
    const int begin = part * len, end = min(B * walk.per_b, begin + len);
    if (threadIdx.x < kMsWaves) sums[threadIdx.x] = y[walk.at(begin + threadIdx.x)];
    __syncthreads();   // read by all before any of it is overwritten
    float t = 0.f;
#pragma unroll
    for (int q = 0; q < kMsWaves; q++) t += sums[q];
    const float mean = t / ((float)B * (float)L);
    if (part == 0 && threadIdx.x == 0) {
        if (mean_out) mean_out[c] = mean;
        if (running_mean) move_running_mean(running_mean, c, mean, momentum);
    }
    for (int i0 = begin + threadIdx.x; i0 < end; i0 += UN * kMsPartThreads) {
        size_t at[UN];
        V v[UN];
#pragma unroll
        for (int u = 0; u < UN; u++) {
            at[u] = walk.at(min(i0 + u * kMsPartThreads, end - 1));
            v[u] = *reinterpret_cast<const V*>(x + at[u]);
        }
#pragma unroll
        for (int u = 0; u < UN; u++)
            if (i0 + u * kMsPartThreads < end) *reinterpret_cast<V*>(y + at[u]) = v[u] - mean;
    }
}

// Parts of a channel: four workgroups per CU, each with a full trip of loads (1024 vectors); 1: one workgroup does it all.
// The lines, us, one workgroup per channel -> shared, images x channels x L with four values to a vector:
//   128 x 32 x 1024 21.5 -> 12.2, 128 x 64 x 1024 24.3 -> 20.3, 128 x 96 x 1024 26.6 -> 26.6, 128 x 128 x 1024 36.4 -> 38.0;
//   77 x 32 x 784 11.9 -> 9.2, 32 x 32 x 1024 7.2 -> 6.7, 128 x 64 x 256 8.0 -> 8.4, 77 x 64 x 196 4.9 -> 7.6
// and with one: 128 x 32 x 841 60.8 -> 21.1, 128 x 128 x 841 66.8 -> 40.9, 128 x 256 x 841 78.8 -> 84.8; 128 x 32 x 101 8.9 -> 7.1,
// 128 x 32 x 49 6.0 -> 6.4.
static int channel_parts(int C, int total, int vec, int num_cu) {
    if (C > num_cu / (vec == 4 ? 4 : 2) || total < 12 * kMsChanThreads) return 1;
    if (total >= (1 << 30)) return 1;   // 31-bit indices, a trip past the end included
    return std::min(std::min(4 * num_cu / C, total / (kMsPartUnroll * kMsPartThreads)), 64);
}

template <int VEC>
static void launch_channels(const float* x, float* y, float* mean_out, float* running_mean, float momentum, int B, int C, int L,
                            int num_cu, hipStream_t stream) {
    const int total = B * (L / VEC), parts = channel_parts(C, total, VEC, num_cu);
    if (parts == 1) {
        hipLaunchKernelGGL(mean_shift_channel_kernel<VEC>, dim3((unsigned)C), dim3(kMsChanThreads), 0, stream, x, y, mean_out,
                           running_mean, momentum, B, C, L);
        return;
    }
    // the last part has at least len - parts + 1 vectors, of 1024 - 63: room for the sixteen sums
    const int len = (total + parts - 1) / parts;
    hipLaunchKernelGGL(mean_shift_sums_kernel<VEC>, dim3((unsigned)(C * kMsWaves)), dim3(64), 0, stream, x, y, B, C, L, parts, len);
    hipLaunchKernelGGL(mean_shift_part_kernel<VEC>, dim3((unsigned)(C * parts)), dim3(kMsPartThreads), 0, stream, x, y, mean_out,
                       running_mean, momentum, B, C, L, parts, len);
}

hipError_t mean_shift(const float* x, float* y, float* mean_out, float* running_mean, float momentum, int B, int C,
                      int L, int num_cu, hipStream_t stream) {
    if (L == 1) {
        const unsigned grid = (unsigned)((C + kMsCols - 1) / kMsCols);
        if (C % 4 == 0 && aligned16(x) && aligned16(y))
            hipLaunchKernelGGL(mean_shift_rows_kernel<true>, dim3(grid), dim3(kMsThreads), 0, stream, x, y, mean_out,
                               running_mean, momentum, B, C);
        else
            hipLaunchKernelGGL(mean_shift_rows_kernel<false>, dim3(grid), dim3(kMsThreads), 0, stream, x, y,
                               mean_out, running_mean, momentum, B, C);
    } else if (L % 4 == 0 && aligned16(x) && aligned16(y)) {
        launch_channels<4>(x, y, mean_out, running_mean, momentum, B, C, L, num_cu, stream);
    } else {
        launch_channels<1>(x, y, mean_out, running_mean, momentum, B, C, L, num_cu, stream);
    }
    return hipGetLastError();
}

}  // namespace ldist
