// Both p-norm gradients of a fully connected layer with few outputs per group (a classification head), p > 1:
//   t[m,n,k] = g[m,n] * (|x[m,k] - w[n,k]| / out[m,n])^(p-1) * sign(x - w)
//   grad_input[m,k] = sum_n t        grad_weight[n,k] += -sum_m t
// (reference model/norm_dist_cuda.cu:294-425, two kernels).
//
// All outputs of a group fit the registers of a lane that owns one column k: a wave walks 16 rows at a time, evaluates every
// term once and adds it to both sums; grad_input leaves with the row, the waves' weight sums meet in LDS after the last.
// g and 1 / out of 64 rows lie in LDS, where all lanes read the same word.  Bound by latency: the terms are 1 to 6 us of a
// launch of 10 to 13.  The two general kernels (norm_backward_kernel.hpp) walk stages of 32 outputs, of which ten are real, and
// leave grad_weight to 40 workgroups of 32 x 128.  Rows x inputs -> outputs, us, both gradients:
//   512 x 5120 -> 10, p = 8: 69 -> 13;  64 x 5120 -> 10, p = 37.3: 50 -> 11;  128 x 512 -> 10, p = 8: 65 -> 10
#include "fwd_engine.hpp"
#include "pow.hpp"
#include "skinny.hpp"

namespace ldist {
namespace {

constexpr int kRows = 64;    // of a stage: 16 per wave
constexpr int kCols = 64;

// IE = p - 1 for 1, 2, 3, 7 by multiplications, with the power of 1 / out taken into g where every output of the stage lies
// in [2^-12, 2^12] (norm_backward_kernel.hpp says why that is safe); IE = 0: any p > 1.  NB: outputs rounded up to four.
template <int NB, int IE>
__global__ void __launch_bounds__(256)
norm_backward_few_kernel(const float* __restrict__ grad_output, const float* __restrict__ input, const float* __restrict__ weight,
                         const float* __restrict__ output, float* __restrict__ grad_input, float* __restrict__ grad_weight, float e,
                         Dims d, int col_blocks, int rows_per_wg, int chunks) {
    __shared__ __align__(16) float cs[kRows][NB], rs[kRows][NB];
    __shared__ float sums[4][NB][kCols];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kb = blockIdx.x % col_blocks, rest = blockIdx.x / col_blocks, chunk = rest % chunks, g = rest / chunks;
    const int K = d.K, NG = d.NG, k = kb * kCols + lane, kc = min(k, K - 1);
    const int m_begin = chunk * rows_per_wg;
    int left = min(d.M - m_begin, rows_per_wg);   // rows to come: what is past them may have no number below 2^31
    const float ev = in_vgpr(e);
    auto spower = [&](float u) {
        if constexpr (IE == 0) return __builtin_copysignf(pow_pos(__builtin_fabsf(u), ev), u);
        else if constexpr (IE == 2) return u * __builtin_fabsf(u);
        else return pow_int<IE>(u);
    };
    float w[NB], gw[NB];
#pragma unroll
    for (int j = 0; j < NB; j++) {
        w[j] = weight[((size_t)g * NG + min(j, NG - 1)) * K + kc];
        gw[j] = 0.f;
    }
    for (int m0 = m_begin;; m0 += kRows) {
        const int rows = min(kRows, left), mine = wave * (kRows / 4);
        float x[kRows / 4];
#pragma unroll
        for (int r = 0; r < kRows / 4; r++) x[r] = input[((size_t)(m0 + min(mine + r, rows - 1)) * d.G + g) * K + kc];
        __syncthreads();   // the stage before is done with
        bool unsafe = false;
        for (int i = tid; i < kRows * NB; i += 256) {
            const int r = i / NB, j = i - r * NB;
            float c = 0.f, ri = 0.f;
            if (r < rows && j < NG) {
                const size_t at = ((size_t)(m0 + r) * d.G + g) * NG + j;
                const float out = output[at];
                c = grad_output[at];
                ri = __builtin_amdgcn_rcpf(out);
                unsafe |= !(out >= 0x1p-12f && out <= 0x1p12f);
            }
            cs[r][j] = c;
            rs[r][j] = ri;
        }
        const bool factored = !__syncthreads_or(unsafe) && IE > 0;
        if constexpr (IE > 0) {
            if (factored) {
                for (int i = tid; i < kRows * NB; i += 256) (&cs[0][0])[i] *= pow_int<IE>((&rs[0][0])[i]);
                __syncthreads();
            }
        }
        auto walk = [&](auto term) {
#pragma unroll
            for (int r = 0; r < kRows / 4; r++) {
                if (mine + r >= rows) break;
                float gi = 0.f;
#pragma unroll
                for (int j = 0; j < NB; j++) {
                    if (j > NB - 4 && j >= NG) break;
                    const float t = term(x[r] - w[j], mine + r, j);
                    gi += t;
                    gw[j] -= t;
                }
                if (k < K) grad_input[((size_t)(m0 + mine + r) * d.G + g) * K + k] = gi;
            }
        };
        if (factored) walk([&](float df, int r, int j) { return cs[r][j] * spower(df); });
        else walk([&](float df, int r, int j) { return cs[r][j] * spower(df * rs[r][j]); });
        if ((left -= kRows) <= 0) break;
    }
#pragma unroll
    for (int j = 0; j < NB; j++) sums[wave][j][lane] = gw[j];
    __syncthreads();
    if (k < K)
        for (int j = wave; j < NG; j += 4) {
            const float s = (sums[0][j][lane] + sums[1][j][lane]) + (sums[2][j][lane] + sums[3][j][lane]);
            float* const dst = grad_weight + ((size_t)g * NG + j) * K + k;
            if (chunks > 1) atomicAdd(dst, s);
            else *dst += s;
        }
}

template <int NB>
hipError_t launch_few(const float* grad_output, const float* input, const float* weight, const float* output, float* grad_input,
                      float* grad_weight, float p, const Problem& pr, hipStream_t stream) {
    const Dims d = make_dims(pr);
    const int col_blocks = (pr.K + kCols - 1) / kCols;
    // rows are shared out until there are four workgroups per CU; every share costs an atomic addition per weight
    const long all = d.M, want = 4L * pr.num_cu / ((long)col_blocks * pr.G), most = (all + kRows - 1) / kRows;
    long chunks = want < 1 ? 1 : want < most ? want : most;
    const int rows_per_wg = (int)((all + chunks * kRows - 1) / (chunks * kRows)) * kRows;   // below 2^31: chunks is 1 for few rows only
    chunks = (all + rows_per_wg - 1) / rows_per_wg;
    const unsigned grid = (unsigned)(col_blocks * chunks * pr.G);
#define LAUNCH(IE)                                                                                                            \
    hipLaunchKernelGGL((norm_backward_few_kernel<NB, IE>), dim3(grid), dim3(256), 0, stream, grad_output, input, weight, output,  \
                       grad_input, grad_weight, p - 1.0f, d, col_blocks, rows_per_wg, (int)chunks)
    switch (small_int_power(p - 1.0f)) {
        case 1: LAUNCH(1); break;
        case 2: LAUNCH(2); break;
        case 3: LAUNCH(3); break;
        case 7: LAUNCH(7); break;
        default: LAUNCH(0); break;
    }
#undef LAUNCH
    return hipGetLastError();
}

}  // namespace

// Every fully connected layer of up to 16 outputs per group, where the order of the sums is free; a launch has fewer than 2^32 lanes.
bool norm_backward_few_applicable(const Problem& pr) {
    return pr.HW == 1 && pr.NG <= kSkinnyMaxNG && g_tile_override < 0 && (long long)((pr.K + kCols - 1) / kCols) * pr.G < (1LL << 23);
}

hipError_t norm_backward_few(const float* grad_output, const float* input, const float* weight, const float* output,
                             float* grad_input, float* grad_weight, float p, const Problem& pr, hipStream_t stream) {
    if (pr.NG <= 4) return launch_few<4>(grad_output, input, weight, output, grad_input, grad_weight, p, pr, stream);
    if (pr.NG <= 8) return launch_few<8>(grad_output, input, weight, output, grad_input, grad_weight, p, pr, stream);
    if (pr.NG <= 12) return launch_few<12>(grad_output, input, weight, output, grad_input, grad_weight, p, pr, stream);
    return launch_few<16>(grad_output, input, weight, output, grad_input, grad_weight, p, pr, stream);
}

}  // namespace ldist
