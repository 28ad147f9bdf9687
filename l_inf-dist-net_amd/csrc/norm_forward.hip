// p-norm distance forward, p > 1:  out[m,n] = (sum_k |x[m,k] - w[n,k]|^p)^(1/p),
// evaluated as  mx * (sum_k (|x-w|/mx)^p)^(1/p)  with a running maximum mx so
// that no power can overflow for any p.  Semantics follow the reference kernel
// model/norm_dist_cuda.cu:228-292: mx and the sum are seeded with 1e-10 (:232-233),
// and whenever a block of k raises mx the sum is rescaled by (mx_old/mx_new)^p
// (:257-261).  Here the block is a 32-wide chunk.  Below p = 128 a chunk is normally
// swept once with the scale left by earlier chunks (see the kernel; a chunk that
// overflows is swept again the reference's way: maximum, rescale, powers);
// from p = 128 the kernel first
// finds the maxima over all of k and then takes only the powers that can matter
// (see MODE 2 in the kernel).  p = 2, 3, 4, 8 use multiplies only; any other p goes
// through v_log_f32 / v_exp_f32.
#include "norm_forward_kernel.hpp"
#include "skinny.hpp"

namespace ldist {

// Few outputs per group: two passes over k, first the exact maximum per (row, output),
// then the sum of (|x-w| / max)^p; lanes split k in both.
template <int RW, int NB, bool VEC>
__global__ void __launch_bounds__(256)
norm_forward_skinny_kernel(const float* __restrict__ input, const float* __restrict__ weight,
                           float* __restrict__ output, float p, Dims d) {
    __shared__ float red[4][RW * NB];
    __shared__ float bcast[RW * NB];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    SkinnyRows<RW> rows;
    rows.init(d);
    for (int nb = 0; nb < d.NG; nb += NB) {
        float acc[RW][NB], rmx[RW][NB];
        // pass 0: maximum; pass 1: power sum
        for (int pass = 0; pass < 2; pass++) {
#pragma unroll
            for (int r = 0; r < RW; r++)
#pragma unroll
                for (int j = 0; j < NB; j++) acc[r][j] = 0.f;
            const float* const ins[1] = {input};
            skinny_sweep<1, RW, NB, VEC>(ins, weight, rows, d, nb, tid, [&](int, const float (&xv)[1][RW], const float (&wv)[NB]) {
#pragma unroll
                for (int r = 0; r < RW; r++)
#pragma unroll
                    for (int j = 0; j < NB; j++) {
                        const float a = __builtin_fabsf(xv[0][r] - wv[j]);
                        if (pass == 0) acc[r][j] = __builtin_fmaxf(acc[r][j], a);
                        else acc[r][j] += pow_pos(a * rmx[r][j], p);
                    }
            });
#pragma unroll
            for (int r = 0; r < RW; r++)
#pragma unroll
                for (int j = 0; j < NB; j++) {
                    const float v = pass == 0 ? wave_max(acc[r][j]) : wave_sum(acc[r][j]);
                    if (lane == 63) red[wave][r * NB + j] = v;
                }
            __syncthreads();
            if (tid < RW * NB) {
                float v = red[0][tid];
#pragma unroll
                for (int q = 1; q < 4; q++) v = pass == 0 ? __builtin_fmaxf(v, red[q][tid]) : v + red[q][tid];
                if (pass == 0) {
                    bcast[tid] = __builtin_fmaxf(v, 1e-10f);   // the reference's seed for the maximum
                } else {
                    const float mx = bcast[tid];
                    const float sum = v + 1e-10f * pow_pos(1e-10f * __builtin_amdgcn_rcpf(mx), p);  // seeded sum
                    const int r = tid / NB, j = tid % NB;
                    if (rows.m0 + r < d.M && nb + j < d.NG)
                        output[rows.ooff[r] + (size_t)(nb + j) * d.HW] = shifted_value(d.mean, d.bias, rows.g * d.NG + nb + j, pow_pos(sum, 1.0f / p) * mx);
                }
            }
            __syncthreads();
            if (pass == 0) {
#pragma unroll
                for (int r = 0; r < RW; r++)
#pragma unroll
                    for (int j = 0; j < NB; j++) rmx[r][j] = __builtin_amdgcn_rcpf(bcast[r * NB + j]);
            }
            __syncthreads();
        }
    }
}

// The fc layout alone (launch_forward names both layouts).
template <class GEO, bool CONV, int VEC>
struct NormForwardColumns {
    static hipError_t launch(unsigned grid, const Dims& d, int device, hipStream_t stream, const float* input,
                             const float* weight, float* output, float p) {
        if constexpr (!CONV) return NormForwardLaunch<GEO, false, VEC, false>::launch(grid, d, device, stream, input, weight, output, p, ImgWin{});
        else return hipErrorInvalidValue;
    }
};

template <class GEO, bool CONV, int VEC>
struct NormForward {
    static hipError_t launch(unsigned grid, const Dims& d, int device, hipStream_t stream, const float* input,
                             const float* weight, float* output, float p) {
        return NormForwardLaunch<GEO, CONV, VEC, false>::launch(grid, d, device, stream, input, weight, output, p, ImgWin{});
    }
};

// Fully connected layers that choose_tile gives tiles of 32 x 32 with eight k-groups (the 128-row tiles would leave the
// device idle): the same eight k-groups, hence the same order of summation, on the tile whose shares load the busiest CU
// least; a CU runs one workgroup of eight waves at a time.  32 x 40: 64 x 5120 -> 5120 is 256 tiles instead of 320, 280 ->
// 189 us at p = 8, 602 -> 386 at p = 37.3.  16 x 32 with two rows per lane: 128 x 12288 -> 512 is 128 tiles instead of 64,
// 290 -> 184 us and 684 -> 369; 100 x 1024 -> 1024 43 -> 27 and 84 -> 48.  A lane of the latter reads six LDS words for
// eight differences instead of eight for sixteen, hence the surcharge.  16 x 16 with two rows and columns: a wave per k-group, so
// that two waves per SIMD stay on every CU where 16 x 32 is 128 workgroups: 128 x 16384 -> 512 237 -> 142 us at p = 8, 489 -> 279
// at p = 37.3, 533 -> 278 at 300; 64 x 3072 -> 1024 54 -> 33; 16 x 784 -> 1024 25 -> 16.  It reads four LDS words for four
// differences, which shows in several rounds of tiles: three of them against one of 32 x 32, 64 x 5120 -> 3072, 134 -> 147 us at
// p = 8, 87 -> 105 at 2, but 303 -> 281 at 37.3 and 404 -> 388 at 300; five against three of 16 x 32, 80 x 4096 -> 4096, 200 -> 202 at
// p = 8, 399 -> 384 at 37.3.  So its price depends on what a difference costs: 1.5 where a power is a few multiplications, 1.3
// where it is a logarithm and an exponential, unless the reduction is short or its loads are single words (64 x 511 -> 3072, p = 37.3,
// three rounds 3 % slower).
template <class GEO>
static hipError_t launch_eight_groups(const Problem& pr, hipStream_t stream, const float* input, const float* weight,
                                      float* output, float p) {
    return launch_forward<NormForwardColumns, GEO>(pr, can_vec4(pr, input, weight), can_vec4_out(pr, output), stream, input,
                                                   weight, output, p);
}

enum class EightGroups { k32x32, k32x40, k16x32, k16x16 };
static EightGroups eight_groups_tile(const Problem& pr, float p, bool vec) {
    auto cost = [&](int bm, int bn, double price) {
        const long tiles = (long)((pr.B + bm - 1) / bm) * ((pr.NG + bn - 1) / bn) * pr.G;
        return (double)((tiles + pr.num_cu - 1) / pr.num_cu) * bm * bn * price;
    };
    const bool dear = small_int_power(p) == 0 || small_int_power(p) == 7;   // the exponents without an instantiation of their own
    const double square = cost(32, 32, 1.0), wide = cost(32, 40, 1.0), flat = cost(16, 32, 1.1);
    const double small = cost(16, 16, dear && vec && pr.K >= 512 ? 1.3 : 1.5);
    if (small < square && small < wide && small < flat) return EightGroups::k16x16;
    if (wide < square && wide <= flat) return EightGroups::k32x40;
    return flat < square ? EightGroups::k16x32 : EightGroups::k32x32;
}

static hipError_t norm_forward_eight_groups(const float* input, const float* weight, float* output, float p, const Problem& pr,
                                            hipStream_t stream) {
    switch (eight_groups_tile(pr, p, can_vec4(pr, input, weight))) {
        case EightGroups::k16x16: return launch_eight_groups<Geo<16, 16, 2, 2, 8>>(pr, stream, input, weight, output, p);
        case EightGroups::k32x40: return launch_eight_groups<Geo<32, 40, 4, 5, 8>>(pr, stream, input, weight, output, p);
        case EightGroups::k16x32: return launch_eight_groups<Geo<16, 32, 2, 4, 8>>(pr, stream, input, weight, output, p);
        default: return launch_eight_groups<Geo<32, 32, 4, 4, 8>>(pr, stream, input, weight, output, p);
    }
}

int norm_forward_tile(const Problem& pr, float p) {
    if (pr.NG <= kSkinnyMaxNG || pr.HW != 1 || g_tile_override >= 0) return 0;
    if (choose_tile(pr.B, pr.NG, pr.G, pr.num_cu) != TileChoice::M32N32K8) return 0;
    switch (eight_groups_tile(pr, p, pr.K % 4 == 0)) {
        case EightGroups::k16x16: return 16016;
        case EightGroups::k32x40: return 32040;
        case EightGroups::k16x32: return 16032;
        default: return 32032;
    }
}

bool norm_forward_shifts(const Problem& pr, float p) {
    return pr.HW == 1 && (pr.NG <= kSkinnyMaxNG || small_forward_tile(pr, ForwardKind::kNorm, p) >= 0);
}

// `values_only`: no gradient follows.  Such a pass may sum in any order and takes whichever kernel is fastest for the
// size.  A forward pass that trains keeps the order of summation it has always had (chunks of 32 k, alternating between
// the k-groups of the tile that fits the size): the batch-mean shift behind a layer of nearly equal distances leaves small
// differences of large numbers, and one unit in the last place of the distances was seen a thousand times as large in the
// gradients of a five-layer net.  The bits of general exponents below 128 depend on the tile all the same: its first stage gives the
// unit that its logarithms are taken in.
hipError_t norm_forward(const float* input, const float* weight, float* output, float p, const Problem& pr,
                        bool values_only, hipStream_t stream) {
    if (pr.NG <= kSkinnyMaxNG && values_only && few_rows_of_few_outputs(pr, true, small_int_power(p) < 2 || small_int_power(p) == 7))
        return norm_forward_few_rows(input, weight, output, p, pr, stream);
    if (pr.NG <= kSkinnyMaxNG) {
        const Dims d = make_dims(pr);
        const bool vec = pr.HW == 1 && pr.K % 4 == 0 && aligned16(input) && aligned16(weight);
#define LDIST_LAUNCH_RW(RW, NB, VEC)                                                                                        \
    hipLaunchKernelGGL((norm_forward_skinny_kernel<RW, NB, VEC>), dim3(skinny_grid(d, RW)), dim3(256), 0, stream, input, \
                       weight, output, p, d)
        // two rows per workgroup share the weight loads; with few rows (up to eight per CU) one each: more workgroups hide more latency
#define LDIST_LAUNCH_1(NB, VEC) LDIST_LAUNCH_RW(1, NB, VEC)
#define LDIST_LAUNCH_2(NB, VEC) LDIST_LAUNCH_RW(2, NB, VEC)
        if ((long)d.M * d.G <= 8L * pr.num_cu) LDIST_SKINNY_DISPATCH(pr.NG, vec, LDIST_LAUNCH_1);
        else LDIST_SKINNY_DISPATCH(pr.NG, vec, LDIST_LAUNCH_2);
#undef LDIST_LAUNCH_1
#undef LDIST_LAUNCH_2
#undef LDIST_LAUNCH_RW
        return hipGetLastError();
    }
    if (const int tile = values_only || g_tile_override >= 10 ? small_forward_tile(pr, ForwardKind::kNorm, p) : -1; tile >= 0)
        return norm_forward_small(input, weight, output, p, pr, tile, stream);
    if (pr.HW == 1 && g_tile_override < 0 && choose_tile(pr.B, pr.NG, pr.G, pr.num_cu) == TileChoice::M32N32K8)
        return norm_forward_eight_groups(input, weight, output, p, pr, stream);
    return dispatch_forward<NormForward>(pr, can_vec4(pr, input, weight), can_vec4_out(pr, output), stream, input,
                                         weight, output, p);
}

}  // namespace ldist
