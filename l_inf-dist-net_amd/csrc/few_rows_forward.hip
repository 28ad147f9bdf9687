// Forward kernels for fully connected layers with a handful of rows (serving one or a few inputs): bound by reading the
// weights once, so they go from memory into registers, never through LDS.
//
// A wave owns RM rows x four outputs (one or two rows: also one or two) and its 64 lanes split k, four consecutive k each per trip
// (a trip is 256 k): a lane loads the weight vectors and RM input vectors with 128-bit loads, the next trip's before the arithmetic of this one.
// The four waves of a workgroup take neighbouring outputs and read the same rows, which they find in the vector
// cache.  At the end the lanes' results meet through LDS: every wave writes its 4 * RM results of 64 lanes and two lanes
// take one output.  k past the end: the last vector of a row is moved back to end with the row, vectors beyond it
// repeat that one, which changes no maximum (sums blank the repeated values).
//
// Against tiles of rows x outputs (32 x 32 is the smallest of fwd_engine.hpp) nothing is computed for absent rows:
// 1 x 5120 -> 5120, values: 60 -> 27 us, of which 21 us are the 105 MB of weights at the rate of a large copy.
#include <cmath>

#include "quad_engine.hpp"
#include "fwd_engine.hpp"
#include "pow.hpp"
#include "skinny.hpp"

namespace ldist {

// Outputs per wave of one and two rows: as many as rows, or four.  Few of them make more waves, with five or three trips' loads
// in flight each: 1 x 5120 -> 5120, values, 17.4 -> 16.7 us; with four its 320 workgroups are 1.25 to a CU.  Four read the rows
// less often, and are better where they fill the CUs and where the rows are short.  Us, as many as rows / four:
//   1 x 5120 -> 1024 4.1 / 6.2, 1 x 3072 -> 4096 9.6 / 9.2, 1 x 800 -> 4096 3.5 / 3.2, -> 5120 3.9 / 3.7; with positions 5.0 / 6.1,
//   10.5 / 10.1, 4.5 / 3.8, 4.8 / 4.3; p = 37.3 7.9 / 12.0, 16.4 / 16.1, 5.8 / 5.0, 6.2 / 6.5
//   2 x 5120 -> 1024 6.3 / 7.3, 2 x 5120 -> 4096 16.2 / 14.1, 2 x 800 -> 5120 4.6 / 4.0; p = 37.3 15.6 / 18.1, 30.6 / 26.6, 9.0 / 8.8;
//   with positions 7.4 / 10.6, 14.9 / 18.8, 5.7 / 5.0
//   bounds, which read two inputs: 1 x 5120 -> 1024 7.0 / 7.9, -> 3000 12.3 / 11.6, 1 x 3072 -> 5120 12.5 / 12.0;
//   2 x 5120 -> 1024 11.8 / 11.1, 2 x 1000 -> 20000 18.5 / 14.8
constexpr int few_cols(int rows) { return rows <= 2 ? rows : 4; }
enum class FewKind { kValues, kPos, kNorm, kBounds };
static int cols_of(const Problem& pr, FewKind kind) {
    if (pr.B > 2) return 4;
    const double per_cu = (double)pr.NG * pr.G / (16.0 * pr.num_cu);   // workgroups, with four
    const bool enough = per_cu >= 0.7, full = per_cu >= 0.7 * std::ceil(per_cu), brief = pr.K < 2048;
    if (kind == FewKind::kBounds) return pr.B == 2 || enough ? 4 : 1;
    if (kind == FewKind::kPos && pr.B == 2) return per_cu > 1 && brief ? 4 : 2;
    return enough && (full || brief) ? 4 : pr.B;
}

typedef float FewF4 __attribute__((ext_vector_type(4)));

template <int RM, int NX, int COLS = few_cols(RM)>
struct FewRows {
    const float* xr[NX][RM];
    const float* wr[COLS];
    int K, lane, m0, n0, g;

    __device__ __forceinline__ FewRows(const float* const (&input)[NX], const float* weight, const Dims& d) {
        const int wave = threadIdx.x >> 6;
        lane = threadIdx.x & 63;
        K = d.K;
        int tm, tn;
        tile_of_block(d, tm, tn, g);
        m0 = tm * RM;
        n0 = (tn * 4 + wave) * COLS;
#pragma unroll
        for (int q = 0; q < NX; q++)
#pragma unroll
            for (int i = 0; i < RM; i++) xr[q][i] = input[q] + ((size_t)min(m0 + i, d.M - 1) * d.G + g) * K;
#pragma unroll
        for (int j = 0; j < COLS; j++) wr[j] = weight + ((size_t)g * d.NG + min(n0 + j, d.NG - 1)) * K;
    }
    __device__ __forceinline__ int trips() const { return (K + 255) / 256; }
    __device__ __forceinline__ int k_of(int trip) const { return trip * 256 + lane * 4; }
    struct Vecs { FewF4 x[NX][RM], w[COLS]; };
    __device__ __forceinline__ void load(Vecs& v, int trip) const {
        const int k = min(k_of(trip), K - 4);
#pragma unroll
        for (int j = 0; j < COLS; j++) v.w[j] = vec(wr[j] + k);
#pragma unroll
        for (int q = 0; q < NX; q++)
#pragma unroll
            for (int i = 0; i < RM; i++) v.x[q][i] = vec(xr[q][i] + k);
    }
    __device__ __forceinline__ static FewF4 vec(const float* p) {
        const float4_any a = *reinterpret_cast<const float4_any*>(p);
        return FewF4{a.v[0], a.v[1], a.v[2], a.v[3]};
    }
    // f(vectors, trip) for every trip, ascending.
    template <class F>
    __device__ __forceinline__ void walk(F&& f) const {
        const int n = trips();
        if constexpr (RM * NX >= 8) {   // enough loads in flight; a third wave per SIMD is worth more than the next trip's
#pragma unroll 1
            for (int t = 0; t < n; t++) {
                Vecs v;
                load(v, t);
                f(v, t);
            }
            return;
        }
        if constexpr (COLS <= 2) {
            constexpr int AHEAD = RM == 1 ? 5 : 3;
#pragma unroll 1
            for (int t = 0; t < n; t += AHEAD) {
                Vecs v[AHEAD];
#pragma unroll
                for (int c = 0; c < AHEAD; c++) load(v[c], min(t + c, n - 1));
#pragma unroll
                for (int c = 0; c < AHEAD; c++)
                    if (t + c < n) f(v[c], t + c);
            }
            return;
        }
        Vecs a, b;
        load(a, 0);
#pragma unroll 1
        for (int t = 0; t < n; t += 2) {
            load(b, min(t + 1, n - 1));
            f(a, t);
            if (t + 1 >= n) break;
            load(a, min(t + 2, n - 1));
            f(b, t + 1);
        }
    }
};

// Sets of 64 lanes' results, one per (row, output) of a wave: row o of `park` holds lane 0..63, padded so that two lanes
// per output read it in vectors.
constexpr int kFewPitch = 68;

// GATED: behind lists of outermost values, which may have left nothing to do; they are for larger batches than the forms of few
// rows.  Looking at the gate costs a launch without one 0.2 us.
// L_inf.  A lane keeps the trip in which its maximum was raised; (trip, lane) is the order of k.
template <int RM, bool POS, int COLS = few_cols(RM), bool GATED = false>
__global__ void __launch_bounds__(256, 3)
inf_forward_few_rows_kernel(const float* __restrict__ input, const float* __restrict__ weight, float* __restrict__ output,
                            int32_t* __restrict__ pos, Dims d) {
    constexpr int kFewCols = COLS, NO = RM * kFewCols;
    if constexpr (GATED) {
        if (gated_off(d)) return;
    }
    __shared__ float park[4][NO][kFewPitch];   // first the values, then the tags: both at once would cost a workgroup per CU
    const float* const ins[1] = {input};
    const FewRows<RM, 1, COLS> rows(ins, weight, d);
    const int wave = threadIdx.x >> 6, lane = rows.lane;
    float acc[RM][kFewCols];
    int trip[RM][kFewCols];
#pragma unroll
    for (int i = 0; i < RM; i++)
#pragma unroll
        for (int j = 0; j < kFewCols; j++) { acc[i][j] = 0.f; trip[i][j] = 0; }
    rows.walk([&](const typename FewRows<RM, 1, COLS>::Vecs& v, int t) {
#pragma unroll
        for (int i = 0; i < RM; i++)
#pragma unroll
            for (int j = 0; j < kFewCols; j++) {
                const FewF4 df = v.x[0][i] - v.w[j];
                float m = __builtin_fmaxf(__builtin_fmaxf(acc[i][j], __builtin_fabsf(df.x)), __builtin_fabsf(df.y));
                m = __builtin_fmaxf(__builtin_fmaxf(m, __builtin_fabsf(df.z)), __builtin_fabsf(df.w));
                if constexpr (POS) trip[i][j] = m > acc[i][j] ? t : trip[i][j];
                acc[i][j] = m;
            }
    });
    // only the wave itself reads what it wrote: no barrier, LDS operations of a wave stay in order
    const int o = lane >> 1, half = lane & 1;
    FewF4 vals[8];
#pragma unroll
    for (int i = 0; i < RM; i++)
#pragma unroll
        for (int j = 0; j < kFewCols; j++) park[wave][i * kFewCols + j][lane] = acc[i][j];
    __builtin_amdgcn_wave_barrier();
    float best = 0.f;
    int tag = 0x7fffffff;
#pragma unroll
    for (int q = 0; q < 8; q++) {
        vals[q] = *reinterpret_cast<const FewF4*>(&park[wave][o < NO ? o : 0][half * 32 + 4 * q]);
#pragma unroll
        for (int e = 0; e < 4; e++) best = __builtin_fmaxf(best, vals[q][e]);
    }
    if constexpr (POS) {
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int i = 0; i < RM; i++)
#pragma unroll
            for (int j = 0; j < kFewCols; j++) park[wave][i * kFewCols + j][lane] = __int_as_float(trip[i][j] * 64 + lane);
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int q = 0; q < 8; q++) {
            const int4 tg = *reinterpret_cast<const int4*>(&park[wave][o < NO ? o : 0][half * 32 + 4 * q]);
            const int ts[4] = {tg.x, tg.y, tg.z, tg.w};
#pragma unroll
            for (int e = 0; e < 4; e++) tag = vals[q][e] == best ? min(tag, ts[e]) : tag;
        }
    }
    const float ov = dpp_move<kDppSwap1, 0xF>(best, best);
    if constexpr (POS) {
        const int ot = dpp_move<kDppSwap1, 0xF>(tag, tag);
        tag = (ov > best || (ov == best && ot < tag)) ? ot : tag;
    }
    best = __builtin_fmaxf(best, ov);
    const int m = rows.m0 + o / kFewCols, n = rows.n0 + o % kFewCols;
    if (half == 0 && o < NO && m < d.M && n < d.NG) {
        const size_t at = ((size_t)m * d.G + rows.g) * d.NG + n;
        output[at] = shifted_value(d.mean, d.bias, rows.g * d.NG + n, best);
        if constexpr (POS) {
            int found = 0;
            if (best > 0.f) {
                const int kc = min((tag >> 6) * 256 + (tag & 63) * 4, d.K - 4);
                const FewF4 df = FewRows<RM, 1, COLS>::vec(input + ((size_t)m * d.G + rows.g) * d.K + kc) -
                                 FewRows<RM, 1, COLS>::vec(weight + ((size_t)rows.g * d.NG + n) * d.K + kc);
#pragma unroll
                for (int e = 3; e >= 0; e--)
                    if (__builtin_fabsf(df[e]) == best) found = (kc + e) | (__float_as_int(df[e]) & 0x80000000);
            }
            pos[at] = found;
        }
    }
}

// The lanes' values of every (row, output) of the wave reduced by op: lanes 2 * o and 2 * o + 1 return output o's.
template <int NO, class OP>
__device__ __forceinline__ float few_reduce(float (*park)[kFewPitch], const float* vals, int lane, float identity, OP&& op) {
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int o = 0; o < NO; o++) park[o][lane] = vals[o];
    __builtin_amdgcn_wave_barrier();
    const int o = lane >> 1, half = lane & 1;
    float r = identity;
    if (o < NO) {
#pragma unroll
        for (int q = 0; q < 8; q++) {
            const FewF4 v = *reinterpret_cast<const FewF4*>(&park[o][half * 32 + 4 * q]);
#pragma unroll
            for (int e = 0; e < 4; e++) r = op(r, v[e]);
        }
    }
    return op(r, dpp_move<kDppSwap1, 0xF>(r, r));
}

// Interval bounds: a trip whose vectors hold l > u, a NaN or an infinity takes the reference's literal predicate.
template <int RM, int COLS, bool GATED = false>
__global__ void __launch_bounds__(256, 3)
bound_forward_few_rows_kernel(const float* __restrict__ lower, const float* __restrict__ upper, const float* __restrict__ weight,
                              float* __restrict__ out_lower, float* __restrict__ out_upper, Dims d) {
    constexpr int kFewCols = COLS, NO = RM * kFewCols;
    if constexpr (GATED) {
        if (gated_off(d)) return;
    }
    __shared__ float park[4][NO][kFewPitch];
    const float* const ins[2] = {lower, upper};
    const FewRows<RM, 2, COLS> rows(ins, weight, d);
    const int wave = threadIdx.x >> 6, lane = rows.lane;
    float lo[NO], up[NO];
#pragma unroll
    for (int o = 0; o < NO; o++) { lo[o] = 0.f; up[o] = 0.f; }
    rows.walk([&](const typename FewRows<RM, 2, COLS>::Vecs& v, int t) {
        // 0 * v is NaN for a NaN or an infinity, and stays in the sum; u - l < 0 betrays l > u
        float zero = 0.f, width = 0.f;
#pragma unroll
        for (int e = 0; e < 4; e++) {
#pragma unroll
            for (int i = 0; i < RM; i++) {
                const float l = v.x[0][i][e], u = v.x[1][i][e];
                zero = __builtin_fmaf(u, 0.f, __builtin_fmaf(l, 0.f, zero));
                width = __builtin_fminf(width, u - l);
            }
#pragma unroll
            for (int j = 0; j < kFewCols; j++) zero = __builtin_fmaf(v.w[j][e], 0.f, zero);
        }
        if (__builtin_amdgcn_ballot_w64(!(zero == 0.f) || width < 0.f) == 0) {
#pragma unroll
            for (int i = 0; i < RM; i++)
#pragma unroll
                for (int j = 0; j < kFewCols; j++)
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const float tl = v.x[0][i][e] - v.w[j][e], tu = v.x[1][i][e] - v.w[j][e];
                        float &L = lo[i * kFewCols + j], &U = up[i * kFewCols + j];
                        U = __builtin_fmaxf(__builtin_fmaxf(U, __builtin_fabsf(tl)), __builtin_fabsf(tu));
                        L = __builtin_fmaxf(__builtin_fmaxf(L, tl), -tu);
                    }
        } else {   // rare: one k at a time, from memory again, so that it adds nothing to the registers of the other path
            const int k = min(rows.k_of(t), d.K - 4);
#pragma unroll 1
            for (int e = 0; e < 4; e++) {
                float w[kFewCols];
#pragma unroll
                for (int j = 0; j < kFewCols; j++) w[j] = rows.wr[j][k + e];
#pragma unroll
                for (int i = 0; i < RM; i++) {
                    const float xl = rows.xr[0][i][k + e], xu = rows.xr[1][i][k + e];
#pragma unroll
                    for (int j = 0; j < kFewCols; j++) {
                        const float tl = xl - w[j], tu = xu - w[j], al = __builtin_fabsf(tl), au = __builtin_fabsf(tu);
                        float &L = lo[i * kFewCols + j], &U = up[i * kFewCols + j];
                        U = __builtin_fmaxf(U, __builtin_fmaxf(al, au));
                        L = __builtin_fmaxf(L, (tl < 0.f && tu > 0.f) ? 0.f : __builtin_fminf(al, au));   // L >= 0
                    }
                }
            }
        }
    });
    auto larger = [](float a, float b) { return __builtin_fmaxf(a, b); };
    const float l = few_reduce<NO>(park[wave], lo, lane, 0.f, larger), u = few_reduce<NO>(park[wave], up, lane, 0.f, larger);
    const int o = lane >> 1, m = rows.m0 + o / kFewCols, n = rows.n0 + o % kFewCols;
    if ((lane & 1) == 0 && o < NO && m < d.M && n < d.NG) {
        const size_t at = ((size_t)m * d.G + rows.g) * d.NG + n;
        out_lower[at] = shifted_value(d.mean, d.bias, rows.g * d.NG + n, l);
        out_upper[at] = shifted_value(d.mean, d.bias, rows.g * d.NG + n, u);
    }
}

// p-norm, as norm_forward_quad_kernel: IP = 2, 3, 4, 8 one walk with the powers as they are, again the general way if a
// sum left [2^-90, 2^100]; IP = 0 a walk for the maxima and one for the sums (the second finds the weights in the caches).
template <int RM, int IP, int COLS = few_cols(RM)>
__global__ void __launch_bounds__(256, 3)
norm_forward_few_rows_kernel(const float* __restrict__ input, const float* __restrict__ weight, float* __restrict__ output,
                             float p, Dims d) {
    constexpr int kFewCols = COLS, NO = RM * kFewCols;
    __shared__ float park[4][NO][kFewPitch];
    const float* const ins[1] = {input};
    const FewRows<RM, 1, COLS> rows(ins, weight, d);
    using Vecs = typename FewRows<RM, 1, COLS>::Vecs;
    const int wave = threadIdx.x >> 6, lane = rows.lane;
    const float pv = in_vgpr(p);
    auto add = [](float a, float b) { return a + b; };
    auto larger = [](float a, float b) { return __builtin_fmaxf(a, b); };
    // the values of a vector that are this lane's own: all, but for the row's last vectors
    auto own = [&](int t, int e) { const int k = rows.k_of(t); return k <= d.K - 4 || (k < d.K && d.K - 4 + e >= k); };
    const bool ragged = d.K % 256 != 0;
    const int last = rows.trips() - 1;
    float acc[NO];
    float result = 0.f;
    bool general = IP == 0;
    if constexpr (IP > 0) {
#pragma unroll
        for (int o = 0; o < NO; o++) acc[o] = 0.f;
        rows.walk([&](const Vecs& v, int t) {
            float keep[4] = {1.f, 1.f, 1.f, 1.f};
            if (ragged && t == last)
#pragma unroll
                for (int e = 0; e < 4; e++) keep[e] = own(t, e) ? 1.f : 0.f;
#pragma unroll
            for (int i = 0; i < RM; i++)
#pragma unroll
                for (int j = 0; j < kFewCols; j++)
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const float df = v.x[0][i][e] - v.w[j][e];
                        const float term = IP % 2 == 0 ? pow_int<IP>(df) : pow_int<IP>(__builtin_fabsf(df));
                        acc[i * kFewCols + j] += keep[e] != 0.f ? term : 0.f;
                    }
        });
        const float sum = few_reduce<NO>(park[wave], acc, lane, 0.f, add);
        general = __builtin_amdgcn_ballot_w64((lane >> 1) < NO && !(sum > 0x1p-90f && sum < 0x1p100f)) != 0;
        const int e = ((int)((__float_as_uint(sum) >> 23) & 0xff) - 127) / IP;   // see norm_forward_quad_kernel
        result = __builtin_ldexpf(pow_pos(__builtin_ldexpf(sum, -e * IP), 1.0f / IP), e);
    }
    if (general) {
#pragma unroll
        for (int o = 0; o < NO; o++) acc[o] = 0.f;
        rows.walk([&](const Vecs& v, int) {
#pragma unroll
            for (int i = 0; i < RM; i++)
#pragma unroll
                for (int j = 0; j < kFewCols; j++) {
                    const FewF4 df = v.x[0][i] - v.w[j];
                    float& a = acc[i * kFewCols + j];
                    a = __builtin_fmaxf(__builtin_fmaxf(a, __builtin_fabsf(df.x)), __builtin_fabsf(df.y));
                    a = __builtin_fmaxf(__builtin_fmaxf(a, __builtin_fabsf(df.z)), __builtin_fabsf(df.w));
                }
        });
        const float mx = __builtin_fmaxf(few_reduce<NO>(park[wave], acc, lane, 0.f, larger), 1e-10f);
        __builtin_amdgcn_wave_barrier();
        if ((lane & 1) == 0 && (lane >> 1) < NO) park[wave][lane >> 1][0] = 1.0f / mx;
        __builtin_amdgcn_wave_barrier();
        float rs[NO];
#pragma unroll
        for (int o = 0; o < NO; o++) { rs[o] = park[wave][o][0]; acc[o] = 0.f; }
        rows.walk([&](const Vecs& v, int t) {
            float keep[4] = {1.f, 1.f, 1.f, 1.f};
            if (ragged && t == last)
#pragma unroll
                for (int e = 0; e < 4; e++) keep[e] = own(t, e) ? 1.f : 0.f;
#pragma unroll
            for (int i = 0; i < RM; i++)
#pragma unroll
                for (int j = 0; j < kFewCols; j++)
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const float term = pow_pos(__builtin_fabsf(v.x[0][i][e] - v.w[j][e]) * rs[i * kFewCols + j], pv);
                        acc[i * kFewCols + j] += keep[e] != 0.f ? term : 0.f;
                    }
        });
        const float sum = few_reduce<NO>(park[wave], acc, lane, 0.f, add) + 1e-10f * pow_pos(1e-10f / mx, pv);
        result = pow_pos(sum, 1.0f / p) * mx;
    }
    const int o = lane >> 1, m = rows.m0 + o / kFewCols, n = rows.n0 + o % kFewCols;
    if ((lane & 1) == 0 && o < NO && m < d.M && n < d.NG)
        output[((size_t)m * d.G + rows.g) * d.NG + n] = shifted_value(d.mean, d.bias, rows.g * d.NG + n, result);
}

static Dims few_dims(const Problem& pr, int rm, int cols) {
    Dims d = make_dims(pr);
    d.tiles_m = (d.M + rm - 1) / rm;
    d.tiles_n = (d.NG + 4 * cols - 1) / (4 * cols);
    return d;
}

#define FEW_LAUNCH(KERNEL, RM, COLS, ...)                                                                               \
    do {                                                                                                                \
        const Dims d = few_dims(pr, RM, COLS);                                                                          \
        hipLaunchKernelGGL(KERNEL, dim3((unsigned)d.tiles_m * d.tiles_n * d.G), dim3(256), 0, stream, __VA_ARGS__, d); \
        return hipGetLastError();                                                                                       \
    } while (0)

// ROWS rows with the outputs per wave of cols_of(); LAUNCH(cols) for either.
#define FEW_EITHER(ROWS, KIND, LAUNCH)                                       \
    if (pr.B == ROWS) {                                                      \
        if (cols_of(pr, KIND) == 4) LAUNCH(ROWS, 4); else LAUNCH(ROWS, few_cols(ROWS)); \
    }

hipError_t inf_forward_few_rows(const float* input, const float* weight, float* output, int32_t* pos, const Problem& pr,
                                hipStream_t stream) {
#define WITH_POS(RM, COLS) FEW_LAUNCH((inf_forward_few_rows_kernel<RM, true, COLS>), RM, COLS, input, weight, output, pos)
#define VALUES(RM, COLS) FEW_LAUNCH((inf_forward_few_rows_kernel<RM, false, COLS>), RM, COLS, input, weight, output, pos)
    if (pos) {
        FEW_EITHER(1, FewKind::kPos, WITH_POS)
        FEW_EITHER(2, FewKind::kPos, WITH_POS)
        if (pr.gate) FEW_LAUNCH((inf_forward_few_rows_kernel<8, true, 4, true>), 8, 4, input, weight, output, pos);
        if (pr.B <= 4) WITH_POS(4, 4);
        WITH_POS(8, 4);
    }
    FEW_EITHER(1, FewKind::kValues, VALUES)
    FEW_EITHER(2, FewKind::kValues, VALUES)
    if (pr.gate) FEW_LAUNCH((inf_forward_few_rows_kernel<8, false, 4, true>), 8, 4, input, weight, output, pos);
    if (pr.B <= 4) VALUES(4, 4);
    VALUES(8, 4);
#undef WITH_POS
#undef VALUES
}

hipError_t bound_forward_few_rows(const float* lower, const float* upper, const float* weight, float* out_lower, float* out_upper,
                                  const Problem& pr, hipStream_t stream) {
#define BOUNDS(RM, COLS) FEW_LAUNCH((bound_forward_few_rows_kernel<RM, COLS>), RM, COLS, lower, upper, weight, out_lower, out_upper)
    FEW_EITHER(1, FewKind::kBounds, BOUNDS)
    if (pr.B == 2) BOUNDS(2, 4);
    if (pr.gate) FEW_LAUNCH((bound_forward_few_rows_kernel<4, 4, true>), 4, 4, lower, upper, weight, out_lower, out_upper);
    BOUNDS(4, 4);
#undef BOUNDS
}

template <int IP>
static hipError_t norm_few_rows(const float* input, const float* weight, float* output, float p, const Problem& pr,
                                hipStream_t stream) {
#define NORM(RM, COLS) FEW_LAUNCH((norm_forward_few_rows_kernel<RM, IP, COLS>), RM, COLS, input, weight, output, p)
    FEW_EITHER(1, FewKind::kNorm, NORM)
    FEW_EITHER(2, FewKind::kNorm, NORM)
    if (pr.B <= 4) NORM(4, 4);
    NORM(8, 4);
#undef NORM
}

hipError_t norm_forward_few_rows(const float* input, const float* weight, float* output, float p, const Problem& pr,
                                 hipStream_t stream) {
    switch (small_int_power(p)) {
        case 2: return norm_few_rows<2>(input, weight, output, p, pr, stream);
        case 3: return norm_few_rows<3>(input, weight, output, p, pr, stream);
        case 4: return norm_few_rows<4>(input, weight, output, p, pr, stream);
        case 8: return norm_few_rows<8>(input, weight, output, p, pr, stream);
        default: return norm_few_rows<0>(input, weight, output, p, pr, stream);
    }
}

}  // namespace ldist
