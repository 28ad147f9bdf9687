// Forward kernels for fully connected layers whose tiles of fwd_engine.hpp would leave CUs idle (quad_engine.hpp says
// how they are built): the L_inf forward with and without pos and the interval bounds.  Same subtractions and maxima of
// the same numbers as inf_forward.hip and bound_forward.hip, so values, indices and bounds are the same bits.
#include "quad_engine.hpp"
#include "fwd_engine.hpp"
#include "pow.hpp"

#include <cmath>

namespace ldist {

// Tile -> global from LDS, four outputs per store where the tensor allows it.
template <class GEO, class T>
__device__ __forceinline__ void q_store_tile(T* __restrict__ dst, const T* cand, const Dims& d, int m0, int n0, int g, int tid) {
    using V4 = typename std::conditional<std::is_same<T, float>::value, float4, int4>::type;
    for (int q = tid; q < GEO::BM * GEO::BN / 4; q += GEO::NT) {
        const int ml = q / (GEO::BN / 4), nl = (q % (GEO::BN / 4)) * 4;
        const int m = m0 + ml, n = n0 + nl;
        if (m >= d.M || n >= d.NG) continue;
        T* at = dst + ((size_t)m * d.G + g) * d.NG + n;
        const T* from = cand + ml * GEO::BN + nl;
        if constexpr (std::is_same<T, float>::value) {
            if (d.mean || d.bias) {
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; e++) v[e] = shifted_value(d.mean, d.bias, g * d.NG + min(n + e, d.NG - 1), from[e]);
                if (d.ovec && n + 3 < d.NG) {
                    *reinterpret_cast<float4*>(at) = make_float4(v[0], v[1], v[2], v[3]);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        if (n + e < d.NG) at[e] = v[e];
                }
                continue;
            }
        }
        if (d.ovec && n + 3 < d.NG) {
            *reinterpret_cast<V4*>(at) = *reinterpret_cast<const V4*>(from);
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (n + e < d.NG) at[e] = from[e];
        }
    }
}

// L_inf forward.  POS: the loop asks once per 32 k of a k-group (REC stages) whether the running maximum moved and
// keeps the number of that record; after the k-groups have met, the 32 k of the winning record and group are looked at
// again.  Two groups may reach the same maximum inside the same record; then which holds the lower k is not known and
// the whole record, all groups, is searched in order.
template <class GEO, bool POS>
__global__ void __launch_bounds__(GEO::NT, GEO::TN == 4 ? 3 : 2)
inf_forward_quad_kernel(const float* __restrict__ input, const float* __restrict__ weight, float* __restrict__ output,
                        int32_t* __restrict__ pos, Dims d) {
    constexpr int TM = GEO::TM, TN = GEO::TN, KK = GEO::KK, NGRP = GEO::NGRP;
    constexpr int REC = GEO::CH >= 32 ? 1 : 32 / GEO::CH;   // stages per record
    constexpr int ANY = 63;                                 // in a tag: several groups hold the maximum
    using Stage = QStager<GEO, 1>;
    extern __shared__ __align__(16) float lds[];
    if (gated_off(d)) return;
    int tm, tn, g;
    tile_of_block(d, tm, tn, g);
    const int m0 = tm * GEO::BM, n0 = tn * GEO::BN;
    const int tid = threadIdx.x, grp = tid / NGRP, t = tid % NGRP, tx = t % GEO::TX, ty = t / GEO::TX;

    Stage st;
    const float* const ins[1] = {input};
    st.init(ins, weight, d, m0, n0, g, tid);
    float acc[TM][TN], prev[POS ? TM : 1][TN];
    int rec[POS ? TM : 1][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) {
            acc[i][j] = 0.f;
            if constexpr (POS) { prev[i][j] = 0.f; rec[i][j] = 0; }
        }

    const int nstage = (d.K + KK - 1) / KK;
    st.load(lds, 0);
    st.arrived();
    __syncthreads();
    for (int s = 0; s < nstage; s++) {
        if (s + 1 < nstage) st.load(lds + ((s + 1) & 1) * Stage::STAGE, (s + 1) * KK);
        q_sweep<GEO, 1>(lds + (s & 1) * Stage::STAGE, q_vectors<GEO>(s, nstage, d.K, grp), grp, tx, ty, [&](const QFrag<GEO, 1>& f) {
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    const float d0 = __builtin_fabsf(f.x[0][i].x - f.w[j].x), d1 = __builtin_fabsf(f.x[0][i].y - f.w[j].y);
                    const float d2 = __builtin_fabsf(f.x[0][i].z - f.w[j].z), d3 = __builtin_fabsf(f.x[0][i].w - f.w[j].w);
                    acc[i][j] = __builtin_fmaxf(__builtin_fmaxf(acc[i][j], d0), d1);
                    acc[i][j] = __builtin_fmaxf(__builtin_fmaxf(acc[i][j], d2), d3);
                }
        });
        if constexpr (POS) {
            if (s % REC == REC - 1 || s + 1 == nstage) {
                const int r = s / REC;
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < TN; j++) {
                        rec[i][j] = acc[i][j] > prev[i][j] ? r : rec[i][j];
                        prev[i][j] = acc[i][j];
                    }
            }
        }
        st.arrived();
        __syncthreads();
    }

    // the k-groups meet; tag = record * 64 + group
    float* pv = lds;                                                             // [KS/2][TM*TN][NGRP]
    int* pt = reinterpret_cast<int*>(lds) + GEO::KS / 2 * TM * TN * NGRP;
    if constexpr (POS) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) rec[i][j] = rec[i][j] * 64 + grp;
    }
    q_merge<GEO>(grp,
        [&](int slot) {
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    const int o = (slot * TM * TN + i * TN + j) * NGRP + t;
                    pv[o] = acc[i][j];
                    if constexpr (POS) pt[o] = rec[i][j];
                }
        },
        [&](int slot) {
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    const int o = (slot * TM * TN + i * TN + j) * NGRP + t;
                    const float v = pv[o];
                    if constexpr (POS) {
                        const int tag = pt[o], mine = rec[i][j];
                        const bool tie = v == acc[i][j];
                        const int both = (tag >> 6) == (mine >> 6) ? (mine | ANY) : (tag >> 6) < (mine >> 6) ? tag : mine;
                        rec[i][j] = v > acc[i][j] ? tag : tie ? both : mine;
                    }
                    acc[i][j] = __builtin_fmaxf(acc[i][j], v);
                }
        });
    __syncthreads();
    float* cand_v = lds;
    int* cand_t = reinterpret_cast<int*>(lds) + GEO::BM * GEO::BN;
    if (grp == 0) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const int o = GEO::row(ty, i) * GEO::BN + GEO::col(tx, j);
                cand_v[o] = acc[i][j];
                if constexpr (POS) cand_t[o] = rec[i][j];
            }
    }
    __syncthreads();

    if constexpr (POS) {
        // LPO neighbouring lanes take one output, one stage of the record each (ascending k).
        constexpr int LPO = REC, STEP = GEO::NT / LPO;
        const int sub = tid % LPO, shift = (tid & 63) - sub;
        for (int base = 0; base < GEO::BM * GEO::BN; base += STEP) {
            const int o = base + tid / LPO;
            const bool live = o < GEO::BM * GEO::BN;
            const int oc = live ? o : 0, m = min(m0 + oc / GEO::BN, d.M - 1), n = min(n0 + oc % GEO::BN, d.NG - 1);
            const float* xr = input + ((size_t)m * d.G + g) * d.K;
            const float* wr = weight + ((size_t)g * d.NG + n) * d.K;
            const float target = cand_v[oc];
            const int tag = cand_t[oc];
            const int k0 = ((tag >> 6) * REC + sub) * KK, grp1 = tag & ANY;
            int found = -1;
            auto look = [&](int k) {   // the four k of one vector; the last vector of a row is the one that ends with it
                const int kc = min(k, d.K - 4);
                const float4_any a = *reinterpret_cast<const float4_any*>(xr + kc), b = *reinterpret_cast<const float4_any*>(wr + kc);
#pragma unroll
                for (int e = 3; e >= 0; e--) {
                    const float df = a.v[e] - b.v[e];
                    if (__builtin_fabsf(df) == target) found = (kc + e) | (__float_as_int(df) & 0x80000000);
                }
            };
            if (live && target > 0.f && k0 < d.K) {
                if (grp1 != ANY) {
#pragma unroll
                    for (int q = GEO::QG - 1; q >= 0; q--) look(k0 + grp1 * GEO::CH + 4 * q);   // descending: the lowest stays
                } else {
                    for (int q = min(GEO::QR, (d.K - k0 + 3) / 4) - 1; q >= 0; q--) look(k0 + 4 * q);
                }
            }
            const bool hit = found != -1;
            const unsigned mine = (unsigned)(__builtin_amdgcn_ballot_w64(hit) >> shift) & ((1u << LPO) - 1u);
            if (live) {
                if (hit && (mine & ((1u << sub) - 1u)) == 0) cand_t[o] = found;
                if (sub == 0 && mine == 0) cand_t[o] = 0;
            }
        }
        __syncthreads();
        q_store_tile<GEO>(pos, cand_t, d, m0, n0, g, tid);
    }
    q_store_tile<GEO>(output, cand_v, d, m0, n0, g, tid);
}

// Interval bounds: the arithmetic of bound_forward.hip (regular boxes; a stage that holds an irregular value anywhere
// is reduced with the reference's literal predicate).
template <class GEO>
__global__ void __launch_bounds__(GEO::NT, GEO::TN == 4 ? 3 : 2)
bound_forward_quad_kernel(const float* __restrict__ lower, const float* __restrict__ upper, const float* __restrict__ weight,
                          float* __restrict__ out_lower, float* __restrict__ out_upper, Dims d) {
    constexpr int TM = GEO::TM, TN = GEO::TN, KK = GEO::KK, NGRP = GEO::NGRP;
    using Stage = QStager<GEO, 2>;
    extern __shared__ __align__(16) float lds[];
    if (gated_off(d)) return;
    int tm, tn, g;
    tile_of_block(d, tm, tn, g);
    const int m0 = tm * GEO::BM, n0 = tn * GEO::BN;
    const int tid = threadIdx.x, grp = tid / NGRP, t = tid % NGRP, tx = t % GEO::TX, ty = t / GEO::TX;
    Stage st;
    const float* const ins[2] = {lower, upper};
    st.init(ins, weight, d, m0, n0, g, tid);
    float lo[TM][TN], up[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) { lo[i][j] = 0.f; up[i][j] = 0.f; }
    // Whether the vectors this lane has fetched of a stage hold l > u, a NaN or an infinity (the panels of l and u have
    // the same layout, so it holds both ends of an interval); looked at as soon as they are in LDS.  vote[stage % 3]
    // carries the answer over the barrier that ends the stage before; the slot two stages ahead is cleared behind it.
    __shared__ int vote[3];
    auto look_at = [&](const float* stage, int s) {
        typedef float F4 __attribute__((ext_vector_type(4)));
        constexpr float INF = __builtin_inff();
        bool bad = false;
#pragma unroll
        for (int i = 0; i < (GEO::BM * GEO::QR + GEO::NT - 1) / GEO::NT; i++) {
            const int at = i * GEO::NT + tid;
            if (GEO::BM * GEO::QR % GEO::NT != 0 && at >= GEO::BM * GEO::QR) continue;
            const F4 l = *reinterpret_cast<const F4*>(stage + 4 * at), u = *reinterpret_cast<const F4*>(stage + Stage::XS + 4 * at);
#pragma unroll
            for (int e = 0; e < 4; e++) bad |= !(l[e] <= u[e] && __builtin_fabsf(l[e]) < INF && __builtin_fabsf(u[e]) < INF);
        }
#pragma unroll
        for (int i = 0; i < (GEO::BN * GEO::QR + GEO::NT - 1) / GEO::NT; i++) {
            const int at = i * GEO::NT + tid;
            if (GEO::BN * GEO::QR % GEO::NT != 0 && at >= GEO::BN * GEO::QR) continue;
            const F4 v = *reinterpret_cast<const F4*>(stage + 2 * Stage::XS + 4 * at);
#pragma unroll
            for (int e = 0; e < 4; e++) bad |= !(__builtin_fabsf(v[e]) < INF);
        }
        if (__builtin_amdgcn_ballot_w64(bad) != 0) vote[s % 3] = 1;
    };
    const int nstage = (d.K + KK - 1) / KK;
    st.load(lds, 0);
    if (tid < 3) vote[tid] = 0;
    __syncthreads();
    st.arrived();
    look_at(lds, 0);
    __syncthreads();
    for (int s = 0; s < nstage; s++) {
        if (s + 1 < nstage) st.load(lds + ((s + 1) & 1) * Stage::STAGE, (s + 1) * KK);
        const float* stage = lds + (s & 1) * Stage::STAGE;
        const int irregular = vote[s % 3], vectors = q_vectors<GEO>(s, nstage, d.K, grp);
        if (tid == 0) vote[(s + 2) % 3] = 0;
        if (!irregular) {
            q_sweep<GEO, 2>(stage, vectors, grp, tx, ty, [&](const QFrag<GEO, 2>& f) {
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < TN; j++)
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            const float tl = f.x[0][i][e] - f.w[j][e], tu = f.x[1][i][e] - f.w[j][e];
                            up[i][j] = __builtin_fmaxf(__builtin_fmaxf(up[i][j], __builtin_fabsf(tl)), __builtin_fabsf(tu));
                            lo[i][j] = __builtin_fmaxf(__builtin_fmaxf(lo[i][j], tl), -tu);
                        }
            });
        } else {
            q_sweep_plain<GEO, 2>(stage, vectors, grp, tx, ty, [&](const float (&x)[2][TM], const float (&w)[TN]) {
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < TN; j++) {
                        const float tl = x[0][i] - w[j], tu = x[1][i] - w[j];
                        const float al = __builtin_fabsf(tl), au = __builtin_fabsf(tu);
                        up[i][j] = __builtin_fmaxf(up[i][j], __builtin_fmaxf(al, au));
                        if (!(tl < 0.f && tu > 0.f)) lo[i][j] = __builtin_fmaxf(lo[i][j], __builtin_fminf(al, au));
                    }
            });
        }
        if (s + 1 < nstage) {
            st.arrived();
            look_at(lds + ((s + 1) & 1) * Stage::STAGE, s + 1);
        }
        __syncthreads();
    }
    float* pl = lds;
    float* pu = lds + GEO::KS / 2 * TM * TN * NGRP;
    q_merge<GEO>(grp,
        [&](int slot) {
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    const int o = (slot * TM * TN + i * TN + j) * NGRP + t;
                    pl[o] = lo[i][j];
                    pu[o] = up[i][j];
                }
        },
        [&](int slot) {
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    const int o = (slot * TM * TN + i * TN + j) * NGRP + t;
                    lo[i][j] = __builtin_fmaxf(lo[i][j], pl[o]);
                    up[i][j] = __builtin_fmaxf(up[i][j], pu[o]);
                }
        });
    __syncthreads();
    float* cl = lds;
    float* cu = lds + GEO::BM * GEO::BN;
    if (grp == 0) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const int o = GEO::row(ty, i) * GEO::BN + GEO::col(tx, j);
                cl[o] = lo[i][j];
                cu[o] = up[i][j];
            }
    }
    __syncthreads();
    q_store_tile<GEO>(out_lower, cl, d, m0, n0, g, tid);
    q_store_tile<GEO>(out_upper, cu, d, m0, n0, g, tid);
}

// p-norm: out = (sum_k |x-w|^p)^(1/p).
// General exponents (IP == 0) walk k twice: the first walk finds every output's maximum mx, the second adds
// (|x-w| / mx)^p, so no power can overflow and every term that counts is near 1.  SPARSE (large p): as in
// norm_forward_kernel.hpp, the second walk takes a row's powers only where one of them is above 2^-32.
// IP = 2, 3, 4, 8: one walk adds the powers as they are, by multiplications only; the tile is walked again the general
// way when one of its sums has left [2^-90, 2^100], where float powers would lose terms or overflow.
// The seeds (1e-10 for maximum and sum) are the reference's (model/norm_dist_cuda.cu:232-233).
// Scratch per lane, as the compiler reports it: the SPARSE instances 156 to 300 bytes, on every tile; IP = 2, 3, 4, 8 on
// 32 x 64 and 16 x 32 28 and 32 bytes under the bound of three waves per SIMD; the others none.
template <class GEO, int IP, bool SPARSE>
__global__ void __launch_bounds__(GEO::NT, GEO::TN == 4 ? 3 : 2)
norm_forward_quad_kernel(const float* __restrict__ input, const float* __restrict__ weight, float* __restrict__ output, float p,
                         Dims d) {
    constexpr int TM = GEO::TM, TN = GEO::TN, KK = GEO::KK, NGRP = GEO::NGRP;
    using Stage = QStager<GEO, 1>;
    extern __shared__ __align__(16) float lds[];
    __shared__ int outside;
    int tm, tn, g;
    tile_of_block(d, tm, tn, g);
    const int m0 = tm * GEO::BM, n0 = tn * GEO::BN;
    const int tid = threadIdx.x, grp = tid / NGRP, t = tid % NGRP, tx = t % GEO::TX, ty = t / GEO::TX;
    const float pv = in_vgpr(p);
    Stage st;
    const float* const ins[1] = {input};
    st.init(ins, weight, d, m0, n0, g, tid);
    const int nstage = (d.K + KK - 1) / KK;
    const bool ragged = d.K % KK != 0;
    if (tid == 0) outside = 0;

    // Calls f(frag) for every vector of every stage.  The last stage of a ragged K is blanked: zero differences add
    // nothing (and raise no maximum).
    auto walk = [&](auto&& f) {
        st.load(lds, 0);
        for (int s = 0; s < nstage; s++) {
            float* stage = lds + (s & 1) * Stage::STAGE;
            st.arrived();
            if (ragged && s + 1 == nstage) st.blank(stage, s * KK);
            __syncthreads();                       // the stage is there, and everybody has left the one before
            if (s + 1 < nstage) st.load(lds + ((s + 1) & 1) * Stage::STAGE, (s + 1) * KK);
            q_sweep<GEO, 1>(stage, q_vectors<GEO>(s, nstage, d.K, grp), grp, tx, ty, f);
        }
        __syncthreads();
    };
    float acc[TM][TN], rs[TM][TN];   // sums; reciprocals of the scales (first the maxima)
    auto clear = [&](float (&v)[TM][TN]) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) v[i][j] = 0.f;
    };
    // Joins the k-groups' values in group 0.
    auto join = [&](float (&v)[TM][TN], auto&& op) {
        q_merge<GEO>(grp,
            [&](int slot) {
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < TN; j++) lds[(slot * TM * TN + i * TN + j) * NGRP + t] = v[i][j];
            },
            [&](int slot) {
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < TN; j++) v[i][j] = op(v[i][j], lds[(slot * TM * TN + i * TN + j) * NGRP + t]);
            });
    };
    auto add = [](float a, float b) { return a + b; };
    auto larger = [](float a, float b) { return __builtin_fmaxf(a, b); };

    clear(acc);
    bool general = IP == 0;
    if constexpr (IP > 0) {
        walk([&](const QFrag<GEO, 1>& f) {
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++)
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const float df = f.x[0][i][e] - f.w[j][e];
                        acc[i][j] += IP % 2 == 0 ? pow_int<IP>(df) : pow_int<IP>(__builtin_fabsf(df));
                    }
        });
        join(acc, add);
        if (grp == 0) {
            bool out_of_range = false;
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) out_of_range |= !(acc[i][j] > 0x1p-90f && acc[i][j] < 0x1p100f);
            if (out_of_range) outside = 1;
        }
        __syncthreads();
        general = outside != 0;
        if (!general) {
            // sum^(1/p) with the sum brought near 1 by an exact power of 2^p first: the logarithm of a large or small
            // number would carry its rounding, times the number's exponent, into the result
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    const int e = ((int)((__float_as_uint(acc[i][j]) >> 23) & 0xff) - 127) / IP;
                    acc[i][j] = __builtin_ldexpf(pow_pos(__builtin_ldexpf(acc[i][j], -e * IP), 1.0f / IP), e);
                }
        }
    }
    if (general) {
        clear(rs);
        walk([&](const QFrag<GEO, 1>& f) {
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    const float d0 = __builtin_fabsf(f.x[0][i].x - f.w[j].x), d1 = __builtin_fabsf(f.x[0][i].y - f.w[j].y);
                    const float d2 = __builtin_fabsf(f.x[0][i].z - f.w[j].z), d3 = __builtin_fabsf(f.x[0][i].w - f.w[j].w);
                    rs[i][j] = __builtin_fmaxf(__builtin_fmaxf(rs[i][j], d0), d1);
                    rs[i][j] = __builtin_fmaxf(__builtin_fmaxf(rs[i][j], d2), d3);
                }
        });
        join(rs, larger);
        __syncthreads();
        if (grp == 0) {
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) lds[(i * TN + j) * NGRP + t] = __builtin_fmaxf(rs[i][j], 1e-10f);
        }
        __syncthreads();
        float cut = __builtin_exp2f(-32.0f / p);
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const float mx = lds[(i * TN + j) * NGRP + t];
                if (!(mx > 1e-10f)) cut = -1.f;   // on the seed scale nothing is negligible
                rs[i][j] = 1.0f / mx;
                acc[i][j] = grp == 0 ? 1e-10f * pow_pos(1e-10f * rs[i][j], pv) : 0.f;
            }
        __syncthreads();
        walk([&](const QFrag<GEO, 1>& f) {
            if constexpr (SPARSE) {
                float top[TM], all = 0.f;
#pragma unroll
                for (int i = 0; i < TM; i++) {
                    top[i] = 0.f;
#pragma unroll
                    for (int j = 0; j < TN; j++) {
                        const float u0 = __builtin_fabsf(f.x[0][i].x - f.w[j].x), u1 = __builtin_fabsf(f.x[0][i].y - f.w[j].y);
                        const float u2 = __builtin_fabsf(f.x[0][i].z - f.w[j].z), u3 = __builtin_fabsf(f.x[0][i].w - f.w[j].w);
                        const float u = __builtin_fmaxf(__builtin_fmaxf(u0, u1), __builtin_fmaxf(u2, u3));
                        top[i] = __builtin_fmaxf(top[i], u * rs[i][j]);
                    }
                    all = __builtin_fmaxf(all, top[i]);
                }
                if (__builtin_amdgcn_ballot_w64(all > cut) == 0) return;
#pragma unroll
                for (int i = 0; i < TM; i++)
                    if (__builtin_amdgcn_ballot_w64(top[i] > cut) != 0) {
#pragma unroll
                        for (int j = 0; j < TN; j++)
#pragma unroll
                            for (int e = 0; e < 4; e++)
                                acc[i][j] += pow_pos(__builtin_fabsf(f.x[0][i][e] - f.w[j][e]) * rs[i][j], pv);
                    }
            } else {
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < TN; j++)
#pragma unroll
                        for (int e = 0; e < 4; e++)
                            acc[i][j] += pow_pos(__builtin_fabsf(f.x[0][i][e] - f.w[j][e]) * rs[i][j], pv);
            }
        });
        join(acc, add);
        const float inv_p = 1.0f / p;
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) acc[i][j] = pow_pos(acc[i][j], inv_p) / rs[i][j];
    }
    __syncthreads();
    if (grp == 0) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) lds[GEO::row(ty, i) * GEO::BN + GEO::col(tx, j)] = acc[i][j];
    }
    __syncthreads();
    q_store_tile<GEO>(output, lds, d, m0, n0, g, tid);
}

template <class GEO>
static Dims quad_dims(const Problem& pr, bool ovec) {
    Dims d = make_dims(pr);
    d.ovec = ovec;
    d.tiles_m = (d.M + GEO::BM - 1) / GEO::BM;
    d.tiles_n = (d.NG + GEO::BN - 1) / GEO::BN;
    return d;
}

template <class GEO, bool POS>
static hipError_t launch_inf(const Problem& pr, hipStream_t stream, const float* input, const float* weight, float* output,
                             int32_t* pos) {
    const Dims d = quad_dims<GEO>(pr, can_vec4_out(pr, output, pos));
    const size_t lds = q_lds_bytes<GEO, 1>();
    auto kern = inf_forward_quad_kernel<GEO, POS>;
    static LdsRecord lds_allowed = {};
    if (hipError_t e = allow_lds(kern, lds, pr.device, lds_allowed); e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, dim3((unsigned)d.tiles_m * d.tiles_n * d.G), dim3(GEO::NT), lds, stream, input, weight, output, pos, d);
    return hipGetLastError();
}

template <class GEO>
static hipError_t launch_bound(const Problem& pr, hipStream_t stream, const float* lower, const float* upper,
                               const float* weight, float* out_lower, float* out_upper) {
    const Dims d = quad_dims<GEO>(pr, can_vec4_out(pr, out_lower, out_upper));
    const size_t lds = q_lds_bytes<GEO, 2>();
    auto kern = bound_forward_quad_kernel<GEO>;
    static LdsRecord lds_allowed = {};
    if (hipError_t e = allow_lds(kern, lds, pr.device, lds_allowed); e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, dim3((unsigned)d.tiles_m * d.tiles_n * d.G), dim3(GEO::NT), lds, stream, lower, upper, weight,
                       out_lower, out_upper, d);
    return hipGetLastError();
}

template <class GEO>
static hipError_t launch_norm(const Problem& pr, hipStream_t stream, const float* input, const float* weight, float* output, float p) {
    const Dims d = quad_dims<GEO>(pr, can_vec4_out(pr, output));
    const size_t lds = q_lds_bytes<GEO, 1>();
    auto go = [&](auto kern, LdsRecord& lds_allowed) {
        if (hipError_t e = allow_lds(kern, lds, pr.device, lds_allowed); e != hipSuccess) return e;
        hipLaunchKernelGGL(kern, dim3((unsigned)d.tiles_m * d.tiles_n * d.G), dim3(GEO::NT), lds, stream, input, weight, output, p, d);
        return hipGetLastError();
    };
    static LdsRecord allowed[6] = {};
    switch (small_int_power(p)) {
        case 2: return go(norm_forward_quad_kernel<GEO, 2, false>, allowed[0]);
        case 3: return go(norm_forward_quad_kernel<GEO, 3, false>, allowed[1]);
        case 4: return go(norm_forward_quad_kernel<GEO, 4, false>, allowed[2]);
        case 8: return go(norm_forward_quad_kernel<GEO, 8, false>, allowed[3]);
        default:
            if (p >= 128.f && d.K >= 2048) return go(norm_forward_quad_kernel<GEO, 0, true>, allowed[4]);
            return go(norm_forward_quad_kernel<GEO, 0, false>, allowed[5]);
    }
}

// The tiles a problem can be cut into; `resident`: workgroups per CU.
struct QuadTile { int bm, bn, resident; };
constexpr QuadTile kQuadTiles[] = {{32, 80, 2}, {32, 40, 2}, {16, 40, 2}, {32, 64, 3}, {32, 32, 3}, {16, 32, 3}, {64, 80, 2}};
constexpr int kQuadTileCount = (int)(sizeof(kQuadTiles) / sizeof(kQuadTiles[0]));
constexpr int kFewRows = 20;    // few_rows_forward.hip
#define QUAD_TILES(CALL)                                    \
    switch (tile) {                                         \
        case 0: return CALL((QGeo<32, 80, 8, 5, 4, 64>));   \
        case 1: return CALL((QGeo<32, 40, 8, 5, 8, 64>));   \
        case 2: return CALL((QGeo<16, 40, 8, 5, 16, 128>)); \
        case 3: return CALL((QGeo<32, 64, 8, 4, 4, 64>));   \
        case 4: return CALL((QGeo<32, 32, 8, 4, 8, 64>));   \
        case 5: return CALL((QGeo<16, 32, 8, 4, 16, 128>)); \
        default: return CALL((QGeo<64, 80, 8, 5, 2, 32>));  \
    }
#define UNPAREN(...) __VA_ARGS__

// What the kernels of a kind reach, fitted to their times on thirty sizes from 1 x 1024 x 1024 to 1024 x 5120 x 5120 (rows
// x outputs x inputs): differences per microsecond of a full device for every tile, for the few-rows kernel and for the
// kernel of fwd_engine.hpp; what a tile or a row costs beside its k, in k (merging, locating, storing); and a constant,
// mostly the launch.  With these the kernel picked is within 5 % of the fastest on all of the thirty but three.
struct ForwardModel {
    double tile[kQuadTileCount], few, big;   // millions per microsecond
    double one_fill;                         // share of the rate that a CU reaches with a single workgroup
    double tile_k, few_k, big_k, tile_us, few_us, big_us;
};
constexpr ForwardModel kModels[] = {
    /* L_inf   */ {{28.2, 23.4, 21.1, 29.4, 26.1, 23.4, 29.7}, 20.4, 31.3, 0.61, 150, 800, 320, 18.9, 2.2, 14.6},
    /* values  */ {{31.3, 31.4, 25.5, 32.0, 30.7, 27.2, 32.7}, 22.9, 0, 0.59, 10, 540, 0, 8.6, 1.4, 0},
    /* bounds  */ {{11.9, 10.2, 9.5, 11.3, 10.7, 9.1, 12.3}, 8.0, 11.6, 0.60, 0, 650, 100, 10.2, 0.0, 4.4},
    /* p = 2, 3, 4, 8 */ {{13.6, 13.2, 12.5, 13.4, 13.2, 12.6, 13.6}, 9.8, 13.2, 0.64, 0, 580, 160, 11.4, 1.5, 5.0},
    /* other p */ {{4.55, 4.75, 4.42, 4.70, 4.81, 4.80, 4.33}, 4.3, 5.2, 0.82, 0, 200, 120, 25.4, 16.1, 4.7},
};

// The kernel with the shortest estimate, and the estimate.  Tiles: the busiest CU's share of them
// at the rate it reaches with that many workgroups (a single one leaves the vector unit idle nearly half the time,
// since a wave issues every 4.3 clocks at best).  A handful of rows: the reading of the weights plus the arithmetic.
static int fastest_forward(const Problem& pr, ForwardKind kind, float p, double cus, double& best) {
    const ForwardModel& model = kModels[kind != ForwardKind::kNorm ? (int)kind : small_int_power(p) >= 2 ? 3 : 4];
    const double M = pr.B, K = pr.K;
    // the busiest CU's time for its tiles of bm x bn (k of them the parts of a tile that do not grow with K)
    auto tiles_us = [&](int bm, int bn, int resident, double k, double rate) {
        const double per_cu = std::ceil(std::ceil(M / bm) * std::ceil((double)pr.NG / bn) * pr.G / cus);
        return per_cu * bm * bn * (K + k) * cus * 1e-6 / (rate * (per_cu < 2 && resident > 1 ? model.one_fill : 1.0));
    };
    best = model.few_us + 4e-6 * pr.G * pr.NG * K / 4.4 + 1e-6 * M * pr.G * pr.NG * (K + model.few_k) / model.few;
    int pick = kFewRows;
    for (int i = 0; i < kQuadTileCount; i++) {
        const QuadTile& t = kQuadTiles[i];
        const double us = model.tile_us + tiles_us(t.bm, t.bn, t.resident, model.tile_k, model.tile[i]);
        if (us < best) { best = us; pick = i; }
    }
    // the kernel of fwd_engine.hpp needs aligned rows for its 128-bit loads; its L_inf form runs tiles of 128 x 80 or two
    // workgroups of 64 x 80 per CU, the others one of 128 x 80
    if (pr.K % 4 == 0 && kind != ForwardKind::kValues) {
        const bool halves = M > 64 && kind == ForwardKind::kInf;
        const double us = model.big_us + tiles_us(halves ? 64 : 128, 80, halves ? 2 : 1, model.big_k, model.big);
        if (us < best) { best = us; pick = -1; }
    }
    return pick;
}

// Which kernel a fully connected layer takes.
int small_forward_tile(const Problem& pr, ForwardKind kind, float p) {
    if (pr.HW != 1 || pr.K < 4 || 4LL * 80 * pr.G * pr.K >= (1LL << 31)) return -1;
    if (g_tile_override >= 10) return g_tile_override - 10;
    if (g_tile_override >= 0) return kind == ForwardKind::kValues ? kQuadTileCount - 1 : -1;   // values: there are no larger tiles
    double us;
    return fastest_forward(pr, kind, p, pr.num_cu, us);
}

double full_walk_us(const Problem& pr, ForwardKind kind, int num_cu) {
    double us;
    fastest_forward(pr, kind, 0.f, num_cu, us);
    return us;
}

hipError_t inf_forward_small(const float* input, const float* weight, float* output, int32_t* pos, const Problem& pr, int tile,
                             hipStream_t stream) {
    if (tile == kFewRows) return inf_forward_few_rows(input, weight, output, pos, pr, stream);
    if (pos) {
#define CALL(G) launch_inf<UNPAREN G, true>(pr, stream, input, weight, output, pos)
        QUAD_TILES(CALL)
#undef CALL
    }
#define CALL(G) launch_inf<UNPAREN G, false>(pr, stream, input, weight, output, nullptr)
    QUAD_TILES(CALL)
#undef CALL
}
hipError_t bound_forward_small(const float* lower, const float* upper, const float* weight, float* out_lower, float* out_upper,
                               const Problem& pr, int tile, hipStream_t stream) {
    if (tile == kFewRows) return bound_forward_few_rows(lower, upper, weight, out_lower, out_upper, pr, stream);
#define CALL(G) launch_bound<UNPAREN G>(pr, stream, lower, upper, weight, out_lower, out_upper)
    QUAD_TILES(CALL)
#undef CALL
}

hipError_t norm_forward_small(const float* input, const float* weight, float* output, float p, const Problem& pr, int tile,
                              hipStream_t stream) {
    if (tile == kFewRows) return norm_forward_few_rows(input, weight, output, p, pr, stream);
#define CALL(G) launch_norm<UNPAREN G>(pr, stream, input, weight, output, p)
    QUAD_TILES(CALL)
#undef CALL
}

}  // namespace ldist
