// L_inf forward passes of large fully connected layers that evaluate only the differences that can be a maximum.
//
// max_k |x[m,k] - w[n,k]| is attained where x[m,k] or w[n,k] lies far out: if a short list of row m holds its q_x
// outermost inputs, and one of row n its q_w outermost weights, then every k in neither list has
//     |x - w| <= max(max x - min w, max w - min x)   over what the two lists left out,
// two numbers per row.  The maximum over the k in either list is therefore the maximum over all k wherever it exceeds
// that bound, which can be read off afterwards: rounding is monotone, so the statement holds for the rounded differences
// too, and the results (argmax with its sign included) are the same bits as those of the full walk.  Outputs that do not
// pass are walked in full by the wave that finds them.  With K = 5120 inputs, lists of 1 to 4 % suffice for all but one
// output in a thousand, for inputs and weights of comparable spread as for very different ones.
//
// Launches, all on the caller's stream:
//   sample   64 x 64 outputs in full, and for their rows what lists of eight lengths would leave out;
//   select   the list lengths that cost least by that sample (or none: `dense`, and the kernels of the full walk, which
//            are launched last and otherwise leave at once, do the work), and every row's list;
//   scan     first every row's list against all outputs, then every weight row's list against all rows.  Where the weights
//            need no list (images, or activations spread far wider than the weights) the first scan checks the bounds itself,
//            and the second leaves at once: 5120 x 5120 with positions at batch 272, 46 + 43 -> 50 + 5 us.
//
// Boxes and the points inside them (certification) share sample, lists and first scan: an entry of a row of x is {lower, upper,
// 32 k, point}.  Where the weights have lists, the second scans of boxes and of values follow it.  Certification of the 5-layer,
// 5120-wide net at batch 1024: 1500 us with passes of their own, 820 together; 5120 x 5120 normal weights and inputs of the same
// spread, batch 512, 171 + 229 -> 330 us, 1024 235 + 385 -> 548.
//
// The reduction is cut into C chunks of at most 2560 k with lists and bounds of their own, so that a chunk of eight rows
// of the other operand fits half a CU's LDS.  Rows with NaN or infinities (bounds: boxes that are not l <= u) get an infinite
// bound: their outputs are walked in full with the comparisons of the other kernels.
//
// 5120 x 5120, full walk -> lists, us: layers of an untrained net on its own inputs, positions at batch 512 445 -> 102, values at 1024
// 780 -> 100, bounds at 1024 2170 -> 142; normal weights and inputs of the same spread 215, 235 and 385.  Data that the lists cannot help (two values in both operands) cost the sample and the lists beside the full walk: 15 to 60 us
// up to 5120 inputs, 75 at 12544, 110 to 140 at 20000.  Weights of a 5 x 5120 net that has been trained through p = 8 ... 1000 and
// infinity need lists of their own, and leave more outputs to be walked: on its own inputs at batch 1024 positions 155 to 169, values 135
// to 160, bounds 211 to 223, values with bounds 297 to 342.
#include <algorithm>

#include "kernels.hpp"
#include "quad_engine.hpp"
#include "wave_reduce.hpp"

namespace ldist {
namespace {

typedef float F4 __attribute__((ext_vector_type(4)));

constexpr int kMaxChunk = 2560;              // eight rows of it: 80 KB of LDS, two workgroups per CU
constexpr int kLengths[8] = {0, 8, 16, 32, 48, 64, 96, 128};   // of a chunk's list
constexpr int kMaxList = 128;
constexpr int kBins = 512;                   // of the histogram of |v - center|: 256 to the octave, the top two octaves
constexpr int kBinShift = 15;
constexpr int kSampled = 64;                 // rows of either operand that the sample looks at
constexpr int kSampleRows = 4;               // of them in one workgroup
constexpr int kSampleGroups = kSampled / kSampleRows;
constexpr int kBoxFails = 1 << 29, kPointFails = 1 << 30;   // beside an index of Search::walk (boxes and points have scratch memory for 2^24 outputs)
constexpr float kNever = 3.402823466e38f;    // bound of an empty remainder; finite, so that infinite bounds stay infinite beside it

// How many entries of a list are meant to be taken, so that those of rows with a few more still fit.
__device__ __forceinline__ constexpr int typical(int length) { return length - length / 8 - length / 16; }

struct Header {
    float center;
    int qx, qw;
    int dense;         // the lists are not worth it
    int full;          // the full walk has to do the work: dense, or the lists left too many outputs unsettled
    int failed;        // how many
    int taken[3][8];   // tiles of a scan (Search::turn) that the workgroups of an XCD have taken beyond their first
};

// One operand: its rows, their lists in blocks of 16 rows (entry-major, so that 16 neighbouring lanes read 128 bytes)
// and per chunk and row what the lists left out.
struct Side {
    const float *v, *v2, *v3;   // v2: the upper ends where v are the lower ends of boxes; v3: the points inside them
    int rows, blocks;
    char* lists;           // [chunk][block][entry][16] of {value, 32 k} or {lower, upper, 32 k, point}
    float* rest;           // [chunk][rests][rows]: max, min; boxes: max of the upper ends, min of the lower, max of the lower, min of the upper; points: max, min
    int rests;             // 2, 4 or 6
};

struct Search {
    Side x, w;
    float *out, *out2, *out3;   // distances, or the lower and upper bounds, and the points' distances
    const float *mean, *bias;   // of Problem
    int32_t* pos;
    Header* head;
    unsigned char* counts; // [workgroup of the sample][combination of lengths]: outputs that would not pass
    float* reach;          // [x, w][length][sampled row]: how far from the center a list of that length begins
    float* partial;        // [row of x][pitch] of the first scan's {value, position}, {upper, lower bound}, or values
    float* partial3;       // [row of x][pitch] of the points' distances
    int pitch;
    int turn;              // which of Header::taken a scan counts in
    int* walk;             // [walk_most]: indices of outputs that fail; boxes and points: with what of them fails
    int walk_most;
    int note;              // boxes and points: what a scan notes as failing, of its boxes, of its points or both
    int K, C, KC;
    int lanes_first, lanes_second, lanes_only;   // rows per workgroup of the two scans, and of a first that no second follows
    float price_x, price_w, price_both, price_fail, price_dense;   // of a list entry, of a second scan after the first, of an output that does not pass, of the full walk
};

__device__ __forceinline__ float wave_max_f(float x) {
#pragma unroll
    for (int o = 32; o; o >>= 1) x = __builtin_fmaxf(x, __shfl_xor(x, o));
    return x;
}
__device__ __forceinline__ float wave_min_f(float x) {
#pragma unroll
    for (int o = 32; o; o >>= 1) x = __builtin_fminf(x, __shfl_xor(x, o));
    return x;
}
__device__ __forceinline__ int sum_from_lane(int x, int lane) {   // over this lane and those above it
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_down(x, o);
        if (lane + o < 64) x += y;
    }
    return x;
}
__device__ __forceinline__ bool not_finite(float v) { return !(__builtin_fabsf(v) < __builtin_inff()); }

// A chunk of a row in a wave's registers: lane l holds k = 64 j + l.
template <int NV>
struct RowChunk {
    float v[NV];
    __device__ __forceinline__ void load(const float* row, int kc, int lane) {
        const auto rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)row, 0, kc * 4, 0x00020000);
#pragma unroll
        for (int j = 0; j < NV; j++)
            v[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, lane * 4, j * 256, 0));
    }
    // k past the chunk as `center`, which no list takes.
    __device__ __forceinline__ void center_past(int kc, int lane, float center) {
        if (kc >= NV * 64) return;
#pragma unroll
        for (int j = 0; j < NV; j++) {
            v[j] = lane < kc - j * 64 ? v[j] : center;
            if (j % 4 == 3) __builtin_amdgcn_sched_barrier(0);   // no more lane masks at a time than there are registers for
        }
    }
    // Keeps the compiler from carrying what one pass over the values derives from them into the next (registers).
    __device__ __forceinline__ void opaque() {
#pragma unroll
        for (int j = 0; j < NV; j++) asm volatile("" : "+v"(v[j]));
    }
};

// The largest of each of 16 values over a wave, NaN where there is one: in lane l that of value l / 4.  Halves, rows of 16, eights
// and fours of lanes trade the values that the other part goes on with (33 instructions; 16 reductions of their own take 96).
__device__ __forceinline__ float wave_max_of_16(float (&v)[16], int lane) {
    auto larger = [](float a, float b) { return __builtin_elementwise_maximum(a, b); };
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[i]), __float_as_uint(v[i + 8]), false, false);
        v[i] = larger(__uint_as_float(r[0]), __uint_as_float(r[1]));
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v[i]), __float_as_uint(v[i + 4]), false, false);
        v[i] = larger(__uint_as_float(r[0]), __uint_as_float(r[1]));
    }
    constexpr int kHalfMirror = 0x141;
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const float keep = lane & 8 ? v[i + 2] : v[i], give = lane & 8 ? v[i] : v[i + 2];
        v[i] = larger(keep, dpp_move<kDppRor8, 0xF>(give, give));
    }
    const float keep = lane & 4 ? v[1] : v[0], give = lane & 4 ? v[0] : v[1];
    float m = larger(keep, dpp_move<kHalfMirror, 0xF>(give, give));
    m = larger(m, dpp_move<kDppSwap1, 0xF>(m, m));
    return larger(m, dpp_move<kDppSwap2, 0xF>(m, m));
}

// ---- sample ----------------------------------------------------------------------------------------------------------
// Distance from the center as a bin of a histogram: 256 to the octave, two octaves below the largest; negative: below.
struct Bins {
    unsigned base;
    __device__ __forceinline__ explicit Bins(float most) : base(__float_as_uint(most) - ((unsigned)(kBins - 1) << kBinShift)) {}
    __device__ __forceinline__ int of(float u) const { return min((int)(__float_as_uint(u) - base) >> kBinShift, kBins - 1); }
    __device__ __forceinline__ float edge(int bin) const {   // lower edge
        return __uint_as_float((unsigned)max((int)(base + ((unsigned)bin << kBinShift)), 0));
    }
};

// found(i, distance from the center at which a list of the i-th length begins), for one row chunk.
template <int NV, class F>
__device__ __forceinline__ void lengths_of(RowChunk<NV>& a, float center, int* hist, int lane, F&& found) {
    float most = 0.f;
#pragma unroll
    for (int j = 0; j < NV; j++) most = __builtin_fmaxf(most, __builtin_fabsf(a.v[j] - center));
    const Bins bins(wave_max_f(most));
    a.opaque();
#pragma unroll
    for (int j = 0; j < kBins / 256; j++) *reinterpret_cast<int4*>(hist + (j * 64 + lane) * 4) = make_int4(0, 0, 0, 0);
#pragma unroll
    for (int j = 0; j < NV; j++) {   // a quarter of normally distributed values get here
        const int bin = bins.of(__builtin_fabsf(a.v[j] - center));
        if (bin >= 0) atomicAdd(hist + bin, 1);
        if (j % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
    constexpr int OWN = kBins / 64;
    int upward[OWN], sum = 0;   // values in this lane's bins, from each bin up; then in all bins from there up
#pragma unroll
    for (int j = OWN / 4 - 1; j >= 0; j--) {
        const int4 h = *reinterpret_cast<const int4*>(hist + lane * OWN + j * 4);
        upward[4 * j + 3] = sum += h.w;
        upward[4 * j + 2] = sum += h.z;
        upward[4 * j + 1] = sum += h.y;
        upward[4 * j] = sum += h.x;
    }
    const int above = sum_from_lane(sum, lane) - sum;
#pragma unroll
    for (int j = 0; j < OWN; j++) upward[j] += above;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        int taken = 0;   // of this lane's bins
#pragma unroll
        for (int j = 0; j < OWN; j++) taken += upward[j] <= typical(kLengths[i]);
        const unsigned long long over = __ballot(upward[0] > typical(kLengths[i]));
        int cut = 0;
        if (over) {
            const int at = 63 - __builtin_clzll(over);
            cut = (at + 1) * OWN - __builtin_amdgcn_readlane(taken, at);
        }
        found(i, bins.edge(cut));
    }
}

// A workgroup looks at 4 x 4 outputs: wave i at row i % 8 (four of x, four of w) in every other chunk, then all at the outputs.
// Bound by a chain of latencies: the outputs' rows are on their way during the histograms, and their 16 (boxes 32, with points 48)
// maxima meet 16 at a time: 5120 -> 5120 17.5 -> 15.9 us, boxes with points 29.9 -> 24.7.
// ENDS: 1 values, 2 boxes, 3 boxes and the points inside them.  Of 40 values per lane 1 is spilled without boxes, and 31 registers with
// points, outside of the loops over the outputs.
template <int NV, int ENDS>
__global__ void __launch_bounds__(1024) extremes_sample_kernel(Search s) {
    constexpr bool PAIR = ENDS >= 2, ALL = ENDS == 3;
    constexpr int NO = kSampleRows * kSampleRows, NB = ENDS, WAVES = 16;
    __shared__ __align__(16) int hist[WAVES][kBins];
    __shared__ float rest[NB][2 * kSampleRows][8][16];   // [bound][row][length][chunk]: the most that the list leaves out
    __shared__ float reach[2 * kSampleRows][8][16];
    __shared__ float outs[WAVES][NB * NO];
    __shared__ float part[WAVES];
    __shared__ int fails[64];
    static_assert(NO == WAVES, "a wave for every output");
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int bx = blockIdx.x / kSampleGroups, bw = blockIdx.x % kSampleGroups;
    auto sampled = [](int i, int rows) { return (int)((long long)i * rows / kSampled); };
    if (tid < 64) fails[tid] = 0;
    const int r = wave & 7;
    const bool of_x = r < kSampleRows;
    const Side& side = of_x ? s.x : s.w;
    const int row = sampled((of_x ? bx : bw) * kSampleRows + (r & (kSampleRows - 1)), side.rows);
    RowChunk<NV> a, b;   // boxes: both ends, then a alone, the middles
    auto load = [&](int ch) {
        const int k0 = ch * s.KC, kc = min(s.KC, s.K - k0);
        a.load(side.v + (size_t)row * s.K + k0, kc, lane);
        if constexpr (PAIR) { if (of_x) b.load(side.v2 + (size_t)row * s.K + k0, kc, lane); }
    };
    const int first = wave >> 3;
    if (first < s.C) load(first);
    const float *xr[kSampleRows], *ur[kSampleRows], *pr[kSampleRows], *wr[kSampleRows];   // of the outputs
#pragma unroll
    for (int i = 0; i < kSampleRows; i++) {
        xr[i] = s.x.v + (size_t)sampled(bx * kSampleRows + i, s.x.rows) * s.K;
        if constexpr (PAIR) ur[i] = s.x.v2 + (size_t)sampled(bx * kSampleRows + i, s.x.rows) * s.K;
        if constexpr (ALL) pr[i] = s.x.v3 + (size_t)sampled(bx * kSampleRows + i, s.x.rows) * s.K;
        wr[i] = s.w.v + (size_t)sampled(bw * kSampleRows + i, s.w.rows) * s.K;
    }
    constexpr int AHEAD = ALL ? 2 : PAIR ? 3 : 5;
    constexpr bool EARLY = ENDS == 1;   // the first of them before the histograms; boxes have no registers for that
    float x[AHEAD][kSampleRows], u[AHEAD][kSampleRows], p[AHEAD][kSampleRows], w[AHEAD][kSampleRows];
    auto fetch = [&](int kb) {
#pragma unroll
        for (int e = 0; e < AHEAD; e++) {
            const int k = min(kb + e * 1024 + tid, s.K - 1);   // past the end: the last k again
#pragma unroll
            for (int i = 0; i < kSampleRows; i++) {
                x[e][i] = xr[i][k];
                w[e][i] = wr[i][k];
                if constexpr (PAIR) u[e][i] = ur[i][k];
                if constexpr (ALL) p[e][i] = pr[i][k];
            }
        }
    };
    // a center common to both operands: the mean of 1024 weights; any number is correct
    float c = s.w.v[(size_t)((long long)tid * s.w.rows / 1024) * s.K + (size_t)((long long)tid * 61 % s.K)];
    if (EARLY) fetch(0);
#pragma unroll
    for (int o = 32; o; o >>= 1) c += __shfl_xor(c, o);
    if (lane == 0) part[wave] = c;
    __syncthreads();
    c = 0.f;
#pragma unroll
    for (int i = 0; i < WAVES; i++) c += part[i];
    const float center = not_finite(c) ? 0.f : c / 1024.f;
    if (blockIdx.x == 0) {
        if (tid == 0) s.head->center = center;
        if (tid < 24) s.head->taken[tid >> 3][tid & 7] = 0;
        if (tid == 24) s.head->failed = 0;
    }
#pragma unroll 1
    for (int ch = first; ch < s.C; ch += WAVES / 8) {
        if (ch != first) load(ch);
        const int kc = min(s.KC, s.K - ch * s.KC);
        float widest = 0.f, width = 0.f, off = 0.f;   // of the boxes, and the mean; half of each; points off the middle
        if constexpr (PAIR) {
            if (of_x) {
#pragma unroll
                for (int j = 0; j < NV; j++) {
                    const float half = 0.5f * (b.v[j] - a.v[j]);
                    widest = __builtin_fmaxf(widest, half);
                    width += half;
                    a.v[j] = 0.5f * (a.v[j] + b.v[j]);
                }
                widest = wave_max_f(widest);
#pragma unroll
                for (int o = 32; o; o >>= 1) width += __shfl_xor(width, o);
                width /= kc;
                if constexpr (ALL) {
                    b.load(s.x.v3 + (size_t)row * s.K + ch * s.KC, kc, lane);   // both 0 past the end
#pragma unroll
                    for (int j = 0; j < NV; j++) off = __builtin_fmaxf(off, __builtin_fabsf(b.v[j] - a.v[j]));
                    off = wave_max_f(off);
                }
            }
        }
        a.center_past(kc, lane, center);
        lengths_of<NV>(a, center, hist[wave], lane, [&](int i, float edge) {
            if (lane == 0) {
                reach[r][i][ch] = edge;
                rest[0][r][i][ch] = edge + widest;                    // upper bounds reach further than the middles,
                if constexpr (PAIR) rest[1][r][i][ch] = edge - width;   // lower bounds less far
                if constexpr (ALL) rest[2][r][i][ch] = edge + off;
            }
        });
    }

    float up[NO], lo[NO], pt[NO];
#pragma unroll
    for (int i = 0; i < NO; i++) up[i] = lo[i] = pt[i] = 0.f;
    for (int kb = 0; kb < s.K; kb += 1024 * AHEAD) {
        if (!EARLY || kb > 0) fetch(kb);
#pragma unroll
        for (int e = 0; e < AHEAD; e++)
#pragma unroll
            for (int i = 0; i < kSampleRows; i++)
#pragma unroll
                for (int j = 0; j < kSampleRows; j++) {
                    const float dl = x[e][i] - w[e][j];
                    float& U = up[i * kSampleRows + j];
                    U = __builtin_fmaxf(U, __builtin_fabsf(dl));
                    if constexpr (PAIR) {
                        const float du = u[e][i] - w[e][j];
                        float& L = lo[i * kSampleRows + j];
                        U = __builtin_fmaxf(U, __builtin_fabsf(du));
                        L = __builtin_fmaxf(__builtin_fmaxf(L, dl), -du);
                    }
                    if constexpr (ALL) pt[i * kSampleRows + j] = __builtin_fmaxf(pt[i * kSampleRows + j], __builtin_fabsf(p[e][i] - w[e][j]));
                }
    }
    auto gather = [&](float (&v)[NO], int q) {
        const float m = wave_max_of_16(v, lane);
        if ((lane & 3) == 0) outs[wave][q * NO + (lane >> 2)] = m;
    };
    gather(up, 0);
    if constexpr (PAIR) gather(lo, 1);
    if constexpr (ALL) gather(pt, 2);
    __syncthreads();
    if (tid < NB * NO) {
        float best = outs[0][tid];
#pragma unroll
        for (int i = 1; i < WAVES; i++) best = __builtin_fmaxf(best, outs[i][tid]);
        outs[0][tid] = best;
    }
    __syncthreads();
    {   // wave: output, lane: combination of lengths
        const int ix = lane >> 3, iw = lane & 7;
        bool ok = true;
#pragma unroll
        for (int q = 0; q < NB; q++) {
            float bound = 0.f;
            for (int ch = 0; ch < s.C; ch++)
                bound = __builtin_fmaxf(bound, rest[q][wave / kSampleRows][ix][ch] + rest[0][kSampleRows + wave % kSampleRows][iw][ch]);
            ok &= PAIR ? outs[0][q * NO + wave] >= bound : outs[0][wave] > bound;
        }
        if (!ok) atomicAdd(&fails[lane], 1);
    }
    __syncthreads();
    if (tid < 64) {
        s.counts[blockIdx.x * 64 + tid] = (unsigned char)fails[tid];
    } else if (tid < 128) {   // 8 rows x 8 lengths; of x from the workgroups with bw == 0, of w from those with bx == 0
        const int rr = (tid >> 3) & 7, i = tid & 7;
        if (rr < kSampleRows ? bw == 0 : bx == 0) {
            float sum = 0.f;
            for (int ch = 0; ch < s.C; ch++) sum += reach[rr][i][ch];
            s.reach[((rr < kSampleRows ? 0 : 1) * 8 + i) * kSampled + (rr < kSampleRows ? bx : bw) * kSampleRows + (rr & (kSampleRows - 1))] = sum / s.C;
        }
    }
}

// ---- select ----------------------------------------------------------------------------------------------------------
// The cheapest lengths by the sample; every workgroup works this out for itself.
__device__ __forceinline__ void choose_lengths(const Search& s, int (&sums)[8][64], int wave, int lane, int& ix, int& iw, int& dense) {
    constexpr int SHARE = kSampleGroups * kSampleGroups / 8;
    int part = 0;
#pragma unroll
    for (int b = 0; b < SHARE; b++) part += s.counts[(wave * SHARE + b) * 64 + lane];
    sums[wave][lane] = part;
    __syncthreads();
    int fails = 0;
#pragma unroll
    for (int i = 0; i < 8; i++) fails += sums[i][lane];
    float cost = s.C * (s.price_x * kLengths[lane >> 3] + s.price_w * kLengths[lane & 7]) +
                 (lane > 7 && (lane & 7) ? s.price_both : 0.f) + s.price_fail * ((float)fails / (kSampled * kSampled));
    int pick = lane;
#pragma unroll
    for (int o = 32; o; o >>= 1) {
        const float c = __shfl_xor(cost, o);
        const int p = __shfl_xor(pick, o);
        if (c < cost || (c == cost && p < pick)) { cost = c; pick = p; }
    }
    pick = __builtin_amdgcn_readfirstlane(pick);
    ix = pick >> 3;
    iw = pick & 7;
    dense = __builtin_amdgcn_readfirstlane(cost > s.price_dense ? 1 : 0);
}

// Resident workgroups take eight rows of a chunk at a time, a wave that of a row: all values beyond `t` from the center,
// where t starts as what the sampled rows needed on the average and is moved where the list would overflow or stay half empty
// (rows of weights are alike: most pass at once).  What the list leaves out lies in [center - t, center + t] then, exactly,
// unless more values tie at the outer end than the list has places: such a row's bounds are those of all its values.
// Bound by reading the operands once.
// Boxes of 40 values per lane spill 18 registers of what all of a workgroup's rows share.
// SPREAD: no positions follow, and the order of a list is free (its own instantiation: the code of both orders in one made the
// kernel 43 -> 48 us).
template <int NV, int ENDS, bool SPREAD>
__global__ void __launch_bounds__(512, ENDS > 1 || NV > 24 ? 4 : 6) extremes_select_kernel(Search s) {
    extern __shared__ __align__(16) char stage[];   // [2 kMaxList][8] entries: half of a block of Side::lists, and what finds no place in its order
    __shared__ int sums[8][64];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int ix, iw, dense;
    choose_lengths(s, sums, wave, tid & 63, ix, iw, dense);
    if (blockIdx.x == 0 && tid == 0) { s.head->qx = kLengths[ix]; s.head->qw = kLengths[iw]; s.head->dense = s.head->full = dense; }
    if (dense) return;
    const float center = s.head->center;
    auto needed = [&](int i) {   // by the sampled rows on the average
        float sum = s.reach[i * kSampled + (tid & 63)];
#pragma unroll
        for (int o = 32; o; o >>= 1) sum += __shfl_xor(sum, o);
        return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(sum * (1.f / kSampled))));
    };
    const float guess_x = needed(ix), guess_w = needed(8 + iw);

    auto lists = [&](auto ends, const Side& side, int q, float guess, int ch, int block) {
        constexpr bool P = decltype(ends)::value >= 2, ALL = decltype(ends)::value == 3;
        int lane = tid & 63;
        asm volatile("" : "+v"(lane));   // what is derived from it is made where it is used, not kept in registers over the loop
        const int k0 = ch * s.KC, r = block * 8 + wave, row = __builtin_amdgcn_readfirstlane(min(r, side.rows - 1));
        RowChunk<NV> a;
        const int kc = min(s.KC, s.K - k0);
        a.load(side.v + (size_t)row * s.K + k0, kc, lane);
        // twice the middle of a box, where values are compared by themselves
        constexpr float F = P ? 2.f : 1.f;
        if constexpr (!P) a.center_past(kc, lane, center);
        float odd = 0.f;   // NaN if there is a NaN or an infinity
        bool crossed = false;
#pragma unroll
        for (int j = 0; j < NV; j++) odd = __builtin_fmaf(a.v[j], 0.f, odd);
        if constexpr (P) {
            RowChunk<NV / 2> b;   // half a row at a time: registers
#pragma unroll
            for (int h = 0; h < 2; h++) {
                b.load(side.v2 + (size_t)row * s.K + k0 + h * NV * 32, max(kc - h * NV * 32, 0), lane);
#pragma unroll
                for (int j = 0; j < NV / 2; j++) {
                    float& mid = a.v[h * NV / 2 + j];
                    odd = __builtin_fmaf(b.v[j], 0.f, odd);
                    crossed |= mid > b.v[j];
                    mid += b.v[j];
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if constexpr (P) a.center_past(kc, lane, F * center);
        bool bad = __any(odd != 0.f || crossed);
        auto key = [&](int j) { return a.v[j]; };
        auto count = [&](float t) {
            const float hi = F * (center + t), lo = F * (center - t);
            int n = 0;
#pragma unroll
            for (int j = 0; j < NV; j++) n += __builtin_popcountll(__ballot(key(j) > hi) | __ballot(key(j) < lo));
            return n;
        };
        float hi, lo;
        if (q == 0) {   // no list: everything is left out
            hi = -kNever;
            lo = kNever;
#pragma unroll
            for (int j = 0; j < NV; j++) { hi = __builtin_fmaxf(hi, key(j)); lo = __builtin_fminf(lo, key(j)); }
            hi = wave_max_f(hi);
            lo = wave_min_f(lo);
        } else {
            float t = guess;
            int n = count(t);
            if (n > q || n < q / 2) {
                float most = 0.f;
#pragma unroll
                for (int j = 0; j < NV; j++) most = __builtin_fmaxf(most, __builtin_fabsf(key(j) - F * center));
                // too long a list, and one of no more than what ties at the outer end: center + t, rounded, may lie inside it
                float in = 0.f, out = wave_max_f(most) * (1.f / F);
                if (n > q) in = t; else out = __builtin_fminf(out, t);
#pragma unroll 1
                for (int step = 0; step < 10; step++) {
                    t = 0.5f * (in + out);
                    n = count(t);
                    if (n > q) { in = t; continue; }
                    out = t;
                    if (n >= q - q / 4) break;
                }
                t = out;
            }
            hi = F * (center + t);
            lo = F * (center - t);
        }
        struct Ends { float a, b, c; } first = {};
        int base = 0;
        float most = -kNever, least = kNever, most_lower = -kNever, least_upper = kNever, most_point = -kNever, least_point = kNever;
        auto before = [](unsigned long long m) { return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0)); };
        auto place = [&](bool in, int j, auto&& write) {
            const unsigned long long m = __ballot(in);
            if (m) {
                const int at = base + before(m);
                if (in && at < q) write(at * 8 + wave, (unsigned)(lane + j * 64) * 32u);
                base += __builtin_popcountll(m);
            }
        };
        if constexpr (P) {
            // Boxes and points come again, in groups of eight, mostly from the L2: there are no registers for all of them (with
            // both ends kept 155, which leave a workgroup alone on its CU, with the points 168 and 290 spilled).
            float odd_point = 0.f;
            const auto from = [&](const float* v) {
                return __builtin_amdgcn_make_buffer_rsrc((void*)(v + (size_t)row * s.K + k0), 0, kc * 4, 0x00020000);
            };
            const auto ra = from(side.v), rb = from(side.v2), rc = from(ALL ? side.v3 : side.v);
            auto gather = [&](bool record) {   // else: bounds of all values
#pragma unroll 1
                for (int j0 = 0; j0 < NV; j0 += 8) {
                    Ends e[8];
                    auto one = [&](auto rsrc, int j) {
                        return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, lane * 4, (j0 + j) * 256, 0));
                    };
#pragma unroll
                    for (int j = 0; j < 8; j++) e[j] = Ends{one(ra, j), one(rb, j), ALL ? one(rc, j) : 0.f};
#pragma unroll
                    for (int j = 0; j < 8; j++) {
                        if (lane >= kc - (j0 + j) * 64) e[j] = Ends{center, center, center};
                        const float mid = e[j].a + e[j].b;
                        const bool in = record && (mid > hi || mid < lo);
                        if (record)
                            place(in, j0 + j, [&](int to, unsigned k32) {
                                reinterpret_cast<uint4*>(stage)[to] =
                                    make_uint4(__float_as_uint(e[j].a), __float_as_uint(e[j].b), k32, __float_as_uint(e[j].c));
                            });
                        most = __builtin_fmaxf(most, in ? -kNever : e[j].b);
                        least = __builtin_fminf(least, in ? kNever : e[j].a);
                        most_lower = __builtin_fmaxf(most_lower, in ? -kNever : e[j].a);
                        least_upper = __builtin_fminf(least_upper, in ? kNever : e[j].b);
                        if constexpr (ALL) {
                            most_point = __builtin_fmaxf(most_point, in ? -kNever : e[j].c);
                            least_point = __builtin_fminf(least_point, in ? kNever : e[j].c);
                            odd_point = __builtin_fmaf(e[j].c, 0.f, odd_point);
                        }
                    }
                    if (j0 == 0) first = e[0];
                }
            };
            gather(true);
            if (__builtin_expect(base > q, 0)) gather(false);   // the list has lost values that no bound above speaks for
            if constexpr (ALL) bad |= __any(odd_point != 0.f);
        } else {
#pragma unroll
            for (int j = 0; j < NV; j++) {
                place(a.v[j] > hi || a.v[j] < lo, j, [&](int to, unsigned k32) {
                    reinterpret_cast<uint2*>(stage)[to] = make_uint2(__float_as_uint(a.v[j]), k32);
                });
                __builtin_amdgcn_sched_barrier(0);
            }
            if (__builtin_expect(base > q, 0)) {   // as above
#pragma unroll
                for (int j = 0; j < NV; j++) {
                    most = __builtin_fmaxf(most, a.v[j]);
                    least = __builtin_fminf(least, a.v[j]);
                }
                hi = wave_max_f(most);
                lo = wave_min_f(least);
            }
        }
        // a list that is not full repeats the chunk's first value, or one of its first eight
        using Entry = typename std::conditional<P, uint4, uint2>::type;
        Entry* mine = reinterpret_cast<Entry*>(stage) + wave;
        auto entry_of = [&](int from) {   // what lane `from` holds of the chunk's first 64
            const unsigned v0 = __shfl(__float_as_uint(P ? first.a : a.v[0]), from);
            if constexpr (P) return make_uint4(v0, __shfl(__float_as_uint(first.b), from), (unsigned)from * 32u, __shfl(__float_as_uint(first.c), from));
            else return make_uint2(v0, (unsigned)from * 32u);
        };
        if constexpr (SPREAD) {
            // Entry s of row r becomes one with k = s + r / 2 (mod 8) where the row has such an entry left, so that 16 neighbouring lanes
            // of a scan read from different banks.  Done on the finished list, 64 entries at a time: where every 64 values were put in
            // order as they were found, with lists for both operands the kernel took 28 instead of 24 us of 512 x 3072 -> 5120, 44 instead
            // of 37 with 5120 inputs, 59 instead of 51 for boxes at batch 1024 (20, 35 and 56 in the order of k).
            const int n = min(base, q);
            int of_class = 0, over = 0, vacant = 0;   // entries with this lane's k mod 8; those beyond an eighth of the list, kept behind it
            Entry own[kMaxList / 64];
#pragma unroll
            for (int i = 0; i < kMaxList / 64; i++) own[i] = i * 64 + lane < n ? mine[(i * 64 + lane) * 8] : Entry{};
            __builtin_amdgcn_wave_barrier();   // all of them, before the first is overwritten
#pragma unroll
            for (int i = 0; i < kMaxList / 64; i++) {
                if (i * 64 >= n) break;
                unsigned k32;
                if constexpr (P) k32 = own[i].z;
                else k32 = own[i].y;
                const unsigned long long all = __ballot(i * 64 + lane < n);
                unsigned long long bit[3];
#pragma unroll
                for (int b = 0; b < 3; b++) bit[b] = __ballot(k32 >> (5 + b) & 1u);
                auto of = [&](unsigned c) {   // which of the 64 have k mod 8 = c
                    unsigned long long m = all;
#pragma unroll
                    for (int b = 0; b < 3; b++) m &= c >> b & 1u ? bit[b] : ~bit[b];
                    return m;
                };
                const unsigned c = k32 >> 5 & 7u;
                const int rank = __shfl(of_class, (int)c) + before(of(c));
                const bool in = i * 64 + lane < n;
                const unsigned long long beyond = __ballot(in && rank >= q / 8);
                if (in) mine[(rank >= q / 8 ? kMaxList + over + before(beyond) : rank * 8 + (((int)c - (r >> 1)) & 7)) * 8] = own[i];
                over += __builtin_popcountll(beyond);
                of_class += __builtin_popcountll(of(lane & 7u));
            }
            __builtin_amdgcn_wave_barrier();
            for (int e0 = 0; e0 < q; e0 += 64) {
                const int e = e0 + lane, from = (e + (r >> 1)) & 7;
                const bool free = e < q && e / 8 >= __shfl(of_class, from);
                const unsigned long long m = __ballot(free);
                const int nth = vacant + before(m);
                Entry put = entry_of(from < kc ? from : 0);
                if (free && nth < over) put = mine[(kMaxList + nth) * 8];   // a conditional expression would choose between their addresses: the pad in memory
                if (free) mine[e * 8] = put;
                vacant += __builtin_popcountll(m);
            }
        } else {
            const Entry pad = entry_of(0);
            for (int e = base + lane; e < q; e += 64) mine[e * 8] = pad;
        }
        if constexpr (P) {
            most = wave_max_f(most);
            least = wave_min_f(least);
            most_lower = wave_max_f(most_lower);
            least_upper = wave_min_f(least_upper);
            if constexpr (ALL) {
                most_point = wave_max_f(most_point);
                least_point = wave_min_f(least_point);
            }
        } else {
            most = hi;
            least = lo;
        }
        if (lane == 0 && r < side.rows) {
            const float inf = __builtin_inff();
            float* rest = side.rest + (size_t)ch * side.rests * side.rows + row;
            rest[0] = bad ? inf : most;
            rest[side.rows] = bad ? -inf : least;
            if constexpr (P) {
                rest[2 * side.rows] = bad ? inf : most_lower;
                rest[3 * side.rows] = bad ? -inf : least_upper;
            }
            if constexpr (ALL) {
                rest[4 * side.rows] = bad ? inf : most_point;
                rest[5 * side.rows] = bad ? -inf : least_point;
            }
        }
        __syncthreads();
        constexpr int E = P ? 16 : 8, S = E / 2;   // bytes of an entry, and 16-byte pieces of the same entry of eight rows
        uint4* dst = reinterpret_cast<uint4*>(side.lists + ((size_t)ch * side.blocks + block / 2) * q * 16 * E) + (block & 1) * S;
        for (int i = tid; i < q * S; i += 512) dst[i / S * 2 * S + i % S] = reinterpret_cast<const uint4*>(stage)[i];
    };
    const int qx = kLengths[ix], qw = kLengths[iw], of_x = 2 * s.x.blocks;
    const int per = of_x + (qw ? 2 * s.w.blocks : 0);   // weights without lists: the first scan finds what bounds their rows as it reads them
#pragma unroll 1
    for (int unit = blockIdx.x; unit < per * s.C; unit += gridDim.x) {
        const int ch = unit / per, block = unit - ch * per;
        if (block < of_x) lists(std::integral_constant<int, ENDS>{}, s.x, qx, guess_x, ch, block);
        else lists(std::integral_constant<int, 1>{}, s.w, qw, guess_w, ch, block - of_x);
        __syncthreads();   // `stage` is free again
    }
}

// ---- scan ------------------------------------------------------------------------------------------------------------
enum { kWithPos, kOnlyValues, kBoxes, kBoxesAndPoints };
__device__ __host__ constexpr int strip_rows(bool pairs) { return pairs ? 4 : 8; }   // 32 bytes per k

// Lanes own rows of one operand (`ln`) and walk their lists; a strip of rows of the other (`sd`) lies in LDS, 32 bytes per
// k, so that an entry costs two 128-bit reads at a place of its own for eight differences (boxes in the strip: four rows,
// lower and upper end).  Odd lanes read the second half first: two lanes at the same k mod 8 then miss each other's banks.
//
// Bound by neither unit but by phases that take turns: the hand-out and the heads of the lists, a strip on its way to LDS, the
// walk.  5120 x 5120 with positions, at 2.7 clocks per instruction: batch 272, weights without lists, 50 us, the vector unit 22 % and
// LDS 13 % busy; batch 512 with both lists 65 + 68 us, 42 % and 37 %, 58 % of the latter bank conflicts of places in the order of k
// (where the order of a list is free, 34 to 42 %).  Boxes and points at batch 1024 136 us, the vector unit 49 %.  Four rows per
// strip with four workgroups per CU read the lists twice as often: 92 + 105 us before, and 73 + 91 with eight rows, both with the first
// pass's results stored one by one to 64 rows at a time (35 us of that pass); a strip's next chunk fetched between the entries made
// their loads wait for it (they return in order): 82 us.
//
// First pass: lanes are rows of x.  Where the weights have lists, its results go into s.partial, and the second pass, whose lanes are
// rows of w, takes them up; whichever is the last checks the bound, stores every output and notes those that fail it.
//
// Two workgroups of eight waves to a CU leave a lane 128 registers, which the first pass of boxes (3 spilled) and that of boxes and
// points (13) exceed: numbers of a tile, stored and fetched once per tile, none of them in the walk.
template <class T, int N>
__device__ __forceinline__ void store_row(T* to, const T (&v)[N]) {   // neighbouring elements, aligned to one
    static_assert(N % 4 == 0);
    typedef T Four __attribute__((ext_vector_type(4)));
    struct __attribute__((packed, aligned(4))) Any { Four v; };
#pragma unroll
    for (int j = 0; j < N; j += 4) reinterpret_cast<Any*>(to + j)->v = Four{v[j], v[j + 1], v[j + 2], v[j + 3]};
}

template <int MODE, bool SECOND>
__global__ void __launch_bounds__(512, 4) extremes_scan_kernel(Search s) {
    constexpr bool ALL = MODE == kBoxesAndPoints, BOX = MODE == kBoxes || ALL, PAIR_ENTRY = BOX && !SECOND, PAIR_STRIP = BOX && SECOND;
    static_assert(!(ALL && SECOND), "the second scans of boxes and points are those of boxes and of values");
    constexpr int RS = strip_rows(PAIR_STRIP), U = kMaxChunk / 512, NT = 512;
    extern __shared__ __align__(16) char lds[];
    if (s.head->dense) return;
    const Side& ln = SECOND ? s.w : s.x;
    const Side& sd = SECOND ? s.x : s.w;
    const int q = SECOND ? s.head->qw : s.head->qx;
    const bool both = s.head->qx != 0;   // second pass: the first has left something
    const bool last = SECOND || s.head->qw == 0;   // no second pass: the first checks the bounds
    if (SECOND ? q == 0 : !both && !last) return;
    const int K = s.K, KC = s.KC, C = s.C, N = s.w.rows;
    const int LG = SECOND ? s.lanes_second : last ? s.lanes_only : s.lanes_first, EG = NT / LG;
    const int tid = threadIdx.x, lane = tid & 63;
    const int eg = __builtin_amdgcn_readfirstlane(tid / LG), at = tid % LG;
    const unsigned odd = (lane & 1) * 16u;   // which half a lane reads first

    // Every XCD takes a contiguous run of tiles.  First pass: the lane blocks of one strip beside each other, so that w
    // streams from memory once.  Second: an eighth of the strips, which then stay in the XCD's L2, under every lane block in
    // turn, whose lists are read once.
    const int strips = (sd.rows + RS - 1) / RS, blocks = (ln.rows + LG - 1) / LG, tiles = strips * blocks;
    const int together = SECOND ? (strips + 7) / 8 : 1;
    auto place = [&](int t, int& strip, int& block) {
        const int group = t / (together * blocks), i = t - group * together * blocks, n = min(together, strips - group * together);
        block = i / n;
        strip = group * together + i - block * n;
    };
    const int xcd = blockIdx.x % 8;
    const int t_begin = (int)((long long)tiles * xcd / 8), t_end = (int)((long long)tiles * (xcd + 1) / 8);
    int tile = t_begin + (int)(blockIdx.x / 8);
    if (tile >= t_end) return;
    // The first tile is fixed, the others are taken as workgroups get there; lane 0 has the next one in hand a tile ahead.
    auto take = [&] { return t_begin + (int)(gridDim.x / 8) + atomicAdd(&s.head->taken[s.turn][xcd], 1); };
    int in_hand = tid == 0 ? take() : 0;

    while (true) {
        int strip, block;
        place(tile, strip, block);
        const int s0 = strip * RS, row0 = block * LG;
        const int l = min(row0 + at, ln.rows - 1);
        const bool live = row0 + at < ln.rows;
        const bool wave_live = __builtin_amdgcn_readfirstlane(row0 + (at & ~63)) < ln.rows;
        // values: the difference of the largest magnitude, with its sign, and 32 k; boxes: upper and lower bound
        float best[RS], low[RS], point[RS];
        unsigned key[RS];
#pragma unroll
        for (int j = 0; j < RS; j++) { best[j] = low[j] = point[j] = 0.f; key[j] = 0u; }
        int next_tile = t_end;
#pragma unroll 1
        for (int ch = 0; ch < C; ch++) {
            const int k0 = ch * KC, kc = min(KC, K - k0);
            __syncthreads();   // everyone is done with the strip before
            if (ch + 1 == C) {   // hand out the next tile
                if (tid == 0) *reinterpret_cast<int*>(lds) = in_hand;
                __syncthreads();
                next_tile = __builtin_amdgcn_readfirstlane(*reinterpret_cast<volatile int*>(lds));
                __syncthreads();
                if (tid == 0 && next_tile < t_end) in_hand = take();
            }
            {
                const auto rl = __builtin_amdgcn_make_buffer_rsrc((void*)(sd.v + (size_t)s0 * K + k0), 0, 0x7fffffff, 0x00020000);
                const auto ru = __builtin_amdgcn_make_buffer_rsrc((void*)((PAIR_STRIP ? sd.v2 : sd.v) + (size_t)s0 * K + k0), 0, 0x7fffffff, 0x00020000);
                float t[U][8];
#pragma unroll
                for (int u = 0; u < U; u++) {
                    if (u * NT >= kc || (q == 0 && !(!SECOND && last))) continue;
                    const unsigned k4 = (unsigned)min(u * NT + tid, kc - 1) * 4u;   // lanes past the chunk store nothing
#pragma unroll
                    for (int j = 0; j < RS; j++) {
                        const int row = min(j, sd.rows - 1 - s0) * K * 4;
                        t[u][PAIR_STRIP ? 2 * j : j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rl, k4, row, 0));
                        if constexpr (PAIR_STRIP) t[u][2 * j + 1] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(ru, k4, row, 0));
                    }
                }
                if (!SECOND && last) {   // weights without lists: what bounds the strip's rows in this chunk is their largest and smallest
                    float v[16];
#pragma unroll
                    for (int j = 0; j < 8; j++) { v[j] = t[0][j]; v[j + 8] = -t[0][j]; }
#pragma unroll
                    for (int u = 1; u < U; u++)
                        if (u * NT < kc) {
#pragma unroll
                            for (int j = 0; j < 8; j++) {
                                v[j] = __builtin_elementwise_maximum(v[j], t[u][j]);
                                v[j + 8] = __builtin_elementwise_maximum(v[j + 8], -t[u][j]);
                            }
                        }
                    float* part = reinterpret_cast<float*>(lds);   // [wave][16]
                    const float m = wave_max_of_16(v, lane);
                    if ((lane & 3) == 0) part[(tid >> 6) * 16 + (lane >> 2)] = m;
                    __syncthreads();
                    if (tid < 16) {
                        float r = part[tid];
#pragma unroll
                        for (int i = 1; i < NT / 64; i++) r = __builtin_elementwise_maximum(r, part[i * 16 + tid]);
                        if (not_finite(r)) r = __builtin_inff();
                        // workgroups that have this strip under other rows write the same
                        if (s0 + (tid & 7) < sd.rows) sd.rest[((size_t)ch * 2 + (tid >> 3)) * sd.rows + s0 + (tid & 7)] = tid < 8 ? r : -r;
                    }
                    __syncthreads();
                }
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const int k = u * NT + tid;
                    if (k < kc && q != 0) {
                        *reinterpret_cast<F4*>(lds + k * 32) = F4{t[u][0], t[u][1], t[u][2], t[u][3]};
                        *reinterpret_cast<F4*>(lds + k * 32 + 16) = F4{t[u][4], t[u][5], t[u][6], t[u][7]};
                    }
                }
            }
            using Entry = typename std::conditional<PAIR_ENTRY, uint4, uint2>::type;
            const Entry* list = reinterpret_cast<const Entry*>(ln.lists) + (((size_t)ch * ln.blocks + l / 16) * q) * 16 + (l & 15);
            const unsigned kb = (unsigned)k0 * 32u;
            auto entry = [&](const Entry& en) {
                unsigned k32;
                if constexpr (PAIR_ENTRY) k32 = en.z;
                else k32 = en.y;
                const float v = __uint_as_float(en.x);
                const unsigned from = k32 ^ odd;
                const F4 half[2] = {*reinterpret_cast<const F4*>(lds + from), *reinterpret_cast<const F4*>(lds + (from ^ 16u))};
#pragma unroll
                for (int j = 0; j < RS; j++) {
                    if constexpr (PAIR_STRIP) {
                        const float dl = half[j / 2][2 * (j & 1)] - v, du = half[j / 2][2 * (j & 1) + 1] - v;
                        best[j] = __builtin_fmaxf(__builtin_fmaxf(best[j], __builtin_fabsf(dl)), __builtin_fabsf(du));
                        low[j] = __builtin_fmaxf(__builtin_fmaxf(low[j], dl), -du);
                    } else {
                        const float other = half[j / 4][j & 3];
                        if constexpr (BOX) {
                            const float dl = v - other, du = __uint_as_float(en.y) - other;
                            best[j] = __builtin_fmaxf(__builtin_fmaxf(best[j], __builtin_fabsf(dl)), __builtin_fabsf(du));
                            low[j] = __builtin_fmaxf(__builtin_fmaxf(low[j], dl), -du);
                            if constexpr (ALL) point[j] = __builtin_fmaxf(point[j], __builtin_fabsf(__uint_as_float(en.w) - other));
                        } else {
                            const float df = SECOND ? other - v : v - other;
                            if constexpr (MODE == kWithPos) {
                                const bool wins = __builtin_fabsf(df) > __builtin_fabsf(best[j]);
                                best[j] = wins ? df : best[j];
                                key[j] = wins ? kb + k32 : key[j];
                            } else {
                                best[j] = __builtin_fmaxf(best[j], __builtin_fabsf(df));
                            }
                        }
                    }
                }
            };
            // entries eg, eg + EG, ... four at a time (boxes two: registers); a place past the end repeats the last
            constexpr int AT = PAIR_ENTRY ? 2 : 4;
            const int quads = ((q - eg + EG - 1) / EG + AT - 1) / AT;
            Entry en[AT], en_next[AT];
            auto read = [&](Entry (&e)[AT], int i) {
#pragma unroll
                for (int c = 0; c < AT; c++) e[c] = list[min(eg + (AT * i + c) * EG, q - 1) * 16];
            };
            if (wave_live && q != 0) read(en, 0);
            __syncthreads();
            if (wave_live && q != 0) {
#pragma unroll 1
                for (int i = 0; i < quads; i++) {
                    read(en_next, i + 1);
#pragma unroll
                    for (int c = 0; c < AT; c++) entry(en[c]);
#pragma unroll
                    for (int c = 0; c < AT; c++) en[c] = en_next[c];
                }
            }
        }

        // odd lanes hold the halves the other way round
        auto swap = [&](auto& p, auto& r) { const auto c = p; p = lane & 1 ? r : p; r = lane & 1 ? c : r; };
#pragma unroll
        for (int j = 0; j < RS / 2; j++) {
            swap(best[j], best[j + RS / 2]);
            if constexpr (BOX) swap(low[j], low[j + RS / 2]);
            if constexpr (ALL) swap(point[j], point[j + RS / 2]);
            if constexpr (MODE == kWithPos) swap(key[j], key[j + RS / 2]);
        }
        if (EG > 1) {   // the groups of lanes that shared a row's list
            float* pa = reinterpret_cast<float*>(lds);
            unsigned* pb = reinterpret_cast<unsigned*>(lds + NT / 2 * RS * 4);
            float* pc = reinterpret_cast<float*>(lds + NT * RS * 4);
            for (int half = EG / 2; half > 0; half /= 2) {
                __syncthreads();
                if (eg >= half && eg < 2 * half) {
#pragma unroll
                    for (int j = 0; j < RS; j++) {
                        pa[j * (NT / 2) + tid - half * LG] = best[j];
                        if constexpr (MODE != kOnlyValues) pb[j * (NT / 2) + tid - half * LG] = BOX ? __float_as_uint(low[j]) : key[j];
                        if constexpr (ALL) pc[j * (NT / 2) + tid - half * LG] = point[j];
                    }
                }
                __syncthreads();
                if (eg < half) {
#pragma unroll
                    for (int j = 0; j < RS; j++) {
                        const float o = pa[j * (NT / 2) + tid];
                        if constexpr (MODE == kWithPos) {
                            const unsigned ok = pb[j * (NT / 2) + tid];
                            const float ao = __builtin_fabsf(o), ab = __builtin_fabsf(best[j]);
                            if (ao > ab || (ao == ab && ok < key[j])) { best[j] = o; key[j] = ok; }
                        } else {
                            best[j] = __builtin_fmaxf(best[j], o);
                            if constexpr (BOX) low[j] = __builtin_fmaxf(low[j], __uint_as_float(pb[j * (NT / 2) + tid]));
                            if constexpr (ALL) point[j] = __builtin_fmaxf(point[j], pc[j * (NT / 2) + tid]);
                        }
                    }
                }
            }
        }
        auto pos_of = [&](int j) { return best[j] == 0.f ? 0 : (int)((key[j] >> 5) | (__float_as_uint(best[j]) & 0x80000000u)); };
        if (eg == 0 && wave_live) {
            if (!last) {
                if (live) {   // 16 * RS bytes of a row (8 * RS without positions): whole sectors, and all of a lane's in few stores
                    if constexpr (MODE == kOnlyValues) {
                        store_row(s.partial + (size_t)l * s.pitch + s0, best);
                    } else {
                        float* to = s.partial + 2 * ((size_t)l * s.pitch + s0);
                        auto second = [&](int j) { return BOX ? low[j] : __int_as_float(pos_of(j)); };
#pragma unroll
                        for (int j = 0; j < RS; j += 2)
                            *reinterpret_cast<F4*>(to + 2 * j) = F4{__builtin_fabsf(best[j]), second(j), __builtin_fabsf(best[j + 1]), second(j + 1)};
                        if constexpr (ALL) store_row(s.partial3 + (size_t)l * s.pitch + s0, point);
                    }
                }
            } else {
                float limit[RS], limit_low[RS], limit_point[RS];   // what neither list holds
#pragma unroll
                for (int j = 0; j < RS; j++) limit[j] = limit_low[j] = limit_point[j] = -kNever;
                for (int ch = 0; ch < C; ch++) {
                    const float* lr = ln.rest + (size_t)ch * ln.rests * ln.rows + l;
                    constexpr int LL = BOX && !SECOND ? 2 : 0, SL = BOX && SECOND ? 2 : 0, LP = ALL ? 4 : 0;   // which of a side's, for lower bounds and points
                    const float lh = lr[0], ll = lr[ln.rows], lh_low = lr[LL * ln.rows], ll_low = lr[(LL + 1) * ln.rows];
                    const float lh_point = lr[LP * ln.rows], ll_point = lr[(LP + 1) * ln.rows];
#pragma unroll
                    for (int j = 0; j < RS; j++) {
                        const float* sr = sd.rest + (size_t)ch * sd.rests * sd.rows + min(s0 + j, sd.rows - 1);
                        limit[j] = __builtin_fmaxf(limit[j], __builtin_fmaxf(sr[0] - ll, lh - sr[sd.rows]));
                        if constexpr (BOX) limit_low[j] = __builtin_fmaxf(limit_low[j], __builtin_fmaxf(sr[SL * sd.rows] - ll_low, lh_low - sr[(SL + 1) * sd.rows]));
                        if constexpr (ALL) limit_point[j] = __builtin_fmaxf(limit_point[j], __builtin_fmaxf(sr[0] - ll_point, lh_point - sr[sd.rows]));
                    }
                }
                float mu[RS], add[RS];   // before the stores, which they might alias
#pragma unroll
                for (int j = 0; j < RS; j++) {
                    const int n = SECOND ? l : min(s0 + j, N - 1);
                    mu[j] = s.mean ? s.mean[n] : 0.f;
                    add[j] = s.bias ? s.bias[n] : 0.f;
                }
                auto stored = [&](float v, int j) {
                    if (s.mean) v = v - mu[j];
                    if (s.bias) v = v + add[j];
                    return v;
                };
                unsigned failed = 0;
                float got[RS], got_low[RS], got_point[RS];
                int got_pos[RS];
#pragma unroll
                for (int j = 0; j < RS; j++) {
                    const size_t from = SECOND ? (size_t)min(s0 + j, sd.rows - 1) * s.pitch + l : 0;   // what the first pass left
                    float have = 0.f, with = 0.f;
                    if constexpr (SECOND) {
                        if constexpr (MODE == kOnlyValues) {
                            if (both) have = s.partial[from];
                        } else if (both) {
                            const float2 left = reinterpret_cast<const float2*>(s.partial)[from];
                            have = left.x;
                            with = left.y;
                        }
                    }
                    // an infinite limit is a row that the lists cannot speak for, whatever they found
                    bool settled;
                    if constexpr (BOX) {
                        const float lo = __builtin_fmaxf(low[j], with), up = __builtin_fmaxf(best[j], have);
                        settled = up >= limit[j] && lo >= limit_low[j] && limit[j] < __builtin_inff();
                        if constexpr (ALL) settled = settled && point[j] >= limit_point[j];
                        got_low[j] = stored(lo, j);
                        got[j] = stored(up, j);
                        if constexpr (ALL) got_point[j] = stored(point[j], j);
                    } else if constexpr (MODE == kOnlyValues) {
                        const float v = __builtin_fmaxf(best[j], have);
                        settled = v >= limit[j] && limit[j] < __builtin_inff();
                        got[j] = stored(v, j);
                    } else {
                        float v = __builtin_fabsf(best[j]);
                        int p = pos_of(j);
                        const int hp = __float_as_int(with);
                        if (have > v || (have == v && (hp & 0x7fffffff) < (p & 0x7fffffff))) { v = have; p = hp; }
                        settled = v > limit[j];   // at the limit a lower k might hold the same value
                        got[j] = stored(v, j);
                        got_pos[j] = p;
                    }
                    if (live && s0 + j < sd.rows && !settled) failed |= 1u << j;
                }
                auto index = [&](int j) { return SECOND ? (s0 + j) * N + l : l * N + s0 + j; };
                // all of them: what has failed is written again by a later launch
                if (SECOND || s0 + RS > N) {
#pragma unroll
                    for (int j = 0; j < RS; j++)
                        if (live && s0 + j < sd.rows) {
                            const int o = index(j);
                            if constexpr (BOX) {
                                s.out[o] = got_low[j];
                                s.out2[o] = got[j];
                                if constexpr (ALL) s.out3[o] = got_point[j];
                            } else {
                                s.out[o] = got[j];
                                if constexpr (MODE == kWithPos) s.pos[o] = got_pos[j];
                            }
                        }
                } else if (live) {
                    const int o = index(0);
                    if constexpr (BOX) {
                        store_row(s.out + o, got_low);
                        store_row(s.out2 + o, got);
                        if constexpr (ALL) store_row(s.out3 + o, got_point);
                    } else {
                        store_row(s.out + o, got);
                        if constexpr (MODE == kWithPos) store_row(s.pos + o, got_pos);
                    }
                }
                if (__ballot(failed != 0)) {
                    int n = 0;
#pragma unroll
                    for (int j = 0; j < RS; j++) n += __builtin_popcountll(__ballot(failed >> j & 1));
                    int first = lane == 0 ? atomicAdd(&s.head->failed, n) : 0;
                    first = __builtin_amdgcn_readfirstlane(first);
#pragma unroll
                    for (int j = 0; j < RS; j++) {
                        const unsigned long long m = __ballot(failed >> j & 1);
                        const int at = first + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0));
                        if ((failed >> j & 1) && at < s.walk_most) s.walk[at] = index(j) | s.note;   // more: the full walk follows
                        first += __builtin_popcountll(m);
                    }
                }
            }
        }
        tile = next_tile;
        if (tile >= t_end) return;
    }
}

// ---- walk ------------------------------------------------------------------------------------------------------------
// The outputs that the lists could not settle, a wave for each, all k and the comparisons of the other kernels.  More than
// `s.walk_most` of them: the full walk of the layer is cheaper, and follows.
template <int MODE>
__global__ void __launch_bounds__(256) extremes_walk_kernel(Search s) {
    if (s.head->dense) return;
    const int failed = s.head->failed;
    if (failed > s.walk_most) {
        if (blockIdx.x == 0 && threadIdx.x == 0) s.head->full = 1;
        return;
    }
    const int lane = threadIdx.x & 63, K = s.K, N = s.w.rows;
    for (int i = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6)); i < failed; i += gridDim.x * 4) {
        const int note = __builtin_amdgcn_readfirstlane(s.walk[i]), o = note & (kBoxFails - 1);
        const float* xr = s.x.v + (size_t)(o / N) * K;
        const float* wr = s.w.v + (size_t)(o % N) * K;
        if constexpr (MODE == kBoxes || MODE == kBoxesAndPoints) {
            auto walk = [&](auto box, auto points) {
                constexpr bool BOX = decltype(box)::value, POINT = decltype(points)::value;
                const float* ur = s.x.v2 + (size_t)(o / N) * K;
                const float* pr = POINT ? s.x.v3 + (size_t)(o / N) * K : nullptr;
                float up = 0.f, lo = 0.f, point = 0.f;
                auto one = [&](float x, float u, float w) {
                    const float tl = x - w, tu = u - w, al = __builtin_fabsf(tl), au = __builtin_fabsf(tu);
                    up = __builtin_fmaxf(up, __builtin_fmaxf(al, au));
                    if (!(tl < 0.f && tu > 0.f)) lo = __builtin_fmaxf(lo, __builtin_fminf(al, au));
                };
                for (int kb = 0; kb < K; kb += 256 * 4) {
                    float4_any x[4], u[4], w[4], p[4];
#pragma unroll
                    for (int c = 0; c < 4; c++) {
                        const int k = min(kb + c * 256 + lane * 4, K - 4);   // the last vector is moved back, those past the end repeat it
                        if constexpr (BOX) x[c] = *reinterpret_cast<const float4_any*>(xr + k);
                        if constexpr (BOX) u[c] = *reinterpret_cast<const float4_any*>(ur + k);
                        if constexpr (POINT) p[c] = *reinterpret_cast<const float4_any*>(pr + k);
                        w[c] = *reinterpret_cast<const float4_any*>(wr + k);
                    }
#pragma unroll
                    for (int c = 0; c < 4; c++)
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            if constexpr (BOX) one(x[c].v[e], u[c].v[e], w[c].v[e]);
                            if constexpr (POINT) point = __builtin_fmaxf(point, __builtin_fabsf(p[c].v[e] - w[c].v[e]));
                        }
                }
                if constexpr (BOX) {
                    up = wave_max(up);
                    lo = wave_max(lo);
                    if (lane == 63) {
                        s.out[o] = shifted_value(s.mean, s.bias, o % N, lo);
                        s.out2[o] = shifted_value(s.mean, s.bias, o % N, up);
                    }
                }
                if constexpr (POINT) {
                    point = wave_max(point);
                    if (lane == 63) s.out3[o] = shifted_value(s.mean, s.bias, o % N, point);
                }
            };
            // The second scans of boxes and of points note an output each, for what it is that fails there: the 23933 outputs of a
            // trained 1024 x 3072 -> 5120 layer, all of them noted twice, took 228 us with both walked for either note, 119 now.
            using Yes = std::true_type;
            using No = std::false_type;
            if (MODE == kBoxes || (note & (kBoxFails | kPointFails)) == kBoxFails) walk(Yes{}, No{});
            else if (note & kBoxFails) walk(Yes{}, Yes{});
            else walk(No{}, Yes{});
        } else {
            float v = 0.f;
            int p = 0;   // k with the sign of the difference
            auto one = [&](float x, float w, int k) {
                const float df = x - w, a = __builtin_fabsf(df);
                const bool wins = a > v;
                v = wins ? a : v;
                p = wins ? (int)((unsigned)k | (__float_as_uint(df) & 0x80000000u)) : p;
            };
            for (int kb = 0; kb < K; kb += 256 * 5) {
                float4_any x[5], w[5];
#pragma unroll
                for (int c = 0; c < 5; c++) {
                    const int k = min(kb + c * 256 + lane * 4, K - 4);   // the last vector is moved back, those past the end repeat it
                    x[c] = *reinterpret_cast<const float4_any*>(xr + k);
                    w[c] = *reinterpret_cast<const float4_any*>(wr + k);
                }
#pragma unroll
                for (int c = 0; c < 5; c++)
#pragma unroll
                    for (int e = 0; e < 4; e++) one(x[c].v[e], w[c].v[e], min(kb + c * 256 + lane * 4, K - 4) + e);
            }
            wave_best(v, p);
            if (lane == 63) {
                s.out[o] = shifted_value(s.mean, s.bias, o % N, v);
                if constexpr (MODE == kWithPos) s.pos[o] = v > 0.f ? p : 0;
            }
        }
    }
}

}  // namespace

// ---- host ------------------------------------------------------------------------------------------------------------
namespace {

struct Layout {
    int C, KC, mb, nb, pitch;
    size_t counts, reach, partial, partial3, walk, x_lists, w_lists, x_rest, w_rest, total;   // byte offsets in the workspace
};

// More outputs than these go to the full walk; forced lists have none after them.
size_t walk_most(const Problem& pr, ForwardKind kind) {   // the two second scans of boxes and points may both note an output
    const size_t outputs = (size_t)pr.B * pr.NG * (kind == ForwardKind::kValueBounds ? 2 : 1);
    return g_extremes > 0 ? outputs : outputs / 16;
}

Layout layout_of(const Problem& pr, ForwardKind kind) {
    const bool all = kind == ForwardKind::kValueBounds, boxes = kind == ForwardKind::kBounds || all;
    Layout l{};
    l.C = (pr.K + kMaxChunk - 1) / kMaxChunk;
    l.KC = ((pr.K + l.C - 1) / l.C + 63) / 64 * 64;
    l.mb = (pr.B + 15) / 16;
    l.nb = (pr.NG + 15) / 16;
    size_t at = 0;
    auto take = [&](size_t bytes) { const size_t here = at; at += (bytes + 255) / 256 * 256; return here; };
    take(sizeof(Header));
    l.counts = take((size_t)kSampleGroups * kSampleGroups * 64);
    l.pitch = (pr.NG + 7) / 8 * 8;
    l.partial = take((size_t)pr.B * l.pitch * (kind == ForwardKind::kValues ? 1 : 2) * sizeof(float));
    l.partial3 = take(all ? (size_t)pr.B * l.pitch * sizeof(float) : 0);
    l.walk = take(walk_most(pr, kind) * sizeof(int));
    l.reach = take(2 * 8 * kSampled * sizeof(float));
    l.x_lists = take((size_t)l.C * l.mb * kMaxList * 16 * (boxes ? 16 : 8));
    l.w_lists = take((size_t)l.C * l.nb * kMaxList * 16 * 8);
    l.x_rest = take((size_t)l.C * (all ? 6 : boxes ? 4 : 2) * pr.B * sizeof(float));
    l.w_rest = take((size_t)l.C * 2 * pr.NG * sizeof(float));
    l.total = at;
    return l;
}

template <int MODE, bool SECOND>
hipError_t launch_scan(const Search& s, const Problem& pr, hipStream_t stream) {
    auto kern = extremes_scan_kernel<MODE, SECOND>;
    static LdsRecord allowed = {};
    const size_t strip = (size_t)s.KC * 32, over = MODE == kBoxesAndPoints ? 24576 : 16384;   // the strip, or what the groups of lanes hand over
    const size_t lds = strip > over ? strip : over;
    if (hipError_t e = allow_lds(kern, (size_t)kMaxChunk * 32, pr.device, allowed); e != hipSuccess) return e;
    const Side &ln = SECOND ? s.w : s.x, &sd = SECOND ? s.x : s.w;
    const int rows = strip_rows(MODE == kBoxes && SECOND), lanes = SECOND ? s.lanes_second : s.lanes_first;
    const long tiles = (long)((sd.rows + rows - 1) / rows) * ((ln.rows + lanes - 1) / lanes);
    const long most = 2L * pr.num_cu / 8 * 8;   // two strips fit a CU
    const unsigned grid = (unsigned)(tiles < most ? (tiles + 7) / 8 * 8 : most);
    hipLaunchKernelGGL(kern, dim3(grid), dim3(512), lds, stream, s);
    return hipGetLastError();
}

template <int ENDS>
hipError_t launch_lists(const Search& s, int num_cu, hipStream_t stream) {
    auto resident = [](int nv) { return nv <= 24 && ENDS == 1 ? 3 : 2; };   // per CU, by registers
    const int units = 2 * s.C * (s.x.blocks + s.w.blocks);
    const size_t stage = (size_t)2 * kMaxList * 8 * (ENDS > 1 ? 16 : 8);
#define LISTS(NV)                                                                                                                 \
    do {                                                                                                                          \
        hipLaunchKernelGGL((extremes_sample_kernel<NV, ENDS>), dim3(kSampleGroups * kSampleGroups), dim3(1024), 0, stream, s);     \
        if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;                                                          \
        const dim3 grid((unsigned)std::min(units, resident(NV) * num_cu));                                                        \
        if (ENDS == 1 && s.pos) hipLaunchKernelGGL((extremes_select_kernel<NV, ENDS, ENDS != 1>), grid, dim3(512), stage, stream, s); \
        else hipLaunchKernelGGL((extremes_select_kernel<NV, ENDS, true>), grid, dim3(512), stage, stream, s);                      \
    } while (0)
    if (s.KC <= 1024) LISTS(16);
    else if (s.KC <= 1536) LISTS(24);
    else if (s.KC <= 2048) LISTS(32);
    else LISTS(40);
#undef LISTS
    return hipGetLastError();
}

// Lanes of a workgroup that own different rows (the others share their lists): as many as leave two tiles per workgroup.
int lanes_for(int rows, int strips, int num_cu) {
    int lanes = 512;
    while (lanes > 128 && (long)strips * ((rows + lanes - 1) / lanes) < 4L * num_cu) lanes /= 2;
    while (lanes > 64 && rows <= lanes / 2) lanes /= 2;
    return lanes;
}

}  // namespace

// The layers for which the lists are expected to be faster, by an estimate of their time on normally distributed values
// (lists of about 50 and 100 entries per chunk), fitted to eight sizes of weights from 1024 x 784 to 5120 x 5120 at
// batches of 32 to 1024, against that of the full walk: e.g. 1024 x 3072 at batch 512 (positions) 92 us in full and
// 80 with lists, at 272 56 and 78; 5120 x 5120 at 64, 128 and 1024 93, 165, 909 and 120, 138, 282 us.
// Few outputs of a long reduction leave the sample and the scans to few workgroups, which walk all its chunks in turn: the terms
// beyond one and two chunks, fitted to 552 layers of 600 to 40000 inputs, normal and uniform inputs, of which 66 were slower
// with lists before (256 x 25088 -> 256 with positions 94 us in full, 174 with lists; 1024 x 25088 -> 64 values 88 and 192), and
// 3 of the 443 that are left are, by 2 to 11 %.  Sample, lists and first scan have become faster since, and points share those of the
// boxes, so that layers stay in full which lists would serve: values and bounds of 256 x 2048 -> 2048 159 us, 60 to 109 with lists,
// 32 x 5120 -> 5120 167, 85 to 142.
// The size alone decides, for the caller asks for the workspace before there is a device to ask.
static bool lists_pay(const Problem& pr, ForwardKind kind) {
    if (g_tile_override >= 0 || pr.K < 512) return false;
    const double outputs = (double)pr.B * pr.NG, weights = (double)pr.NG * pr.K;
    const bool boxes = kind != ForwardKind::kInf && kind != ForwardKind::kValues;   // with points: where the boxes alone pay
    if (boxes) kind = ForwardKind::kBounds;
    const double beyond_one = std::max(0, pr.K - kMaxChunk), beyond_two = std::max(0, pr.K - 2 * kMaxChunk);
    const double us = (boxes ? 65 : 55) + 2.1e-6 * weights + (boxes ? 5.3e-5 : 3.5e-5) * outputs +
                      (boxes ? 3.4e-6 : 1.1e-6) * pr.B * beyond_one + (3.3e-3 + (boxes ? 5.4e-9 : 4.2e-9) * outputs) * beyond_two;
    return 1.1 * us + 5 <= full_walk_us(pr, kind, 256);
}

// Rows of one sequence of launches: all of them where its scratch memory stays below kScratchMost, else equal shares of whole
// blocks (each lists the weights again, 17 + 32 us of some 900 at 4096 x 5120 x 5120).  0: the lists of the weights alone leave
// room for less than kFewestRows, or the layer has none.
constexpr size_t kScratchMost = (size_t)256 << 20;
constexpr int kFewestRows = 256;
static int rows_at_once(const Problem& pr, ForwardKind kind) {
    if (g_extremes == 0 || pr.HW != 1 || pr.G != 1 || pr.NG <= 16 || pr.K < 4 || pr.K > 16 * kMaxChunk) return 0;
    if (kind == ForwardKind::kValueBounds && pr.K % 4 != 0) return 0;   // no full walk of values to follow
    Problem part = pr;
    for (int shares = 1;; shares++) {
        part.B = shares == 1 ? pr.B : ((pr.B + shares - 1) / shares + 15) / 16 * 16;
        if (shares > 1 && part.B < kFewestRows) return 0;
        if (layout_of(part, kind).total <= kScratchMost) break;
    }
    return g_extremes > 0 || lists_pay(part, kind) ? part.B : 0;
}

size_t extremes_workspace(const Problem& pr, ForwardKind kind, int& rows) {
    rows = rows_at_once(pr, kind);
    if (rows == 0) return 0;
    Problem part = pr;
    part.B = rows;
    return layout_of(part, kind).total;
}

hipError_t extremes_forward(const float* x, const float* x2, const float* x3, const float* w, float* out, float* out2, float* out3,
                            int32_t* pos, void* workspace, const Problem& pr, hipStream_t stream, const int** gate) {
    const bool all = x3 != nullptr, boxes = x2 != nullptr;
    const ForwardKind kind = all ? ForwardKind::kValueBounds : boxes ? ForwardKind::kBounds : pos ? ForwardKind::kInf : ForwardKind::kValues;
    const Layout l = layout_of(pr, kind);
    char* ws = static_cast<char*>(workspace);
    Search s{};
    s.head = reinterpret_cast<Header*>(ws);
    s.counts = reinterpret_cast<unsigned char*>(ws + l.counts);
    s.reach = reinterpret_cast<float*>(ws + l.reach);
    s.partial = reinterpret_cast<float*>(ws + l.partial);
    s.partial3 = reinterpret_cast<float*>(ws + l.partial3);
    s.pitch = l.pitch;
    s.walk = reinterpret_cast<int*>(ws + l.walk);
    s.walk_most = (int)std::min<size_t>(walk_most(pr, kind), INT32_MAX);
    s.x = Side{x, x2, x3, pr.B, l.mb, ws + l.x_lists, reinterpret_cast<float*>(ws + l.x_rest), all ? 6 : boxes ? 4 : 2};
    s.w = Side{w, nullptr, nullptr, pr.NG, l.nb, ws + l.w_lists, reinterpret_cast<float*>(ws + l.w_rest), 2};
    s.out = out; s.out2 = out2; s.out3 = out3; s.pos = pos;
    s.mean = pr.mean; s.bias = pr.bias;
    s.K = pr.K; s.C = l.C; s.KC = l.KC;
    s.note = all ? kBoxFails | kPointFails : 0;
    s.lanes_first = lanes_for(pr.B, (pr.NG + 7) / 8, pr.num_cu);
    // Without a list for the weights the lists of x are short, and a strip on its way to LDS costs more than its walk: where two blocks of
    // rows fit a workgroup with an eighth of its lanes to spare, they share it (200 to 448 rows, 5120 -> 5120, a whole pass 91 -> 83 and
    // 97 -> 92 us; 3072 -> 4096 76 -> 67).  512 rows of 5120 outputs would leave the last round of strips to a quarter of the
    // workgroups (64 -> 73 us of the scan), and with both lists two blocks are as fast at best.
    s.lanes_only = s.lanes_first;
    while (s.lanes_only < 512 && pr.B > s.lanes_only && pr.B <= s.lanes_only * 7 / 4) s.lanes_only *= 2;
    const int second_rows = strip_rows(boxes);
    s.lanes_second = lanes_for(pr.NG, (pr.B + second_rows - 1) / second_rows, pr.num_cu);
    s.price_x = 1.f;
    s.price_w = all ? 3.f : boxes ? 2.f : 1.f;
    s.price_both = all ? 120.f : 60.f;
    // in list entries of one row: a walked output reads two rows, 3 ns with all waves at it, an entry takes 0.1 ps per output; with
    // points five rows in two walks, 10 ns, and 0.2 ps.  The price there is higher than that, for what a sample of 64 x 64 outputs
    // does not see: with 12 instead of 18 1024 x 3072 -> 5120 normal values take 533 instead of 437 us, 512 x 4096 -> 4096 291 and 254,
    // and nothing is faster by more than 1 %.
    s.price_fail = (all ? 18.f : boxes ? 9.f : 6.f) * pr.K;
    s.price_dense = g_extremes > 0 ? 3e38f : (all ? 0.7f : boxes ? 0.5f : 0.2f) * pr.K;
    *gate = &s.head->full;
    if (hipError_t e = all ? launch_lists<3>(s, pr.num_cu, stream) : boxes ? launch_lists<2>(s, pr.num_cu, stream) : launch_lists<1>(s, pr.num_cu, stream); e != hipSuccess) return e;
    auto walk = [&](auto mode) {
        hipLaunchKernelGGL(extremes_walk_kernel<decltype(mode)::value>, dim3(4 * pr.num_cu), dim3(256), 0, stream, s);
        return hipGetLastError();
    };
    auto second_of = [&](int turn, int note = 0) { Search t = s; t.turn = turn; t.note = note; return t; };
    if (all) {
        if (hipError_t e = launch_scan<kBoxesAndPoints, false>(s, pr, stream); e != hipSuccess) return e;
        if (hipError_t e = launch_scan<kBoxes, true>(second_of(1, kBoxFails), pr, stream); e != hipSuccess) return e;
        Search points = second_of(2, kPointFails);
        points.x.v = x3;
        points.x.rest = s.x.rest + (size_t)4 * pr.B;
        points.out = out3;
        points.partial = s.partial3;
        points.lanes_second = lanes_for(pr.NG, (pr.B + 7) / 8, pr.num_cu);
        if (hipError_t e = launch_scan<kOnlyValues, true>(points, pr, stream); e != hipSuccess) return e;
        return walk(std::integral_constant<int, kBoxesAndPoints>{});
    }
#define SCANS(MODE)                                                                                                       \
    do {                                                                                                                  \
        if (hipError_t e = launch_scan<MODE, false>(s, pr, stream); e != hipSuccess) return e;                   \
        if (hipError_t e = launch_scan<MODE, true>(second_of(1), pr, stream); e != hipSuccess) return e;         \
        return walk(std::integral_constant<int, MODE>{});                                                                 \
    } while (0)
    if (boxes) SCANS(kBoxes);
    if (pos) SCANS(kWithPos);
    SCANS(kOnlyValues);
#undef SCANS
}

}  // namespace ldist
