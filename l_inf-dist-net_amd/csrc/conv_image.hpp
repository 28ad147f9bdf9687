// Launch shape shared by the kernels that run the 3x3 distance layer straight from images
// (inf_conv_forward.hip: values and argmax; bound_conv_forward.hip: interval bounds).
#pragma once
#include "kernels.hpp"
#include "tile.hpp"

namespace ldist {
namespace convimg {

constexpr int kTM = 8, kTN = 4;   // positions x outputs per lane
constexpr int kCC = 4;            // channels per weight stage
constexpr int kTrack = 1;         // channels per recorded unit
constexpr int kKC = kCC * 9;      // k values per weight stage
constexpr int kMaxThreads = 256;
constexpr int kBNP = 68;          // row length of the weight stage: 64 outputs + 4, a constant so that reads take immediate offsets
constexpr int kWRegs = 9;         // weight words a lane carries from global to LDS per stage (64 outputs x 36 / 256)
constexpr int kRest = 6;          // weight words a lane has in flight beyond those, where a workgroup has fewer lanes (values only)
// image words a lane carries per stage when the channels are staged (4 channels x rows held x padded width / lanes)
__host__ __device__ constexpr int x_regs(int S) { return S == 1 ? 7 : 10; }

struct ConvFwd {
    int B, G, CG, NG, K;         // images, groups, channels and outputs per group, K = 9*CG
    int H, W, HO, WO, P;         // image, output positions, padding
    int R, NR, WP, CGP;          // output rows per workgroup, image rows held, padded row length, CG rounded up to kCC
    int SEG, ML, NL, BN;         // 8-position segments per output row, lanes along positions / outputs, outputs per
                                 // workgroup
    int tiles_h, tiles_n;
    int vec_in, vec_out;         // 128-bit global loads of image rows / stores of results allowed
    int resident;                // 1: all channels of the image rows stay in LDS; 0: staged kCC channels at a time
    int xwords;                  // floats of the image area in LDS
    int cstride;                 // resident: floats between channels (NR*WP padded to 4 mod 8); staged: unused
    const float *mean, *bias;    // per channel: (v - mean) + bias is stored; either may be null
    int KG, GT;                  // groups of lanes that share a tile's channels, lanes of one
};

constexpr size_t kLdsLimit = 160 * 1024;

// Fills the launch shape; false when this kernel does not cover the geometry.
// Channel stride of the resident image area: rows stay 16-byte aligned (a multiple of 4) and consecutive
// channels start 4 banks apart modulo 8, so that channel c begins at bank 4c mod 64.
inline int channel_stride(int plane) { return plane % 8 == 4 ? plane : plane + (4 - plane % 8 + 8) % 8; }

// nx: images staged side by side (1: the input; 2: lower and upper interval ends, which are always staged and may
// have any number of channels: that kernel masks the channels a last stage does not have).
inline bool plan(const ConvGeom& q, int G, int CO, ConvFwd& a, int nx = 1) {
    if (q.KH != 3 || q.KW != 3 || q.D != 1 || (q.S != 1 && q.S != 2)) return false;
    if (G <= 0 || q.C % G != 0 || CO % G != 0) return false;
    if ((long long)kCC * q.H * q.W >= (1LL << 28)) return false;   // staged loads pack the channel above 28 offset bits
    const int S = q.S, NXR = (7 * S + 2) / 4 + 1;
    a.B = q.B; a.G = G; a.CG = q.C / G; a.NG = CO / G; a.K = a.CG * 9;
    a.H = q.H; a.W = q.W; a.HO = q.HO; a.WO = q.WO; a.P = q.P;
    a.CGP = (a.CG + kCC - 1) / kCC * kCC;
    a.SEG = (q.WO + kTM - 1) / kTM;                  // a last segment may reach past the row: those positions are not stored
    // the last lane of a row reads NXR*4 words from column (SEG-1)*8*S; the image with its padding is W + 2P wide
    int wp = (a.SEG - 1) * kTM * S + NXR * 4;
    if (q.W + 2 * q.P > wp) wp = q.W + 2 * q.P;
    a.WP = (wp + 3) / 4 * 4;
    if (a.WP % 32 == 0) a.WP += 4;                     // rows of one lane's window in different banks
    // Outputs per workgroup: at most 64, split evenly over the tiles; more tiles when a workgroup of that
    // width would have too many lanes (wide images).
    const int quads = (a.NG + kTN - 1) / kTN;
    for (int pass = 0; pass < 2; pass++) {
        // pass 0: all channels resident in LDS; pass 1: channels staged (needs CG % kCC == 0, so that no
        // stage holds a channel that does not exist)
        const bool resident = pass == 0;
        if (resident && nx > 1) continue;
        if (g_conv_staging_override == 3) continue;
        if (g_conv_staging_override == 1 && !resident) continue;
        if (g_conv_staging_override == 2 && resident) continue;
        if (!resident && nx == 1 && a.CG % kCC != 0) continue;
        // Candidates: the fewest output tiles that fit and up to three more (a narrower workgroup may take more
        // rows, or rows that divide the image evenly); each further tile re-reads the image rows once more,
        // priced at 3 %.  Past those, more tiles are only tried until something fits at all.
        const int first_tiles = (quads + 15) / 16;
        bool have = false;
        double haveScore = -1.0;
        ConvFwd pick = a;
        for (int tiles_n = first_tiles; tiles_n <= quads; tiles_n++) {
            if (have && tiles_n > first_tiles + 3) break;
            const int NL = (quads + tiles_n - 1) / tiles_n;
            if (a.SEG * NL > kMaxThreads) continue;
            const int BN = NL * kTN;
            // rows per workgroup: the choice that keeps most lanes busy on a CU (LDS limit, 8 waves of this
            // register footprint, rows computed past the image bottom count as idle); ties take more rows
            int bestR = 0, bestWords = 0;
            double bestScore = -1.0;
            const int maxR = kMaxThreads / (a.SEG * NL);
            int forced = g_conv_rows_override;
            if (forced > maxR) forced = maxR;
            if (forced > q.HO) forced = q.HO;
            for (int R = 1; R <= maxR && R <= q.HO; R++) {
                if (forced > 0 && R != forced) continue;
                const int NR = (R - 1) * S + 3;
                const int NT = R * a.SEG * NL;
                int xwords;
                if (resident) {
                    xwords = a.CGP * channel_stride(NR * a.WP);
                } else {
                    // a lane carries kXRegs image words per stage in registers; what a small workgroup cannot
                    // carry that way it copies directly, which is slow: only taken when forced
                    const int kXRegs = x_regs(S);
                    const int stage = kCC * NR * a.WP;
                    if (stage > kXRegs * NT && forced <= 0) continue;
                    const int half = stage > kXRegs * NT ? stage : kXRegs * NT;
                    xwords = 2 * ((half + 3) / 4 * 4);
                }
                const size_t lds = ((size_t)nx * xwords + 2 * (size_t)kKC * kBNP) * sizeof(float);
                if (lds > kLdsLimit - (nx > 1 ? 1024 : 0)) { if (resident) break; else continue; }   // nx > 1: room for the kernel's static LDS
                const long waves_wg = (NT + 63) / 64;
                long wgs = (long)(kLdsLimit / lds);
                if (wgs * waves_wg > 8) wgs = 8 / waves_wg;
                const int tiles_h = (q.HO + R - 1) / R;
                const double score = (double)wgs * NT * q.HO / ((double)tiles_h * R);
                if (score >= bestScore) { bestScore = score; bestR = R; bestWords = xwords; }
            }
            // below six resident waves per CU this variant does badly: try the other, or leave the layer to
            // the column kernels
            if (bestR == 0 || (bestScore < 384.0 && forced <= 0)) continue;
            const int real_tiles = (quads + NL - 1) / NL;
            const double priced = bestScore * (1.0 - 0.03 * (real_tiles - first_tiles));
            if (have && priced <= haveScore) continue;
            have = true;
            haveScore = priced;
            pick = a;
            pick.NL = NL; pick.BN = BN; pick.tiles_n = real_tiles;
            pick.R = bestR; pick.NR = (bestR - 1) * S + 3; pick.ML = bestR * a.SEG;
            pick.tiles_h = (q.HO + bestR - 1) / bestR;
            pick.resident = resident ? 1 : 0;
            pick.xwords = bestWords;
            pick.cstride = channel_stride(pick.NR * a.WP);
        }
        if (have) {
            a = pick;
            a.KG = 1;
            a.GT = a.ML * a.NL;
            return (long long)q.B * G * a.tiles_h * a.tiles_n < (1LL << 31);
        }
    }
    return false;
}

inline size_t lds_bytes(const ConvFwd& a, int nx) {
    const size_t weights = 2 * (size_t)kKC * kBNP;
    return sizeof(float) * (a.resident ? a.xwords + a.KG * weights : a.KG * (nx * (size_t)a.xwords + weights));
}

// Clocks of a launch: what the busiest CU's workgroups take, one set of as many as fit after the other.  `one` and `two`: a stage's
// clocks with one wave per SIMD and with two; `fixed`, `search`: what a workgroup's start and end take, and what the groups
// divide at the end (the search for the position).
struct StageClocks { double one, two, fixed, search; int rest; };   // rest: weight words in flight beyond the parked ones
inline double launch_clocks(const ConvFwd& a, int nx, int num_cu, const StageClocks& c) {
    const int waves = (a.KG * a.GT + 63) / 64, stages = (a.CGP / kCC + a.KG - 1) / a.KG;
    long at_once = (long)(kLdsLimit / (lds_bytes(a, nx) + (nx > 1 ? 256 : 0)));
    if (at_once * waves > 8) at_once = 8 / waves;
    if (at_once < 1) at_once = 1;
    const long per_cu = ((long)a.B * a.G * a.tiles_h * a.tiles_n + num_cu - 1) / num_cu;
    const int unparked = kKC * a.BN - kWRegs * a.GT;   // weights of a stage that lanes fetch without having them in flight
    const double extra = unparked > 0 ? (c.rest > 1 ? 4e3 : 2e3) * ((unparked + c.rest * a.GT - 1) / (c.rest * a.GT)) : 0.0;
    auto set = [&](long workgroups) {
        return stages * ((workgroups * waves > 4 ? c.two : c.one) + extra) + c.fixed + c.search / (a.KG < kTN ? a.KG : kTN);
    };
    return per_cu / at_once * set(at_once) + (per_cu % at_once ? set(per_cu % at_once) : 0.0);
}

// The launch shape of layers that would leave CUs idle: plan() fills a CU, not the device.  77 images of 14 x 14 and 64
// outputs are 154 workgroups of four waves then, three tenths of what the device can issue.  Here the tile may be smaller
// and its channels are shared by up to eight groups of lanes (eight waves in all, two per SIMD), which have stages of their
// own and meet in LDS at the end.  That layer with 64 channels: bounds 190 -> 117 us, values 85 -> 46; the same images at
// 28 x 28, 32 channels, 32 outputs: 141 -> 119 and 47 -> 47.  The clocks were fitted to these.  A shape is changed where that gains
// what asked() says, and only below four rounds of workgroups: beyond, the last round's share is small.  Measured over layers of
// 1 to 512 images of 7 to 32 pixels, 3 to 160 channels and 8 to 256 outputs: for values and bounds (134 layers) the estimate is
// within a third of the time, and a gain of 7 % is one.  With positions it promises too much: two groups gain from three quarters
// on where there are stages to share, 59.1 -> 49.7 us for 64 images of 32 x 28 x 28 -> 32 at 0.67 of the clocks, and small ones
// of a stage each from two thirds on (0.68: 23 -> 25.9); more groups or two large ones of a stage took 1.1 to 1.54 of the time at 0.62
// to 0.93, and so did launches of more than two workgroups to a CU before (267 images of 74 x 16 x 16 -> 44 in two groups of
// channels 123 -> 189 us).  A smaller tile that is not shared gains where much is promised (146 images of 3 x 15 x 15 -> 100 at
// 0.53: 46 -> 33) and not elsewhere (2 of 4 x 20 x 20 -> 222 at 0.75: 16.2 -> 20.2).  194 layers with positions whose shape
// changes for some rule take 0.785 of their time in all, 5 of them 1.05 to 1.11; with 7 % asked for 0.802, 32 of them up to 1.54.
inline void share_channels(const ConvGeom& q, ConvFwd& a, int nx, int num_cu, const StageClocks& clocks_of) {
    if (g_conv_rows_override > 0 && g_conv_groups_override <= 0) return;
    const int forced = g_conv_groups_override;
    const double before = launch_clocks(a, nx, num_cu, clocks_of);
    double best = forced > 0 ? 1e300 : before;
    if (forced <= 0 && (double)a.B * a.G * a.tiles_h * a.tiles_n > 4.0 * 2 * num_cu) return;   // at least four rounds
    const int S = q.S, quads = (a.NG + kTN - 1) / kTN, first_tiles = (quads + 15) / 16, nstage = a.CGP / kCC;
    auto asked = [&](const ConvFwd& c) {   // share of the clocks before; with positions there is a search to divide
        if (c.KG == 1) return 0.62;
        if (clocks_of.search == 0.0) return 0.93;
        return (double)a.B * a.G * a.tiles_h * a.tiles_n > 2.0 * num_cu ? 0.0 : c.KG > 2 ? 0.6 : nstage > 3 ? 0.75 : c.GT <= 128 ? 0.65 : 0.6;
    };
    ConvFwd pick = a;
    int last_nl = 0;
    for (int tiles_n = first_tiles; tiles_n <= quads && tiles_n <= 8 * first_tiles; tiles_n++) {
        ConvFwd c = a;
        c.NL = (quads + tiles_n - 1) / tiles_n;
        if (c.NL == last_nl || a.SEG * c.NL > kMaxThreads) continue;
        last_nl = c.NL;
        c.BN = c.NL * kTN;
        c.tiles_n = (quads + c.NL - 1) / c.NL;
        for (int R = 1; R <= q.HO && R * a.SEG * c.NL <= kMaxThreads; R++) {
            if (g_conv_rows_override > 0 && R != g_conv_rows_override) continue;
            c.R = R; c.NR = (R - 1) * S + 3; c.ML = R * a.SEG;
            c.tiles_h = (q.HO + R - 1) / R;
            c.GT = c.ML * c.NL;
            c.cstride = channel_stride(c.NR * a.WP);
            const int words = kCC * c.NR * a.WP, carried = x_regs(S) * c.GT;
            if (!a.resident && words > carried) continue;
            c.xwords = a.resident ? a.CGP * c.cstride : 2 * ((carried + 3) / 4 * 4);
            int last_per = nstage + 1;
            for (c.KG = 1; c.KG * c.GT <= 2 * kMaxThreads && c.KG <= nstage; c.KG++) {
                const int per = (nstage + c.KG - 1) / c.KG;
                if (per == last_per || (forced > 0 && c.KG != forced)) continue;   // a group more than the stages are worth
                last_per = per;
                if (lds_bytes(c, nx) > kLdsLimit - (nx > 1 ? 1024 : 0)) break;
                const double clocks = launch_clocks(c, nx, num_cu, clocks_of);
                if (clocks < best && (forced > 0 || clocks < asked(c) * before)) { best = clocks; pick = c; }
            }
        }
    }
    if (pick.KG != a.KG || pick.R != a.R || pick.NL != a.NL) {
        const long long grid = (long long)pick.B * pick.G * pick.tiles_h * pick.tiles_n;
        if (grid < (1LL << 31)) a = pick;
    }
}

// Which group of lanes finishes output t of a lane.
__device__ __forceinline__ int owner_of(int t, int groups) { return t % groups; }

// The groups' results of a lane's outputs meet with the owner of each: mine(e, t) gives an output's
// two numbers, take(e, t, numbers) sees those of every other group.  Lies over the weight stages (64 bytes per lane of at
// most 256, where a group has 19 KB), which nothing reads any more when the caller has passed a barrier.
template <class MINE, class TAKE>
__device__ __forceinline__ void meet_groups(float* park, const ConvFwd& a, int kg, int tid, MINE&& mine, TAKE&& take) {
    float2* const p = reinterpret_cast<float2*>(park);
    const int all = a.KG * a.GT;
#pragma unroll
    for (int t = 0; t < kTN; t++) {
        const int owner = owner_of(t, a.KG);
        if (t > 0) __syncthreads();
        if (kg != owner) {
#pragma unroll
            for (int e = 0; e < kTM; e++) p[e * all + kg * a.GT + tid] = mine(e, t);
        }
        __syncthreads();
        if (kg == owner) {
            for (int g = 0; g < a.KG; g++) {
                if (g == kg) continue;
#pragma unroll
                for (int e = 0; e < kTM; e++) take(e, t, p[e * all + g * a.GT + tid]);
            }
        }
    }
}

}  // namespace convimg
}  // namespace ldist
