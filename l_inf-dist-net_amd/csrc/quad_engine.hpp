// Building blocks of the forward kernels for problems whose (row, output) plane is too small for the tiles of
// fwd_engine.hpp to fill the device (fully connected layers at small and middling batches, or narrow ones).
//
// A workgroup of 256 lanes owns a BM x BN tile and splits the reduction over KS groups of lanes, KS up to 16, so that a
// tile can be as small as 16 x 32 and still occupy two waves per SIMD together with one more workgroup.  The panels of a
// stage lie in LDS as they lie in memory, rows of KK consecutive k: a lane reads four k of a row with one 128-bit read
// (TM + TN reads for 4 * TM * TN differences, the same bytes per difference as the k-major panels of tile.hpp), nothing
// is transposed on the way in, and any number of k >= 4 works, aligned or not: the last vector of a row is moved back so
// that it ends with the row, which for a maximum only repeats values already seen (sums blank them).
//
// A row's vectors are permuted by the XOR of the vector number with the row's number modulo the lanes that read
// different rows at once (TY along m, TX along n; see spread): those rows lie in different banks, and since row i of a lane's
// patch has the same remainder for every i, one address serves all its reads of a panel with constant offsets.
#pragma once
#include "kernels.hpp"
#include "tile.hpp"

namespace ldist {

struct __attribute__((packed, aligned(4))) float4_any { float v[4]; };   // a 128-bit global access at any 4-byte address

template <int BM_, int BN_, int TM_, int TN_, int KS_, int KK_>
struct QGeo {
    static constexpr int BM = BM_, BN = BN_, TM = TM_, TN = TN_, KS = KS_, KK = KK_;
    static constexpr int TX = BN / TN, TY = BM / TM, NGRP = TX * TY, NT = NGRP * KS;
    static constexpr int QR = KK / 4;            // vectors of a panel row
    static constexpr int QG = QR / KS;           // of which a k-group takes this many per stage
    static constexpr int CH = QG * 4;            // k values per k-group and stage
    static_assert(BM % TM == 0 && BN % TN == 0 && NT == 256 && QR % KS == 0 && NT % QR == 0, "tile");
    static_assert((TX & (TX - 1)) == 0 && (TY & (TY - 1)) == 0 && (QR & (QR - 1)) == 0 && QR >= 8, "powers of two");
    static constexpr int GX = TY, GW = TX;       // rows that are read at once
    // What a row's vector numbers are permuted with: 16 rows of 256 bytes, or of 128 bytes (two to the 256 bytes that
    // the banks hold), read at the same vector fall into different banks.
    __device__ static constexpr int spread(int r) { return (QR == 8 ? r >> 1 : r) & (QR - 1) & 15; }
    __device__ static constexpr int row(int ty, int i) { return ty + TY * i; }
    __device__ static constexpr int col(int tx, int j) { return tx + TX * j; }
};

// One panel's share of a stage for a lane, memory -> LDS without a register in between (buffer loads with the lds bit:
// the 64 lanes of a wave fill 64 consecutive vectors of LDS, so the permutation of a row's vectors is applied to the
// addresses they are fetched from).  Written as inline assembly: the compiler, which cannot tell the two stages of the
// LDS array apart, would wait for the loads of the next stage before the first read of the current one.  Nobody but
// arrived() waits for them.
typedef int int4v __attribute__((ext_vector_type(4)));

template <class GEO, int ROWS, int SPREAD>
struct QPanel {
    static constexpr int TOTAL = ROWS * GEO::QR, N = (TOTAL + GEO::NT - 1) / GEO::NT, STEP = GEO::NT / GEO::QR;
    static_assert(STEP % SPREAD == 0, "a lane keeps its vector number over its rows");
    static_assert(TOTAL % 64 == 0, "whole waves");
    unsigned off[N];   // byte offset of the lane's vector in each of its rows, from the tile's first row
    int4v rsrc;

    __device__ __forceinline__ static int vector_of(int tid) { return (tid % GEO::QR) ^ GEO::spread((tid / GEO::QR) % SPREAD); }
    __device__ __forceinline__ void init(const float* base, int ld, int rows_valid, int tid) {
        const uint64_t at = reinterpret_cast<uint64_t>(base);
        rsrc = int4v{__builtin_amdgcn_readfirstlane((int)(unsigned)at), __builtin_amdgcn_readfirstlane((int)(unsigned)(at >> 32)),
                     (int)0x80000000u, 0x00020000};
#pragma unroll
        for (int i = 0; i < N; i++)   // rows past the matrix read its last row; their results are never stored
            off[i] = 4u * ((unsigned)min(tid / GEO::QR + i * STEP, rows_valid - 1) * (unsigned)ld + (unsigned)vector_of(tid) * 4u);
    }
    // panel: LDS byte address; wave: number of the wave (in a scalar register); back: bytes by which this lane's vector
    // of the stage starts beyond the last whole vector of the row (0 inside).  All of it in the lane's offset: the range
    // check looks at that alone, without the scalar one, and a moved vector may begin before k0 in the tile's first row.
    __device__ __forceinline__ void load(unsigned panel, int k0, unsigned back, int wave) const {
#pragma unroll
        for (int i = 0; i < N; i++) {
            if (TOTAL % GEO::NT != 0 && (i * GEO::NT + wave * 64) >= TOTAL) continue;
            // A load that takes its LDS address from M0 needs one wait state behind a scalar write of M0, which nobody
            // adds inside inline assembly.
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                         :: "s"(panel + (unsigned)(i * GEO::NT + wave * 64) * 16u), "v"(off[i] + (4u * (unsigned)k0 - back)), "s"(rsrc), "s"(0)
                         : "memory", "m0");
        }
    }
    // Zeros over what does not belong to the stage in the row's last vectors: the values before the vector that ends
    // with the row, and whole vectors past the end.  For sums; after the loads have arrived.
    __device__ __forceinline__ void blank(float* panel, unsigned back, int tid) const {
        for (int i = 0; i < N; i++)
            if (i * GEO::NT + tid < TOTAL)
                for (unsigned e = 0; e < 4 && 4u * e < back; e++) panel[(i * GEO::NT + tid) * 4 + e] = 0.f;
    }
};

// NX input panels and the weight panel of a stage.
template <class GEO, int NX>
struct QStager {
    static constexpr int XS = GEO::BM * GEO::KK, STAGE = NX * XS + GEO::BN * GEO::KK;   // floats
    static constexpr size_t LDS_BYTES = 2 * (size_t)STAGE * sizeof(float);
    QPanel<GEO, GEO::BM, GEO::GX> x[NX];
    QPanel<GEO, GEO::BN, GEO::GW> w;
    int K, tid, wave;

    __device__ __forceinline__ void init(const float* const (&input)[NX], const float* weight, const Dims& d, int m0, int n0,
                                         int g, int tid_) {
        tid = tid_;
        wave = __builtin_amdgcn_readfirstlane(tid_ >> 6);
        K = d.K;
        w.init(weight + ((size_t)g * d.NG + n0) * K, K, d.NG - n0, tid);
#pragma unroll
        for (int q = 0; q < NX; q++) x[q].init(input[q] + ((size_t)m0 * d.G + g) * K, d.G * K, d.M - m0, tid);
    }
    __device__ __forceinline__ unsigned back(int k0, int vector) const {
        const int k = k0 + vector * 4;
        return k > K - 4 ? 4u * (unsigned)(k - (K - 4)) : 0u;
    }
    __device__ __forceinline__ void load(float* stage, int k0) const {
        const unsigned at = lds_address(stage);
        w.load(at + NX * XS * 4u, k0, back(k0, w.vector_of(tid)), wave);
#pragma unroll
        for (int q = 0; q < NX; q++) x[q].load(at + q * XS * 4u, k0, back(k0, x[q].vector_of(tid)), wave);
    }
    // This wave's loads are in LDS (the others' after the barrier that follows).
    __device__ __forceinline__ static void arrived() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
    __device__ __forceinline__ void blank(float* stage, int k0) const {
#pragma unroll
        for (int q = 0; q < NX; q++) x[q].blank(stage + q * XS, back(k0, x[q].vector_of(tid)), tid);
        w.blank(stage + NX * XS, back(k0, w.vector_of(tid)), tid);
    }
};

// Dynamic LDS of a kernel: the two stages, or the parking places of q_merge with two words per output if larger (they
// also hold the finished tile: KS / 2 * NGRP lanes' patches are at least one tile).
template <class GEO, int NX>
constexpr size_t q_lds_bytes() {
    constexpr size_t stages = QStager<GEO, NX>::LDS_BYTES, parked = (size_t)GEO::NT * GEO::TM * GEO::TN * 4;
    static_assert(GEO::KS >= 2, "a k-group to merge with");
    return stages > parked ? stages : parked;
}

// Four k of a lane's patch operands.
template <class GEO, int NX>
struct QFrag {
    typedef float F4 __attribute__((ext_vector_type(4)));
    F4 x[NX][GEO::TM], w[GEO::TN];
};

// How many vectors of stage s are the k-group's: all of its share, less what lies past the end in the last stage.
template <class GEO>
__device__ __forceinline__ int q_vectors(int s, int nstage, int K, int grp) {
    if (s + 1 < nstage) return GEO::QG;
    return min(GEO::QG, max(0, (K - s * GEO::KK - grp * GEO::CH + 3) / 4));
}

// Walks the first `vectors` of the k-group's share of a stage: f(frag) once per vector, k ascending.
template <class GEO, int NX, class F>
__device__ __forceinline__ void q_sweep(const float* stage, int vectors, int grp, int tx, int ty, F&& f) {
    typedef float F4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) const F4 lds_f4;
    const unsigned base = lds_address(stage);
    const unsigned xb = base + (unsigned)ty * (GEO::KK * 4u);
    const unsigned wb = base + NX * GEO::BM * GEO::KK * 4u + (unsigned)tx * (GEO::KK * 4u);
    auto read = [&](QFrag<GEO, NX>& fr, int j) {
        const unsigned q = (unsigned)(grp * GEO::QG + j);
        const unsigned xa = xb + ((q ^ (unsigned)GEO::spread(ty)) << 4), wa = wb + ((q ^ (unsigned)GEO::spread(tx)) << 4);
#pragma unroll
        for (int p = 0; p < NX; p++)
#pragma unroll
            for (int i = 0; i < GEO::TM; i++)
                fr.x[p][i] = *(lds_f4*)(uintptr_t)(xa + (p * GEO::BM + GEO::TY * i) * (GEO::KK * 4u));
#pragma unroll
        for (int c = 0; c < GEO::TN; c++) fr.w[c] = *(lds_f4*)(uintptr_t)(wa + (GEO::TX * c) * (GEO::KK * 4u));
    };
#pragma unroll 1
    for (int j = 0; j < vectors; j++) {
        QFrag<GEO, NX> a;
        read(a, j);
        f(a);
    }
}

// The same walk one k at a time with few registers: for rarely taken paths that must not add to those of the hot loop.
template <class GEO, int NX, class F>
__device__ __forceinline__ void q_sweep_plain(const float* stage, int vectors, int grp, int tx, int ty, F&& f) {
#pragma unroll 1
    for (int k = 0; k < vectors * 4; k++) {
        const int q = grp * GEO::QG + k / 4;
        const float* xa = stage + ty * GEO::KK + ((q ^ GEO::spread(ty)) << 2) + (k & 3);
        const float* wa = stage + NX * GEO::BM * GEO::KK + tx * GEO::KK + ((q ^ GEO::spread(tx)) << 2) + (k & 3);
        float x[NX][GEO::TM], w[GEO::TN];
#pragma unroll
        for (int p = 0; p < NX; p++)
#pragma unroll
            for (int i = 0; i < GEO::TM; i++) x[p][i] = xa[(p * GEO::BM + GEO::TY * i) * GEO::KK];
#pragma unroll
        for (int j = 0; j < GEO::TN; j++) w[j] = wa[GEO::TX * j * GEO::KK];
        f(x, w);
    }
}

// Hands the k-groups' results to the first group: `park(slot)` leaves a lane's results in LDS, `take(slot)` merges
// what the group half as far again left there; slot numbers the parking places.  A tree of log2(KS) steps.
template <class GEO, class PARK, class TAKE>
__device__ __forceinline__ void q_merge(int grp, PARK&& park, TAKE&& take) {
#pragma unroll
    for (int half = GEO::KS / 2; half > 0; half /= 2) {
        __syncthreads();
        if (grp >= half && grp < 2 * half) park(grp - half);
        __syncthreads();
        if (grp < half) take(grp);
    }
}

}  // namespace ldist
