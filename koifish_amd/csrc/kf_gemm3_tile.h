// kf_gemm3_tile.h -- the 64-deep bf16 MFMA tile of kf_gemm3.hip (operand staging, fragments, main loop): shared by that file's GEMMs and by the row-batch products of
// kf_rb_gemm.hip, which add their own epilogues and a gathered token operand.
#pragma once
#include <type_traits>

#include "kf_gemm_common.h"

namespace kf {

constexpr int G3_BM = 256, G3_BN = 256, G3_BK = 64;
// the workgroup tile: BM rows x BN tokens, NW waves as NW / WN_ (rows; 2 by default) x WN_ (tokens), NBUF LDS buffers: the loads of NBUF - 1 later k-steps are in flight under the step that is multiplied.
// A step is bound by those loads, not by its MFMAs (loads alone take 85 - 95 % of every configuration's time), and with two buffers a lone workgroup of a CU waits out their latency: us per
// step with one workgroup on every CU, two buffers | more: 64 x 64 0.41 | 0.23 (3), 128 x 128 on 8 waves 0.89 | 0.58 (3), 128 x 256 0.75 (3) against 1.26 of 192 x 256 (2: three do not fit).
// Where an operand's instructions are no multiple of the waves (EVEN false: 160 rows are 20) the first waves issue one more; the others' last one has an empty descriptor and
// a KiB of its own behind the buffers (SPARE), so that every wave counts the same loads.  SMEM then is the whole LDS: the tile in 32 bits fits.
template <int BM_, int BN_, int NW_, int NBUF_ = 2, int WN_ = NW_ / 2>
struct G3Cfg {
    static constexpr int BM = BM_, BN = BN_, NW = NW_, WN = WN_, MT = BM_ / (16 * (NW_ / WN_)), NT = BN_ / (16 * WN_), NBUF = NBUF_;
    static constexpr int NIA = (BM_ / 8 + NW_ - 1) / NW_, NIB = (BN_ / 8 + NW_ - 1) / NW_; /* global_load_lds instructions per wave, operand and k-step (8 rows of 128 bytes each) */
    static constexpr bool EVEN = BM_ % (8 * NW_) == 0 && BN_ % (8 * NW_) == 0;
    static constexpr int STAGE = (BM_ + BN_) * G3_BK * 2, NTH = 64 * NW_, SPARE = NBUF_ * STAGE, SMEM = EVEN ? SPARE : 160 * 1024, WGS_PER_CU = (160 * 1024) / SMEM;
    static_assert(EVEN || SPARE + 1024 <= SMEM, "the spare KiB");
};
// an operand of ROWS rows: the first of wave `wid`'s load instructions, and whether it has an i-th one
template <int ROWS, int NW>
struct G3Share {
    static constexpr int ALL = ROWS / 8, Q = ALL / NW, REST = ALL % NW;
    static __device__ __forceinline__ int first(int wid) { return Q * wid + (REST == 0 || wid < REST ? (REST ? wid : 0) : REST); }
    static __device__ __forceinline__ bool has(int wid, int i) { return i < Q || wid < REST; }
};
using G3Big = G3Cfg<256, 256, 8>;      /* 128 KiB of LDS: one workgroup per CU */
using G3Wide = G3Cfg<192, 256, 8>;
using G3Half = G3Cfg<128, 256, 8, 3>;  /* 144 KiB */
using G3Long = G3Cfg<128, 384, 8>;     /* 128 KiB: as many outputs as 192 x 256, where a tile is a head */
using G3Duo = G3Cfg<128, 128, 8, 3>;   /* 96 KiB */
using G3Small = G3Cfg<128, 128, 4>;    /* 64 KiB: two workgroups per CU; the split-K tile of the k-major products */
using G3Few = G3Cfg<64, 64, 4, 3>;     /* 48 KiB: three */
// k-pieces where a workspace is lent (gemm3_launch)
using G3Slim = G3Cfg<160, 256, 8, 3>;  /* 156 KiB: three buffers where 192 rows leave two, five eighths of the big tile's outputs */
using G3Flat = G3Cfg<256, 160, 8, 3, 2>;
using G3Mid = G3Cfg<64, 128, 4>;
using G3Tiny = G3Cfg<64, 64, 4>;

// x, which the compiler cannot trace: addresses formed from it are formed behind this point and take no registers in front of it
__device__ __forceinline__ int g3_opaque(int x) {
    asm volatile("" : "+v"(x));
    return x;
}
// One operand tile (256 rows x 128 bytes) = 32 wave instructions of 1 KiB; wave `wid` issues NI of them.  8 rows per instruction, chunk c of row r at position
// c ^ ((r >> 1) & 7): a fragment read (16 rows x one 16-byte chunk) touches all 64 banks once.
// An instruction's address is a scalar part (the tile's origin, the k-step, whole groups of rows) and a lane's part, which the swizzle makes one of two: even and odd
// instructions.  Rows past the operand's end lie past the descriptor's end: the load writes zeros (their outputs are not stored).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t g3_rsrc(const void* p, uint32_t bytes) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00020000); }
constexpr uint32_t G3_ALL = 0x7FFFFFF0u; /* a descriptor's size that no lane part reaches */
struct G3Src {
    const unsigned char* base; /* uniform: the tile's origin at k-step 0 */
    long long left, step, inst; /* bytes from there to the operand's end (< 0: no row past the end); bytes per k-step; bytes per instruction */
    uint32_t lane[3]; /* [2]: 160-row k-major images */
};
__device__ __forceinline__ G3Src g3_src(const uint16_t* __restrict__ src, long long ld, int row0, int nrows, int first, int lane) { /* first: the wave's first instruction */
    G3Src s;
    s.base = reinterpret_cast<const unsigned char*>(src + ((size_t)row0 + (size_t)first * 8) * ld);
    s.left = ((long long)nrows - row0 - (long long)first * 8) * ld * 2, s.step = G3_BK * 2, s.inst = ld * 16;
#pragma unroll
    for (int v = 0; v < 2; v++) {
        const int r = (first + v) * 8 + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
        s.lane[v] = (uint32_t)(lane >> 3) * (uint32_t)(ld * 2) + c * 16;
    }
    return s;
}
__device__ __forceinline__ bf16x8 g3_frag(const unsigned char* tile, int row, int c) {
    const int p = c ^ ((row >> 1) & 7);
    return *reinterpret_cast<const bf16x8*>(tile + row * (2 * G3_BK) + (p << 4));
}

// the same tile from a K-MAJOR operand (src[k][row], `row` contiguous: an activation or a weight as it lies in memory when the contraction runs over its ROWS --
// both GEMMs of SLP::Back): the LDS image is [BK k][ROWS rows] (512- or 256-byte k-rows), one wave instruction = two or four k-rows; its 32-byte blocks are XOR-swizzled by k & 3 and
// its 128-byte quarters by bit 3 of k, so that the transposing fragment read below (per 32 lanes: k-rows k .. k+3 and k+8 .. k+11, 32 bytes of each) touches all 64
// banks once (without the second term the two 16-lane halves meet in the same 32 banks: SQ_LDS_BANK_CONFLICT = 50 % of the LDS cycles, measured).
// A k-row of 160 rows is 20 chunks, 64 bytes past whole turns of the banks, so four k-rows meet in no bank as they are and only bit 3 of k moves a block, to its neighbour; five instructions are 16 k-rows.
// A base serves the loads of a wave and step (of a step, 160 rows): the k-rows between them are scalar offsets, a lane's own k-row and column the lane part, all below the descriptor's end, G3_ALL.
template <int ROWS>
struct G3Km {
    static constexpr int INST = ROWS == 160 ? 16 : 512 / ROWS;      /* k-rows of a scalar step: of an instruction, of five (160) */
    static constexpr int SPAN = 4 * INST;                            /* k-rows that a base's offsets lie in */
    static constexpr int part(int i) { return ROWS == 160 ? i : ROWS == 128 ? i >> 1 : i & 1; }        /* which lane part instruction i of a wave takes */
    static constexpr int steps(int first, int i) { return ROWS == 160 ? (first + i) / 5 : i; }        /* and how many scalar steps */
};
template <int ROWS>
static constexpr bool g3_km_reach(long long ld) { return 2 * ld * G3Km<ROWS>::SPAN <= (long long)G3_ALL; } /* a row of ld values in reach: up to 2^24 - 8 (160), 2^26 - 8 (128), 2^27 - 8 (256) */
// ROWS = the tile's rows (256, 160 or 128): a k-row of the image is 2 ROWS bytes = CPK chunks of 16 bytes, one wave instruction covers 64 / CPK k-rows, wave `wid` issues
// instructions NI wid .. NI wid + NI - 1 of the ROWS / 8
template <int ROWS, int NI>
__device__ __forceinline__ G3Src g3_src_km(const uint16_t* __restrict__ src, long long ld, int row0, int nrows, int wid, int lane) {
    constexpr int CPK = ROWS / 8, KPI = 64 / CPK, UNIT = ROWS == 256 ? 1 : 2; /* 256: the swizzle tells even from odd instructions, 128: pairs of them */
    G3Src s;
    if constexpr (ROWS == 160) {
        static_assert(NI == 3, "a lane part per instruction");
        const int first = G3Share<160, 8>::first(wid);
        s.base = reinterpret_cast<const unsigned char*>(src), s.left = -1, s.step = (long long)G3_BK * ld * 2, s.inst = (long long)G3Km<ROWS>::INST * ld * 2;
#pragma unroll
        for (int v = 0; v < 3; v++) {
            const int at = (first + v) % 5 * 64 + lane, kr = at / CPK, p = at % CPK, c = p ^ (((kr >> 3) & 1) << 1);
            int col = row0 + c * 8;
            col = col + 8 <= nrows ? col : (nrows - 8 > 0 ? nrows - 8 : 0); /* as below */
            s.lane[v] = G3Share<160, 8>::has(wid, v) ? (uint32_t)kr * (uint32_t)(ld * 2) + col * 2 : G3_ALL; /* (none: past the descriptor's end) */
        }
        return s;
    }
    static_assert(ROWS == 160 || ((ROWS == 256 || ROWS == 128) && NI == 4), "two lane parts per wave");
    s.base = reinterpret_cast<const unsigned char*>(src + (size_t)wid * NI * KPI * ld);
    s.left = -1, s.step = (long long)G3_BK * ld * 2, s.inst = (long long)G3Km<ROWS>::INST * ld * 2; /* every k-row of the steps exists; chunks past a row's end are clamped here */
#pragma unroll
    for (int v = 0; v < 2; v++) {
        const int kr = (wid * NI + v * UNIT) * KPI + lane / CPK, p = lane % CPK, c = p ^ ((kr & 3) << 1) ^ (((kr >> 3) & 1) << 3);
        int col = row0 + c * 8;
        col = col + 8 <= nrows ? col : (nrows - 8 > 0 ? nrows - 8 : 0); /* chunks past the end re-read the last whole chunk: their outputs are not stored (rows % 8 == 0) */
        s.lane[v] = (uint32_t)(lane / CPK) * (uint32_t)(ld * 2) + col * 2;
    }
    return s;
}
// fragment (8 consecutive k of row `row`, k = kbase .. kbase + 7) of a k-major tile: two ds_read_b64_tr_b16, each a 4 (k) x 16 (rows) block transposed across 16 lanes
// (lane i of the 16 receives D[(i >> 2) + 4 j][i & 3], scratch/dbg/ds_read_tr_probe.hip): lane l16 reads k-row kbase + (l16 >> 2), 8-byte piece l16 & 3 of the 16-row block
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
// The row block only flips three bits of a lane's offset (the swizzle's), so one register serves all blocks.
// 160 rows: the swizzle puts a block behind or in front of its place by the block's parity, one offset for each (odd: of the blocks 1, 3, .. of a wave whose first block is odd or even, `odd` says which)
__device__ __forceinline__ int g3_km_lane160(int l16, int q4, int odd) {
    const int k = 8 * q4 + (l16 >> 2);
    return k * 320 + ((l16 & 3) >> 1) * 16 + 8 * (l16 & 1) + ((q4 & 1) ? (odd ? -32 : 32) : 0);
}
__device__ __forceinline__ int g3_km_lane(int rows, int l16, int q4) { /* the lane's offset in a tile at row block 0, k 0 */
    const int k = 8 * q4 + (l16 >> 2), swz = ((k & 3) << 1) ^ (((k >> 3) & 1) << 3);
    return k * (2 * rows) + ((((l16 & 3) >> 1) ^ swz) << 4) + 8 * (l16 & 1);
}
template <int ROWS>
__device__ __forceinline__ bf16x8 g3_frag_km(const unsigned char* tile, int km_lane, int rowblk16, int kk) {
    bf16x4 h[2];
    const unsigned char* const at = tile + (ROWS == 160 ? km_lane + rowblk16 * 32 : (km_lane ^ ((rowblk16 & 7) << 5)) + ((rowblk16 >> 3) << 8));
#pragma unroll
    for (int t = 0; t < 2; t++) h[t] = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) bf16x4*)(at + (kk * 32 + 4 * t) * (2 * ROWS)));
    return bf16x8{h[0][0], h[0][1], h[0][2], h[0][3], h[1][0], h[1][1], h[1][2], h[1][3]};
}

// k-steps kt0 .. kt1 - 1 (of BK) of the output tile at (m0, t0) accumulated into acc (the caller zeroes it).  See g3_mainloop below for the schedule.
// `rows` (G3Rows: plain; G3Gather: row r of the token tile is row map[r] of x) says where the tile's token rows lie.
// TILED: w is stored in MFMA tiles (kf_rb.h: 16 rows x 32 columns, piece (r, q) at number 16 q + r) instead of rows: a load
// instruction moves one tile, contiguous in memory and in LDS, and a fragment read is lane-linear -- no swizzle on this operand.
// F32: both operands are 32-bit floats, their strides counted in 16-bit units like the others' (K = twice the floats): a step is 32 of them, the tile's bytes, chunks and swizzle are
// the same, and a lane's 16-byte chunk is the operand of four v_mfma_f32_16x16x4_f32 (lane group q, float i: k = 4 q + i on both sides).
struct G3Rows {
    static constexpr bool GATHER = false, TILED = false, F32 = false;
};
struct G3Tiled {
    static constexpr bool GATHER = false, TILED = true, F32 = false;
};
struct G3GatherTiled {
    static constexpr bool GATHER = true, TILED = true, F32 = false;
    const int32_t* map; /* [BN] rows of x, every entry valid */
};
struct G3RowsF32 {
    static constexpr bool GATHER = false, TILED = false, F32 = true;
};
struct G3GatherF32 {
    static constexpr bool GATHER = true, TILED = false, F32 = true;
    const int32_t* map;
};
// The schedule.  A wave's outputs are four quadrants (row half x token half); the fragments of a quadrant are read from LDS under the MFMAs of the quadrant before it:
//   quadrant (0,0): read token half 1          (0,1): read row half 1          -- step kt + 1 has landed, every wave holds its last fragments of step kt: ONE barrier --
//   loads of step kt + 2 into the buffer of step kt          (1,1): read row half 0 of step kt + 1          (1,0): read token half 0 of step kt + 1
// so neither the LDS reads (1.5 k of the 2 k cycles that a 256 x 256 x 64 step's MFMAs take) nor the barrier leave the matrix pipe without issued work, and a load has a
// whole step to arrive.  The form before it read a step's fragments right behind the barrier, two at a time in front of the four MFMAs that use them, and waited there for the
// loads it had issued one barrier earlier.  Same products in the same order: same bits.
// f over LDS buffers that the compiler may tell apart (restrict).  Otherwise it takes a transposing LDS read (k-major operands) for one that may read what any load on its way writes, and puts a wait for
// all of them in front of it: a step of the weight gradients then took what its loads took (8192 x 6400 x 1600: 2.4 us a step of 256 x 256 against 1.5 with K-contiguous operands)
template <class F>
static __device__ void g3_told_apart(unsigned char* __restrict__ a0, unsigned char* __restrict__ a1, unsigned char* __restrict__ b0, unsigned char* __restrict__ b1, F&& f) {
    f(a0, a1, b0, b1);
}
template <class F>
static __device__ void g3_told_apart(unsigned char* __restrict__ a0, unsigned char* __restrict__ a1, unsigned char* __restrict__ a2, unsigned char* __restrict__ b0, unsigned char* __restrict__ b1,
                                     unsigned char* __restrict__ b2, F&& f) {
    f(a0, a1, a2, b0, b1, b2);
}
template <int M, int N, int V, int I>
__device__ __forceinline__ void g3_issue() { /* an MFMA, then its share of N reads and of V loads among M MFMAs */
    constexpr int P = N < M ? N : M, Q = V < M - 1 ? V : M - 1;
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    if constexpr (I < P) __builtin_amdgcn_sched_group_barrier(0x100, N * (I + 1) / P - N * I / P, 0);
    if constexpr (I < Q) __builtin_amdgcn_sched_group_barrier(0x010, V * (I + 1) / Q - V * I / Q, 0);
    if constexpr (I + 1 < (P > Q ? P : Q)) g3_issue<M, N, V, I + 1>();
}
struct G3Nothing {
    __device__ __forceinline__ void operator()(int) const {}
};
// between(kt): in front of step kt, behind all MFMAs of the step before
template <bool AKM, bool BKM, int BK, class C, class ROWS = G3Rows, class BETWEEN = G3Nothing>
__device__ __forceinline__ void g3_mainloop(const GemmArgs& a, int m0, int t0, int kt0, int kt1, f32x4 (&acc)[C::MT][C::NT], unsigned char* smem_raw, int wid_, int lane, ROWS rows = ROWS(),
                                            BETWEEN between = BETWEEN()) {
    static_assert(BK == G3_BK && C::MT > 1 && C::NT > 1, "two k-halves of 32 per step, two halves of rows and of tokens per wave");
    constexpr int LPW = C::NIA + C::NIB, HM = (C::MT + 1) / 2, HN = (C::NT + 1) / 2; /* loads per wave and step; MFMA blocks of the first half (five: three and two) */
    constexpr std::integral_constant<int, 0> lo{};
    constexpr std::integral_constant<int, 1> hi{};
    using ShareA = G3Share<C::BM, C::NW>;
    using ShareB = G3Share<C::BN, C::NW>;
    constexpr int BYTES_A = C::BM * BK * 2, BYTES_B = C::BN * BK * 2;
    const int wid = __builtin_amdgcn_readfirstlane(wid_), wm = wid / C::WN, wn = wid % C::WN;
    auto bufA = [&](int b) { return smem_raw + b * BYTES_A; }; /* an operand's two buffers side by side: both in reach of an LDS instruction's 16-bit offset */
    auto bufB = [&](int b) { return smem_raw + C::NBUF * BYTES_A + b * BYTES_B; };
    [[maybe_unused]] const int firstA = ShareA::first(wid), firstB = ShareB::first(wid);
    // AKM: W is [K][M] with row stride a.ldr (re-used field: the residual is not served by the k-major forms); BKM: x is [K][n] with row stride a.ldx.
    G3Src sa, sb;
    const uint16_t* gat[ROWS::GATHER ? C::NIB : 1];
    const uint16_t* const W = reinterpret_cast<const uint16_t*>(a.w);
    if constexpr (ROWS::TILED) {
        static_assert(!AKM, "an instruction is a tile, two tiles per row block and step");
        const long long rb = m0 >> 4, row = (long long)(a.K / 32) * 1024; /* row block of the first tile; bytes of a row block */
        sa.base = a.w + rb * row, sa.left = ((a.M + 15) / 16 - rb) * row, sa.step = 2048, sa.inst = row;
        sa.lane[0] = lane * 16, sa.lane[1] = lane * 16;
    } else if constexpr (AKM)
        sa = g3_src_km<C::BM, C::NIA>(W, a.ldr, m0, a.M, wid, lane);
    else
        sa = g3_src(W, a.K, m0, a.M, firstA, lane);
    if constexpr (ROWS::GATHER) {
        static_assert(!BKM && ShareB::REST == 0, "gathered rows: K-contiguous operands, every load has a row");
#pragma unroll
        for (int i = 0; i < C::NIB; i++) {
            const int r = (firstB + i) * 8 + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
            gat[i] = a.x + (size_t)rows.map[r] * a.ldx + c * 8;
        }
    } else if constexpr (BKM)
        sb = g3_src_km<C::BN, C::NIB>(a.x, a.ldx, t0, a.n, wid, lane);
    else
        sb = g3_src(a.x, a.ldx, t0, a.n, firstB, lane);
    // K-contiguous operands: one descriptor per instruction for the whole tile, a step is the scalar offset (a row past the end lies past the descriptor's end at every
    // step, whether or not the check counts that offset; a row inside never does).  k-major: every step has a base of its own, of any size, and an instruction the scalar offset.
    // Past the last step the descriptors are empty: the load moves nothing and puts zeros where nobody reads, and the steps need no branch.
    uint32_t restA[C::NIA], restB[C::NIB];
    auto rest = [](long long left) { return (uint32_t)(left < 0 ? 0 : (left > 0xFFFFFFFFll ? 0xFFFFFFFFll : left)); };
    auto atA = [&](int i) {
        const int j = firstA + i; /* tile (row block j / 2, k-half j % 2) of the workgroup's */
        return ROWS::TILED ? sa.inst * (j >> 1) + (j & 1) * 1024 : AKM ? sa.inst * G3Km<C::BM>::steps(firstA, i) : sa.inst * i;
    };
    [[maybe_unused]] auto atB = [&](int i) { return BKM ? sb.inst * G3Km<C::BN>::steps(firstB, i) : sb.inst * i; };
#pragma unroll
    for (int i = 0; i < C::NIA; i++) restA[i] = !ShareA::has(wid, i) ? 0 : AKM ? G3_ALL : rest(sa.left - atA(i));
#pragma unroll
    for (int i = 0; i < C::NIB; i++) restB[i] = !ShareB::has(wid, i) ? 0 : BKM || ROWS::GATHER ? G3_ALL : rest(sb.left - atB(i));
    [[maybe_unused]] auto to = [&](unsigned char* tile, int i, bool has) { return (__attribute__((address_space(3))) void*)(has ? tile + i * 1024 : smem_raw + C::SPARE); };
    [[maybe_unused]] const unsigned char *nextA = sa.base + (AKM ? sa.step * kt0 : 0), *nextB = BKM ? sb.base + sb.step * kt0 : nullptr; /* k-major: the base of the step staged next */
    auto stageA = [&](int kt, unsigned char* tile) {
#ifdef __HIP_DEVICE_COMPILE__
#pragma unroll
        for (int i = 0; i < C::NIA; i++) {
            [[maybe_unused]] const auto at = to(tile, firstA + i, ShareA::has(wid, i));
            [[maybe_unused]] const uint32_t n = kt < kt1 ? restA[i] : 0;
            if constexpr (AKM) __builtin_amdgcn_raw_ptr_buffer_load_lds(g3_rsrc(nextA, kt < kt1 ? G3_ALL : 0), at, 16, sa.lane[G3Km<C::BM>::part(i)], (int)atA(i), 0, 0);
            else __builtin_amdgcn_raw_ptr_buffer_load_lds(g3_rsrc(sa.base + atA(i), n), at, 16, sa.lane[ROWS::TILED ? 0 : i & 1], (int)sa.step * kt, 0, 0);
        }
        if constexpr (AKM) nextA += sa.step;
#endif
    };
    auto stageB = [&](int kt, unsigned char* tile) {
#ifdef __HIP_DEVICE_COMPILE__
#pragma unroll
        for (int i = 0; i < C::NIB; i++) {
            [[maybe_unused]] const auto at = to(tile, firstB + i, ShareB::has(wid, i));
            [[maybe_unused]] const uint32_t n = kt < kt1 ? restB[i] : 0;
            if constexpr (ROWS::GATHER) __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(gat[i] + (size_t)(kt < kt1 ? kt : kt1 - 1) * BK), at, 16, 0, 0); /* (past the end: the last step again) */
            else if constexpr (BKM) __builtin_amdgcn_raw_ptr_buffer_load_lds(g3_rsrc(nextB, kt < kt1 ? G3_ALL : 0), at, 16, sb.lane[G3Km<C::BN>::part(i)], (int)atB(i), 0, 0);
            else __builtin_amdgcn_raw_ptr_buffer_load_lds(g3_rsrc(sb.base + atB(i), n), at, 16, sb.lane[i & 1], (int)sb.step * kt, 0, 0);
        }
        if constexpr (BKM) nextB += sb.step;
#endif
    };
    const int r16 = lane & 15, q4 = lane >> 4;
    int kmA[2], kmB[2]; /* [1]: odd blocks of a 160-row operand */
#pragma unroll
    for (int odd = 0; odd < 2; odd++) {
        kmA[odd] = C::BM == 160 ? g3_km_lane160(r16, q4, (wm * C::MT + odd) & 1) : g3_km_lane(C::BM, r16, q4);
        kmB[odd] = C::BN == 160 ? g3_km_lane160(r16, q4, (wn * C::NT + odd) & 1) : g3_km_lane(C::BN, r16, q4);
    }
    auto readA = [&](const unsigned char* tile, auto half, bf16x8 (&f)[HM][2]) {
        constexpr int H = decltype(half)::value, BLOCKS = H ? C::MT - HM : HM;
        const int km = AKM && C::BM != 160 && HM > 2 ? g3_opaque(kmA[0]) : kmA[0]; /* eight blocks' addresses kept would not leave room for the fragments */
#pragma unroll
        for (int mh = 0; mh < BLOCKS; mh++)
#pragma unroll
            for (int kk = 0; kk < 2; kk++) {
                const int mt = H * HM + mh;
                if constexpr (ROWS::TILED) f[mh][kk] = *reinterpret_cast<const bf16x8*>(tile + ((wm * C::MT + mt) * 2 + kk) * 1024 + lane * 16);
                else if constexpr (AKM) f[mh][kk] = g3_frag_km<C::BM>(tile, C::BM == 160 && (mt & 1) ? kmA[1] : km, wm * C::MT + mt, kk);
                else f[mh][kk] = g3_frag(tile, (wm * C::MT + mt) * 16 + r16, kk * 4 + q4);
            }
    };
    auto readB = [&](const unsigned char* tile, auto half, bf16x8 (&f)[HN][2]) {
        constexpr int H = decltype(half)::value, BLOCKS = H ? C::NT - HN : HN;
        const int km = BKM && C::BN != 160 && C::BN > 128 ? g3_opaque(kmB[0]) : kmB[0];
#pragma unroll
        for (int nh = 0; nh < BLOCKS; nh++)
#pragma unroll
            for (int kk = 0; kk < 2; kk++) {
                const int nt = H * HN + nh;
                if constexpr (BKM) f[nh][kk] = g3_frag_km<C::BN>(tile, C::BN == 160 && (nt & 1) ? kmB[1] : km, wn * C::NT + nt, kk);
                else f[nh][kk] = g3_frag(tile, wn * (16 * C::NT) + nt * 16 + r16, kk * 4 + q4);
            }
    };
    constexpr int PIECES = ROWS::F32 ? 4 : 1; /* MFMAs per pair of fragments */
    auto mul = [&](auto mh0, auto nh0, const bf16x8 (&fa)[HM][2], const bf16x8 (&fb)[HN][2]) {
        constexpr int I0 = decltype(mh0)::value * HM, J0 = decltype(nh0)::value * HN;
#pragma unroll
        for (int kk = 0; kk < 2; kk++)
#pragma unroll
            for (int e = 0; e < PIECES; e++)
#pragma unroll
                for (int i = 0; i < (I0 ? C::MT - HM : HM); i++)
#pragma unroll
                    for (int j = 0; j < (J0 ? C::NT - HN : HN); j++) {
                        f32x4& d = acc[I0 + i][J0 + j];
                        if constexpr (ROWS::F32) d = __builtin_amdgcn_mfma_f32_16x16x4f32(__builtin_bit_cast(f32x4, fa[i][kk])[e], __builtin_bit_cast(f32x4, fb[j][kk])[e], d, 0, 0, 0);
                        else d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[i][kk], fb[j][kk], d, 0, 0, 0);
                    }
    };
    // the issue order of quadrant (row half, token half): its LDS reads and its loads one by one among its first MFMAs, the rest of the MFMAs behind them
    auto order = [&](auto mh, auto nh, auto n_reads, auto n_loads) {
        constexpr int N = decltype(n_reads)::value, V = decltype(n_loads)::value, M = (decltype(mh)::value ? C::MT - HM : HM) * (decltype(nh)::value ? C::NT - HN : HN) * 2 * PIECES;
        constexpr int P = N < M ? N : M, Q = V < M - 1 ? V : M - 1, X = P > Q ? P : Q;
        g3_issue<M, N, V, 0>();
        if (M > X) __builtin_amdgcn_sched_group_barrier(0x008, M - X, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    constexpr std::integral_constant<int, HM * 2 * (AKM ? 2 : 1)> ra0{};
    constexpr std::integral_constant<int, (C::MT - HM) * 2 * (AKM ? 2 : 1)> ra1{};
    constexpr std::integral_constant<int, HN * 2 * (BKM ? 2 : 1)> rb0{};
    constexpr std::integral_constant<int, (C::NT - HN) * 2 * (BKM ? 2 : 1)> rb1{};
    bf16x8 a0[HM][2], a1[HM][2], b0[HN][2], b1[HN][2];
    if (kt0 >= kt1) return;
    constexpr std::integral_constant<int, 0> none{};
    constexpr std::integral_constant<int, C::NIA> la{};
    constexpr std::integral_constant<int, C::NIB> lb{};
    // step kt on the tiles ca, cb (which hold the step's loads, and then those of step kt + NBUF); those of step kt + 1 are at na, nb.  Behind the last step the reads of "step kt + 1" take what lies there: never used
    auto step = [&](int kt, unsigned char* ca, unsigned char* cb, const unsigned char* na, const unsigned char* nb, bf16x8 (&bx)[HN][2], bf16x8 (&by)[HN][2]) __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        readB(cb, hi, by);
        mul(lo, lo, a0, bx);
        order(lo, lo, rb1, none);
        readA(ca, hi, a1);
        mul(lo, hi, a0, by);
        order(lo, hi, ra1, none);
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((C::NBUF - 2) * LPW) : "memory");
        __builtin_amdgcn_s_barrier(); /* step kt + 1 has landed for every wave, and every wave has read all of step kt: its buffer may be filled again */
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        stageA(kt + C::NBUF, ca);
        readA(na, lo, a0);
        mul(hi, hi, a1, by);
        order(hi, hi, ra0, la);
        stageB(kt + C::NBUF, cb);
        readB(nb, lo, by);
        mul(hi, lo, a1, bx);
        order(hi, lo, rb0, lb);
    };
    // the steps are unrolled by two: the two token halves' registers swap roles with them, and of two buffers every LDS address of a step is base + an immediate
    [[maybe_unused]] auto two = [&](unsigned char* a_even, unsigned char* a_odd, unsigned char* b_even, unsigned char* b_odd) {
        stageA(kt0, a_even), stageB(kt0, b_even), stageA(kt0 + 1, a_odd), stageB(kt0 + 1, b_odd);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LPW) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory"); /* no read moves up */
        readA(a_even, lo, a0), readB(b_even, lo, b0);
        for (int kt = kt0; kt < kt1; kt += 2) {
            between(kt);
            step(kt, a_even, b_even, a_odd, b_odd, b0, b1);
            if (kt + 1 < kt1) between(kt + 1), step(kt + 1, a_odd, b_odd, a_even, b_even, b1, b0);
        }
    };
    // three buffers: by six, so that every buffer is a name too.  With the buffer's number in a register a step had 14 - 21 vector additions for its LDS addresses in front of its MFMAs: us, numbered | named,
    // 128 x 256 tiles: 5120 x 5120 at 1000 rows 65 | 60, 6400 x 1600 at 8192 rows 188 | 180; 128 x 128 on 8 waves: 2048 x 2048 at 2047 rows 22.6 | 20.7, 1024 x 2048 at 2608 19.0 | 18.0; 64 x 64: 1024 x 2048 at 2047 14.7 | 14.6
    [[maybe_unused]] auto three = [&](unsigned char* a_0, unsigned char* a_1, unsigned char* a_2, unsigned char* b_0, unsigned char* b_1, unsigned char* b_2) {
        stageA(kt0, a_0), stageB(kt0, b_0), stageA(kt0 + 1, a_1), stageB(kt0 + 1, b_1), stageA(kt0 + 2, a_2), stageB(kt0 + 2, b_2);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * LPW) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory"); /* no read moves up */
        readA(a_0, lo, a0), readB(b_0, lo, b0);
        for (int kt = kt0;;) {
            between(kt), step(kt, a_0, b_0, a_1, b_1, b0, b1);
            if (++kt >= kt1) break;
            between(kt), step(kt, a_1, b_1, a_2, b_2, b1, b0);
            if (++kt >= kt1) break;
            between(kt), step(kt, a_2, b_2, a_0, b_0, b0, b1);
            if (++kt >= kt1) break;
            between(kt), step(kt, a_0, b_0, a_1, b_1, b1, b0);
            if (++kt >= kt1) break;
            between(kt), step(kt, a_1, b_1, a_2, b_2, b0, b1);
            if (++kt >= kt1) break;
            between(kt), step(kt, a_2, b_2, a_0, b_0, b1, b0);
            if (++kt >= kt1) break;
        }
    };
    static_assert(C::NBUF == 2 || C::NBUF == 3, "two or three buffers");
    if constexpr (C::NBUF == 3) g3_told_apart(bufA(0), bufA(1), bufA(2), bufB(0), bufB(1), bufB(2), three);
    else if constexpr (AKM || BKM) g3_told_apart(bufA(0), bufA(1), bufB(0), bufB(1), two);
    else two(bufA(0), bufA(1), bufB(0), bufB(1));
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier(); /* the buffers are free: for a following segment's first loads, for an epilogue's exchange */
    asm volatile("" ::: "memory");
}

// The output tile on its way out: the accumulators go to LDS as they are, where the operands' buffers were, and a LOOP over eight rows of a token applies the epilogue and stores 16 bytes a lane, whole rows of the
// tile at a time.  What bounds an epilogue is its CODE: it runs once, so every line of it is an instruction-cache miss (two CUs share 64 KiB), and unrolled over the 32 MFMA tiles of a wave it was 40 - 60 KB:
// a 256 x 256 tile took 14.4 us to store (4096 x 4096 in one round), from this loop it takes 8.4 (writing as much alone: 4).  Storing rows instead of 32-byte pieces from code as long changed nothing.
// PASSES: the tile in 32 bits may be more than the buffers hold; then half of every wave's tokens at a time.  16-byte chunks of a token are XOR-swizzled by the token: a wave's writes (16 tokens x one chunk) and its
// reads (consecutive chunks) touch all banks once.
template <class C>
struct G3Out {
    static constexpr int PASSES = (C::BM * C::BN * 4 + C::SMEM - 1) / C::SMEM, TN = C::BN / PASSES, HT = C::NT / PASSES; /* tokens, and 16-token blocks of a wave, per pass */
    static constexpr int P = C::BM % 64 == 0 ? 1 : 2; /* tokens whose rows start at different banks */
    static_assert(PASSES <= 2 && C::NT % PASSES == 0 && C::BM % 32 == 0, "a token is whole or half turns of the banks");
    static __device__ __forceinline__ int swz(int lt) { return (lt / P) & (16 / P - 1); }
    static __device__ __forceinline__ int at(int lt, int chunk) { return lt * (4 * C::BM) + ((chunk ^ swz(lt)) << 4); } /* rows 4 chunk .. + 3 of the pass's token lt */
    static __device__ __forceinline__ int token(int pass, int lt) { return PASSES == 1 ? lt : lt / (16 * HT) * (16 * C::NT) + pass * (16 * HT) + lt % (16 * HT); } /* its place in the tile */
    static __device__ __forceinline__ void spill(const f32x4 (&acc)[C::MT][C::NT], unsigned char* smem, int pass, int wid, int lane) {
        const int wm = wid / C::WN, wn = wid % C::WN, r16 = lane & 15, q4 = lane >> 4;
        unsigned char* const to = smem + (wn * (16 * HT) + r16) * (4 * C::BM); /* (16 tokens further the swizzle is the same) */
#pragma unroll
        for (int mt = 0; mt < C::MT; mt++) {
            unsigned char* const b = to + ((((wm * C::MT + mt) * 4 + q4) ^ swz(r16)) << 4);
#pragma unroll
            for (int nt = 0; nt < HT; nt++) *reinterpret_cast<f32x4*>(b + nt * 16 * (4 * C::BM)) = PASSES == 2 && pass ? acc[mt][nt + C::NT - HT] : acc[mt][nt];
        }
    }
    /* rows 8 c .. 8 c + 7 of token lt; which of the two chunks is read first alternates every eight lanes, so that sixteen lanes in a row meet in no bank */
    static __device__ __forceinline__ void rows8(const unsigned char* smem, int lt, int c, int lane, float (&v)[8]) {
        const bool odd = (lane >> 3) & 1;
        const f32x4 p = *reinterpret_cast<const f32x4*>(smem + at(lt, 2 * c + (odd ? 1 : 0))), q = *reinterpret_cast<const f32x4*>(smem + at(lt, 2 * c + (odd ? 0 : 1)));
#pragma unroll
        for (int j = 0; j < 4; j++) v[j] = odd ? q[j] : p[j], v[4 + j] = odd ? p[j] : q[j];
    }
    /* f(token of the tile, token of the pass, unit) for this thread's share of TN tokens x U units, after a barrier */
    template <int U, class F>
    static __device__ __forceinline__ void each(int pass, int tid, F&& f) {
        __syncthreads();
#pragma unroll 1
        for (int id = tid; id < TN * U; id += C::NTH) f(token(pass, id / U), id / U, id % U);
    }
    /* PASSES times: the accumulators to LDS, then each<U> */
    template <int U, class F>
    static __device__ __forceinline__ void all(const f32x4 (&acc)[C::MT][C::NT], unsigned char* smem, int tid, F&& f) {
#pragma unroll
        for (int pass = 0; pass < PASSES; pass++) {
            if (pass) __syncthreads();
            spill(acc, smem, pass, tid >> 6, tid & 63);
            each<U>(pass, tid, f);
        }
    }
};
// 16 bytes to base + off (base: uniform), written through: left to the write-back of the XCDs' L2s at the launch's end a one-round product is 1.5 - 2.5 us longer
__device__ __forceinline__ void g3_store16(void* base, uint32_t off, u32x4 v) { __builtin_amdgcn_raw_buffer_store_b128(v, g3_rsrc(base, G3_ALL), off, 0, 16 /* sc1 */); }
/* the same to `byte` of token tk's row of a tile at `base`, rows ld values apart: out of a 32-bit offset's reach by its own address */
__device__ __forceinline__ void g3_store_row(uint16_t* base, int tk, long long ld, int byte, u32x4 v) {
    if (ld < (1 << 22)) g3_store16(base, (uint32_t)tk * (uint32_t)(2 * ld) + byte, v);
    else *reinterpret_cast<u32x4*>(reinterpret_cast<unsigned char*>(base + tk * ld) + byte) = v;
}
__device__ __forceinline__ u32x4 g3_pack8(const float (&v)[8]) { return u32x4{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7])}; }
__device__ __forceinline__ void g3_unpack8(u32x4 p, float (&v)[8]) {
#pragma unroll
    for (int j = 0; j < 4; j++) v[2 * j] = bf_lo(p[j]), v[2 * j + 1] = bf_hi(p[j]);
}
// The same where a result is a bf16 rounding of the sum (plus a bias) and nothing else: it is rounded in front of LDS, half the bytes, never two passes.  us, 32 bits | so, K = 64: 4096 x 4096 in 256 x 256 tiles 13.8 | 11.6, in 192 x 256 20.3 | 15.1; 4800 x 1600
// at 8192 rows 125.7 | 120.3
template <class C>
struct G3Out16 {
    static constexpr int ROW = (C::BM / 2) % 64, P = ROW == 0 ? 1 : ROW == 32 ? 2 : 4; /* tokens whose rows start at different banks */
    static_assert(C::BM * C::BN * 2 <= C::SMEM && C::BM % 32 == 0, "the tile fits, its chunks of eight rows in eights");
    static __device__ __forceinline__ int at(int tok, int chunk) { return tok * (2 * C::BM) + ((chunk ^ ((tok / P) & (16 / P - 1))) << 4); } /* rows 8 chunk .. + 7 of a token */
    template <bool BIAS>
    static __device__ __forceinline__ void spill(const f32x4 (&acc)[C::MT][C::NT], unsigned char* smem, int tid, const uint16_t* bias, int rows) { /* bias: of the tile's rows, `rows` of them exist */
        const int wid = tid >> 6, lane = tid & 63, wm = wid / C::WN, wn = wid % C::WN, r16 = lane & 15, q4 = lane >> 4;
#pragma unroll
        for (int mt = 0; mt < C::MT; mt++) {
            const int blk = wm * C::MT + mt; /* the wave's 16-row block mt in the tile */
            float b[4] = {0.f, 0.f, 0.f, 0.f};
            if constexpr (BIAS) {
                u32x2 b4 = u32x2{0, 0};
                if (blk * 16 + 4 * q4 < rows) b4 = *reinterpret_cast<const u32x2*>(bias + blk * 16 + 4 * q4);
                b[0] = bf_lo(b4.x), b[1] = bf_hi(b4.x), b[2] = bf_lo(b4.y), b[3] = bf_hi(b4.y);
            }
            unsigned char* const to = smem + at(wn * (16 * C::NT) + r16, 2 * blk + (q4 >> 1)) + 8 * (q4 & 1); /* (16 tokens further the swizzle is the same) */
#pragma unroll
            for (int nt = 0; nt < C::NT; nt++) {
                f32x4 v = acc[mt][nt];
                if constexpr (BIAS) {
#pragma unroll
                    for (int j = 0; j < 4; j++) v[j] = v[j] + b[j];
                }
                *reinterpret_cast<u32x2*>(to + nt * 16 * (2 * C::BM)) = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
            }
        }
    }
    static __device__ __forceinline__ u32x4 rows8(const unsigned char* smem, int tok, int chunk) { return *reinterpret_cast<const u32x4*>(smem + at(tok, chunk)); }
    static __device__ __forceinline__ u32x2 rows4(const unsigned char* smem, int tok, int u) { return *reinterpret_cast<const u32x2*>(smem + at(tok, u >> 1) + 8 * (u & 1)); } /* rows 4 u .. + 3 */
    template <int U, class F>
    static __device__ __forceinline__ void each(int tid, F&& f) { /* f(token of the tile, unit) for this thread's share of BN tokens x U units, after a barrier */
        __syncthreads();
#pragma unroll 1
        for (int id = tid; id < C::BN * U; id += C::NTH) f(id / U, id % U);
    }
};
// 256 x 256 or 192 x 256: with one big workgroup per CU a launch takes whole rounds of 256 tiles, and a round of the smaller ones takes 0.79 to 0.95 of a round, so the smaller tile pays where it needs no
// more rounds.  us, big | wide: 6144 x 1024 at 2608 rows (264 | 352 tiles) 66.7 | 54.3, x 4096 176 | 143, x 25600 1230 | 1036; 5120 x 12288 at 4096 rows (320 | 432) 543 | 518; 10240 x 8192 at 3500 rows
// (560 | 756) 522 | 449.  One round more pays for 5 and 6 of them at K <= 2048, where the round is shortest against its start: 12288 x 2048 at 5888 rows (1104 | 1472) 280 | 269, at 6912 (1296 | 1728) 332 |
// 312; at K 4096 486 | 498 and 585 | 606.  Two more never: 12288 x 2048 at 11008 rows (2064 | 2752) 515 | 562.
static constexpr bool g3_prefer_wide(int M, int n, int K) {
    const long by = (n + 255) / 256, rb = ((M + 255) / 256 * by + 255) / 256, rw = ((M + 191) / 192 * by + 255) / 256;
    return rw <= rb || (rw == rb + 1 && (rb == 5 || rb == 6) && K <= 2048);
}
// The tile of a product whose rows are whole tiles of any of them (`wide` = 192-row ones may be taken): the smallest that makes ONE round of the CUs; of several rounds the cheaper of the big
// tiles and 128 x 128 on 4 waves (512 at a time), a round of R us taking R (ceil r + 0.8 r + 0.55) / 2 for r rounds (the last one is dealt out early and finds the caches warm) --
// R = E + S (K / 64): 19.7 us at K = 1024 (128 x 128), 29.2 (192 x 256), 33.3 (256 x 256).  us, 128 x 128 on 8 | 128 x 256 | 128 x 128 on 4 | 192 x 256 | 256 x 256:
//   4096 x 1024   at 2047 rows 22.6 | 18.9 | 19.7 | 22.9 | 28.3, at 2608 32.6 | 34.5 | 31.1 | 24.6 | 30.1, at 4096 48.0 | 39.3 | 38.5 | 48.1 | 33.3
//   6144 x 1024 with SwiGLU at 2047 rows 36.9 | 40.0 | 35.1 | 29.2 | 36.0, at 2608 47.5 | 58.3 | 39.9 | 53.5 | 67.9
//   6400 x 1600 at 8192 rows 191 | 174 | 169 | 164 | 169, 12288 x 2048 with SwiGLU at 8190 rows 448 | 372 | 368 | 339 | 327
enum G3Pick { G3_DUO, G3_HALF, G3_SMALL, G3_WIDE, G3_BIG, G3_SLIM, G3_FLAT };
static constexpr G3Pick g3_pick(int M, int n, int K, bool wide) {
    const long r128 = (M + 127) / 128, c128 = (n + 127) / 128, c256 = (n + 255) / 256, n128 = r128 * c128, nw = (M + 191) / 192 * c256, nb = (M + 255) / 256 * c256;
    if (n128 <= 256) return G3_DUO;
    if (r128 * c256 <= 256) return G3_HALF;
    if (n128 <= 512 || n < 256 || M < 256) return G3_SMALL;
    if (wide && nw <= 256) return G3_WIDE;
    if (nb <= 256) return G3_BIG;
    const bool w = wide && g3_prefer_wide(M, n, K);
    const double k = K / 64, rs = n128 / 512.0, rb = (w ? nw : nb) / 256.0, Rs = 3.7 + k, Rb = w ? 9.0 + 1.26 * k : 10.1 + 1.45 * k;
    const double ts = Rs * ((n128 + 511) / 512 + 0.8 * rs + 0.55), tb = Rb * (((w ? nw : nb) + 255) / 256 + 0.8 * rb + 0.55);
    return ts < 0.97 * tb ? G3_SMALL : w ? G3_WIDE : G3_BIG;
}
// Products with a k-major W (both GEMMs of a backward pass): 160 x 256 or 256 x 160 instead of 256 x 256 where they need no more rounds.  A big tile's round on three quarters of the CUs was cut in k-pieces over all of
// them, whose partial tiles (256 KiB each, written and read) took what the idle CUs had been worth and more; five eighths of a tile on nearly all CUs needs none.  us, pieces | 256 x 256 whole | 160 x 256 | 256 x 160:
//   weight gradients (bkm)  1600 x 6400 from 8192 tokens 167 | 166 | 136 | 241, 6400 x 1600 166 | 170 | 233 | 147, 1600 x 6400 from 2560 80 | 62 | 51 | 88, 4096 x 2560 from 8192 154 | 167 | 236 | 150,
//                           3000 x 3000 from 4096 95 | 90 | 75 | 72, 2400 x 3600 from 2048 63 | 52 | 42 | 41
//   input gradients         1600 x 5120 rows, K 6400: 112 | 119 | 93 | 99, 1600 x 6000, K 1600: 37 | 37 | 29 | 53, 6400 x 3000, K 1600 (two rounds each) - | 75 | 59 | 61
// One round more for four big ones gains at most 3 % (6400 x 8192, K 1600: - | 158 | 155 | 171) and is not taken.  Of both with as many rounds: us of weight gradients 75 | 72, of input gradients 92 | 97.
// One walk over k where there were two to five pieces: error of a sum of 8192 products of normal values against 64 bits 2.9e-7 of its norm, in pieces 2.1e-7; of the bf16 result 1.6613e-3 either way (restated on the host).
// 160-row tiles of an operand whose rows are in their reach (ldw: of W, ldx: of x where it is k-major too, else 0); a row beyond it is 2^24 values and more, and the big tiles reach to 2^27.
// Up to K = 8192, the longest of these rows.  Behind it nothing was timed, and pieces gain there: their partial tiles cost the same at any K, and T big tiles then take T / 256 of a big tile's time where
// 160 x 256 takes five eighths of it.  By the steps of the rows above 4096 x 2560 from 16384 tokens would be about 260 us in pieces and 290 whole (154 | 150 from 8192), the input gradient of a 50304-wide head at 5120
// rows, 786 steps, about 560 and 700 (112 | 93 with 100).
static constexpr int G3_KM_160_MAX_K = 8192;
static constexpr G3Pick g3_km_pick(int M, int n, int K, bool bkm, long long ldw, long long ldx) {
    const long nb = (long)((M + 255) / 256) * ((n + 255) / 256), rb = (nb + 255) / 256, rs = ((long)((M + 159) / 160) * ((n + 255) / 256) + 255) / 256, rf = ((long)((M + 255) / 256) * ((n + 159) / 160) + 255) / 256;
    if (K > G3_KM_160_MAX_K || nb <= 128 || (rs < rf ? rs : rf) > rb) return G3_BIG; /* (up to 128: two and more pieces of a tile, or tiles of 128 x 128) */
    const G3Pick p = rs < rf || (rs == rf && !bkm) ? G3_SLIM : G3_FLAT;
    return g3_km_reach<160>(p == G3_SLIM ? ldw : ldx) ? p : G3_BIG;
}
// Where a launch of more than half a round may be cut in owners and tails (gemm3_sk_kernel, S = 1): k-steps.  The tails of 256 x 256 tiles are 256 KiB each, about 50 us of writing and reading at any K; up to K = 4096 that is
// what the idle CUs are worth or more.  us, cut | whole, tiles in brackets: from 2048 tokens 2400 x 3600 (150) 64 | 52, from 2560 1600 x 6400 (175) 80 | 62, from 4096 3000 x 3000 (144) 95 | 90, 3072 x 3072 (144) 89 | 88, 5120 x
// 2048 (160) 94 | 91; K 6400, 1600 x 5120 (140) 112 | 119; from 8192 4096 x 2560 (160) 154 | 167, 2560 x 4096 149 | 161, 1600 x 6400 (175) 167 | 166.  Between 4096 and 6400 nothing was timed: cut.
static constexpr int g3_tails_from(int bm) { return bm == 256 ? 65 : 32; }
// workgroup number -> tile number: workgroups go to the 8 XCDs round robin, so the tiles an XCD runs back to back are made neighbours
__device__ __forceinline__ int g3_remap(int orig, int nwg) {
    const int q = nwg / 8, rr = nwg % 8, xcd = orig % 8;
    return (xcd < rr ? xcd * (q + 1) : rr * (q + 1) + (xcd - rr) * q) + orig / 8;
}
// tile number -> (row tile, token tile): bands of at most 8 row tiles, token tile after token tile inside a band, so that the 32 tiles an XCD multiplies at a time are a block of about
// 8 x 4.  What a step of those 32 brings into that XCD's L2 is 12 operand tiles; numbered row tile by row tile through all of M it was 33, and the link of an XCD (1.1 TB/s) was what the main loop
// waited for: 8192 x 8192 x 8192 with its MFMAs left out took as long as with them.
__device__ __forceinline__ void g3_tile(int t, int nbx, int nby, int& bx, int& by) {
    const int nb = (nbx + 7) / 8, h = nbx / nb, tall = nbx % nb, cut = tall * (h + 1) * nby; /* the first `tall` bands have h + 1 row tiles, the others h */
    const bool up = t < cut;
    const int r = up ? t : t - cut, w = up ? h + 1 : h, band = r / (w * nby), in = r - band * (w * nby);
    by = in / w, bx = (up ? band * (h + 1) : tall * (h + 1) + band * h) + in % w;
}
}  // namespace kf
