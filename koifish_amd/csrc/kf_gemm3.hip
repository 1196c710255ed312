// kf_gemm3.hip -- large-batch bf16 GEMM on tiles of 64 x 64 to 256 x 256 outputs, 64 deep: y[n, M] (+)= x[n, K] . W[M, K]^T (SLP::Forw's product for a dequantised or bf16
// weight) and, with either operand stored K-MAJOR, both GEMMs of SLP::Back without a transpose of anything:
//   * both operand tiles go global -> LDS by buffer loads (16 bytes per lane, no VGPR round trip; a scalar base and step, one lane offset, an empty descriptor past the last step).  The LDS image of
//     such a load is lane-linear, so the bank-conflict-free layout is produced on the SOURCE side: a tile row is 128 bytes = 8 chunks of 16 bytes, chunk c of row r
//     is stored at position c ^ ((r >> 1) & 7); a fragment read (16 rows x one chunk, ds_read_b128) then touches all 64 banks exactly once;
//     a k-major operand's image is [64 k][rows], two-term swizzle, fragments by the transposing ds_read_b64_tr_b16 (g3_frag_km);
//   * two or three LDS buffers (G3Cfg::NBUF): the loads of a later k-step are issued among the MFMAs of this one, the fragments of a quadrant are read while the one before is multiplied, and ONE raw
//     s_barrier per step, behind a wait, by count, for the next step's loads;
//   * 256 x 256: 8 waves as 2 (rows) x 4 (tokens), 128 x 64 outputs per wave = 32 accumulator tiles of v_mfma_f32_16x16x32_bf16, one workgroup per CU.  A product takes the smallest tile that makes one
//     round of the CUs, of several rounds the cheaper one (g3_pick; of k-major operands g3_km_pick; kf_gemm3_tile.h lists the tiles).  All of them add up a k in the same order;
//   * workgroup order remapped so that the blocks an XCD runs back to back share their W row-tile in that XCD's L2;
//   * split-K forms (gemm3_sk_kernel) with an ordered in-kernel fix-up for launches with fewer tiles than resident workgroups: deterministic, no atomics on data;
//   * up to three matrices stacked along M (Q | K | V, gate | up) in one launch, each tile's rows routed to its matrix's output (gemm3_multi_launch).
// Measured: 8192 x 8192 x 8192 about 1.45 PFLOP/s (1.0 with the fragments of a step read behind its barrier and per-lane global pointers); the MFMAs alone, without a load, reach 2.0 - 2.06 at the card's
// power limit.  BK = 32 with four buffers, stream-K ranges and 4 waves of 128 x 128 were slower.
// The epilogue is gemm_epilogue's (alpha, beta, bias, one bf16 store, residual added to the rounded value), a loop over the tile in LDS (G3Out).
#include <string.h>

#include <type_traits>

#include <mutex>

#include "kf_gemm3_tile.h"

namespace kf {

// ROPE::cuInfer on a 128-row tile that is one head (hd 128) of Q or K, in the epilogue of the stacked Q | K | V launch (the arithmetic of prep_head_cs, kf_attn_common.h: the
// projection rounded to bf16 as the plain epilogue stores it, fp64 sum of squares, s rounded to bf16, (x s) w rounded, rotate-half pairs (j, j + 64) with every product and the
// sum rounded once).  A thread has eight pairs of a token, the eight threads of a token are neighbours.
template <class C>
__device__ __forceinline__ void g3_epilogue_qkrope(const GemmArgs& a, int m0, int t0, const f32x4 (&acc)[C::MT][C::NT], int tid, unsigned char* smem_raw, uint16_t* ybase, long long ldy, int mshift,
                                                   const uint16_t* nw) {
    static_assert(C::BM == 128, "one head per tile");
    using Out = G3Out16<C>;
    static_assert(C::BN * 8 % C::NTH == 0, "the eight threads of a token run the loop together");
    Out::template spill<false>(acc, smem_raw, tid, nullptr, 0);
    Out::template each<8>(tid, [&](int tk, int u) {
        const int tok = t0 + tk < a.n ? t0 + tk : a.n - 1; /* (a token past the end: the last one's angles, not stored) */
        float x[2][8]; /* rows 8 u .. and 64 + 8 u .., as the plain epilogue stores them (alpha 1, no bias) */
#pragma unroll
        for (int e = 0; e < 2; e++) g3_unpack8(Out::rows8(smem_raw, tk, 8 * e + u), x[e]);
        if (nw) {
            double ss = 0.0;
#pragma unroll
            for (int e = 0; e < 2; e++)
#pragma unroll
                for (int j = 0; j < 8; j++) ss = fma((double)x[e][j], (double)x[e][j], ss);
#pragma unroll
            for (int d = 1; d < 8; d *= 2) ss += __shfl_xor(ss, d, 64);
            const float s = round_bf16(1.0f / sqrtf((float)ss / 128.0f + a.qk_eps));
#pragma unroll
            for (int e = 0; e < 2; e++) {
                float w[8];
                g3_unpack8(*reinterpret_cast<const u32x4*>(nw + 64 * e + 8 * u), w);
#pragma unroll
                for (int j = 0; j < 8; j++) x[e][j] = round_bf16(x[e][j] * s * w[j]);
            }
        }
        if (a.rope_table) { /* (cos, sin) of the eight pairs: 64 contiguous bytes of the table */
            const f32x4* const table = reinterpret_cast<const f32x4*>(a.rope_table + (size_t)(a.rope_pos0 + (a.rope_seq > 0 ? tok % a.rope_seq : tok)) * 128 + 16 * u);
#pragma unroll
            for (int p = 0; p < 4; p++) {
                const f32x4 cs = table[p];
#pragma unroll
                for (int e = 0; e < 2; e++) {
                    const int j = 2 * p + e;
                    const float c = cs[2 * e], sn = cs[2 * e + 1], lo = x[0][j], hi = x[1][j], p0 = lo * c, p1 = hi * sn, p2 = lo * sn, p3 = hi * c;
                    x[0][j] = p0 - p1, x[1][j] = p2 + p3;
                }
            }
        }
        if (t0 + tk < a.n) {
#pragma unroll
            for (int e = 0; e < 2; e++) g3_store_row(ybase + (size_t)t0 * ldy + (m0 - mshift), tk, ldy, 128 * e + 16 * u, g3_pack8(x[e]));
        }
    });
}

// epilogue (gemm_epilogue's order) of the tile at (m0, t0)
template <bool AKM, class C>
__device__ __forceinline__ void g3_epilogue(const GemmArgs& a, int m0, int t0, const f32x4 (&acc)[C::MT][C::NT], int tid, unsigned char* smem_raw) {
    using Out = G3Out<C>;
    if (!AKM && a.swiglu) { /* Relu::Forw (CU_swiglu_v0, Activation.cu:85-93) on the two bf16-rounded projections, as swiglu_kernel: 16-row block 2i holds gate rows, block 2i + 1 the up rows of
                               the same 16 FFN rows (the operand was dequantised interleaved) */
        const int F = a.M >> 1; /* a multiple of 16 (gemm3_swiglu_launch) */
        using Half = G3Out16<C>;
        Half::template spill<false>(acc, smem_raw, tid, nullptr, 0);
        Half::template each<C::BM / 16>(tid, [&](int tk, int u) {
            const int tok = t0 + tk, f = (m0 >> 1) + 8 * u, c = (u >> 1) * 4 + (u & 1);
            if (tok >= a.n || f >= F) return;
            float g[8], p[8];
            g3_unpack8(Half::rows8(smem_raw, tk, c), g), g3_unpack8(Half::rows8(smem_raw, tk, c + 2), p);
#pragma unroll
            for (int j = 0; j < 8; j++) g[j] = (g[j] * p[j]) / (1.0f + kf_expf(-g[j]));
            g3_store_row(a.y + (size_t)t0 * a.ldy + (m0 >> 1), tk, a.ldy, 16 * u, g3_pack8(g));
        });
        return;
    }
    // up to three matrices stacked along M (Q | K | V or gate | up, each a multiple of the 256-row tile: a.rb_end[j] = cumulative rows / 32): the tile's rows go to
    // that matrix's own output (the K and V rows of a prompt land in the cache, Q in its buffer)
    uint16_t* ybase = a.y;
    long long ldy = a.ldy;
    int mshift = 0, Mlim = a.M;
    if (a.njobs > 1) {
        const int e0 = a.rb_end[0] * 32, e1 = a.rb_end[1] * 32;
        if (m0 >= e1 && a.njobs > 2) ybase = a.xy[1], ldy = a.xldy[1], mshift = e1, Mlim = a.rb_end[2] * 32;
        else if (m0 >= e0) ybase = a.xy[0], ldy = a.xldy[0], mshift = e0, Mlim = e1;
        else Mlim = e0;
    }
    if constexpr (!AKM && C::BM == 128) {
        if (a.qkrope) { /* workgroup-uniform: a tile lies inside one job */
            const int job = a.njobs > 1 ? (m0 >= a.rb_end[1] * 32 ? 2 : (m0 >= a.rb_end[0] * 32 ? 1 : 0)) : 0;
            if (job < 2) {
                g3_epilogue_qkrope<C>(a, m0, t0, acc, tid, smem_raw, ybase, ldy, mshift, a.qk_norm[job]);
                return;
            }
        }
    }
    const uint16_t* const res = AKM ? nullptr : a.residual;
    // eight rows of a token, every operand of theirs 16 aligned bytes; else four rows, in 8 aligned bytes or one by one.  us, four rows straight from the accumulators | one row at a time | as here, without and with a
    // residual: 6148 x 1600 at 2608 rows 67 86 | 89 136 | 60 74, 50260 x 768 at 2048 rows 215 397 | 315 667 | 169 303, 50257 x 768 287 620 | 316 666 | 238 368
    const bool whole = ((ldy | Mlim) & 7) == 0 && ldy < (1 << 22) && ((reinterpret_cast<uintptr_t>(ybase) | reinterpret_cast<uintptr_t>(res) | reinterpret_cast<uintptr_t>(a.bias)) & 15) == 0 && (!res || (a.ldr & 7) == 0);
    const bool quads = ((ldy | Mlim) & 3) == 0 && ((reinterpret_cast<uintptr_t>(ybase) | reinterpret_cast<uintptr_t>(res) | reinterpret_cast<uintptr_t>(a.bias)) & 7) == 0 && (!res || (a.ldr & 3) == 0);
    if ((whole || quads) && a.alpha == 1.0f && a.beta == 0.0f) {
        using Half = G3Out16<C>;
        uint16_t* const yt = ybase + (size_t)t0 * ldy + (m0 - mshift);
        if (a.bias) Half::template spill<true>(acc, smem_raw, tid, a.bias + m0, Mlim - m0);
        else Half::template spill<false>(acc, smem_raw, tid, nullptr, 0);
        if (!whole) {
            Half::template each<C::BM / 4>(tid, [&](int tk, int u) {
                const int tok = t0 + tk, m = m0 + 4 * u;
                if (tok >= a.n || m >= Mlim) return;
                u32x2 v = Half::rows4(smem_raw, tk, u);
                if (res) {
                    const u32x2 r = *reinterpret_cast<const u32x2*>(res + (size_t)tok * a.ldr + m);
#pragma unroll
                    for (int j = 0; j < 2; j++) v[j] = pack_bf16x2(bf_lo(r[j]) + bf_lo(v[j]), bf_hi(r[j]) + bf_hi(v[j]));
                }
                *reinterpret_cast<u32x2*>(yt + (size_t)tk * ldy + 4 * u) = v;
            });
            return;
        }
        Half::template each<C::BM / 8>(tid, [&](int tk, int u) {
            const int tok = t0 + tk, m = m0 + 8 * u;
            if (tok >= a.n || m >= Mlim) return;
            u32x4 v = Half::rows8(smem_raw, tk, u);
            if (res) {
                const u32x4 r = *reinterpret_cast<const u32x4*>(res + (size_t)tok * a.ldr + m);
#pragma unroll
                for (int j = 0; j < 4; j++) v[j] = pack_bf16x2(bf_lo(r[j]) + bf_lo(v[j]), bf_hi(r[j]) + bf_hi(v[j]));
            }
            g3_store16(yt, (uint32_t)tk * (uint32_t)(2 * ldy) + 16 * u, v);
        });
        return;
    }
    if (whole) {
        Out::template all<C::BM / 8>(acc, smem_raw, tid, [&](int tk, int lt, int u) {
            const int tok = t0 + tk, m = m0 + 8 * u;
            if (tok >= a.n || m >= Mlim) return;
            u32x4 r4 = u32x4{0, 0, 0, 0};
            if (res) r4 = *reinterpret_cast<const u32x4*>(res + (size_t)tok * a.ldr + m);
            float v[8], o[8];
            Out::rows8(smem_raw, lt, u, tid, v);
            if (a.alpha != 1.0f) {
#pragma unroll
                for (int j = 0; j < 8; j++) v[j] = a.alpha * v[j];
            }
            if (a.beta != 0.0f) {
                g3_unpack8(*reinterpret_cast<const u32x4*>(ybase + (size_t)tok * ldy + (m - mshift)), o);
#pragma unroll
                for (int j = 0; j < 8; j++) v[j] = v[j] + a.beta * o[j];
            }
            if (a.bias) {
                g3_unpack8(*reinterpret_cast<const u32x4*>(a.bias + m), o);
#pragma unroll
                for (int j = 0; j < 8; j++) v[j] = v[j] + o[j];
            }
            if (res) {
                g3_unpack8(r4, o);
#pragma unroll
                for (int j = 0; j < 8; j++) v[j] = o[j] + round_bf16(v[j]);
            }
            g3_store16(ybase + (size_t)t0 * ldy + (m0 - mshift), (uint32_t)tk * (uint32_t)(2 * ldy) + 16 * u, g3_pack8(v));
        });
        return;
    }
    Out::template all<C::BM / 4>(acc, smem_raw, tid, [&](int tk, int lt, int u) {
        const int tok = t0 + tk, m = m0 + 4 * u;
        if (tok >= a.n || m >= Mlim) return;
        uint16_t* const yp = ybase + (size_t)tok * ldy + (m - mshift);
        const uint16_t* const rp = res ? res + (size_t)tok * a.ldr + m : nullptr;
        const int rows = Mlim - m < 4 ? Mlim - m : 4;
        auto get4 = [&](const uint16_t* p) {
            if (quads) return *reinterpret_cast<const u32x2*>(p);
            uint32_t w[4];
#pragma unroll
            for (int j = 0; j < 4; j++) w[j] = p[j < rows ? j : 0];
            return u32x2{w[0] | w[1] << 16, w[2] | w[3] << 16};
        };
        u32x2 r4 = u32x2{0, 0}, y4 = u32x2{0, 0}, b4 = u32x2{0, 0};
        if (res) r4 = get4(rp);
        if (a.beta != 0.0f) y4 = get4(yp);
        if (a.bias) b4 = get4(a.bias + m);
        const f32x4 d = *reinterpret_cast<const f32x4*>(smem_raw + Out::at(lt, u));
        uint32_t o[2];
#pragma unroll
        for (int e = 0; e < 2; e++) {
            float v[2] = {d[2 * e], d[2 * e + 1]};
            const float y[2] = {bf_lo(y4[e]), bf_hi(y4[e])}, b[2] = {bf_lo(b4[e]), bf_hi(b4[e])}, r[2] = {bf_lo(r4[e]), bf_hi(r4[e])};
#pragma unroll
            for (int j = 0; j < 2; j++) {
                if (a.alpha != 1.0f) v[j] = a.alpha * v[j];
                if (a.beta != 0.0f) v[j] = v[j] + a.beta * y[j];
                if (a.bias) v[j] = v[j] + b[j];
                if (res) v[j] = r[j] + round_bf16(v[j]);
            }
            o[e] = pack_bf16x2(v[0], v[1]);
        }
        if (quads) {
            *reinterpret_cast<u32x2*>(yp) = u32x2{o[0], o[1]};
            return;
        }
#pragma unroll
        for (int j = 0; j < 4; j++)
            if (j < rows) yp[j] = (uint16_t)(o[j >> 1] >> (16 * (j & 1)));
    });
}

template <bool AKM, bool BKM, int BK, class C>
__global__ void __launch_bounds__(C::NTH, C::WGS_PER_CU * C::NW / 4) gemm3_kernel(const GemmArgs a) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int nbx = (a.M + C::BM - 1) / C::BM, nby = (a.n + C::BN - 1) / C::BN, nwg = nbx * nby;
    const int wg = g3_remap(blockIdx.x, nwg);
    int bx, by;
    g3_tile(wg, nbx, nby, bx, by);
    const int m0 = bx * C::BM, t0 = by * C::BN;
    f32x4 acc[C::MT][C::NT];
#pragma unroll
    for (int i = 0; i < C::MT; i++)
#pragma unroll
        for (int j = 0; j < C::NT; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    g3_mainloop<AKM, BKM, BK, C>(a, m0, t0, 0, a.K / BK, acc, smem_raw, wid, lane);
    const int e = g3_opaque(tid);
    g3_epilogue<AKM, C>(a, m0, t0, acc, e, smem_raw);
}

// a tile by one workgroup, its k in S equal pieces that are added up in order: the sums of the S >= 2 split-K form below, bit for bit, where no workgroup is idle that would take a piece
template <class C>
__global__ void __launch_bounds__(C::NTH, C::WGS_PER_CU * C::NW / 4) gemm3_pieces_kernel(const GemmArgs a, int S) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    const int tid = threadIdx.x, nbx = (a.M + C::BM - 1) / C::BM, nby = (a.n + C::BN - 1) / C::BN, nkt = a.K / G3_BK;
    int bx, by;
    g3_tile(g3_remap(blockIdx.x, nbx * nby), nbx, nby, bx, by);
    const int m0 = bx * C::BM, t0 = by * C::BN;
    f32x4 acc[C::MT][C::NT], sum[C::MT][C::NT];
#pragma unroll
    for (int i = 0; i < C::MT; i++)
#pragma unroll
        for (int j = 0; j < C::NT; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    int piece = 1, next = nkt / S;
    auto between = [&](int kt) __attribute__((always_inline)) {
        if (kt != next) return;
#pragma unroll
        for (int i = 0; i < C::MT; i++)
#pragma unroll
            for (int j = 0; j < C::NT; j++) sum[i][j] = piece == 1 ? acc[i][j] : sum[i][j] + acc[i][j], acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        piece++, next = (int)((long long)nkt * piece / S);
    };
    g3_mainloop<false, false, G3_BK, C>(a, m0, t0, 0, nkt, acc, smem_raw, tid >> 6, tid & 63, G3Rows(), between);
#pragma unroll
    for (int i = 0; i < C::MT; i++)
#pragma unroll
        for (int j = 0; j < C::NT; j++) acc[i][j] = sum[i][j] + acc[i][j];
    const int e = g3_opaque(tid);
    g3_epilogue<false, C>(a, m0, t0, acc, e, smem_raw);
}

// SPLIT-K forms for launches with fewer tiles than CUs (a weight gradient [OC, IC] of 49 tiles, its contraction 8192 token rows long; where tiles of 160 make one round they are taken instead).  The pieces are cut so
// that the workgroups an XCD runs side by side stay at (nearly) the SAME k: they share operand strips in that XCD's L2.  (Ranges of a plain stream-K cut drift apart
// in k and every workgroup then streams its own strips through the fabric -- measured: 496 TFLOP/s.)
//   S >= 2 (2 P <= 256):  every tile's k-steps are cut in S equal pieces, P S workgroups; piece 0 owns the tile;
//   S == 1 (P < 256 < 2 P): workgroup t < P owns tile t and multiplies k-steps [0, kp), kp = nkt P / 256; the 256 - P helpers cut the tails [kp, nkt) of all tiles,
//                          laid end to end, into equal ranges (a helper's range covers pieces of 2 .. 5 tiles; neighbours start a few steps apart).  Owners and
//                          helpers finish together.
// A non-owner leaves each fp32 partial in a slot of `ws` with write-through stores and raises the slot's flag; the owner adds its tile's partials in slot order -- a
// fixed order: the result does not depend on timing -- and runs the epilogue.  a raised flag holds the launch's own value (g3_sk_epoch below: no clearing between launches); only owners wait, for pieces that
// were dispatched before them and wait for nobody.
struct G3SkArgs {
    float* ws;       /* [<= 256][256 * 256] */
    uint32_t* flags; /* [<= 256] */
    int P, S, kp, R;
    uint32_t epoch; /* the value a raised flag holds in THIS launch (g3_sk_epoch): no memset between launches */
};
template <class C>
__device__ __forceinline__ void g3_publish(const G3SkArgs& s, int slot, const f32x4 (&acc)[C::MT][C::NT], int tid) {
    const __amdgpu_buffer_rsrc_t rs = g3_rsrc(s.ws + (size_t)slot * (C::BM * C::BN), C::BM * C::BN * 4);
#pragma unroll
    for (int i = 0; i < C::MT * C::NT; i++)
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[i / C::NT][i % C::NT]), rs, (i * C::NTH + tid) * 16, 0, 16 /* sc1 */);
    // the partial went out with write-through (sc1) stores and every lane has their acknowledgements (vmcnt 0) before the flag is raised -- itself a write-through
    // store.  A release fence here (buffer_wbl2) would write back every dirty line of this XCD's L2, the finished output tiles of its other workgroups included:
    // measured 37 vs 27 us on a 128-tile product.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0) __builtin_amdgcn_raw_buffer_store_b32(s.epoch, g3_rsrc(s.flags + slot, 4), 0, 0, 16 /* sc1 */);
}
template <class C>
__device__ __forceinline__ void g3_collect(const G3SkArgs& s, int slot, f32x4 (&acc)[C::MT][C::NT], int tid) {
    if (tid == 0) {
        for (int spins = 0; spins < (1 << 24); spins++) {
            if (__builtin_amdgcn_raw_buffer_load_b32(g3_rsrc(s.flags + slot, 4), 0, 0, 16 /* sc1 */) == s.epoch) break; /* the partial is read with sc1 loads too: nothing cached to invalidate */
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_sleep(4);
        }
    }
    __syncthreads();
    const __amdgpu_buffer_rsrc_t rs = g3_rsrc(s.ws + (size_t)slot * (C::BM * C::BN), C::BM * C::BN * 4);
    constexpr int B = C::MT * C::NT < 8 ? C::MT * C::NT : 8; /* loads in flight at a time: the big tile's accumulators hold half the register file */
    static_assert(C::MT * C::NT % B == 0, "whole batches");
#pragma unroll
    for (int g = 0; g < C::MT * C::NT / B; g++) {
        f32x4 pv[B];
#pragma unroll
        for (int i = 0; i < B; i++) pv[i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, ((g * B + i) * C::NTH + tid) * 16, 0, 16 /* sc1 */));
#pragma unroll
        for (int i = 0; i < B; i++) acc[(g * B + i) / C::NT][(g * B + i) % C::NT] += pv[i];
        asm volatile("" ::: "memory");
    }
}
template <bool AKM, bool BKM, int BK, class C>
__global__ void __launch_bounds__(C::NTH, C::WGS_PER_CU * C::NW / 4) gemm3_sk_kernel(const GemmArgs a, const G3SkArgs s) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    const int tid = threadIdx.x;
    const int nbx = (a.M + C::BM - 1) / C::BM, nby = (a.n + C::BN - 1) / C::BN, nkt = a.K / BK;
    // Roles by DISPATCH order: every non-owner piece of a tile has a smaller blockIdx than the tile's owner, and non-owners wait for nobody -- so when an owner runs, the
    // pieces it waits for have at least started, whatever else occupies the chip (a collective on another stream): the waits end, no residency assumption.
    // S >= 2: blockIdx group g = blockIdx / P holds piece S - 1 - g of every tile (the owners, piece 0, are the last group); S == 1: the helpers first, then the owners.
    // Inside a group the XCD remap keeps neighbouring tiles on one XCD (the group offset only rotates the XCD labels).
    const int nhelp = (int)gridDim.x - s.P; /* S == 1 */
    const bool helper = s.S < 2 && (int)blockIdx.x < nhelp;
    const int w = s.S >= 2 ? (s.S - 1 - (int)blockIdx.x / s.P) * s.P + g3_remap((int)blockIdx.x % s.P, s.P)
                           : (helper ? s.P + g3_remap((int)blockIdx.x, nhelp) : g3_remap((int)blockIdx.x - nhelp, s.P));
    // tail mode: tail length L, T = P L tail steps in all, cut into ranges of R = s.R steps (the host's ceil(T / helpers)); 32-bit: the host checks T < 2^31
    const int L = nkt - s.kp, T = s.P * L, R = s.R;
    int hb = 0, he = 1; /* a helper's range of tail steps; the other roles make one pass */
    if (helper) hb = (w - s.P) * R, he = hb + R < T ? hb + R : T;
    for (int it = hb; it < he;) {
        int tile, k0, k1, slot = 0, c0 = 0, c1 = 0; /* c0 .. c1 - 1: the slots an owner collects */
        bool owner;
        if (s.S >= 2) {
            const int sp = w / s.P;
            tile = w % s.P, k0 = (int)((long long)nkt * sp / s.S), k1 = (int)((long long)nkt * (sp + 1) / s.S);
            owner = sp == 0, slot = tile * (s.S - 1) + sp - 1, c0 = tile * (s.S - 1), c1 = c0 + s.S - 1;
        } else if (!helper) {
            tile = w, k0 = 0, k1 = s.kp, owner = true;
            const int lo = tile * L; /* helpers lo / R .. (lo + L - 1) / R meet this tile's tail; the piece of helper h in tile t has slot h + t */
            c0 = lo / R + tile, c1 = (lo + L - 1) / R + tile + 1;
        } else {
            tile = it / L;
            const int o = it - tile * L, len = L - o < he - it ? L - o : he - it;
            k0 = s.kp + o, k1 = k0 + len, owner = false, slot = (w - s.P) + tile; /* pieces in range order: one slot each, < P + helpers */
        }
        c0 = __builtin_amdgcn_readfirstlane(c0), c1 = __builtin_amdgcn_readfirstlane(c1), slot = __builtin_amdgcn_readfirstlane(slot);
        int bx, by;
        g3_tile(tile, nbx, nby, bx, by);
        const int m0 = bx * C::BM, t0 = by * C::BN;
        f32x4 acc[C::MT][C::NT];
#pragma unroll
        for (int i = 0; i < C::MT; i++)
#pragma unroll
            for (int j = 0; j < C::NT; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        const int b = g3_opaque(tid);
        g3_mainloop<AKM, BKM, BK, C>(a, m0, t0, k0, k1, acc, smem_raw, b >> 6, b & 63);
        const int e = g3_opaque(tid);
        if (!owner) {
            g3_publish<C>(s, slot, acc, e);
        } else {
            for (int c = c0; c < c1; c++) g3_collect<C>(s, c, acc, e);
            g3_epilogue<AKM, C>(a, m0, t0, acc, e, smem_raw);
        }
        it += helper ? k1 - k0 : 1;
    }
}

// The flag value of one split-K launch.  Launches outside a capture take a fresh value each (a process-wide counter from 2 up), so the flags of the launch before need
// no clearing -- that was a dependent 2-3 us node in front of every such product; a flag area seen for the first time is cleared once.  A launch that is being
// CAPTURED is replayed with the arguments it was recorded with: it keeps the clearing node and the value 1.
constexpr size_t G3_SK_FLAG_BYTES = 8192; /* up to 2048 resident workgroups (64 x 64 tiles, eight per CU) */
static std::mutex g_sk_mu;
static uint32_t g_sk_epoch = 1;
static const void* g_sk_seen[8] = {nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
__global__ void __launch_bounds__(256) g3_clear_kernel(u32x4* flags, int n4) {
    for (int i = threadIdx.x; i < n4; i += 256) flags[i] = u32x4{0, 0, 0, 0};
}
static int g3_sk_epoch(hipStream_t st, uint32_t* flags, int n, uint32_t* epoch) {
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(st, &cs) != hipSuccess) return KF_HIP_CHECK;
    std::lock_guard<std::mutex> lk(g_sk_mu);
    bool seen = false;
    for (int i = 0; i < 8; i++) seen = seen || g_sk_seen[i] == flags;
    if (cs != hipStreamCaptureStatusNone || !seen) {
        const int n4 = seen ? n / 4 : (int)(G3_SK_FLAG_BYTES / 16); /* first seen: the whole area (the next launch may be of smaller tiles, with more flags) */
        hipLaunchKernelGGL(g3_clear_kernel, dim3(1), dim3(256), 0, st, (u32x4*)flags, n4); /* a kernel: memset nodes of a replayed graph have left their memory as it was on this part */
        if (hipGetLastError() != hipSuccess) return KF_HIP_CHECK;
    }
    if (cs != hipStreamCaptureStatusNone) {
        *epoch = 1;
        return KF_OK;
    }
    if (!seen) {
        static int next = 0;
        g_sk_seen[next] = flags, next = (next + 1) & 7;
    }
    if (++g_sk_epoch < 2) g_sk_epoch = 2;
    *epoch = g_sk_epoch;
    return KF_OK;
}

void gemm3_sk_forget(void* ws) { /* something else was (or will be) written where this workspace's flags lie: its next launch clears them */
    const void* const flags = (char*)ws + gemm3_sk_ws_bytes() - G3_SK_FLAG_BYTES;
    std::lock_guard<std::mutex> lk(g_sk_mu);
    for (const void*& p : g_sk_seen)
        if (p == flags) p = nullptr;
}

// Whether nwg tiles of C go in k-pieces, and how (P, S, kp, R; the number of workgroups): when they are fewer than 4/5 of the resident workgroups and the pieces stay >= 512 deep in k; a K-contiguous product of
// K < 3072 (KM: either operand k-major) only where three pieces of every tile find room.  us per layer of prompts on resident copies, never | from K = 3072 | three pieces: 0.6B 320 rows 134 | 116 | 106, 1024 rows
// 149 | 143 | 137, 2047 rows 198 | 190 | 187; 1.7B 320 rows 196 | 165 | 156.  Two pieces below K = 3072: 16 prompts of 131 tokens 6.12 -> 6.18 ms; a piece and tails: 1.7B at 1800 rows 325 -> 332 us.
template <bool KM, class C>
static bool g3_cut(long nwg, int nkt, G3SkArgs& s, int& nlaunch) {
    const int G = 256 * C::WGS_PER_CU, min_steps = 512 / G3_BK;
    if (5 * nwg >= 4 * G || !(KM || 3 * nwg <= G || nkt >= 48)) return false;
    if (2 * nwg > G && nkt < g3_tails_from(C::BM)) return false;
    s.P = (int)nwg, s.S = G / s.P, s.kp = 0, s.R = 1;
    if (s.S >= 2) {
        while (s.S > 1 && nkt / s.S < min_steps) s.S--;
        nlaunch = s.P * s.S;
        return s.S >= 2;
    }
    s.kp = (int)(((long long)nkt * s.P + G / 2) / G);
    nlaunch = G;
    const long long T = (long long)s.P * (nkt - s.kp);
    s.R = (int)((T + (G - s.P) - 1) / (G - s.P));
    return nkt - s.kp >= 1 && T * 2 < (1LL << 31) && s.kp > 0;
}
// KF_OK launched, 1 = not for this kernel (the caller's other tile kernels take the shape), < 0 error.  bf16 "weights" only: quantised ones are dequantised first.
// BK = 32 (4 LDS buffers, three steps in flight) was measured 8-10 % slower than BK = 64 (2 buffers) on every shape, forward and backward: the per-step costs
// (barrier, counted wait, loop) double, and the loop is not waiting for memory.  Only BK = 64 is instantiated.
template <bool AKM, bool BKM, class C>
static int g3_go_c(hipStream_t st, const GemmArgs& a, long nwg, void* ws, size_t ws_bytes, long min_plain) {
    constexpr int BK = G3_BK, SMEM = C::SMEM;
    static int attr_set = 0;
    if (!attr_set && SMEM > 64 * 1024) {
        if (hipFuncSetAttribute((const void*)gemm3_kernel<AKM, BKM, BK, C>, hipFuncAttributeMaxDynamicSharedMemorySize, SMEM) != hipSuccess) return KF_HIP_CHECK;
        if (hipFuncSetAttribute((const void*)gemm3_sk_kernel<AKM, BKM, BK, C>, hipFuncAttributeMaxDynamicSharedMemorySize, SMEM) != hipSuccess) return KF_HIP_CHECK;
        attr_set = 1;
    }
    G3SkArgs s;
    int nlaunch;
    if (ws && ws_bytes >= gemm3_sk_ws_bytes() && g3_cut<AKM || BKM, C>(nwg, a.K / BK, s, nlaunch)) {
        // the flags live in the LAST 8 KiB of the lent workspace whatever the tile configuration (behind the partial tiles of THIS configuration they would move with it,
        // and another configuration's fp32 partials could overwrite words already marked "seen" with values that pass for an epoch)
        static_assert((size_t)256 * C::WGS_PER_CU * C::BM * C::BN * 4 <= (size_t)256 * G3_BM * G3_BN * 4 && 256 * C::WGS_PER_CU * 4 <= G3_SK_FLAG_BYTES, "partials and flags fit the lent workspace");
        s.ws = (float*)ws, s.flags = (uint32_t*)((char*)ws + gemm3_sk_ws_bytes() - G3_SK_FLAG_BYTES);
        if (g3_sk_epoch(st, s.flags, 256 * C::WGS_PER_CU, &s.epoch) != KF_OK) return KF_HIP_CHECK;
        hipLaunchKernelGGL((gemm3_sk_kernel<AKM, BKM, BK, C>), dim3(nlaunch), dim3(C::NTH), SMEM, st, a, s);
        return hipGetLastError() == hipSuccess ? KF_OK : KF_HIP_CHECK;
    }
    if (nwg < min_plain) return 1;
    hipLaunchKernelGGL((gemm3_kernel<AKM, BKM, BK, C>), dim3((unsigned)nwg), dim3(C::NTH), SMEM, st, a);
    return hipGetLastError() == hipSuccess ? KF_OK : KF_HIP_CHECK;
}
template <bool AKM, bool BKM>
static int g3_go(hipStream_t st, const GemmArgs& a, long nwg, void* ws, size_t ws_bytes) {
    return g3_go_c<AKM, BKM, G3Big>(st, a, nwg, ws, ws_bytes, 64);
}
size_t gemm3_sk_ws_bytes() { return (size_t)256 * G3_BM * G3_BN * 4 + G3_SK_FLAG_BYTES; }
static long g3_tiles_of(int M, int n, int bm, int bn) { return (long)((M + bm - 1) / bm) * ((n + bn - 1) / bn); }
template <class C, bool AKM = false, bool BKM = false>
static int g3_whole(hipStream_t st, const GemmArgs& a) { /* one workgroup per tile */
    static int attr_set = 0;
    if (!attr_set && C::SMEM > 64 * 1024) {
        if (hipFuncSetAttribute((const void*)gemm3_kernel<AKM, BKM, G3_BK, C>, hipFuncAttributeMaxDynamicSharedMemorySize, C::SMEM) != hipSuccess) return KF_HIP_CHECK;
        attr_set = 1;
    }
    hipLaunchKernelGGL((gemm3_kernel<AKM, BKM, G3_BK, C>), dim3((unsigned)g3_tiles_of(a.M, a.n, C::BM, C::BN)), dim3(C::NTH), C::SMEM, st, a);
    return hipGetLastError() == hipSuccess ? KF_OK : KF_HIP_CHECK;
}
template <class C>
static int g3_pieces(hipStream_t st, const GemmArgs& a, int S) {
    static int attr_set = 0;
    if (!attr_set && C::SMEM > 64 * 1024) {
        if (hipFuncSetAttribute((const void*)gemm3_pieces_kernel<C>, hipFuncAttributeMaxDynamicSharedMemorySize, C::SMEM) != hipSuccess) return KF_HIP_CHECK;
        attr_set = 1;
    }
    hipLaunchKernelGGL((gemm3_pieces_kernel<C>), dim3((unsigned)g3_tiles_of(a.M, a.n, C::BM, C::BN)), dim3(C::NTH), C::SMEM, st, a, S);
    return hipGetLastError() == hipSuccess ? KF_OK : KF_HIP_CHECK;
}
static int g3_picked(hipStream_t st, const GemmArgs& a, bool wide) {
    switch (g3_pick(a.M, a.n, a.K, wide && g_knobs.g3_wide)) {
        case G3_DUO: return g3_whole<G3Duo>(st, a);
        case G3_HALF: return g3_whole<G3Half>(st, a);
        case G3_SMALL: return g3_whole<G3Small>(st, a);
        case G3_WIDE: return g3_whole<G3Wide>(st, a);
        default: return g3_whole<G3Big>(st, a);
    }
}
int gemm3_launch(hipStream_t st, int fmt, const GemmArgs& a, void* ws, size_t ws_bytes) {
    if (fmt != FMT_BF16 || a.K % G3_BK != 0 || a.K < G3_BK) return 1;
    if ((a.ldx & 7) != 0 || (reinterpret_cast<uintptr_t>(a.x) & 15) != 0 || (reinterpret_cast<uintptr_t>(a.w) & 15) != 0 || (a.K & 7) != 0) return 1;
    if (a.n < 128 || a.M < 128) return 1;
    const int nkt = a.K / G3_BK;
    const long n128 = g3_tiles_of(a.M, a.n, 128, 128), n64 = g3_tiles_of(a.M, a.n, 64, 64);
    if (n128 < 32 && n64 < 64) return 1;
    // Where the workspace is lent (resident copies, and a layer's own from K = 3072) products go in k-pieces, cut as g3_cut says for 64 x 128 or 64 x 64 tiles.  Which products are cut, and where, is part of their result,
    // and stays: other cuts are other sums in every layer of a prompt, and a 1.7B or 32B prompt in 4 bits is then farther from itself than its error allows.  Who adds the pieces up is free: other workgroups
    // (gemm3_sk_kernel) or, of a layer's own copies (a.own_pieces), the tile's workgroup one after the other (gemm3_pieces_kernel), of 64 x 64 tiles or of 128 x 128 on 8 waves.  us, M x K at rows (64 x 64 tiles | 128 x 128): others' | 64 x 64 | 128 x 128:
    //   1024 x 3072 at 515 rows (144 | 40) 17.8 | 16.4 | 28.0, at 1500 (384 | 96) 23.3 | 20.8 | 26.7, at 2047 (512 | 128) 25.7 | 21.6 | 26.2, at 2608 (656 | 168) 31.1 | 29.0 | 25.6; 1024 x 2048 at 2047 20.6 | 16.2 | 19.9;
    //   2048 x 4096 at 1030 (544 | 144) 37.0 | 35.6 | 31.5; 2048 x 6144 at 330 (192) 28.7 | 27.3 | 46.8, at 700 (352 | 96) 34.2 | 38.7 | 46.0, at 1300 (672 | 176) 55.7 | 59.7 | 46.2; 2560 x 9728 at 330 (240) 46.7 | 40.2 |
    //   65.4, at 515 (360) 52.0 | 56.7 | 64.2, at 900 (600 | 160) 71.9 | 85.9 | 64.3; 5120 x 8192 at 330 (480) 49.1 | 51.7 | 55.8, at 450 (640 | 160) 62.1 | 70.0 | 54.2
    if (ws && ws_bytes >= gemm3_sk_ws_bytes() && n128 < 256) {
        const long nmid = g3_tiles_of(a.M, a.n, 64, 128);
        G3SkArgs s;
        int nl;
        if (nmid >= 192 ? g3_cut<false, G3Mid>(nmid, nkt, s, nl) : g3_cut<false, G3Tiny>(n64, nkt, s, nl)) {
            if (a.own_pieces && s.S >= 2 && n64 <= (nkt < 96 ? 512 : 256)) return g3_pieces<G3Few>(st, a, s.S);
            if (a.own_pieces && s.S >= 2 && n64 > 512) return g3_pieces<G3Duo>(st, a, s.S);
            return nmid >= 192 ? g3_go_c<false, false, G3Mid>(st, a, nmid, ws, ws_bytes, 1) : g3_go_c<false, false, G3Tiny>(st, a, n64, ws, ws_bytes, 1);
        }
    }
    // Otherwise the smallest tile that makes ONE round of the CUs (g3_pick; in front of it 64 x 64: up to two side by side, from K = 6144 one).  us with a residual, 64 x 64 | 64 x 128 (three buffers) | 128 x 128 on 8 waves |
    // 128 x 256 | 128 x 128 on 4 waves:  M 1024 x K 2048 at 515 rows 12.5 | 17.4 | 20.7 | 31.0 | 28.3, at 2047 rows 18.0 | 18.5 | 21.4 | 32.0 | 29.2, at 2608 rows (656 tiles) 22.8 | 23.9 | 21.8 | 32.3 | 29.4;
    // M 2048 x K 6144 at 1540 rows 99 | 87 | 66 | 100 | 90, at 2608 rows (1312 | 672 | 336 | 176) 146 | 133 | 132 | 102 | 122
    if (n64 <= (nkt < 96 ? 512 : 256)) return g3_whole<G3Few>(st, a);
    return g3_picked(st, a, true);
}
// y[n, M] = alpha * sum_k B(k, tok) A(k, m) + beta * y (+ bias) with either operand stored K-MAJOR: akm: A = w[K][lda] (element (k, m) at k * lda + m), else w[M][K];
// bkm: B = x[K][ldb], else x[n][ldb].  The two GEMMs of SLP::Back without a transpose of anything:  delta[n, IC] = deltaIn[n, OC] . W[OC, IC]  (A = W k-major),
// gW[OC, IC] += deltaIn^T . inp  (A = inp[n][IC] k-major, B = deltaIn[n][OC] k-major, contraction over the n token rows).  1 = shape not served.
// ws (gemm3_sk_ws_bytes() bytes, 16-byte aligned) lends the stream-K form its partial-tile slots; NULL = one workgroup per tile only.
int gemm3_km_launch(hipStream_t st, const uint16_t* A, long long lda, bool akm, const uint16_t* B, long long ldb, bool bkm, int n, int M, int K, uint16_t* y, long long ldy,
                    const uint16_t* bias, float alpha, float beta, void* ws, size_t ws_bytes) {
    if (K % G3_BK != 0 || K < G3_BK || n < G3_BN || M < G3_BM || (M & 7) || (n & 7) || (lda & 7) || (ldb & 7)) return 1;
    if ((reinterpret_cast<uintptr_t>(A) & 15) || (reinterpret_cast<uintptr_t>(B) & 15)) return 1;
    if ((akm && !g3_km_reach<G3_BM>(lda)) || (bkm && !g3_km_reach<G3_BN>(ldb))) return 1;
    const long nwg = (long)((M + G3_BM - 1) / G3_BM) * ((n + G3_BN - 1) / G3_BN);
    GemmArgs a;
    memset(&a, 0, sizeof(a));
    a.w = reinterpret_cast<const unsigned char*>(A), a.M = M, a.K = K, a.x = B, a.ldx = ldb, a.n = n, a.y = y, a.ldy = ldy, a.bias = bias, a.alpha = alpha, a.beta = beta;
    a.ldr = lda; /* the k-major A operand's row stride */
    if (!akm && lda != K) return 1; /* the row-major A form reads rows of K */
    // big tiles that fill less than 4/5 of the CUs: 128 x 128 tiles instead when they make (nearly) whole rounds of the 512 resident workgroups, or -- with the
    // workspace -- their split-K form (partials of 64 KiB instead of 256 KiB, twice the workgroups)
    // (measured: Qwen3-0.6B training step 99.3 -> 95.7 ms with the first rule alone, -> 87.2 ms with both; GPT2-1558M 166.0 -> 163.7 -> 161.2 ms)
    const long nws = (long)((M + 127) / 128) * ((n + 127) / 128), rounds = (nws + 511) / 512;
    const bool small = 5 * nwg < 4 * 256 && akm && g3_km_reach<128>(lda) && (!bkm || g3_km_reach<128>(ldb)) && (20 * nws >= 17 * rounds * 512 || (ws && ws_bytes >= gemm3_sk_ws_bytes() && 5 * nws < 4 * 512));
    if (small) return bkm ? g3_go_c<true, true, G3Small>(st, a, nws, ws, ws_bytes, 1) : g3_go_c<true, false, G3Small>(st, a, nws, ws, ws_bytes, 1);
    switch (akm ? g3_km_pick(M, n, K, bkm, lda, bkm ? ldb : 0) : G3_BIG) {
        case G3_SLIM: return bkm ? g3_whole<G3Slim, true, true>(st, a) : g3_whole<G3Slim, true, false>(st, a);
        case G3_FLAT: return bkm ? g3_whole<G3Flat, true, true>(st, a) : g3_whole<G3Flat, true, false>(st, a);
        default: break;
    }
    if (akm && bkm) return g3_go<true, true>(st, a, nwg, ws, ws_bytes);
    if (akm) return g3_go<true, false>(st, a, nwg, ws, ws_bytes);
    if (bkm) return g3_go<false, true>(st, a, nwg, ws, ws_bytes);
    return g3_go<false, false>(st, a, nwg, ws, ws_bytes);
}

// up to three bf16 matrices stacked along M in ONE contiguous buffer (the caller dequantised them back to back: Q | K | V, or gate | up), each a multiple of 256
// rows, multiplied by the same x in one launch; matrix j's rows go to y[j] (row stride M[j]).  1 = shape not served.
// rope != NULL (n_w == 3: Q | K | V, head_dim 128): q/k-norm + RoPE in the epilogue (GemmArgs::qkrope), on tiles of 128 rows: one head; 1 where Q and K are not whole heads
// or a pointer is not 16-byte aligned: the caller then runs the plain stacked launch and qknorm_rope_launch
int gemm3_multi_launch(hipStream_t st, int n_w, const uint16_t* Wcat, const int* M, int K, const uint16_t* x, long long ldx, int n, uint16_t* const* y, const G3Rope* rope) {
    if (n_w < 2 || n_w > 3 || K % G3_BK != 0 || K < G3_BK || n < G3_BN || (ldx & 7) || (reinterpret_cast<uintptr_t>(x) & 15) || (reinterpret_cast<uintptr_t>(Wcat) & 15)) return 1;
    GemmArgs a;
    memset(&a, 0, sizeof(a));
    int tot = 0;
    for (int j = 0; j < 3; j++) {
        if (j < n_w) {
            if (M[j] < G3_BM || M[j] % G3_BM != 0) return 1;
            tot += M[j];
        }
        a.rb_end[j] = tot / 32;
        if (j >= 1 && j < n_w) a.xy[j - 1] = y[j], a.xldy[j - 1] = M[j];
    }
    a.njobs = n_w;
    a.w = reinterpret_cast<const unsigned char*>(Wcat), a.M = tot, a.K = K, a.x = x, a.ldx = ldx, a.n = n, a.y = y[0], a.ldy = M[0], a.alpha = 1.0f, a.beta = 0.0f;
    const long nwg = (long)(tot / G3_BM) * ((n + G3_BN - 1) / G3_BN);
    if (nwg < 64 && (long)(tot / 128) * ((n + 127) / 128) < 64) return 1;
    const long n128 = g3_tiles_of(tot, n, 128, 128);
    if (rope) { /* a head-sized tile: one round of the wider or the deeper one where it is one */
        if (n_w != 3 || M[0] % 128 != 0 || M[1] % 128 != 0 || ((reinterpret_cast<uintptr_t>(y[0]) | reinterpret_cast<uintptr_t>(y[1]) | reinterpret_cast<uintptr_t>(rope->wq) | reinterpret_cast<uintptr_t>(rope->wk) | reinterpret_cast<uintptr_t>(rope->table)) & 15)) return 1;
        a.qkrope = 1, a.qk_norm[0] = rope->wq, a.qk_norm[1] = rope->wk, a.rope_table = rope->table, a.rope_pos0 = rope->pos0, a.rope_seq = rope->seq_len, a.qk_eps = rope->eps;
    }
    // us, 128 x 128 on 4 waves | 128 x 384 where that is one round: 16 + 8 + 8 heads x 128, K 1024, at 2100 rows 37.1 | 30.5, at 3000 36.5 | 31.0; K 2048, 2608 rows 57.7 | 47.9; 8 + 2 + 2 heads, K 1024, 7500 rows
    // 36.5 | 31.4; 32 + 8 + 8, K 4096, 1600 rows 98.0 | 80.8; 64 + 8 + 8, K 5120, 1000 rows 127.8 | 96.4
    if (rope) return n128 <= 256 ? g3_whole<G3Duo>(st, a) : g3_tiles_of(tot, n, 128, 256) <= 256 ? g3_whole<G3Half>(st, a) : g3_tiles_of(tot, n, 128, 384) <= 256 ? g3_whole<G3Long>(st, a) : g3_whole<G3Small>(st, a);
    return g3_picked(st, a, false); /* a tile's rows are one matrix's: no 192-row ones */
}

// gate | up dequantised INTERLEAVED in blocks of 16 rows (dequant_launch ilv_n = 2) x the same x, SwiGLU in the epilogue: act[n, ffn] in one launch (the stacked route
// wrote both projections and ran swiglu_kernel over them: 12 us and 38 MB of traffic per layer of a 2047-token prompt).  1 = shape not served.
int gemm3_swiglu_launch(hipStream_t st, const uint16_t* Wilv, int ffn, int K, const uint16_t* x, long long ldx, int n, uint16_t* act) {
    const int M = 2 * ffn;
    if (ffn % 16 != 0 || M % G3_BM != 0 || K % G3_BK != 0 || K < G3_BK || n < G3_BN || (ldx & 7) || (ffn & 3) || (reinterpret_cast<uintptr_t>(x) & 15) || (reinterpret_cast<uintptr_t>(Wilv) & 15) ||
        (reinterpret_cast<uintptr_t>(act) & 15))
        return 1;
    GemmArgs a;
    memset(&a, 0, sizeof(a));
    a.njobs = 1, a.swiglu = 1;
    a.w = reinterpret_cast<const unsigned char*>(Wilv), a.M = M, a.K = K, a.x = x, a.ldx = ldx, a.n = n, a.y = act, a.ldy = ffn, a.alpha = 1.0f, a.beta = 0.0f;
    const long nwg = (long)(M / G3_BM) * ((n + G3_BN - 1) / G3_BN);
    if (nwg < 64 && (long)(M / 128) * ((n + 127) / 128) < 64) return 1;
    return g3_picked(st, a, true);
}

}  // namespace kf
