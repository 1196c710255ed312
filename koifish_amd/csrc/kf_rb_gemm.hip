// kf_rb_gemm.hip -- row-batch products on MFMA tiles: the 64-deep tile of kf_gemm3_tile.h (both operands global -> LDS by global_load_lds, swizzled at the source) with the
// row-batch epilogues (fp32 residual with alpha, gated activation of interleaved rows, fp32 store) and, for experts, a gathered token operand: the rows of a token tile are
// the pairs of one expert, each lane's source pointer is set up once from the pair list, so routed rows are never copied together.
#include <string.h>

#include "kf_gemm3_tile.h"
#include "kf_rb_common.h"

namespace kf {

using RbTiny = G3Cfg<64, 64, 4>;      /* 32-bit storage: five to a CU */
using RbPairs = G3Cfg<128, 64, 4>;    /* experts of about a hundred pairs: half the padding of 128-pair tiles, each weight tile read about once; three to a CU (with three buffers, two: 64 experts of 3072 x 2048, 7884 pairs 259 -> 268 us) */

// eight values from a multiple of 8 columns; rows of 16-bit values are at least 8-byte aligned.  base: uniform, off: in elements.  In reach of 32 bits they are written through (g3_store16)
__device__ __forceinline__ void rb_st8(uint16_t* base, size_t off, const float (&v)[8], int64_t ld, bool reach) {
    const u32x4 o = g3_pack8(v);
    if ((ld & 7) == 0 && reach) g3_store16(base, (uint32_t)off * 2, o);
    else if ((ld & 7) == 0) *reinterpret_cast<u32x4*>(base + off) = o;
    else reinterpret_cast<u32x2*>(base + off)[0] = u32x2{o.x, o.y}, reinterpret_cast<u32x2*>(base + off)[1] = u32x2{o.z, o.w};
}
__device__ __forceinline__ void rb_st8(float* base, size_t off, const float (&v)[8], int64_t, bool) {
    reinterpret_cast<f32x4*>(base + off)[0] = f32x4{v[0], v[1], v[2], v[3]}, reinterpret_cast<f32x4*>(base + off)[1] = f32x4{v[4], v[5], v[6], v[7]};
}

// The list's tiles up to the last that holds pairs: those at its end are empty (-1).  Only these are dealt to the XCDs, in equal runs of neighbours; dealt with the others an XCD that the list's end falls to, once per band of row tiles,
// has little to do.  us, 128 experts of 15768 pairs, about 300 of 374 tiles filled, dealt all | filled: gated 1536 x 2048 252 | 220 (1.08 GB from memory, 0.8 of it weights: 4.9 TB/s), 2048 x 768 145 | 131; bands of all 12 or 16 row tiles
// instead of g3_tile's, the token rows read once by an XCD, 229 and 131; bands of 4 the same as of 6 and 8.
__device__ __forceinline__ int rb_filled(const int32_t* tile_expert, int n, int lane) {
    int c = 0;
    for (int i0 = 0; i0 < n; i0 += 512) {
        int v[8];
#pragma unroll
        for (int j = 0; j < 8; j++) v[j] = tile_expert[i0 + 64 * j + lane < n ? i0 + 64 * j + lane : 0];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const unsigned long long b = __ballot(i0 + 64 * j + lane < n && v[j] >= 0);
            if (b) c = i0 + 64 * j + 64 - __builtin_clzll(b);
        }
    }
    return c;
}

// T: the storage, uint16_t (bf16: weights in MFMA tiles) or float (true 32-bit: weights in rows)
template <class C, bool EXPERTS, class T>
__global__ void __launch_bounds__(C::NTH, C::WGS_PER_CU * C::NW / 4) rb_gemm_kernel(const RbProduct q) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    __shared__ int32_t s_src[EXPERTS ? C::BN : 1], s_dst[EXPERTS ? C::BN : 1];
    const kf_rb_product& p = q.p;
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int nbx = (p.m + C::BM - 1) / C::BM;
    int bx, by, ex = 0;
    if constexpr (EXPERTS) {
        const int n_act = rb_filled(q.e.tile_expert, (int)gridDim.x / nbx, lane);
        if ((int)blockIdx.x / 8 >= (nbx * n_act + 7 - (int)blockIdx.x % 8) / 8) return; /* workgroup-uniform */
        g3_tile(g3_remap(blockIdx.x, nbx * n_act), nbx, n_act, bx, by);
        ex = q.e.tile_expert[by];
        if (ex < 0) return; /* workgroup-uniform */
    } else
        g3_tile(g3_remap(blockIdx.x, gridDim.x), nbx, (int)gridDim.x / nbx, bx, by);
    const int m0 = bx * C::BM, t0 = by * C::BN;
    GemmArgs a; /* what the main loop reads */
    constexpr int U = sizeof(T) / 2, KT = G3_BK / U; /* 16-bit units of an element, elements of a step */
    a.w = reinterpret_cast<const unsigned char*>(p.w), a.M = p.m, a.K = p.k * U, a.x = reinterpret_cast<const uint16_t*>(p.x), a.ldx = p.ldx * U, a.n = p.n, a.ldr = 0;
    f32x4 acc[C::MT][C::NT];
#pragma unroll
    for (int i = 0; i < C::MT; i++)
#pragma unroll
        for (int j = 0; j < C::NT; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    if constexpr (EXPERTS) {
        a.w += (size_t)ex * q.e.w_stride * sizeof(T);
        for (int i = tid; i < C::BN; i += C::NTH) {
            const int pair = q.e.list[(size_t)by * C::BN + i];
            s_dst[i] = pair, s_src[i] = pair < 0 ? 0 : (p.mode == KF_RB_UP ? pair / q.e.top : pair);
        }
        __syncthreads();
        using Rows = std::conditional_t<U == 2, G3GatherF32, G3GatherTiled>;
        g3_mainloop<false, false, G3_BK, C, Rows>(a, m0, 0, 0, p.k / KT, acc, smem_raw, wid, lane, Rows{s_src});
    } else {
        g3_mainloop<false, false, G3_BK, C, std::conditional_t<U == 2, G3RowsF32, G3Tiled>>(a, m0, t0, 0, p.k / KT, acc, smem_raw, wid, lane);
    }
    // the tile by way of LDS (G3Out); rows of y: the token itself, or the pair in the token tile's place
    using Out = G3Out<C>;
    T* const y = reinterpret_cast<T*>(p.y);
    const bool reach = !EXPERTS && (size_t)p.n * p.ldy < ((size_t)1 << 29); /* (experts' tiles leave at different times: 5.54 | 5.58 ms for 4 x 509 tokens) */
    auto row_of = [&](int tk) { return EXPERTS ? s_dst[EXPERTS ? tk : 0] : (t0 + tk < p.n ? t0 + tk : -1); };
    if (p.epilogue == KF_RB_GATED) {
        auto gated = [&](auto act) { /* a loop per activation: decided inside it costs a branch per value */
            Out::template all<C::BM / 16>(acc, smem_raw, tid, [&](int tk, int lt, int u) { /* rows of 16 gates and of the 16 ups behind them: eight outputs */
                const int row = row_of(tk), f = (m0 >> 1) + 8 * u, c = (u >> 1) * 4 + (u & 1);
                if (row < 0 || 2 * f >= p.m) return;
                const float scale = EXPERTS && p.mode == KF_RB_UP ? q.e.weight[row] : 1.f;
                float g[8], v[8];
                Out::rows8(smem_raw, lt, c, tid, g), Out::rows8(smem_raw, lt, c + 2, tid, v);
#pragma unroll
                for (int j = 0; j < 8; j++) g[j] = scale * (rb_activate(act, g[j]) * v[j]);
                rb_st8(y, (size_t)row * p.ldy + f, g, p.ldy, reach);
            });
        };
        if (p.act == KF_RB_SILU) gated(std::integral_constant<int, KF_RB_SILU>());
        else gated(p.act);
    } else if (p.epilogue == KF_RB_STORE && U == 1) {
        Out::template all<C::BM / 8>(acc, smem_raw, tid, [&](int tk, int lt, int u) {
            const int row = row_of(tk), m = m0 + 8 * u;
            if (row < 0 || m >= p.m) return;
            float v[8];
            Out::rows8(smem_raw, lt, u, tid, v);
            if (m + 7 >= p.act_lo && m < p.act_hi) {
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    const float w = rb_activate(p.act, v[j]);
                    v[j] = m + j >= p.act_lo && m + j < p.act_hi ? w : v[j];
                }
            }
            rb_st8(y, (size_t)row * p.ldy + m, v, p.ldy, reach);
        });
    } else {
        Out::template all<C::BM / 4>(acc, smem_raw, tid, [&](int tk, int lt, int u) {
            const int row = row_of(tk), m = m0 + 4 * u;
            if (row < 0 || m >= p.m) return;
            f32x4 d = *reinterpret_cast<const f32x4*>(smem_raw + Out::at(lt, u));
            if (U == 2 && p.epilogue == KF_RB_STORE && m + 3 >= p.act_lo && m < p.act_hi) {
#pragma unroll
                for (int j = 0; j < 4; j++)
                    if (m + j >= p.act_lo && m + j < p.act_hi) d[j] = rb_activate(p.act, d[j]);
            }
            if (p.epilogue == KF_RB_RESIDUAL) {
                const f32x4 r = rb_ld4(p.res + (size_t)row * p.ldr + m);
#pragma unroll
                for (int j = 0; j < 4; j++) d[j] = fmaf(p.alpha, r[j], d[j]);
            }
            const size_t off = (size_t)row * p.ldy + m;
            if (reach) g3_store16(p.y, (uint32_t)off * 4, __builtin_bit_cast(u32x4, d));
            else rb_st4(reinterpret_cast<float*>(p.y) + off, d);
        });
    }
}
template <class C, bool EXPERTS, class T = uint16_t>
static int rb_go(hipStream_t st, const RbProduct& q, long nwg) {
    constexpr int SMEM = C::SMEM;
    static int attr_set = 0;
    if (!attr_set && SMEM + 2 * 4 * C::BN > 64 * 1024) { /* the pair rows of the experts form sit in static LDS */
        if (hipFuncSetAttribute((const void*)rb_gemm_kernel<C, EXPERTS, T>, hipFuncAttributeMaxDynamicSharedMemorySize, SMEM) != hipSuccess) return KF_HIP_CHECK;
        attr_set = 1;
    }
    hipLaunchKernelGGL((rb_gemm_kernel<C, EXPERTS, T>), dim3((unsigned)nwg), dim3(C::NTH), SMEM, st, q);
    return KF_OK;
}
static long rb_tiles(const kf_rb_product& p, int bm, int bn) { return (long)((p.m + bm - 1) / bm) * ((p.n + bn - 1) / bn); }
int rb_gemm_launch(hipStream_t st, const RbProduct& q) {
    const kf_rb_product& p = q.p;
    if (p.mode != KF_RB_ALL) {
        if (q.e.tile == 128) return rb_go<G3Small, true>(st, q, (long)((p.m + 127) / 128) * q.e.n_tile);
        if (q.e.tile == 64) return rb_go<RbPairs, true>(st, q, (long)((p.m + 127) / 128) * q.e.n_tile);
        return 1;
    }
    // the smallest tile that makes one round of the CUs, as for the products of kf_gemm3.hip (g3_pick has the figures): same main loop
    const long n64 = rb_tiles(p, 64, 64);
    if (n64 <= (p.k < 96 * G3_BK ? 512 : 256)) return rb_go<G3Few, false>(st, q, n64);
    switch (g3_pick(p.m, p.n, p.k, true)) {
        case G3_DUO: return rb_go<G3Duo, false>(st, q, rb_tiles(p, 128, 128));
        case G3_HALF: return rb_go<G3Half, false>(st, q, rb_tiles(p, 128, 256));
        case G3_SMALL: return rb_go<G3Small, false>(st, q, rb_tiles(p, 128, 128));
        case G3_WIDE: return rb_go<G3Wide, false>(st, q, rb_tiles(p, 192, 256));
        default: return rb_go<G3Big, false>(st, q, rb_tiles(p, 256, 256));
    }
}
// The 32-bit product on v_mfma_f32_16x16x4_f32 (157 TFLOP/s; the vector pipe without packed instructions: 78).  It is bound by the MFMAs, 16 x slower than bf16's, so the tile only has to share them
// out evenly: 64 x 64 tiles, five to a CU; a lone one of a CU waits for its loads, so with three buffers.  us at 512 rows, two buffers | three: 2048 x 6144 (256 tiles) 127.6 | 108.6, x 2048 46.3 | 40.9; 5120 x 2048
// (640) 95.6 | 100.5, 12288 x 2048 190 | 201.
int rb_f32_launch(hipStream_t st, const RbProduct& q) {
    const kf_rb_product& p = q.p;
    if (p.mode == KF_RB_SUM || (p.mode != KF_RB_ALL && q.e.tile != 64)) return 1;
    if (p.mode != KF_RB_ALL) return rb_go<RbTiny, true, float>(st, q, (long)(p.m / 64) * q.e.n_tile);
    const long nwg = rb_tiles(p, 64, 64);
    return nwg <= 256 ? rb_go<G3Few, false, float>(st, q, nwg) : rb_go<RbTiny, false, float>(st, q, nwg);
}

}  // namespace kf
