// kf_attn_bwd_mfma.hip -- causal multi-head attention backward on MFMA (flash form), gfx950 / wave64.  Same contract as kf_attn_bwd.hip (its
// header has the mathematics and the reference), same two-launch split, the tile algebra of the forward kernel (kf_flash.h):
//
//   dQ launch, workgroup = 128 query columns (32 per wave), key tiles of 32, two walks:
//              S^T[key][col] = K . Q^T, dP^T[key][col] = V . dO^T     A = K / V rows (ds_read_b128), B = Q / dO rows (registers, loaded once)
//              first walk: the column's log-sum-exp L (running maximum and sum, a column lives in one lane pair); L and D = dO . O go to launch 2, side by side
//              P = exp(scale S^T - L), dS^T = P o (dP^T - D)          element-wise on the accumulators
//              dQ^T[d][col] += K^T[d][key] . dS^T[key][col]           the dS^T registers, packed to bf16, ARE the B operand (free contraction order)
//   dK/dV launch, workgroup = 128 key columns, query tiles of 32 from the diagonal down (Q, dO, and L | D of the tile's queries):
//              S[q][key] = Q . K^T, dP[q][key] = dO . V^T   A = Q / dO rows, B = K / V rows of the column (registers)
//              P = exp(scale S - L_q), dS = P o (dP - D_q)  L, D per accumulator ROW: two ds_read_b128 per four rows
//              dV^T[d][key] += dO^T[d][q] . P[q][key],  dK^T[d][key] += Q^T[d][q] . dS[q][key]
// P and dS enter their products as single bf16 values (gradients are compared at 2^-7 of scale); everything else fp32.
//
// What bounds it: per 32 x 32 tile the two launches' MFMAs take 384 + 512 cycles of a SIMD at dim 64 and their vector instructions about as many.  A tile goes global -> LDS by buffer loads, AB_NB buffers, ONE barrier per
// tile (the first walk: per two); it lies there once, under a swizzle that suits the row reads and the transposing reads of the same rows (ab_swz); two or three waves to a SIMD do the rest.  25 heads x 64, 8 x 1024
// tokens: 410 us with tiles staged through registers, twice each, two barriers a tile; 193 so, the same bits.  With one walk, dQ divided by the sum of p at its end, 165, but other roundings of every dS.
#include "kf_kernels.h"

namespace kf {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr long long AB_NEAR = 1ll << 24; /* elements between rows of which 32 are in reach of a load's 32-bit offset */
constexpr int AB_T = 32, AB_NB = 4; /* rows of a tile; buffers: two to three tiles are on their way */
constexpr float AB_LOG2E = 1.44269502162933349609375f;

__device__ __forceinline__ f32x16 ab_zero() {
    f32x16 z;
#pragma unroll
    for (int i = 0; i < 16; i++) z[i] = 0.f;
    return z;
}
__device__ __forceinline__ f32x16 ab_mfma(u32x4 A, u32x4 B, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, A), __builtin_bit_cast(bf16x8, B), c, 0, 0, 0);
}
// the place of 16-byte chunk c of row r: 16 rows of a chunk (row reads) and four rows, from a multiple of four, of four chunks (transposing reads) touch all 64 banks once
template <int HD>
__device__ __forceinline__ int ab_swz(int r, int c) {
    return HD == 128 ? c ^ (((r & 3) << 2) | ((r >> 2) & 3)) : c ^ ((((r >> 1) & 1) << 2) | (((r >> 2) & 1) << 1) | ((r >> 3) & 1));
}
template <int HD, bool FAR>
struct AbTile {
    static constexpr int RB = 2 * HD, PART = AB_T * RB, RPI = 1024 / RB, NI = PART / 4096; /* bytes of a row, of a tile; rows per load instruction; instructions per wave (four to a workgroup) */
    int rf[HD / 16], tl[HD / 32], th[HD / 32]; /* this lane's offsets: row fragments per MFMA step, transposing reads per 32 columns (tile rows 4 h + (l16 >> 2), and 8 further) */
    int off_row[NI], off_chunk[NI];
    __device__ __forceinline__ void init(int lane, int wave) {
        const int r = lane & 31, h = lane >> 5;
#pragma unroll
        for (int s = 0; s < HD / 16; s++) rf[s] = r * RB + ab_swz<HD>(r, 2 * s + h) * 16;
#pragma unroll
        for (int db = 0; db < HD / 32; db++) { /* lane l16 of a 16-lane group addresses row (l16 >> 2) of its 4, piece 4 (l16 & 3) of the group's 16 columns; it receives the 4 rows' values of column l16 */
            const int row = 4 * h + ((lane & 15) >> 2), c = 4 * db + ((lane & 16) >> 3) + ((lane & 3) >> 1);
            tl[db] = row * RB + ab_swz<HD>(row, c) * 16 + 8 * (lane & 1);
            th[db] = (row + 8) * RB + ab_swz<HD>(row + 8, c) * 16 + 8 * (lane & 1);
        }
#pragma unroll
        for (int i = 0; i < NI; i++) off_row[i] = (wave * NI + i) * RPI + lane / (HD / 8), off_chunk[i] = ab_swz<HD>(off_row[i], lane % (HD / 8)) * 16;
    }
    __device__ __forceinline__ u32x4 rows(const unsigned char* tile, int s) const { return *reinterpret_cast<const u32x4*>(tile + rf[s]); }
    // contraction slots j <-> tile rows 16 s2 + (j & 3) + 8 (j >> 2) + 4 h
    __device__ __forceinline__ u32x4 turned(const unsigned char* tile, int db, int s2) const {
        const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) bf16x4*)(tile + tl[db] + 16 * s2 * RB));
        const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) bf16x4*)(tile + th[db] + 16 * s2 * RB));
        return __builtin_bit_cast(u32x4, bf16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]});
    }
    // 32 rows from `base`, rows `row_bytes` apart, into LDS: this wave's share.  `left` of them exist (<= 0: the sequence ended that far in front of base).  The others become zeros, and so does everything unless
    // `wanted`; FAR (a lane's offset does not fit 32 bits): rows of the sequence instead: nobody may look at what they hold
    __device__ __forceinline__ void load(const uint16_t* base, long long row_bytes, int left, bool wanted, unsigned char* to, int wave) const {
#ifdef __HIP_DEVICE_COMPILE__
        if constexpr (!FAR) {
            const uint32_t rb = (uint32_t)row_bytes, n = left <= 0 || !wanted ? 0 : (uint32_t)(left < AB_T ? left : AB_T) * rb;
            const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(base), 0, (int)n, 0x00020000);
#pragma unroll
            for (int i = 0; i < NI; i++) __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)(to + (wave * NI + i) * 1024), 16, (uint32_t)off_row[i] * rb + off_chunk[i], 0, 0, 0);
        } else {
#pragma unroll
            for (int i = 0; i < NI; i++) {
                const int row = off_row[i] < left ? off_row[i] : left - 1;
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(reinterpret_cast<const unsigned char*>(base) + row * row_bytes + off_chunk[i]),
                                                 (__attribute__((address_space(3))) void*)(to + (wave * NI + i) * 1024), 16, 0, 0);
            }
        }
#endif
    }
};
template <int N>
__device__ __forceinline__ void ab_landed() { /* all but the wave's N latest loads have landed, for every wave, and every wave has read what it wanted */
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}
// f over a tile and the place that the loads set out for meanwhile, told apart (restrict): the compiler otherwise puts a wait for those loads in front of every transposing read
template <class F>
__device__ __forceinline__ void ab_apart(const unsigned char* __restrict__ tile, unsigned char* __restrict__ to, F&& f) {
    f(tile, to);
}

template <int HD, bool FAR>
__global__ void __launch_bounds__(256, HD == 64 ? 3 : 2) attn_bwd_dq_mfma_kernel(const uint16_t* q, const uint16_t* k, const uint16_t* v, long long ld_qkv, const uint16_t* o, const uint16_t* dO, long long ld_o,
                                                                                 uint16_t* dq, long long ld_d, float* LD, int T, float scale, int gq, long long ld_kv) {
    using Tile = AbTile<HD, FAR>;
    constexpr int NS = HD / 16, NDB = HD / 32, SET = 2 * Tile::PART, LPS = 2 * Tile::NI; /* K and V of a tile; loads per wave and tile */
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 31, h = lane >> 5;
    /* consecutive workgroups go to consecutive XCDs: a head's blocks stay on the same one(s); the longest columns first */
    const int wg = (int)blockIdx.x + (int)gridDim.x * (int)blockIdx.y, head = wg % (int)gridDim.y, tok0 = ((int)gridDim.x - 1 - wg / (int)gridDim.y) * 128;
    const size_t hoff = (size_t)head * HD, hoff_kv = (size_t)(head / gq) * HD; /* GQA: gq query heads share a kv head */
    { /* sequence blockIdx.z: T rows further on in every tensor */
        const size_t ro = (size_t)blockIdx.z * T;
        q += ro * ld_qkv, k += ro * ld_kv + hoff_kv, v += ro * ld_kv + hoff_kv, o += ro * ld_o, dO += ro * ld_o, dq += ro * ld_d;
        LD += (size_t)blockIdx.z * gridDim.y * T * 2;
    }
    const int tok_last = tok0 + 127 < T ? tok0 + 127 : T - 1, ntile = tok_last / AB_T + 1, first = tok0 + wave * 32; /* first: this wave's first column */
    Tile W;
    W.init(lane, wave);
    const int n1 = (ntile + 1) / 2;
    auto load = [&](int i, unsigned char* to) { /* step i: two K tiles of the first walk, then K and V of each of the second (keys past the sequence's end lie behind every column: masked) */
        const bool one = i < n1;
        const int ta = one ? 2 * i : i - n1, tb = one ? ta + 1 : ta;
        const uint16_t* const second = one ? k : v;
        W.load(k + (size_t)ta * AB_T * ld_kv, 2 * ld_kv, T - ta * AB_T, ta < ntile, to, wave);
        W.load(second + (size_t)tb * AB_T * ld_kv, 2 * ld_kv, T - tb * AB_T, tb < ntile, to + Tile::PART, wave);
    };
    int tok = first + r;
    const bool col_ok = tok < T;
    if (!col_ok) tok = T - 1;
    u32x4 qf[NS], dof[NS];
    float Dp = 0.f;
    {
        const uint16_t* qrow = q + (size_t)tok * ld_qkv + hoff;
        const uint16_t* drow = dO + (size_t)tok * ld_o + hoff;
        const uint16_t* orow = o + (size_t)tok * ld_o + hoff;
#pragma unroll
        for (int s = 0; s < NS; s++) {
            qf[s] = *reinterpret_cast<const u32x4*>(qrow + 16 * s + 8 * h);
            dof[s] = *reinterpret_cast<const u32x4*>(drow + 16 * s + 8 * h);
            const u32x4 of = *reinterpret_cast<const u32x4*>(orow + 16 * s + 8 * h);
            const uint32_t a[4] = {dof[s].x, dof[s].y, dof[s].z, dof[s].w}, b[4] = {of.x, of.y, of.z, of.w};
#pragma unroll
            for (int e = 0; e < 4; e++) Dp = fmaf(bf_lo(a[e]), bf_lo(b[e]), Dp), Dp = fmaf(bf_hi(a[e]), bf_hi(b[e]), Dp);
        }
    }
    const float D = Dp + __shfl_xor(Dp, 32, 64);
#pragma unroll
    for (int b = 0; b < AB_NB - 1; b++) load(b, smem_raw + b * SET);

    const float c1 = scale * AB_LOG2E;
    int b = 0;
    auto step = [&](int i, auto&& f) { /* step i is here; step i + NB - 1 goes where step i - 1 was */
        ab_landed<(AB_NB - 2) * LPS>();
        ab_apart(smem_raw + b * SET, smem_raw + (b ? b - 1 : AB_NB - 1) * SET, [&](const unsigned char* tile, unsigned char* to) __attribute__((always_inline)) {
            load(i + AB_NB - 1, to);
            f(tile);
        });
        b = b + 1 < AB_NB ? b + 1 : 0;
    };
    // the log-sum-exp of every column, in log2 units: running maximum and sum of 2^(s - M)
    float M = -__builtin_inff(), l = 0.f;
    for (int i = 0; i < n1; i++)
        step(i, [&](const unsigned char* tile) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const int t = 2 * i + u;
                if (t * AB_T > first + 31) return; /* every key of the tile follows this wave's columns */
                f32x16 st = ab_zero();
#pragma unroll
                for (int s = 0; s < NS; s++) st = ab_mfma(W.rows(tile + u * Tile::PART, s), qf[s], st);
#pragma unroll
                for (int e = 0; e < 16; e++) st[e] *= c1;
                if (t * AB_T + AB_T - 1 > first) { /* else every key of the tile precedes every column of this wave */
#pragma unroll
                    for (int e = 0; e < 16; e++) st[e] = t * AB_T + 4 * h + (e & 3) + 8 * (e >> 2) <= tok ? st[e] : -__builtin_inff();
                }
                float mt = st[0];
#pragma unroll
                for (int e = 1; e < 16; e++) mt = fmaxf(mt, st[e]);
                mt = xmax32(mt);
                if (mt > M) l *= __builtin_amdgcn_exp2f(M - mt), M = mt; /* M = -inf on the first tile: 0 */
#pragma unroll
                for (int e = 0; e < 16; e++) l += __builtin_amdgcn_exp2f(st[e] - M);
            }
        });
    const float L2 = (M + __log2f(xsum32(l))) * 0.693147182464599609375f * AB_LOG2E; /* (by way of natural units) */

    f32x16 acc[NDB];
#pragma unroll
    for (int db = 0; db < NDB; db++) acc[db] = ab_zero();
    for (int t = 0; t < ntile; t++)
        step(n1 + t, [&](const unsigned char* tile) __attribute__((always_inline)) {
            if (t * AB_T > first + 31) return;
            f32x16 st = ab_zero(), dpt = ab_zero();
#pragma unroll
            for (int s = 0; s < NS; s++) {
                st = ab_mfma(W.rows(tile, s), qf[s], st);
                dpt = ab_mfma(W.rows(tile + Tile::PART, s), dof[s], dpt);
            }
            if (t * AB_T + AB_T - 1 > first) {
#pragma unroll
                for (int i = 0; i < 16; i++) st[i] = t * AB_T + 4 * h + (i & 3) + 8 * (i >> 2) <= tok ? st[i] : -__builtin_inff();
            }
            uint32_t dw[8];
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const float p0 = __builtin_amdgcn_exp2f(fmaf(st[2 * i], c1, -L2)), p1 = __builtin_amdgcn_exp2f(fmaf(st[2 * i + 1], c1, -L2));
                dw[i] = pack_bf16x2(p0 * (dpt[2 * i] - D), p1 * (dpt[2 * i + 1] - D));
            }
#pragma unroll
            for (int s2 = 0; s2 < 2; s2++) {
                const u32x4 B = u32x4{dw[4 * s2], dw[4 * s2 + 1], dw[4 * s2 + 2], dw[4 * s2 + 3]};
#pragma unroll
                for (int db = 0; db < NDB; db++) acc[db] = ab_mfma(W.turned(tile, db, s2), B, acc[db]);
            }
        });
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); /* loads past the last tile write zeros: none may be on its way when the workgroup's LDS goes to another */
    if (!col_ok) return;
    if (h == 0) LD[((size_t)head * T + tok) * 2] = L2, LD[((size_t)head * T + tok) * 2 + 1] = D; /* log-sum-exp of the scaled scores, log2 units */
    uint16_t* out = dq + (size_t)tok * ld_d + hoff;
#pragma unroll
    for (int db = 0; db < NDB; db++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const int d = 32 * db + 8 * g + 4 * h;
            *reinterpret_cast<u32x2*>(out + d) = u32x2{pack_bf16x2(acc[db][4 * g] * scale, acc[db][4 * g + 1] * scale), pack_bf16x2(acc[db][4 * g + 2] * scale, acc[db][4 * g + 3] * scale)};
        }
}

template <int HD, bool FAR>
__global__ void __launch_bounds__(256, HD == 64 ? 3 : 2) attn_bwd_dkv_mfma_kernel(const uint16_t* q, const uint16_t* k, const uint16_t* v, long long ld_qkv, const uint16_t* dO, long long ld_o, uint16_t* dk,
                                                                                  uint16_t* dv, long long ld_d, const float* LD, int T, float scale, int gq, long long ld_kv, long long ld_dkv) {
    using Tile = AbTile<HD, FAR>;
    constexpr int NS = HD / 16, NDB = HD / 32, SET = 2 * Tile::PART + 1024, LPS = 2 * Tile::NI + 1; /* Q and dO of a tile, and each wave's own copy of its L | D; loads per wave and tile */
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 31, h = lane >> 5;
    const int wg = (int)blockIdx.x + (int)gridDim.x * (int)blockIdx.y, kvh = wg % (int)gridDim.y, key0 = wg / (int)gridDim.y * 128; /* the first key columns see the most query tiles: first */
    const size_t hoff = (size_t)kvh * HD;
    {
        const size_t ro = (size_t)blockIdx.z * T;
        q += ro * ld_qkv, k += ro * ld_kv, v += ro * ld_kv, dO += ro * ld_o, dk += ro * ld_dkv, dv += ro * ld_dkv;
        LD += (size_t)blockIdx.z * gridDim.y * gq * T * 2;
    }
    const int ntq = (T + AB_T - 1) / AB_T, tg0 = (key0 / AB_T) * gq, tg1 = ntq * gq; /* (query tile, query head of the group) pairs */
    Tile W;
    W.init(lane, wave);
    int lt = tg0 / gq, lh = 0; /* the pair loaded next */
    auto load = [&](unsigned char* to) {
        const int left = T - lt * AB_T, head = kvh * gq + lh;
        W.load(q + (size_t)lt * AB_T * ld_qkv + (size_t)head * HD, 2 * ld_qkv, left, true, to, wave);
        W.load(dO + (size_t)lt * AB_T * ld_o + (size_t)head * HD, 2 * ld_o, left, true, to + Tile::PART, wave);
#ifdef __HIP_DEVICE_COMPILE__
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(LD + ((size_t)head * T + lt * AB_T) * 2), 0, left < 0 ? 0 : left * 8, 0x00020000);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)(to + 2 * Tile::PART + wave * 256), 4, lane * 4, 0, 0, 0);
#endif
        if (++lh == gq) lh = 0, lt++;
    };
    const int wave_key0 = key0 + wave * 32;
    int key = wave_key0 + r;
    const bool key_ok = key < T;
    if (!key_ok) key = T - 1;
    u32x4 kf_[NS], vf[NS];
    {
        const uint16_t* krow = k + (size_t)key * ld_kv + hoff;
        const uint16_t* vrow = v + (size_t)key * ld_kv + hoff;
#pragma unroll
        for (int s = 0; s < NS; s++) kf_[s] = *reinterpret_cast<const u32x4*>(krow + 16 * s + 8 * h), vf[s] = *reinterpret_cast<const u32x4*>(vrow + 16 * s + 8 * h);
    }
#pragma unroll
    for (int b = 0; b < AB_NB - 1; b++) load(smem_raw + b * SET);
    f32x16 dka[NDB], dva[NDB];
#pragma unroll
    for (int db = 0; db < NDB; db++) dka[db] = ab_zero(), dva[db] = ab_zero();
    const float c1 = scale * AB_LOG2E;
    int b = 0, t = tg0 / gq, th = 0;
    for (int tg = tg0; tg < tg1; tg++) {
        ab_landed<(AB_NB - 2) * LPS>();
        ab_apart(smem_raw + b * SET, smem_raw + (b ? b - 1 : AB_NB - 1) * SET, [&](const unsigned char* tile, unsigned char* to) __attribute__((always_inline)) {
            load(to);
            if (t * AB_T + AB_T - 1 < wave_key0) return; /* every query of the tile precedes this wave's keys */
            f32x16 st = ab_zero(), dpt = ab_zero();
#pragma unroll
            for (int s = 0; s < NS; s++) {
                st = ab_mfma(W.rows(tile, s), kf_[s], st);
                dpt = ab_mfma(W.rows(tile + Tile::PART, s), vf[s], dpt);
            }
            if (t * AB_T < wave_key0 + 31 || t * AB_T + AB_T > T) { /* else every query of the tile exists and follows every key of this wave */
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const int query = t * AB_T + 4 * h + (i & 3) + 8 * (i >> 2);
                    st[i] = query >= key && query < T ? st[i] : -__builtin_inff();
                }
            }
            uint32_t pw[8], dw[8];
            const f32x4* const ld = reinterpret_cast<const f32x4*>(tile + 2 * Tile::PART + wave * 256);
#pragma unroll
            for (int g = 0; g < 4; g++) /* accumulator rows 8 g + 4 h + {0..3} */
#pragma unroll
                for (int e = 0; e < 2; e++) {
                    const f32x4 w = ld[4 * g + 2 * h + e]; /* L, D of two queries */
                    const int i = 4 * g + 2 * e;
                    const float p0 = __builtin_amdgcn_exp2f(fmaf(st[i], c1, -w[0])), p1 = __builtin_amdgcn_exp2f(fmaf(st[i + 1], c1, -w[2]));
                    pw[2 * g + e] = pack_bf16x2(p0, p1);
                    dw[2 * g + e] = pack_bf16x2(p0 * (dpt[i] - w[1]), p1 * (dpt[i + 1] - w[3]));
                }
#pragma unroll
            for (int s2 = 0; s2 < 2; s2++) {
                const u32x4 BP = u32x4{pw[4 * s2], pw[4 * s2 + 1], pw[4 * s2 + 2], pw[4 * s2 + 3]}, BS = u32x4{dw[4 * s2], dw[4 * s2 + 1], dw[4 * s2 + 2], dw[4 * s2 + 3]};
#pragma unroll
                for (int db = 0; db < NDB; db++) {
                    dva[db] = ab_mfma(W.turned(tile + Tile::PART, db, s2), BP, dva[db]);
                    dka[db] = ab_mfma(W.turned(tile, db, s2), BS, dka[db]);
                }
            }
        });
        b = b + 1 < AB_NB ? b + 1 : 0;
        if (++th == gq) th = 0, t++;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (!key_ok) return;
    uint16_t* okp = dk + (size_t)key * ld_dkv + hoff;
    uint16_t* ovp = dv + (size_t)key * ld_dkv + hoff;
#pragma unroll
    for (int db = 0; db < NDB; db++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const int d = 32 * db + 8 * g + 4 * h;
            *reinterpret_cast<u32x2*>(okp + d) = u32x2{pack_bf16x2(dka[db][4 * g] * scale, dka[db][4 * g + 1] * scale), pack_bf16x2(dka[db][4 * g + 2] * scale, dka[db][4 * g + 3] * scale)};
            *reinterpret_cast<u32x2*>(ovp + d) = u32x2{pack_bf16x2(dva[db][4 * g], dva[db][4 * g + 1]), pack_bf16x2(dva[db][4 * g + 2], dva[db][4 * g + 3])};
        }
}

template <int HD, bool FAR>
static int ab_go(hipStream_t st, const uint16_t* q, const uint16_t* k, const uint16_t* v, long long ld_qkv, const uint16_t* o, const uint16_t* dO, long long ld_o, uint16_t* dq, uint16_t* dk, uint16_t* dv,
                 long long ld_d, int T, int n_head, int n_seq, float* LD, int n_kv, long long ld_kv, long long ld_dkv) {
    constexpr int smem_q = AB_NB * 2 * AbTile<HD, FAR>::PART, smem_kv = AB_NB * (2 * AbTile<HD, FAR>::PART + 1024);
    static int attr_set = 0;
    if (!attr_set && smem_kv > 64 * 1024) {
        if (hipFuncSetAttribute((const void*)attn_bwd_dq_mfma_kernel<HD, FAR>, hipFuncAttributeMaxDynamicSharedMemorySize, smem_q) != hipSuccess) return KF_HIP_CHECK;
        if (hipFuncSetAttribute((const void*)attn_bwd_dkv_mfma_kernel<HD, FAR>, hipFuncAttributeMaxDynamicSharedMemorySize, smem_kv) != hipSuccess) return KF_HIP_CHECK;
        attr_set = 1;
    }
    const float scale = 1.0f / sqrtf((float)HD);
    const dim3 grid((T + 127) / 128, n_head, n_seq), grid_kv((T + 127) / 128, n_kv, n_seq);
    hipLaunchKernelGGL((attn_bwd_dq_mfma_kernel<HD, FAR>), grid, dim3(256), smem_q, st, q, k, v, ld_qkv, o, dO, ld_o, dq, ld_d, LD, T, scale, n_head / n_kv, ld_kv);
    hipLaunchKernelGGL((attn_bwd_dkv_mfma_kernel<HD, FAR>), grid_kv, dim3(256), smem_kv, st, q, k, v, ld_qkv, dO, ld_o, dk, dv, ld_d, LD, T, scale, n_head / n_kv, ld_kv, ld_dkv);
    return hipGetLastError() == hipSuccess ? KF_OK : KF_HIP_CHECK;
}
// KF_OK launched; 1 = shape not covered by the MFMA form
int attn_backward_mfma_launch(hipStream_t st, const uint16_t* q, const uint16_t* k, const uint16_t* v, long long ld_qkv, const uint16_t* o, const uint16_t* dO, long long ld_o,
                              uint16_t* dq, uint16_t* dk, uint16_t* dv, long long ld_d, int T, int n_head, int hd, int n_seq, float* scratch, int n_kv, long long ld_kv, long long ld_dkv) {
    if ((hd != 64 && hd != 128) || n_kv < 1 || n_head % n_kv != 0) return 1;
    float* const LD = scratch; /* [n_seq][n_head][T][2]: log-sum-exp and dO . O of a query */
    const bool far = ld_qkv >= AB_NEAR || ld_o >= AB_NEAR || ld_kv >= AB_NEAR;
    const auto go = hd == 64 ? (far ? &ab_go<64, true> : &ab_go<64, false>) : (far ? &ab_go<128, true> : &ab_go<128, false>);
    return go(st, q, k, v, ld_qkv, o, dO, ld_o, dq, dk, dv, ld_d, T, n_head, n_seq, LD, n_kv, ld_kv, ld_dkv);
}

}  // namespace kf
