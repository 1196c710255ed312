// kf_attn_prefill.hip -- causal GQA attention for a batch of prompt tokens on MFMA (flash form), gfx950 / wave64.
//
// Reference: none on the inference side (Fish::Chat prefills token by token through attention_qk_kernel / CU_softmax_multihead /
// attention_v_kernel, QKV.cu:669-673); its batched forward is cuDNN SDPA on the training side (QKV.cu:130-315), removed here.
// Same arithmetic contract as the decode kernel (kf_attn.hip): score = bf16(dot / sqrt(hd)) -- the store the reference makes --, fp32
// softmax statistics with exp as v_exp_f32(x * log2 e), out = (sum_t p_t v_t) / (sum_t p_t) with one bf16 store; the probabilities
// enter the P.V product as a bf16 pair (high part + remainder, ~16 significant bits; the reference keeps them in plain bf16,
// operator.cuh:251-277), the sum of p stays fp32.
//
// Workgroup = one kv-head x TQ = 128/GQ consecutive tokens: 128 "columns" (token, query head of the group), 32 per wave (kf_flash.h: a wave's walk over the keys, 32 at a time).
// A tile of K and V goes global -> LDS by buffer loads (no VGPR round trip), AP_NB buffers: up to three tiles of 16 KiB are on their way while one is multiplied, which is what a load from another
// XCD's memory side takes (about 2 us; one tile ahead, the step took what the load took).  The LDS image of such a load is lane-linear, so rows are unpadded and the swizzle is made at the
// source (ap_swz_k, ap_swz_v): 16 lanes of a K read and 32 of a transposing V read touch all 64 banks once.
#include <type_traits>

#include "kf_flash.h"
#include "kf_kernels.h"

namespace kf {

struct AttnPrefillArgs {
    const uint16_t* q;
    const uint16_t* kcache;
    const uint16_t* vcache;
    uint16_t* out;
    int pos0, n_tok, n_kv, kv_stride;
    int n_seq; /* sequences of n_tok rows each, back to back in q / out and in the K / V rows (blockIdx.z); 1 for prompt prefill */
    long long q_stride;
    long long out_stride; /* row stride of out (a training step reads q out of the fused [rows, 3C] buffer and writes a dense [rows, C] out) */
    float rden;
};

// rows of K or V from memory into LDS: N instructions per wave, from row `first` of those the workgroup loads at a time.  Rows past `left` bytes from `base` become zeros
template <int HD, int N, bool V>
struct ApLoad {
    uint32_t off[N];
    __device__ __forceinline__ void init(int first, long long row_bytes, int lane) {
#pragma unroll
        for (int i = 0; i < N; i++) {
            const int row = first + i * ApTile<HD>::RPI + lane / (HD / 8), p = lane % (HD / 8);
            off[i] = (uint32_t)row * (uint32_t)row_bytes + (V ? ap_swz_v<HD>(row, p) : ap_swz_k<HD>(row, p)) * 16;
        }
    }
    __device__ __forceinline__ void go(const unsigned char* base, long long left, unsigned char* to) const {
#ifdef __HIP_DEVICE_COMPILE__
        const int n = (int)(left < 0 ? 0 : (left > 0x7FFFFFFFll ? 0x7FFFFFFFll : left));
        const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned char*>(base), 0, n, 0x00020000);
#pragma unroll
        for (int i = 0; i < N; i++) __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)(to + i * 1024), 16, off[i], 0, 0, 0);
#endif
    }
};
// this lane's column of a workgroup whose first token is `first`
struct ApCol {
    int tok, head; /* clamped to the last token */
    bool ok;
};
template <int GQ>
__device__ __forceinline__ ApCol ap_col(const AttnPrefillArgs& a, int first, int col, int g) {
    ApCol c;
    c.tok = first + col / GQ, c.head = g * GQ + col % GQ, c.ok = c.tok < a.n_tok;
    if (!c.ok) c.tok = a.n_tok - 1;
    return c;
}
template <int HD>
__device__ __forceinline__ void ap_query(FlashWave<HD>& W, const AttnPrefillArgs& a, size_t seq_row, const ApCol& c, int h) { /* B operand of S^T: lane (col, h) holds Q[col][16 s + 8 h .. + 8] */
    const uint16_t* const q = a.q + (seq_row + c.tok) * a.q_stride + (size_t)c.head * HD;
#pragma unroll
    for (int s = 0; s < HD / 16; s++) W.qf[s] = *reinterpret_cast<const u32x4*>(q + 16 * s + 8 * h);
}
constexpr float AP_LOG2E = 1.44269502162933349609375f;

// One tile (its K at `k`, the tile before's V at `v`) while others are loaded to `to_k`, `to_v`.  The pointers are told apart (restrict): the compiler otherwise takes every transposing LDS read for one that may
// read what those loads write, and puts a wait for all of them in front of it -- a tile then takes what a load takes.  What has to have landed is waited for by ap_landed.
template <int HD, class LK, class LV>
__device__ __forceinline__ void ap_tile_step(FlashWave<HD>& W, const ApTile<HD>& T, const unsigned char* __restrict__ k, const unsigned char* __restrict__ v, fl_f32x16& cur, float& mt, fl_f32x16& nxt, float by,
                                             bool own, unsigned char* __restrict__ to_k, unsigned char* __restrict__ to_v, LK&& load_k, LV&& load_v) {
    load_k(to_k), load_v(to_v);
    if (own) mt = W.template tile<true, true>(cur, mt, nxt, by, [&](int s) { return T.k(k, s); }, [&](int s2, int db) { return T.v(v, s2, db); });
}

// Many workgroups: 128 columns each, 32 per wave, every wave walks all keys; the blocks with the most keys are dispatched first, two or three workgroups to a CU.
template <int HD, int GQ>
__global__ void __launch_bounds__(256, 2) attn_prefill_kernel(const AttnPrefillArgs a) {
    using Wave = FlashWave<HD>;
    using Tile = ApTile<HD>;
    constexpr int NDB = Wave::NDB, TQ = 128 / GQ, TILE = 2 * Tile::PART, NI = Tile::PART / 4096; /* tokens per workgroup; bytes of a K and a V tile; load instructions per wave and part */
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5;
    // consecutive workgroups go to consecutive XCDs: the workgroups of a kv-head stay on the same one(s), its K / V rows (1 MB at 2047 tokens) in their L2
    const int wg_id = (int)blockIdx.x + (int)gridDim.x * (int)blockIdx.y, g = wg_id % a.n_kv, bx = (int)gridDim.x - 1 - wg_id / a.n_kv;
    const size_t seq_row = (size_t)blockIdx.z * a.n_tok;
    const int first = bx * TQ, last = first + TQ - 1 < a.n_tok - 1 ? first + TQ - 1 : a.n_tok - 1, kmax = a.pos0 + last, ntile = kmax / 32 + 1; /* last key any column needs */
    const ApCol c = ap_col<GQ>(a, first, wave * 32 + (lane & 31), g);
    Wave W;
    W.init();
    ap_query<HD>(W, a, seq_row, c, h);
    const long long row_bytes = (long long)a.kv_stride * 2;
    const unsigned char* const kb = reinterpret_cast<const unsigned char*>(a.kcache + seq_row * a.kv_stride + (size_t)g * HD);
    const unsigned char* const vb = reinterpret_cast<const unsigned char*>(a.vcache + seq_row * a.kv_stride + (size_t)g * HD);
    ApLoad<HD, NI, false> lk;
    ApLoad<HD, NI, true> lv;
    lk.init(wave * NI * Tile::RPI, row_bytes, lane), lv.init(wave * NI * Tile::RPI, row_bytes, lane);
    auto left = [&](int t) { return ((long long)kmax + 1 - 32 * t) * row_bytes; };
    auto load_k = [&](int t, unsigned char* to) { lk.go(kb + 32 * t * row_bytes, left(t), to + wave * NI * 1024); };
    auto load_v = [&](int t, unsigned char* to) { lv.go(vb + 32 * t * row_bytes, left(t), to + wave * NI * 1024); };
    auto part = [&](int b, bool v) { return smem_raw + b * TILE + (v ? Tile::PART : 0); };
#pragma unroll
    for (int b = 0; b < AP_NB - 1; b++) load_k(b, part(b, false)), load_v(b, part(b, true));
    Tile T;
    T.init(lane);
    // score = bf16(dot / sqrt(hd)); a tile is masked unless every key of it precedes every column of this wave
    const int before = first + TQ <= a.n_tok ? a.pos0 + first + wave * 32 / GQ : -1, pos_q = a.pos0 + c.tok;
    auto maximum = [&](fl_f32x16& st, int t, float m) {
        if (32 * t + 31 > before) m = Wave::mask(st, 32 * t, 0, pos_q, h);
        return xmax32(m) * AP_LOG2E;
    };
    fl_f32x16 sa, sb;
    ap_landed<(AP_NB - 3) * 2 * NI>(); /* tiles 0 and 1 */
    W.scores(sa, [&](int s) { return T.k(part(0, false), s); });
    float mt = maximum(sa, 0, Wave::template scale<true>(sa, a.rden));
    int b = 0;
    auto step = [&](int t, fl_f32x16& cur, fl_f32x16& nxt) { /* K of tile t + 1 and V of tile t are here; tile t + NB - 1 goes where tile t - 1 was */
        const int b1 = b + 1 < AP_NB ? b + 1 : 0, bl = b ? b - 1 : AP_NB - 1;
        ap_tile_step<HD>(W, T, part(b1, false), part(b, true), cur, mt, nxt, a.rden, true, part(bl, false), part(bl, true), [&](unsigned char* to) { load_k(t + AP_NB - 1, to); },
                         [&](unsigned char* to) { load_v(t + AP_NB - 1, to); });
        mt = maximum(nxt, t + 1, mt);
        ap_landed<(AP_NB - 3) * 2 * NI>(); /* tile t + 2 */
        b = b1;
    };
    for (int t = 0; t < ntile; t += 2) {
        step(t, sa, sb);
        if (t + 1 < ntile) step(t + 1, sb, sa);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); /* loads past the last tile write zeros: none may be on its way when the workgroup's LDS goes to another */
    // out[col][d] = O^T[d][col] / l ; lane (col, h) holds d = 32 db + (i & 3) + 8 (i >> 2) + 4 h
    const float inv = 1.0f / xsum32(W.l);
    if (!c.ok) return;
    uint16_t* const orow = a.out + (seq_row + c.tok) * a.out_stride + (size_t)c.head * HD;
#pragma unroll
    for (int db = 0; db < NDB; db++)
#pragma unroll
        for (int q = 0; q < 4; q++)
            *reinterpret_cast<u32x2*>(orow + 32 * db + 8 * q + 4 * h) = u32x2{pack_bf16x2(W.o[db][4 * q] * inv, W.o[db][4 * q + 1] * inv), pack_bf16x2(W.o[db][4 * q + 2] * inv, W.o[db][4 * q + 3] * inv)};
}

// Eight waves = CG column groups of 32 x KP key parts (32 of every 32 KP keys each), whose sums meet in LDS at the end.  A wave alone on its SIMD starts an instruction every 5 - 8 cycles, two side by
// side fill each other's gaps, so both waves of a SIMD walk equally far; and a set of tiles serves CG column groups, which is what the loads can deliver.
template <int HD, int CG>
constexpr int ap_sets = HD == 128 && CG == 2 ? 2 : 4; /* sets of K and V in LDS: 128 KiB (64 KiB at dim 64, four column groups: two workgroups to a CU) */
template <int HD, int GQ, int CG>
__global__ void __launch_bounds__(512, 2) attn_prefill_parts_kernel(const AttnPrefillArgs a) {
    using Wave = FlashWave<HD>;
    using Tile = ApTile<HD>;
    constexpr int KP = 8 / CG, TQ = 32 * CG / GQ, SET = KP * Tile::PART, NI = SET / 8192, KEYS = 32 * KP; /* tokens per workgroup; bytes of a set's K rows; load instructions per wave and set; keys of a set */
    constexpr int NB = ap_sets<HD, CG>;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[]; /* NB x (K set, V set) */
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), cg = wave % CG, kp = wave / CG, h = lane >> 5;
    // consecutive workgroups go to consecutive XCDs: the workgroups of a kv-head stay on the same one(s), its K / V rows (1 MB at 2047 tokens) in their L2; the longest first
    const int wg_id = (int)blockIdx.x + (int)gridDim.x * (int)blockIdx.y, g = wg_id % a.n_kv, bx = (int)gridDim.x - 1 - wg_id / a.n_kv;
    const size_t seq_row = (size_t)blockIdx.z * a.n_tok;
    const int first = bx * TQ, last = first + TQ - 1 < a.n_tok - 1 ? first + TQ - 1 : a.n_tok - 1, kmax = a.pos0 + last, nset = kmax / KEYS + 1; /* last key any column needs */
    const ApCol c = ap_col<GQ>(a, first, cg * 32 + (lane & 31), g);
    const long long row_bytes = (long long)a.kv_stride * 2;
    const unsigned char* const kb = reinterpret_cast<const unsigned char*>(a.kcache + seq_row * a.kv_stride + (size_t)g * HD);
    const unsigned char* const vb = reinterpret_cast<const unsigned char*>(a.vcache + seq_row * a.kv_stride + (size_t)g * HD);
    ApLoad<HD, NI, false> lk;
    ApLoad<HD, NI, true> lv;
    lk.init(wave * NI * Tile::RPI, row_bytes, lane), lv.init(wave * NI * Tile::RPI, row_bytes, lane);
    auto left = [&](int j) { return ((long long)kmax + 1 - KEYS * j) * row_bytes; };
    auto load_k = [&](int j, unsigned char* to) { lk.go(kb + KEYS * j * row_bytes, left(j), to + wave * NI * 1024); };
    auto load_v = [&](int j, unsigned char* to) { lv.go(vb + KEYS * j * row_bytes, left(j), to + wave * NI * 1024); };
    auto set = [&](int b, bool v) { return smem_raw + (2 * b + (v ? 1 : 0)) * SET; };
    Wave W;
    W.init();
    ap_query<HD>(W, a, seq_row, c, h);
    load_k(0, set(0, false));
#pragma unroll
    for (int b = 1; b < NB; b++) load_k(b, set(b, false)), load_v(b - 1, set(b - 1, true));
    Tile T;
    T.init(lane);
    // score = bf16(dot / sqrt(hd)); a tile is masked unless every key of it precedes every column of this wave
    const int before = first + TQ <= a.n_tok ? a.pos0 + first + cg * 32 / GQ : -1, pos_q = a.pos0 + c.tok;
    auto maximum = [&](fl_f32x16& st, int j, float m) {
        const int k0 = KEYS * j + 32 * kp;
        if (k0 + 31 > before) m = Wave::mask(st, k0, 0, pos_q, h);
        return xmax32(m) * AP_LOG2E;
    };
    const int nown = (kmax / 32 + KP - kp) / KP; /* this part's tiles */
    fl_f32x16 sa, sb;
    float mt = 0.f;
    int b = 0;
    ap_landed<(NB - 2) * 2 * NI>(); /* K sets 0 and 1, V set 0 */
    if (nown > 0) {
        W.scores(sa, [&](int s) { return T.k(set(0, false) + kp * Tile::PART, s); });
        mt = maximum(sa, 0, Wave::template scale<true>(sa, a.rden));
    }
    ap_landed<(NB - 2) * 2 * NI>(); /* every wave has read K set 0 */
    auto step = [&](int j, fl_f32x16& cur, fl_f32x16& nxt) { /* K set j + 1 and V set j are here; K set j + NB goes where set j was, V set j + NB - 1 where set j - 1 was */
        const int b1 = b + 1 < NB ? b + 1 : 0, bl = b ? b - 1 : NB - 1;
        ap_tile_step<HD>(W, T, set(b1, false) + kp * Tile::PART, set(b, true) + kp * Tile::PART, cur, mt, nxt, a.rden, j < nown, set(b, false), set(bl, true),
                         [&](unsigned char* to) { load_k(j + NB, to); }, [&](unsigned char* to) { load_v(j + NB - 1, to); });
        if (j < nown) mt = maximum(nxt, j + 1, mt);
        ap_landed<(NB - 2) * 2 * NI>(); /* K set j + 2, V set j + 1 */
        b = b1;
    };
    for (int j = 0; j < nset; j += 2) {
        step(j, sa, sb);
        if (j + 1 < nset) step(j + 1, sb, sa);
    }
    ap_landed<0>(); /* loads past the last set write zeros */
    // the parts meet: (M, l) first, then every wave leaves the scaled sums that others finish and finishes HD / KP rows of d for its columns
    constexpr int NE = HD / 8, OWN = NE / KP;                    /* groups of four rows of d per lane; those a part finishes */
    float* const ml = reinterpret_cast<float*>(smem_raw);        /* [CG][KP][2][32] */
    f32x4* const ex = reinterpret_cast<f32x4*>(smem_raw + 4096); /* [CG][KP][NE][64 lanes]: d 32 db + 8 q + 4 h .. + 3 at number 4 db + q */
    W.l = xsum32(W.l);
    if (h == 0) ml[(cg * KP + kp) * 64 + lane] = W.M, ml[(cg * KP + kp) * 64 + 32 + lane] = W.l;
    __syncthreads();
    float M = W.M, l = 0.f;
#pragma unroll
    for (int k = 0; k < KP; k++) M = fmaxf(M, ml[(cg * KP + k) * 64 + (lane & 31)]); /* the part of key 0 has seen it: finite */
#pragma unroll
    for (int k = 0; k < KP; k++) l += ml[(cg * KP + k) * 64 + 32 + (lane & 31)] * __builtin_amdgcn_exp2f(ml[(cg * KP + k) * 64 + (lane & 31)] - M);
    const float f = __builtin_amdgcn_exp2f(W.M - M), inv = 1.0f / l;
#pragma unroll
    for (int e = 0; e < NE; e++) ex[((cg * KP + kp) * NE + e) * 64 + lane] = f32x4{W.o[e >> 2][4 * (e & 3)] * f, W.o[e >> 2][4 * (e & 3) + 1] * f, W.o[e >> 2][4 * (e & 3) + 2] * f, W.o[e >> 2][4 * (e & 3) + 3] * f};
    __syncthreads();
    if (!c.ok) return;
    uint16_t* const orow = a.out + (seq_row + c.tok) * a.out_stride + (size_t)c.head * HD;
#pragma unroll
    for (int i = 0; i < OWN; i++) {
        const int e = kp * OWN + i;
        f32x4 s = ex[(cg * KP * NE + e) * 64 + lane];
#pragma unroll
        for (int k = 1; k < KP; k++) s += ex[((cg * KP + k) * NE + e) * 64 + lane];
        *reinterpret_cast<u32x2*>(orow + 8 * e + 4 * h) = u32x2{pack_bf16x2(s[0] * inv, s[1] * inv), pack_bf16x2(s[2] * inv, s[3] * inv)};
    }
}

template <int HD, int GQ>
static int ap_whole(hipStream_t st, const AttnPrefillArgs& a, dim3 grid) {
    constexpr int smem = AP_NB * 2 * ApTile<HD>::PART;
    static int attr_set = 0;
    if (!attr_set && smem > 64 * 1024) {
        if (hipFuncSetAttribute((const void*)attn_prefill_kernel<HD, GQ>, hipFuncAttributeMaxDynamicSharedMemorySize, smem) != hipSuccess) return KF_HIP_CHECK;
        attr_set = 1;
    }
    grid.x = (a.n_tok * GQ + 127) / 128;
    hipLaunchKernelGGL((attn_prefill_kernel<HD, GQ>), grid, dim3(256), smem, st, a);
    return 0;
}
template <int HD, int GQ, int CG>
static int ap_parts(hipStream_t st, const AttnPrefillArgs& a, dim3 grid) {
    constexpr int sets = ap_sets<HD, CG> * 2 * (8 / CG) * ApTile<HD>::PART, merge = 4096 + 8 * (HD / 8) * 64 * 16, smem = sets > merge ? sets : merge;
    static_assert(smem <= 160 * 1024, "LDS");
    static int attr_set = 0;
    if (!attr_set && smem > 64 * 1024) {
        if (hipFuncSetAttribute((const void*)attn_prefill_parts_kernel<HD, GQ, CG>, hipFuncAttributeMaxDynamicSharedMemorySize, smem) != hipSuccess) return KF_HIP_CHECK;
        attr_set = 1;
    }
    grid.x = (a.n_tok * GQ + 32 * CG - 1) / (32 * CG);
    hipLaunchKernelGGL((attn_prefill_parts_kernel<HD, GQ, CG>), grid, dim3(512), smem, st, a);
    return 0;
}
template <int HD, int GQ>
static int ap_go(hipStream_t st, const AttnPrefillArgs& a, dim3 grid) {
    // One 128-column workgroup to a CU or fewer: two column groups, four key quarters, from the second set of 128 keys on.  Up to two, of long prompts: four groups, two halves.  us, four waves over all keys | four groups, two halves | two groups, four
    // quarters:  16 / 8 heads x 128, 2047 tokens (256 workgroups) 69 | 58 | 44, 1000 tokens (125) 35 | 31 | 20, 128 tokens 9.0 | 10.6 | 9.0; 64 / 8 heads, 700 tokens (352) 32 | 26 | 35; 16 / 8 heads, 4095 tokens
    // (512) 145 | 123 | 130, 16 prompts of 163 tokens (384) 16 | 22 | 27; 25 heads x 64, 8 x 1024 tokens (1600) 88 | 90 | 94
    const long wgs = (long)((a.n_tok * GQ + 127) / 128) * a.n_kv * a.n_seq;
    if (wgs <= g_knobs.attn_parts_max && a.pos0 + a.n_tok > 128) return ap_parts<HD, GQ, 2>(st, a, grid);
    if (wgs <= 2l * g_knobs.attn_parts_max && a.pos0 + a.n_tok >= 512) return ap_parts<HD, GQ, 4>(st, a, grid);
    return ap_whole<HD, GQ>(st, a, grid);
}
template <int HD>
static int ap_launch_gq(hipStream_t st, const AttnPrefillArgs& a, int GQ, dim3 grid) {
    switch (GQ) {
        case 1: return ap_go<HD, 1>(st, a, grid);
        case 2: return ap_go<HD, 2>(st, a, grid);
        case 4: return ap_go<HD, 4>(st, a, grid);
        case 8: return ap_go<HD, 8>(st, a, grid);
        default: return 1;
    }
}

// KF_OK launched; 1 = shape not covered (the caller falls back to the per-token kernel)
int attn_prefill_mfma_launch(hipStream_t st, const uint16_t* q, const uint16_t* kc, const uint16_t* vc, uint16_t* out, int pos0, int n_tok, long long q_stride,
                             int n_head, int n_kv, int hd, int kv_stride, int n_seq, long long out_stride) {
    if (out_stride <= 0) out_stride = q_stride;
    if (out_stride & 3) return 1;
    if ((hd != 64 && hd != 128) || n_kv <= 0 || n_head % n_kv != 0) return 1;
    if ((q_stride & 7) != 0 || (kv_stride & 7) != 0 || (reinterpret_cast<uintptr_t>(q) & 15) != 0 || (reinterpret_cast<uintptr_t>(out) & 7) != 0) return 1;
    const int GQ = n_head / n_kv;
    if (GQ != 1 && GQ != 2 && GQ != 4 && GQ != 8) return 1;
    AttnPrefillArgs a;
    a.q = q, a.kcache = kc, a.vcache = vc, a.out = out, a.pos0 = pos0, a.n_tok = n_tok, a.n_kv = n_kv, a.kv_stride = kv_stride, a.q_stride = q_stride, a.out_stride = out_stride;
    a.rden = 1.0f / sqrtf((float)hd);
    a.n_seq = n_seq;
    const dim3 grid(1, n_kv, n_seq);
    const int rc = hd == 128 ? ap_launch_gq<128>(st, a, GQ, grid) : ap_launch_gq<64>(st, a, GQ, grid);
    if (rc) return rc;
    return hipGetLastError() == hipSuccess ? KF_OK : KF_HIP_CHECK;
}

}  // namespace kf
