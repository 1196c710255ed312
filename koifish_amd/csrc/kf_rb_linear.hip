// kf_rb_linear.hip -- row-batch products y[t][m] = W[m] . x[t] for few rows (decode batches) and in 32-bit, and the ABI entry that picks the form.
//
// Decode batches stream the weights: a workgroup owns one to four blocks of 16 weight rows (GATED: of 8 gate rows and their 8 up rows), its waves take runs of 32-deep k-steps -- a
// step's 16 x 32 weights are one stored tile, a contiguous kilobyte -- and multiply them against up to 64 token columns by v_mfma_f32_16x16x32_bf16 (A = weight rows, B = token rows from
// L2, where the activations of a decode batch stay: more than 8 rows by way of RbTokens), the next run's weights in flight.  The waves' partial tiles meet in LDS, one thread
// per output finishes it.  The RMS norm in front of a product (NORM: few rows of the 32-bit residual sum) costs no pass: the product that formed the sum left its squares
// per 16 columns, every wave adds them up for itself and norms its token fragments as it reads them.  With experts a workgroup's columns are the pairs of one expert (UP, DOWN), or it walks all chosen experts' k-steps as one list dealt to its waves,
// columns that did not choose an expert held at zero (SUM): an expert's rows are read once per workgroup whoever chose them.
#include "kf_ctx.h"
#include "kf_rb_common.h"

namespace kf {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

// k-steps a wave takes in a row (part of a result's last bits: which steps a wave adds up), its token rows' run in LDS
constexpr int rb_deal(int nt) { return nt >= 4 ? 2 : 4; }
// k-steps of weights loaded at a time, one run ahead: a wave of several weight blocks has its bytes in flight with two (us at four | two, 32 rows, two blocks of 32768 x 2048 27.7 | 26.0, three of 12288 x 2048 12.9 | 12.3;
// with one block two are the slower: one row of 2048 x 6144 6.2 | 7.0)
constexpr int rb_run(int nt, int mg) { return nt >= 4 || mg >= 2 ? 2 : 4; }

__device__ __forceinline__ f32x4 rb_mfma16(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

// the run of U k-steps from step s of MG blocks of 16 weight rows; wr[g]: this lane's piece of block g's first tile (a tile per step)
template <int MG, int U>
__device__ __forceinline__ void rb_load_w(u32x4 (&a)[U][MG], const uint16_t* const (&wr)[MG], int s, int s_end) {
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
        for (int g = 0; g < MG; g++) {
            a[u][g] = u32x4{0, 0, 0, 0};
            if (s + u < s_end) a[u][g] = ld_nt(reinterpret_cast<const u32x4*>(wr[g] + 512 * (s + u))); /* wave-uniform */
        }
}
// token fragments of the same steps; xp[t]: this lane's token row + its k octet; steps past s_end read step s_end - 1 against zero weights
template <int NT, int U>
__device__ __forceinline__ void rb_load_x(u32x4 (&b)[U][NT], const uint16_t* const (&xp)[NT], int s, int s_end) {
#pragma unroll
    for (int u = 0; u < U; u++) {
        const int st = s + u < s_end ? s + u : s_end - 1;
#pragma unroll
        for (int t = 0; t < NT; t++) b[u][t] = *reinterpret_cast<const u32x4*>(xp[t] + 32 * st);
    }
}
template <int NT, int MG, int U, int B>
__device__ __forceinline__ void rb_multiply(const u32x4 (&a)[U][MG], const u32x4 (&b)[B][NT], int first, f32x4 (&acc)[MG][NT]) {
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
        for (int g = 0; g < MG; g++)
#pragma unroll
            for (int t = 0; t < NT; t++) acc[g][t] = rb_mfma16(a[u][g], b[first + u][t], acc[g][t]);
}
// the waves' partial tiles of the blocks from unit0 -> outputs; list: the columns are pairs; units: blocks past them repeat the last one.  GATED: a block is 8 gate rows and their 8 up rows; WHOLE: two blocks,
// 16 gate rows and their 16 up rows
template <int NT, int MG, int NW, bool GATED, bool WHOLE = false>
__device__ __forceinline__ void rb_stream_finish(const RbProduct& q, const f32x4 (&acc)[MG][NT], float (&red)[NW][MG][16 * NT][17], const int32_t* list, int unit0, int units, int tid, int part = 0) {
    const kf_rb_product& p = q.p;
    const int lane = tid & 63, wid = tid >> 6, r16 = lane & 15, q4 = lane >> 4;
#pragma unroll
    for (int g = 0; g < MG; g++)
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int j = 0; j < 4; j++) red[wid][g][t * 16 + r16][4 * q4 + j] = acc[g][t][j];
    __syncthreads();
    constexpr int OUT = GATED ? 8 : 16, ROWS = MG * OUT; /* a block's outputs, the workgroup's */
    const int cols = list ? 16 * NT : p.n, rows = (MG == 1 || units - unit0 >= MG ? MG : units - unit0) * OUT;
    for (int i = tid; i < cols * ROWS; i += 64 * NW) {
        const int row = i % ROWS, col = i / ROWS, g = row / OUT, rg = row % OUT, m = unit0 * OUT + row;
        if (MG > 1 && row >= rows) continue;
        int yr = col;
        float scale = 1.f;
        if (list) {
            yr = list[col];
            if (yr < 0) continue;
            if (p.mode == KF_RB_UP) scale = q.e.weight[yr];
        }
        float d = 0.f;
#pragma unroll
        for (int w = 0; w < NW; w++) d += red[w][WHOLE ? 0 : g][col][WHOLE ? row : rg];
        if constexpr (GATED) {
            float u = 0.f;
#pragma unroll
            for (int w = 0; w < NW; w++) u += red[w][WHOLE ? 1 : g][col][WHOLE ? row : 8 + rg];
            reinterpret_cast<uint16_t*>(p.y)[(size_t)yr * p.ldy + m] = f2bf(scale * (rb_activate(p.act, d) * u));
        } else if (p.epilogue == KF_RB_STORE) {
            reinterpret_cast<uint16_t*>(p.y)[(size_t)yr * p.ldy + m] = f2bf(m >= p.act_lo && m < p.act_hi ? rb_activate(p.act, d) : d);
        } else if (p.epilogue == KF_RB_STORE_F32) {
            reinterpret_cast<float*>(p.y)[part * (size_t)p.part_stride + (size_t)yr * p.ldy + m] = d;
        } else {
            const float z = fmaf(p.alpha, p.res[(size_t)yr * p.ldr + m], d);
            reinterpret_cast<float*>(p.y)[(size_t)yr * p.ldy + m] = z;
            if (NT == 1 && p.ssq) { /* 16 lanes = the 16 columns of one row */
                float ss = z * z;
                ss += dpp_f<0xB1>(ss);
                ss += dpp_f<0x4E>(ss);
                ss += dpp_f<0x141>(ss);
                ss += dpp_f<0x140>(ss);
                if (rg == 0) p.ssq[(size_t)(unit0 + g) * KF_RB_NORM_ROWS + yr] = ss;
            }
        }
    }
}

// A run's token rows on their way to the fragments: loaded in whole lines (a row's U x 64 bytes by neighbouring lanes) a run ahead, turned round in this wave's own LDS, no barrier.  A fragment read
// straight from memory takes half a line of each of 16 rows, and a workgroup of 32 rows reads twice as many token bytes as weight bytes: the CU's way to its L2 was the bound, not HBM.  32 rows,
// 2048 x 6144 (128 workgroups): 16.9 -> 12.4 us; gate and up 12288 x 2048: 17.8 -> 15.5; 32768 x 2048: 43.2 -> 32.6 (each with one block of weight rows, or two gated, to a workgroup).  Prefetching alone, without the lines, gave 1 %, and 16 waves
// instead of 8 where workgroups are few cost 10 %.
template <int NT, int U>
struct RbTokens {
    static constexpr int CH = 4 * U, ROW = 8 * CH + 8; /* 16-byte pieces of a row, a row's LDS stride in elements (16 bytes of padding: 16 rows' equal pieces lie in different banks) */
    static constexpr int LDS = 16 * NT * ROW;
    const uint16_t* x;
    uint16_t* lds;
    uint32_t off[NT * U]; /* load i's row */
    u32x4 v[NT * U];
    int lane;
    __device__ __forceinline__ void load(int s, int s_end) {
        const int c = lane % CH, st = s + c / 4 < s_end ? s + c / 4 : s_end - 1; /* steps past the end meet zero weights */
        const uint16_t* at = x + 32 * st + 8 * (c % 4);
#pragma unroll
        for (int i = 0; i < NT * U; i++) v[i] = *reinterpret_cast<const u32x4*>(at + off[i]);
    }
    __device__ __forceinline__ int row(int i) const { return i * (64 / CH) + lane / CH; }
    // Other lanes read what a lane stores, and store over what it has read.  A wave's LDS accesses are in order; only the compiler has to be told, which sees one lane's addresses and could swap them.
    static __device__ __forceinline__ void in_order() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    __device__ __forceinline__ void turn(u32x4 (&b)[U][NT]) {
        in_order();
#pragma unroll
        for (int i = 0; i < NT * U; i++) *reinterpret_cast<u32x4*>(lds + row(i) * ROW + 8 * (lane % CH)) = v[i];
        in_order();
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int t = 0; t < NT; t++) b[u][t] = *reinterpret_cast<const u32x4*>(lds + (16 * t + (lane & 15)) * ROW + 32 * u + 8 * (lane >> 4));
    }
};

// TURN: the token rows go through RbTokens (rows in order, no experts); else every lane reads its fragments itself.  PARTS: blockIdx.y is a part of k (a form of its own: 1 % of a decode step of products
// that have none)
template <int NT, int MG, bool GATED, int NW, bool NORM, bool TURN, bool PARTS = false, bool WHOLE = false, int U = rb_run(NT, MG)>
__global__ void __launch_bounds__(64 * NW) rb_stream_kernel(const RbProduct q) {
    const kf_rb_product& p = q.p;
    constexpr int DEAL = rb_deal(NT);
    static_assert(DEAL % U == 0 && (!WHOLE || (GATED && MG == 2)), "a deal is whole runs; a gate block and its up block");
    static_assert(!(NORM && TURN), "normed fragments are made from the residual sum");
    using Tokens = RbTokens<NT, DEAL>;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    auto& red = *reinterpret_cast<float(*)[NW][MG][16 * NT][17]>(smem); /* [wave][block][column][row], padded; after the waves' token rows */
    const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6), r16 = lane & 15, q4 = lane >> 4;
    const int unit0 = blockIdx.x * MG, units = p.m / 16, part = PARTS ? (int)blockIdx.y : 0, steps = p.k / 32, nstep = PARTS ? steps * (part + 1) / p.parts : steps; /* this part's steps end here */
    const uint16_t* W = reinterpret_cast<const uint16_t*>(p.w);
    const uint16_t* X = reinterpret_cast<const uint16_t*>(p.x);
    const int32_t* list = nullptr;
    if (p.mode != KF_RB_ALL) {
        const int ex = q.e.tile_expert[blockIdx.y];
        if (ex < 0) return;
        W += (size_t)ex * q.e.w_stride;
        list = q.e.list + (size_t)blockIdx.y * q.e.tile;
    }
    const uint16_t* wr[MG];
#pragma unroll
    for (int g = 0; g < MG; g++) {
        const int unit = MG == 1 || unit0 + g < units ? unit0 + g : units - 1;
        if (GATED && !WHOLE) wr[g] = W + (size_t)(2 * (unit >> 1) + (r16 >> 3)) * 16 * p.k + 8 * (16 * q4 + 8 * (unit & 1) + (r16 & 7)); /* half of the gate's tile, half of the up rows': whole lines of both */
        else wr[g] = W + (size_t)unit * 16 * p.k + 8 * lane;
    }
    u32x4 a[U][MG], b[TURN ? DEAL : U][NT];
    int s = (PARTS ? steps * part / p.parts : 0) + wid * DEAL;
    rb_load_w<MG, U>(a, wr, s, nstep);
    const uint16_t* xp[NT];
    Tokens tok;
    const float* zp = nullptr;   /* NORM: this lane's row of the residual sum, and 1 / its root mean square */
    const uint16_t* gp = nullptr;
    float rs = 0.f;
    if constexpr (NORM) {
        static_assert(NT == 1, "a few rows");
        const int row = r16 < p.n ? r16 : p.n - 1, parts = p.k / 16;
        zp = p.norm_z + (size_t)row * p.ldx + 8 * q4, gp = reinterpret_cast<const uint16_t*>(p.norm_w) + 8 * q4;
        for (int t = 0; t < p.n; t++) { /* the sums of squares the product in front left per 16 columns: no barrier, every wave for itself */
            float ss = 0.f;
            for (int i = lane; i < parts; i += 64) ss += p.norm_ssq[(size_t)i * KF_RB_NORM_ROWS + t];
            ss = wave_sum(ss);
            if (row == t) rs = 1.0f / sqrtf(ss / (float)p.norm_dim + p.norm_eps);
        }
        xp[0] = nullptr;
    } else if constexpr (TURN) {
        tok.x = X, tok.lds = reinterpret_cast<uint16_t*>(smem) + wid * Tokens::LDS, tok.lane = lane;
#pragma unroll
        for (int i = 0; i < NT * DEAL; i++) {
            const int row = tok.row(i);
            tok.off[i] = (uint32_t)(row < p.n ? row : p.n - 1) * (uint32_t)p.ldx; /* <= 64 rows: below 2^32 (the launch sees to it) */
        }
        tok.load(s < nstep ? s : nstep - 1, nstep);
    } else {
#pragma unroll
        for (int t = 0; t < NT; t++) { /* columns past the end repeat a row: their outputs are not stored */
            const int col = t * 16 + r16;
            int row = col < p.n ? col : p.n - 1;
            if (list) {
                const int pair = list[col];
                row = pair < 0 ? 0 : (p.mode == KF_RB_UP ? pair / q.e.top : pair);
            }
            xp[t] = X + (size_t)row * p.ldx + 8 * q4;
        }
    }
    f32x4 acc[MG][NT];
#pragma unroll
    for (int g = 0; g < MG; g++)
#pragma unroll
        for (int t = 0; t < NT; t++) acc[g][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (; s < nstep; s += NW * DEAL) {
        if constexpr (TURN) {
            tok.turn(b);
            if (s + NW * DEAL < nstep) tok.load(s + NW * DEAL, nstep); /* wave-uniform */
        }
#pragma unroll
        for (int run = 0; run < DEAL; run += U) { /* (one that begins past the end meets zero weights) */
            const int s0 = s + run, s1 = run + U < DEAL ? s0 + U : s + NW * DEAL;
            u32x4 an[U][MG];
            if constexpr (NORM) {
                f32x4 z0[U], z1[U];
                u32x4 g[U];
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const int k0 = 32 * (s0 + u < nstep ? s0 + u : nstep - 1);
                    z0[u] = rb_ld4(zp + k0), z1[u] = rb_ld4(zp + k0 + 4), g[u] = *reinterpret_cast<const u32x4*>(gp + k0);
                }
                rb_load_w<MG, U>(an, wr, s1, nstep);
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const f32x4 o0 = f32x4{z0[u].x * rs * bf_lo(g[u].x), z0[u].y * rs * bf_hi(g[u].x), z0[u].z * rs * bf_lo(g[u].y), z0[u].w * rs * bf_hi(g[u].y)};
                    const f32x4 o1 = f32x4{z1[u].x * rs * bf_lo(g[u].z), z1[u].y * rs * bf_hi(g[u].z), z1[u].z * rs * bf_lo(g[u].w), z1[u].w * rs * bf_hi(g[u].w)};
                    b[u][0] = u32x4{pack_bf16x2(o0.x, o0.y), pack_bf16x2(o0.z, o0.w), pack_bf16x2(o1.x, o1.y), pack_bf16x2(o1.z, o1.w)};
                    if (blockIdx.x == 0 && r16 < p.n && s0 + u < nstep) { /* the normed rows themselves, once */
                        const size_t at = (size_t)r16 * p.ldx + 32 * (s0 + u) + 8 * q4;
                        rb_st4(p.norm_x + at, o0), rb_st4(p.norm_x + at + 4, o1);
                        *reinterpret_cast<u32x4*>(reinterpret_cast<uint16_t*>(const_cast<void*>(p.x)) + at) = b[u][0];
                    }
                }
            } else {
                if constexpr (!TURN) rb_load_x<NT, U>(b, xp, s0, nstep);
                rb_load_w<MG, U>(an, wr, s1, nstep);
            }
            rb_multiply<NT, MG, U>(a, b, TURN ? run : 0, acc);
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int g = 0; g < MG; g++) a[u][g] = an[u][g];
        }
    }
    if constexpr (TURN) __syncthreads(); /* the token rows make way */
    rb_stream_finish<NT, MG, NW, GATED, WHOLE>(q, acc, red, list, unit0, units, tid, part);
}

// RESIDUAL with the rows' experts summed: (chosen expert, k-step) pairs as one list, cut evenly over the waves
template <int NT, int NW>
__global__ void __launch_bounds__(64 * NW) rb_stream_sum_kernel(const RbProduct q) {
    const kf_rb_product& p = q.p;
    constexpr int U = NT >= 4 ? 2 : 4;
    __shared__ float red[NW][1][16 * NT][17];
    __shared__ int32_t s_ex[KF_RB_SUM_PAIRS], s_ids[KF_RB_SUM_PAIRS];
    __shared__ int s_n;
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, r16 = lane & 15, q4 = lane >> 4;
    const int m0 = blockIdx.x * 16, nstep = p.k / 32, pairs = p.n * q.e.top;
    const uint16_t* X = reinterpret_cast<const uint16_t*>(p.x);
    for (int i = tid; i < pairs; i += 64 * NW) s_ids[i] = q.e.ids[i];
    if (wid == 0) { /* the chosen experts, each once: a tile per expert (a tile holds as many pairs as the batch has rows) */
        int cnt = 0;
        for (int i0 = 0; i0 < q.e.n_tile; i0 += 64) {
            const int ex = i0 + lane < q.e.n_tile ? q.e.tile_expert[i0 + lane] : -1;
            const unsigned long long on = __ballot(ex >= 0);
            if (ex >= 0) s_ex[cnt + __popcll(on & ((1ull << lane) - 1))] = ex;
            cnt += __popcll(on);
        }
        if (lane == 0) s_n = cnt;
    }
    __syncthreads();
    const int total = s_n * nstep, span = (total + NW - 1) / NW;
    int at = wid * span;
    const int end = at + span < total ? at + span : total;
    f32x4 acc[1][NT];
#pragma unroll
    for (int t = 0; t < NT; t++) acc[0][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    while (at < end) { /* an expert's part of this wave's range (wave-uniform) */
        const int i = at / nstep, s0 = at - i * nstep, s1 = s0 + (end - at) < nstep ? s0 + (end - at) : nstep;
        const int ex = s_ex[i];
        const uint16_t* wr = reinterpret_cast<const uint16_t*>(p.w) + (size_t)ex * q.e.w_stride + (size_t)m0 * p.k + 8 * lane;
        // every load is unconditional and no run is copied from one set of registers to another: either makes the wave wait for what it has just asked for.  Past the range its last step is read again and columns of
        // another expert read row 0, and zeros are multiplied instead.  us per call of four tokens, 2048 wide, 64 experts, 1, 4, 8, 14, 32 sequences: 2565 4089 5414 6853 9913 -> 2469 3723 4769 5965 8399
        const uint16_t* xp[NT];
        bool on[NT];
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const int row = t * 16 + r16;
            xp[t] = X + 8 * q4, on[t] = false;
            if (row < p.n)
                for (int j = 0; j < q.e.top; j++)
                    if (s_ids[row * q.e.top + j] == ex) xp[t] = X + (size_t)(row * q.e.top + j) * p.ldx + 8 * q4, on[t] = true;
        }
        auto weights = [&](u32x4 (&w)[U][1], int s) {
#pragma unroll
            for (int u = 0; u < U; u++) w[u][0] = ld_nt(reinterpret_cast<const u32x4*>(wr + 512 * (s + u < s1 ? s + u : s1 - 1)));
        };
        auto run = [&](u32x4 (&w)[U][1], u32x4 (&next)[U][1], int s) {
            u32x4 b[U][NT];
            rb_load_x<NT, U>(b, xp, s, s1);
            weights(next, s + U);
#pragma unroll
            for (int u = 0; u < U; u++) {
                if (s + u >= s1) w[u][0] = u32x4{0, 0, 0, 0}; /* (both factors: the other one may be an infinity) */
#pragma unroll
                for (int t = 0; t < NT; t++)
                    if (!(on[t] && s + u < s1)) b[u][t] = u32x4{0, 0, 0, 0};
            }
            rb_multiply<NT, 1, U>(w, b, 0, acc);
        };
        u32x4 w0[U][1], w1[U][1];
        weights(w0, s0);
        for (int s = s0; s < s1; s += 2 * U) {
            run(w0, w1, s);
            if (s + U < s1) run(w1, w0, s + U);
        }
        at += s1 - s0;
    }
    rb_stream_finish<NT, 1, NW, false>(q, acc, red, nullptr, blockIdx.x, p.m / 16, tid);
}
template <int NT, int MG, bool GATED, int NW, bool NORM, bool TURN, bool PARTS = false, bool WHOLE = false, int U = rb_run(NT, MG)>
static int stream_form(hipStream_t st, const RbProduct& q, dim3 grid) {
    constexpr int RED = NW * MG * 16 * NT * 17 * 4, STAGE = TURN ? NW * RbTokens<NT, rb_deal(NT)>::LDS * 2 : 0, SMEM = RED > STAGE ? RED : STAGE;
    static_assert(SMEM <= 160 * 1024, "LDS");
    const auto kernel = rb_stream_kernel<NT, MG, GATED, NW, NORM, TURN, PARTS, WHOLE, U>;
    if constexpr (SMEM > 64 * 1024) {
        static bool done = false;
        if (!done && hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, SMEM) != hipSuccess) return KF_HIP_CHECK;
        done = true;
    }
    hipLaunchKernelGGL(kernel, grid, dim3(64 * NW), SMEM, st, q);
    return KF_OK;
}
template <int NT, int MG, int NW>
static int stream_go(hipStream_t st, const RbProduct& q, dim3 grid) {
    const kf_rb_product& p = q.p;
    // whole lines for more than 8 rows in order: below, a fragment's 16 half lines are few distinct ones and the way round costs more than it saves (one token of a 2048-wide model: 1.79 -> 1.87 ms
    // over four steps; 6 rows 2.04 -> 2.08; 14 rows 2.42 -> 2.35; 32 rows 4.62 -> 4.23)
    const bool turn = p.n > 8 && p.ldx <= (1 << 24), gated = p.epilogue == KF_RB_GATED;
    // what stream_blocks gives, and nothing else.  Four waves: one block or two of up to 16 rows; any of more, but one only where not gated and four not of 33 to 48 rows.  Eight: four only where gated.  In front of a
    // gated product a norm has four waves.
    constexpr bool THREE = NT == 3 && MG == 4, GATED = NW == 8 || (NT == 1 ? MG <= 2 : MG >= 2 && !THREE), PLAIN = NW == 8 ? MG <= 3 : NT == 1 ? MG <= 2 : !THREE;
    if constexpr (NT == 1 && GATED && NW == 4) {
        // a pair as a gate block and its up block of 16 rows each, four k-steps at a time, instead of two blocks of 8 and 8 (the same sums): behind a norm (768 blocks x 2048, 4 rows, us 15.5 | 16.6) up to 1024 blocks, and
        // for rows that go through LDS from there (6144 x 512, 12 rows, 20.3 | 21.7)
        if constexpr (MG == 2) {
            if (gated && p.norm_z && p.m <= 16 * 1024) return stream_form<1, 2, true, 4, true, false, false, true, rb_deal(1)>(st, q, grid);
            if (gated && turn && p.m > 16 * 1024) return stream_form<1, 2, true, 4, false, true, false, true, rb_deal(1)>(st, q, grid);
        }
        if (p.norm_z && gated) return stream_form<1, MG, true, 4, true, false>(st, q, grid);
    }
    if constexpr (NT == 1 && PLAIN) {
        if (p.norm_z && !gated) return stream_form<1, MG, false, NW, true, false>(st, q, grid);
    }
    if (p.norm_z) return KF_INTERNAL_ERR;
    if constexpr (MG == 1) {
        if (p.parts > 1) return turn ? stream_form<NT, 1, false, NW, false, true, true>(st, q, grid) : stream_form<NT, 1, false, NW, false, false, true>(st, q, grid);
    }
    if constexpr (GATED) {
        if (gated) return turn ? stream_form<NT, MG, true, NW, false, true>(st, q, grid) : stream_form<NT, MG, true, NW, false, false>(st, q, grid);
    }
    if constexpr (PLAIN) {
        if (!gated) return turn ? stream_form<NT, MG, false, NW, false, true>(st, q, grid) : stream_form<NT, MG, false, NW, false, false>(st, q, grid);
    }
    return KF_INTERNAL_ERR;
}
// experts: one gate block and its up rows a workgroup; the tiles are mostly padding, which repeats row 0, and the way round by LDS does not pay (32 rows of 64 experts: 10.15 -> 10.36 ms)
template <int NT, int NW>
static int expert_go(hipStream_t st, const RbProduct& q, dim3 grid) {
    if (q.p.mode == KF_RB_SUM) hipLaunchKernelGGL((rb_stream_sum_kernel<NT, NW>), grid, dim3(64 * NW), 0, st, q);
    else if (q.p.epilogue == KF_RB_GATED) return stream_form<NT, 2, true, NW, false, false, false, true, rb_deal(NT)>(st, q, grid);
    else return stream_form<NT, 1, false, NW, false, false>(st, q, grid);
    return KF_OK;
}
template <int NT, int NW>
static int stream_any(hipStream_t st, const RbProduct& q, dim3 grid, int mg) {
    if (q.p.mode != KF_RB_ALL) return expert_go<NT, NW>(st, q, grid);
    return mg == 1 ? stream_go<NT, 1, NW>(st, q, grid) : mg == 2 ? stream_go<NT, 2, NW>(st, q, grid) : mg == 3 ? stream_go<NT, 3, NW>(st, q, grid) : stream_go<NT, 4, NW>(st, q, grid);
}
// How many 16-row blocks a workgroup takes.  A workgroup takes in its weight rows and, once, all of the batch's token rows by its CU's way to the L2 (about 46 bytes a ns), which, and not HBM, bounds products of
// one block each: with 32 rows two bytes of tokens to one of weights.  More blocks: fewer token bytes, fewer and longer workgroups.  us, one block (gated: 8 gate rows and their 8 up rows) | two | three | four, by blocks of
// the matrix x k:
//  - one round of the CUs (eight waves each, up to 1024 blocks): as many as fill it.  12 rows 640 x 2048 plain 11.4 | 11.6 | 10.2 | 10.8; 32 rows 12288 x 2048 gated 15.6 before, three 12.3.  Not where the tokens are
//    few: plain, 4 rows or fewer (1 row 512 x 1024 5.0 | 5.5), up to 12 where k is short too; gated, 1024 x 512 8 rows two 5.5, four 6.0, 1024 x 4096 9 rows two 27.2, four 28.7.
//  - up to 10 rows of more than 1024 blocks, plain: one.  1 row 2048 x 1024 13.6 | 14.9; 9 14.4 | 14.7; 12 14.7 | 14.8; 16 rows 2048 x 2048 28.3 | 26.1.  Behind a norm, which every workgroup makes for itself: two.
//  - a norm in front of a gated product: one up to 256 blocks (128 x 2048 7.9 | 9.3), then pairs: 768 x 2048 4 rows 16.4 | 15.5.
//  - more than 16 rows of up to 1024 blocks, four waves: two where the CUs still get one workgroup each.  128 x 2048 33 rows 8.4 | 9.8, 320 x 1024 48 rows 7.5 | 7.5, 1024 x 256 24 rows 6.3 | 5.0; short k moves the line up
//    (40 x 256 3.1 | 4.1, 512 x 256 3.8 | 4.4), since the products are over before the tokens are in.
//  - more than 1024 blocks: pairs, many workgroups that follow each other, up to 24 rows; then the least work for the busiest CU.  32 rows 32768 weight rows x 2048 33.4 | 26.0, 64 rows 45.8 | 28.8 with four.  33 to 48
//    rows: three, two workgroups to a CU (four need registers of which only one goes): 3072 x 1024 gated 33.3 | 28.0 | 25.9 | 31.5, but two where the second round of them would be nearly empty: 2048 x 1024 25.6 | 21.1 |
//    22.8 | 23.4.  49 rows and more of a short k: two (3072 x 256 gated 15.4 | 13.7 | 15.1 | 15.3).
// The number of waves is part of a result's last bits (each adds up a part of k) and the same for every count: four for more than 32 rows, behind a norm where gated, and for 768 to 1024 blocks of one matrix.
static int stream_blocks(const kf_rb_product& p, bool wide) {
    const bool gated = p.epilogue == KF_RB_GATED, norm = p.norm_z != nullptr;
    const int units = p.m / 16, n = p.n, k = p.k, round = (units + 255) / 256;
    if (units <= 1024) {
        if (wide && gated) return units > 768 && n <= 16 && (n > 8 || k < 1024) ? 2 : round;
        if (wide) return !norm && (n <= 4 || (n <= 12 && k <= 1024 && units <= 512)) ? 1 : round;
        if (gated) return n > 16 || (norm && units > 256) ? 2 : 1;
        return n > 16 && units >= (k >= 1024 ? 257 : n > 32 && n <= 48 ? 513 : 768) ? 2 : 1;
    }
    if (n <= 16) return gated || norm || n > 10 ? 2 : 1;
    if (n <= 24 || (n > 48 && k < 512)) return 2;
    if (n > 32 && n <= 48) return units > 1536 && units <= 2048 ? 2 : 3;
    int best = 2;
    long least = 0;
    for (int mg = 2; mg <= 4; mg++) {
        const long cost = ((units + mg - 1) / mg + 255) / 256 * (16 * mg + n);
        if (mg == 2 || cost < least) best = mg, least = cost;
    }
    return best;
}
int rb_stream_launch(hipStream_t st, const RbProduct& q) {
    const kf_rb_product& p = q.p;
    const bool tiles = p.mode == KF_RB_UP || p.mode == KF_RB_DOWN, all = p.mode == KF_RB_ALL;
    const int cols = tiles ? q.e.tile : p.n, nt = (cols + 15) / 16, units = p.m / 16;
    if (nt > 4 || (tiles && q.e.tile % 16)) return 1;
    if (p.mode == KF_RB_SUM && ((long)p.n * q.e.top > KF_RB_SUM_PAIRS || q.e.tile < p.n)) return 1;
    const bool gated = p.epilogue == KF_RB_GATED;
    const long small = (long)units / (gated ? 2 : 1) * (tiles ? q.e.n_tile : p.parts > 1 ? p.parts : 1); /* workgroups of 16 rows, of 16 gates and 16 ups */
    const bool wide = p.k >= 512 && nt <= 2 && !(p.norm_z && gated) && small < 768;                        /* few workgroups: more waves each, more loads in flight per CU */
    const int mg = !all ? (gated ? 2 : 1) : p.parts > 1 ? 1 : stream_blocks(p, wide);
    const dim3 grid((units + mg - 1) / mg, tiles ? q.e.n_tile : (p.parts > 1 ? p.parts : 1));
    if (nt > 2) return nt == 3 ? stream_any<3, 4>(st, q, grid, mg) : stream_any<4, 4>(st, q, grid, mg);
    return nt == 1 ? (wide ? stream_any<1, 8>(st, q, grid, mg) : stream_any<1, 4>(st, q, grid, mg)) : (wide ? stream_any<2, 8>(st, q, grid, mg) : stream_any<2, 4>(st, q, grid, mg));
}

}  // namespace kf

using namespace kf;
// Up to half a workgroup per CU: two parts of k, a chip full of workgroups.  us per step of 8 recurrent / windowed layers behind 300 tokens, whole | two | four parts: 2048 wide, 32 rows 867 | 828 | 850, 8 rows 537 | 514 | 523, one
// 473 | 457 | 467; 4096 wide (256 workgroups) 1 row 969 | 978, 16 rows 1238 | 1252.  A product and its norm, us, whole | two parts, one row, 32: 1024 x 2048 6.6 | 6.2, 8.8 | 7.6; 1024 x 6144 10.1 | 8.4, 15.2 | 11.0;
// 1536 x 4096 9.2 | 8.2, 12.7 | 10.3; 2048 x 2048 7.7 | 7.6, 9.7 | 8.8; 2048 x 6144 11.4 | 9.9, 16.4 | 12.6
extern "C" int kf_rb_linear_parts(int type, int m, int k, int n) { return type == KF_BF16 && n >= 1 && n <= KF_RB_DECODE_MAX && m >= 1 && m / 16 <= 128 && k >= 2048 ? 2 : 1; }
extern "C" int kf_rb_linear_norms(int type, int n, int k) { return type == KF_BF16 && n >= 1 && n <= KF_RB_NORM_ROWS && k % KF_RB_PAD == 0; }
extern "C" int kf_rb_linear(kf_ctx* c, const kf_rb_product* p) {
    CHKCTX(c);
    if (!p || !p->w || !p->x || !p->y) return abi_fail(KF_INVALID_ARGS, "kf_rb_linear: null pointer");
    if (p->type != KF_BF16 && p->type != KF_F32) return abi_fail(KF_UNSUPPORTED_DATATYPE, "kf_rb_linear: storage %d", p->type);
    if (p->m < 1 || p->k < 1 || p->n < 1 || p->m % KF_RB_PAD || p->k % KF_RB_PAD) return abi_fail(KF_INVALID_ARGS, "kf_rb_linear: %d x %d weight, %d rows", p->m, p->k, p->n);
    if (p->ldx < p->k || p->ldy < (p->epilogue == KF_RB_GATED ? p->m / 2 : p->m) || p->ldx % 8 || p->ldy % 4) return abi_fail(KF_INVALID_ARGS, "kf_rb_linear: row strides");
    if (!al16(p->w) || !al16(p->x) || !al16(p->y)) return abi_fail(KF_BLAS_UNALIGN, "kf_rb_linear: unaligned pointer");
    if (p->epilogue < KF_RB_STORE || p->epilogue > KF_RB_GATED || p->mode < KF_RB_ALL || p->mode > KF_RB_SUM) return abi_fail(KF_INVALID_ARGS, "kf_rb_linear: epilogue or mode");
    if (p->epilogue == KF_RB_RESIDUAL && (!p->res || !al16(p->res) || p->ldr < p->m || p->ldr % 4)) return abi_fail(KF_INVALID_ARGS, "kf_rb_linear: residual");
    if (p->act_lo < p->act_hi && (p->epilogue != KF_RB_STORE || p->mode != KF_RB_ALL || p->act_lo < 0 || p->act_hi > p->m)) return abi_fail(KF_INVALID_ARGS, "kf_rb_linear: activated columns");
    if (p->parts > 1 && (p->type != KF_BF16 || p->epilogue != KF_RB_STORE_F32 || p->mode != KF_RB_ALL || p->n > KF_RB_DECODE_MAX || p->parts > KF_RB_MAX_PARTS || p->part_stride < (int64_t)(p->n - 1) * p->ldy + p->m || p->norm_z))
        return abi_fail(KF_INVALID_ARGS, "kf_rb_linear: %d parts", p->parts);
    if (p->ssq && (!kf_rb_linear_norms(p->type, p->n, p->m) || p->epilogue != KF_RB_RESIDUAL)) return abi_fail(KF_INVALID_ARGS, "kf_rb_linear: sums of squares");
    if (p->norm_z && (!kf_rb_linear_norms(p->type, p->n, p->k) || p->mode != KF_RB_ALL || p->epilogue == KF_RB_RESIDUAL || !p->norm_w || !p->norm_x || !p->norm_ssq || p->norm_dim < 1 || p->norm_dim > p->k || p->ldx != p->k || !al16(p->norm_z) ||
                      !al16(p->norm_w) || !al16(p->norm_x)))
        return abi_fail(KF_INVALID_ARGS, "kf_rb_linear: norm in front of the product");
    RbProduct q;
    q.p = *p;
    q.e = kf_rb_experts{};
    if (p->mode != KF_RB_ALL) {
        const kf_rb_experts* e = p->experts;
        if (!e || e->n_expert < 1 || e->top < 1 || e->tile < 1 || e->n_tile < 1 || !e->tile_expert || !e->list || !e->ids || !e->weight) return abi_fail(KF_INVALID_ARGS, "kf_rb_linear: experts");
        if (e->w_stride < (int64_t)p->m * p->k || e->w_stride % 8) return abi_fail(KF_INVALID_ARGS, "kf_rb_linear: expert stride");
        if ((p->mode == KF_RB_UP) != (p->epilogue == KF_RB_GATED) || (p->mode == KF_RB_DOWN && p->epilogue != KF_RB_STORE) || (p->mode == KF_RB_SUM && p->epilogue != KF_RB_RESIDUAL))
            return abi_fail(KF_INVALID_ARGS, "kf_rb_linear: this mode has another epilogue");
        q.e = *e;
    }
    int rc;
    if (p->type == KF_F32) rc = rb_f32_launch(c->stream, q);
    else {
        rc = 1;
        if (p->n <= KF_RB_DECODE_MAX) rc = rb_stream_launch(c->stream, q);
        if (rc == 1 && p->mode != KF_RB_SUM) rc = rb_gemm_launch(c->stream, q);
    }
    if (rc == 1) return abi_fail(KF_UNSUPPORTED_DATATYPE, "kf_rb_linear: no kernel for mode %d, %d rows, tiles of %d, storage %d", p->mode, p->n, q.e.tile, p->type);
    if (rc != KF_OK) return abi_fail(rc, "kf_rb_linear: launch failed");
    return hipGetLastError() == hipSuccess ? KF_OK : abi_fail(KF_HIP_CHECK, "kf_rb_linear: launch failed");
}
