// kf_flash.h -- a wave's walk over key tiles of flash attention on MFMA (32 columns, 32 keys at a time), shared by the prompt kernels of kf_attn_prefill.hip and kf_rb_attn.hip.
//   S^T[key][col] = sum_d K[key][d] Q[col][d]      v_mfma_f32_32x32x16_bf16, A = K rows (ds_read_b128), B = Q rows (registers): a column's 32 scores sit in ONE lane pair (lane l and l ^ 32)
//   O^T[d][col]  += sum_key V^T[d][key] P^T[key][col]   the S^T registers, packed to bf16, ARE the B operand (slot (step s, half h, j) <-> key 16 s + (j & 3) + 8 (j >> 2) + 4 h on both operands);
//      A = V^T fragments straight from the row-major V tile (ds_read_b64_tr_b16).  p enters as a bf16 pair (high part + remainder, ~16 significant bits), its sum stays fp32.
// What bounds it: a tile's MFMAs take 768 cycles of a SIMD at dim 128, its vector instructions about as many, and one after the other they leave both pipes idle half the time -- a SIMD has two
// waves at most here, often one.  So a step holds a tile's exponentials and P.V beside the next tile's scores, their scaling and maximum: independent instructions that the compiler mixes.
// A column's reference exponent M is the maximum of the keys seen so far, subtracted before any factor: the largest p is 1 whatever the scores' size, and a sum does not depend on the tiles' way through LDS.
#pragma once
#include "kf_device.h"

namespace kf {

typedef __bf16 fl_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 fl_bf16x4 __attribute__((ext_vector_type(4)));
typedef float fl_f32x16 __attribute__((ext_vector_type(16)));

constexpr float FL_LOG2E = 1.44269502162933349609375f;

template <int HD, bool NAT> /* NAT: scores in natural units; else in log2 units */
struct FlashWave {
    static constexpr int NS = HD / 16, NDB = HD / 32; /* MFMA steps over d of S^T; 32-row blocks of O^T */
    fl_f32x16 o[NDB];
    float M, l; /* the column's reference exponent (units of the scores; -inf: nothing seen) and this lane's half of the sum of p */
    u32x4 qf[NS];
    __device__ __forceinline__ void init() {
#pragma unroll
        for (int db = 0; db < NDB; db++)
#pragma unroll
            for (int i = 0; i < 16; i++) o[db][i] = 0.f;
        M = -__builtin_inff(), l = 0.f;
    }
    // scores of a tile: kfrag(s) = this lane's K fragment of MFMA step s
    template <class KF>
    __device__ __forceinline__ void scores(fl_f32x16& st, KF&& kfrag) const {
        fl_f32x16 z;
#pragma unroll
        for (int i = 0; i < 16; i++) z[i] = 0.f;
#pragma unroll
        for (int s = 0; s < NS; s++) st = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(fl_bf16x8, kfrag(s)), __builtin_bit_cast(fl_bf16x8, qf[s]), s ? st : z, 0, 0, 0);
    }
    // scaled scores and their maximum over this lane's 16 keys.  ROUND: the score is stored in bf16 on its way (the reference's store)
    template <bool ROUND>
    static __device__ __forceinline__ float scale(fl_f32x16& st, float by) {
        float mt = -__builtin_inff();
#pragma unroll
        for (int i = 0; i < 16; i += 2) {
            st[i] *= by, st[i + 1] *= by;
            if (ROUND) {
                const uint32_t w = pack_bf16x2(st[i], st[i + 1]);
                st[i] = bf_lo(w), st[i + 1] = bf_hi(w);
            }
            mt = fmaxf(mt, fmaxf(st[i], st[i + 1]));
        }
        return mt;
    }
    // keys of the tile that the column does not see: first key k0, it sees lo .. hi
    static __device__ __forceinline__ float mask(fl_f32x16& st, int k0, int lo, int hi, int h) {
        float mt = -__builtin_inff();
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int key = k0 + 4 * h + (i & 3) + 8 * (i >> 2);
            st[i] = key >= lo && key <= hi ? st[i] : -__builtin_inff();
            mt = fmaxf(mt, st[i]);
        }
        return mt;
    }
    static __device__ __forceinline__ float power(float d) { return __builtin_amdgcn_exp2f(NAT ? d * FL_LOG2E : d); } /* of a difference of scores */
    // mt: the column's maximum over the tile (both lanes of the pair)
    __device__ __forceinline__ void move(float mt) {
        if (mt > M) {
            const float alpha = power(M - mt); /* M = -inf on the first tile: 0 */
            l *= alpha;
#pragma unroll
            for (int db = 0; db < NDB; db++)
#pragma unroll
                for (int i = 0; i < 16; i++) o[db][i] *= alpha;
            M = mt;
        }
    }
    // p = 2^(score - M) or e^(score - M) as bf16 pairs.  A column that has seen nothing (M = -inf): p = 0
    __device__ __forceinline__ void weights(const fl_f32x16& st, uint32_t (&ph)[8], uint32_t (&pl)[8]) {
        const float ref = M == -__builtin_inff() ? 0.f : M;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const float p0 = power(st[2 * i] - ref), p1 = power(st[2 * i + 1] - ref);
            l += p0;
            l += p1;
            ph[i] = pack_bf16x2(p0, p1);
            pl[i] = pack_bf16x2(p0 - bf_lo(ph[i]), p1 - bf_hi(ph[i]));
        }
    }
    // O^T += V^T P^T: vfrag(s2, db) = this lane's V^T fragment of keys 16 s2 .. + 15, d 32 db .. + 31
    template <class VF>
    __device__ __forceinline__ void accumulate(const uint32_t (&ph)[8], const uint32_t (&pl)[8], VF&& vfrag) {
#pragma unroll
        for (int s2 = 0; s2 < 2; s2++) {
            const u32x4 B = u32x4{ph[4 * s2], ph[4 * s2 + 1], ph[4 * s2 + 2], ph[4 * s2 + 3]}, B2 = u32x4{pl[4 * s2], pl[4 * s2 + 1], pl[4 * s2 + 2], pl[4 * s2 + 3]};
#pragma unroll
            for (int db = 0; db < NDB; db++) {
                const fl_bf16x8 A = vfrag(s2, db);
                o[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A, __builtin_bit_cast(fl_bf16x8, B), o[db], 0, 0, 0);
                o[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A, __builtin_bit_cast(fl_bf16x8, B2), o[db], 0, 0, 0);
            }
        }
    }
    // one tile of the pipeline: its scores are in `cur` (scaled, masked; mt their maximum), those of the tile behind it come out in `nxt` (scaled; the result: this lane's maximum)
    template <bool ROUND, class KF, class VF>
    __device__ __forceinline__ float tile(fl_f32x16& cur, float mt, fl_f32x16& nxt, float by, KF&& kfrag, VF&& vfrag) {
        move(mt);
        uint32_t ph[8], pl[8];
        scores(nxt, kfrag);
        weights(cur, ph, pl);
        accumulate(ph, pl, vfrag);
        return scale<ROUND>(nxt, by);
    }
};

// ---- tiles that went global -> LDS by buffer loads: the LDS image of such a load is lane-linear, so rows are unpadded and the swizzle is made at the source: 16 lanes of a K read and 32 of a transposing V read touch
// all 64 banks once
constexpr int AP_NB = 5; /* buffers: up to three tiles of 16 KiB are on their way while one is multiplied, which is what a load from another XCD's memory side takes */
// the place of 16-byte chunk c of row r of a tile
template <int HD>
__device__ __forceinline__ int ap_swz_k(int r, int c) { return HD == 128 ? c ^ (r & 15) : c ^ ((r >> 1) & 7); }
template <int HD>
__device__ __forceinline__ int ap_swz_v(int r, int c) { return HD == 128 ? c ^ ((r & 3) << 2) : c ^ (((r >> 1) & 1) << 2); }

// where a wave's K and V rows lie in a tile of 32 keys (K, then V, each row-major) in LDS
template <int HD>
struct ApTile {
    static constexpr int RB = HD * 2, PART = 32 * RB, RPI = 1024 / RB; /* bytes of a row, of 32 rows; rows per load instruction */
    int kf[HD / 16], vf[HD / 32]; /* a swizzle flips bits of the chunk, so one offset per MFMA step (K) and per block of d (V) */
    __device__ __forceinline__ void init(int lane) {
        const int r = lane & 31, h = lane >> 5;
#pragma unroll
        for (int s = 0; s < HD / 16; s++) kf[s] = r * RB + ap_swz_k<HD>(r, 2 * s + h) * 16;
#pragma unroll
        for (int db = 0; db < HD / 32; db++) { /* lane l16 of a 16-lane group addresses key-row (l16 >> 2) of its 4, d-piece 4 (l16 & 3) of the group's 16 d; it receives the 4 keys of d = l16 */
            const int row = 4 * h + ((lane & 15) >> 2);
            vf[db] = row * RB + ap_swz_v<HD>(row, 4 * db + ((lane & 16) >> 3) + ((lane & 3) >> 1)) * 16 + 8 * (lane & 1);
        }
    }
    __device__ __forceinline__ u32x4 k(const unsigned char* tile, int s) const { return *reinterpret_cast<const u32x4*>(tile + kf[s]); }
    __device__ __forceinline__ fl_bf16x8 v(const unsigned char* tile, int s2, int db) const {
        const unsigned char* const at = tile + vf[db] + 16 * s2 * RB;
        const fl_bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) fl_bf16x4*)(at));
        const fl_bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) fl_bf16x4*)(at + 8 * RB));
        return fl_bf16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    }
};
template <int N>
__device__ __forceinline__ void ap_landed() { /* all but the wave's N latest loads have landed, for every wave, and every wave has read what it wanted */
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}
// f while loads set out for to_k, to_v.  The pointers are told apart (restrict): the compiler otherwise takes every transposing LDS read for one that may read what those loads write, and puts a wait for all of them
// in front of it -- a tile then takes what a load takes.  What has to have landed is waited for by ap_landed.
template <class F>
__device__ __forceinline__ void ap_apart(const unsigned char* __restrict__ k, const unsigned char* __restrict__ v, unsigned char* __restrict__ to_k, unsigned char* __restrict__ to_v, F&& f) {
    f(k, v, to_k, to_v);
}

}  // namespace kf
