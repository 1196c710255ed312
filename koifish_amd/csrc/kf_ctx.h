// kf_ctx.h -- the context object behind the C ABI and the argument-check plumbing shared by the files that define ABI entries.
#pragma once
#include <hip/hip_runtime.h>

#include <vector>

#include "../../include/kf_abi.h"

struct kf_ctx {
    int device;
    hipStream_t stream;
    bool own_stream;
    bool capturing;
    float* amax_val; /* per-workgroup partial maxima for kf_lm_head when the caller passes no scratch */
    int* amax_idx;
    int canonical;    /* 1: the decode kernels sum in the canonical order of oracle/kf_oracle.c sections 4c / 6 (bit-exact against the oracle; the default); 0: v_dot2c / fp32 forms */
    void* scratch;    /* caller-owned workspace of kf_linear (kf_set_scratch): AWQ slice partials, or a weight dequantised to bf16 */
    size_t scratch_bytes;
    // resident GetDataX copies for token batches (kf_set_dequant_arena): caller-owned memory, filled on first use, keyed by the data pointers and shapes of the matrices a route
    // multiplies in one launch and the form they are laid out in (DEQ_STACK: back to back; DEQ_ILV: gate | up interleaved in blocks of 16 rows).  A descriptor of a matrix's
    // first rows has the matrix's pointer, but the rows behind its own lie elsewhere in a set: another key.
    struct DeqCopy {
        const void* key[3];
        int rows[3], cols, form;
        size_t off;
        DeqCopy(int n_w, const kf_weight* const* w, int form_, size_t off_) : cols(w[0]->ne1), form(form_), off(off_) {
            for (int i = 0; i < 3; i++) key[i] = i < n_w ? w[i]->data : nullptr, rows[i] = i < n_w ? w[i]->ne0 : 0;
        }
        bool of(int n_w, const kf_weight* const* w, int form_) const {
            bool same = form == form_;
            for (int i = 0; i < 3; i++) same = same && key[i] == (i < n_w ? w[i]->data : nullptr) && (i >= n_w || (rows[i] == w[i]->ne0 && cols == w[i]->ne1));
            return same;
        }
    };
    void* arena;
    size_t arena_bytes, arena_used;
    std::vector<DeqCopy> copies;
    // bf16 copies of one layer's matrices for the calls between kf_layer_copies and kf_layer_copies_end, at the front of the scratch (call_used bytes of it)
    std::vector<DeqCopy> call;
    size_t call_used;
    bool call_live() const { return !call.empty() && !capturing; } /* a captured launch is replayed after the copies are gone: it does without them */
    char* scratch_tail() const { return scratch ? (char*)scratch + call_used : nullptr; } /* what the copies leave: 256-byte steps */
    size_t scratch_left() const { return scratch_bytes > call_used ? scratch_bytes - call_used : 0; }
    /* the split-K slots of the tile kernels lie at the scratch's END, whether or not copies leave room to lend them now: their flags stay where they were as long as nothing is written there (scratch_written) */
    void* slots_at(size_t bytes) const { return scratch && scratch_bytes >= bytes + 256 ? (void*)(((uintptr_t)scratch + scratch_bytes - bytes) & ~(uintptr_t)255) : nullptr; }
    void* scratch_end(size_t bytes) const { return scratch_left() >= bytes + 256 ? slots_at(bytes) : nullptr; }
};
enum { DEQ_STACK = 0, DEQ_ILV = 1 };

namespace kf {
int abi_fail(int code, const char* fmt, ...); /* records the text kf_last_error() returns, gives `code` back (kf_abi.hip) */
}

#define HIPCHK(expr)                                                                                   \
    do {                                                                                               \
        hipError_t e_ = (expr);                                                                        \
        if (e_ != hipSuccess) return kf::abi_fail(KF_HIP_CHECK, "%s: %s (%s:%d)", #expr, hipGetErrorString(e_), __FILE__, __LINE__); \
    } while (0)
#define CHKCTX(c) \
    if (!(c)) return kf::abi_fail(KF_INVALID_ARGS, "%s: null kf_ctx", __func__)
#define RET(code) \
    do {          \
        int c_ = (code); \
        if (c_ != KF_OK) return kf::abi_fail(c_, "%s failed with %d", __func__, c_); \
        return KF_OK;    \
    } while (0)

static inline bool al16(const void* p) { return (((uintptr_t)p) & 15) == 0; }
