// Launch parameters of the MLA prolog kernels (internal to the library).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace pto {

constexpr int MLAP_NOPE = 128;       // query channels per head that meet w_uk
constexpr int MLAP_ROPE = 64;        // rotated channels per head and of the key
constexpr int MLAP_KV = 512;         // latent width
constexpr int MLAP_QHEAD = MLAP_NOPE + MLAP_ROPE;
constexpr int MLAP_XBLOCK = 64;      // block length of the fixed-order sums over the hidden axis
constexpr int MLAP_XGROUP = 8;       // block sums per group (one workgroup of the first kernel)
constexpr int MLAP_MAX_XGROUPS = 32; // h <= 32 * 8 * 64 = 16384
constexpr int MLAP_MIN_QLORA = 512;  // (512, 1024 or 1536)
constexpr int MLAP_MAX_QLORA = 1536;
constexpr int QPROJ_KSPLIT_HOST = 4; // partial sums of the int8 projection (prolog_common.h: QPROJ_KSPLIT)
constexpr int MLAP_XTOK = 8;         // tokens per job of the first and of the last kernel
constexpr int MLAP_MFMA_MIN_TOKENS = 9;    // from here on the first launch sums on the matrix cores unless absorb_exact (the fixed-order
                                           // form works on 8 tokens at a time and its cost grows with every 8 tokens)
constexpr int MLAP_UNSPLIT_MIN_TOKENS = 64;   // with absorb_exact the projection still runs unsplit from here on
// ranges of the hidden axis (partial sums per token) of the matrix-core form, at most (what a launch takes: mlap_launch_front);
// the workspace is sized for it
constexpr int MLAP_XM_MAX_SPLITS = 14;

// rows [T, q_lora + 576] of partial sums over the hidden axis the workspace holds: the group sums of the
// fixed-order form, or the ranges of the matrix-core form where that may run
inline int mlap_xpart_rows(const int h, const int T)
{
    const int nblk = h / MLAP_XBLOCK;
    const int groups = (nblk + MLAP_XGROUP - 1) / MLAP_XGROUP;
    const int splits = T >= MLAP_MFMA_MIN_TOKENS ? (nblk < MLAP_XM_MAX_SPLITS ? nblk : MLAP_XM_MAX_SPLITS) : 0;
    return groups > splits ? groups : splits;
}

struct MlapParams {
    const uint16_t *x;            // [T, h] bf16
    const uint16_t *w_dq;         // [h, q_lora] bf16
    const int8_t *w_uqqr;         // [q_lora, n_heads*192] int8
    const float *w_qb_scale;      // [n_heads*192]
    const uint16_t *w_uk;         // [n_heads, 128, 512] bf16
    const uint16_t *w_dkvkr;      // [h, 576] bf16
    const uint16_t *gamma_cq;     // [q_lora] bf16
    const uint16_t *gamma_ckv;    // [512] bf16
    const uint16_t *cos;          // [T, 64] bf16
    const uint16_t *sin;          // [T, 64] bf16
    const long long *cache_index; // [T]
    int8_t *kv_cache;             // [cache_rows, 512]
    uint16_t *kr_cache;           // [cache_rows, 64] bf16
    float *k_scale_cache;         // [cache_rows, 4]
    int8_t *q_norm;               // [T, q_lora]         written, then read by the projection
    float *q_norm_scale;          // [T]
    uint16_t *q_nope;             // [T, n_heads, 512] bf16
    uint16_t *q_rope;             // [T, n_heads, 64] bf16
    float *xpart;                 // workspace [ceil(h/512), T, q_lora + 576]
    int32_t *qpart;               // workspace [4, T, n_heads*192]
    long long cache_rows;
    int T, h, q_lora, n_heads;
    float eps_cq, eps_ckv;
    int absorb_exact;             // 1: the product with w_uk as fixed-order fp32 sums (bit-reproducible against the
                                  // sequential statement); 0: on the matrix cores (bf16 x bf16 exact, fp32 sums in the
                                  // cores' own order: differs in the last bit of some results), and from
                                  // MLAP_MFMA_MIN_TOKENS tokens on the sums over the hidden axis as well
};

// Work of the lightning-indexer prolog that the decode form's launches can carry along (the fused operator): its
// sums over the hidden axis have the same fixed order as this prolog's and its int8 projection reads the same
// q_norm, so wk rides as one more column slab of the first launch, w_proj shares the slab of w_dkv_kr's 64 rope
// columns, and the projection's jobs follow this prolog's in the third launch.
struct MlapRider {
    const uint16_t *wk;      // [h, 128] bf16
    const uint16_t *w_proj;  // [h, 64] bf16
    float *xpart;            // group sums [ceil(h/512), T, 192]: wk's columns, then w_proj's
    const int8_t *w_qb;      // [q_lora, 128 * q_slabs] int8
    int32_t *qpart;          // partial sums [4, T, 128 * q_slabs]
    int q_slabs;
};

// whether the first launch sums on the matrix cores
__host__ __device__ inline bool mlap_prefill_forms(const MlapParams &p) { return p.T >= MLAP_MFMA_MIN_TOKENS && !p.absorb_exact; }
// unless every sum is to keep its fixed order the projection and the last stage are one launch (prolog_small.h up to
// PROLOG_SMALL_TOKENS tokens, prolog_prefill.h beyond)
constexpr int PROLOG_SMALL_TOKENS = 32;
// Heads 2m and 2m + 1 are workgroups of the same XCD, eight apart: a head's rows of w_uq_qr are 192 bytes, a pair's three cache
// lines, the middle one of which they share.  (With neighbours on different XCDs every such line crossed into two L2s, 81 MB
// read for 67 MB of weights; fused prolog: 1 token 33.4 us per pass, now 32.5, 8 tokens 34.4 and 33.8, 16: 39.6 and 39.2.)
__host__ __device__ inline int prolog_small_head(const int wg, const int n_heads)
{
    return (n_heads & 15) == 0 ? 2 * (8 * (wg >> 4) + (wg & 7)) + ((wg >> 3) & 1) : wg;
}
__host__ __device__ inline bool mlap_fused_projection(const MlapParams &p) { return !p.absorb_exact; }
// partial sums per output the int8 projection leaves where it is a launch of its own (absorb_exact): 1 = unsplit (de-quantised
// bf16), else QPROJ_KSPLIT_HOST int32 partials
__host__ __device__ inline int mlap_qsplits(const MlapParams &p) { return p.T >= MLAP_UNSPLIT_MIN_TOKENS ? 1 : QPROJ_KSPLIT_HOST; }
// whether the launches of `p` take a rider at all: the decode forms only
inline bool mlap_takes_rider(const MlapParams &p) { return !mlap_prefill_forms(p) && p.T < MLAP_UNSPLIT_MIN_TOKENS; }

hipError_t mlap_launch(const MlapParams &p, hipStream_t stream);
// all launches but the last (which unless absorb_exact holds the projection too), and the number of workgroups of the last with
// absorb_exact (for the fused operator's last launch)
// lip_rider (prefill forms only): the indexer prolog whose fixed-order sums over the hidden axis (left as group sums:
// LipParams::x_in_groups) ride in this operator's first launch
struct LipParams;
hipError_t mlap_launch_front(const MlapParams &p, hipStream_t stream, const MlapRider *rider = nullptr, const LipParams *lip_rider = nullptr);
int mlap_finish_wgs(const MlapParams &p);
// the last launch alone
hipError_t mlap_launch_finish(const MlapParams &p, hipStream_t stream);
// projections and last stages of both prologs, either of which may be absent (prolog_fused.hip)
hipError_t prolog_prefill_launch(const MlapParams *pm, const LipParams *pl, hipStream_t stream);

}  // namespace pto
