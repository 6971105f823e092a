// MLA prolog for gfx950, the variant with bf16 down-projections, an int8 query up-projection and an
// int8 latent cache with four fp32 scales per token: from a decode batch of hidden states it produces
// the absorbed query (nope and rope parts), the int8 normalised query latent with its scale (input of
// the indexer prolog), and writes the new latent / rope / scale rows of the paged caches.
//
// Arithmetic (reference golden: examples/models/deepseek_v32_exp/deepseekv32_mla_prolog_quant.py:137-282;
// operator graph: examples/models/deepseek_v32_exp/mla_prolog_quant_impl.py:502-707).  Every fp32 sum
// has a fixed order (all products are bf16 x bf16, exact in fp32): sums over the hidden axis in blocks of
// 64 ascending, eight block sums ascending into a group sum, group sums ascending; the RMS sums as a
// balanced tree over the 128 channels of a slab, slab sums ascending; the 128-term sums against w_uk
// ascending.  In that form only the exact integer projection runs on the matrix cores; the caller may let the
// sums against w_uk, and from MLAP_MFMA_MIN_TOKENS tokens on the sums over the hidden axis, run there as well
// (MlapParams::absorb_exact = 0: the same exact products in the cores' own summation order).
//
// Three launches -- sums over the hidden axis, latents, and one for the projection and everything behind it -- or, with every
// sum in its fixed order (absorb_exact), four:
//   mlap_xlinear_kernel  x . [w_dq | w_dkv_kr] (xlinear_fixed.h): one workgroup of eight waves per (slab of 128
//                        columns, group of 512 hidden rows, 8 tokens); each wave takes a 64-row block (staged by
//                        LDS-DMA, hidden states widened to fp32 in LDS), block sums meet in LDS and are
//                        chained into the group sum.  Below MLAP_MFMA_MIN_TOKENS tokens, and with absorb_exact.
//   mlap_xlinear_mfma_kernel   the same sums on the matrix cores (xlinear_mfma.h): per workgroup a 128-column slab x
//                        tokens x a range of the hidden axis, v_mfma_f32_32x32x16_bf16 with the row-major weight chunk as
//                        the transposed operand.  The launch's first workgroups (beyond 128 tokens its last) take the 64
//                        rope columns of w_dkv_kr in their fixed order instead (the rotated key allows no outlier under the
//                        reference's acceptance rule), and the indexer prolog's sums with them in the fused operator.
//   mlap_mid_kernel      per token: group sums chained, bf16, RMS norm (one wave per slab), per-token
//                        int8 quantisation of the query latent; RMS norm and per-slab quantisation of
//                        the key latent, rope of the key, scatter into the caches.
//   mlap_mid_prefill_kernel    the same as a wave per token and latent (64 tokens and more)
//   prolog_small_kernel, prolog_prefill_kernel (prolog_fused.hip)   a head's int8 projection, rope and product with w_uk
// With absorb_exact instead of the last:
//   qproj_kernel         int8 projection of the query latent (shared job code: LDS-DMA tile,
//                        transposing 8-bit LDS reads, v_mfma_i32_32x32x32_i8), partial sums per quarter; from
//                        MLAP_UNSPLIT_MIN_TOKENS tokens on qproj_prefill_kernel, qproj_prefill256_kernel (prolog_common.h):
//                        unsplit, a workgroup per tile over the whole reduction axis, results de-quantised.
//   mlap_finish_kernel   per (head, half of the 512 output columns, 8 tokens): partial sums added and
//                        de-quantised, rope part rotated and stored, nope part times the head's w_uk
//                        slice (staged in LDS by LDS-DMA), one output column per lane.
// For the fused operator the fixed-order first launch and qproj_kernel carry the lightning-indexer prolog's first stage along
// (MlapRider in mlap_kernels.h: its hidden-axis sums have this prolog's fixed order, its projection this one's q_norm).
#include <cstring>

#include "mlap_kernels.h"
#include "prolog_common.h"
#include "prolog_finish.h"
#include "lip_xjob.h"
#include "xlinear_fixed.h"
#include "xlinear_mfma.h"

#pragma clang fp contract(off)

namespace pto {
namespace {

static_assert(QPROJ_KSPLIT == QPROJ_KSPLIT_HOST, "workspace sizing and kernels disagree");

static_assert(XL_BLOCK == MLAP_XBLOCK && XL_GROUP == MLAP_XGROUP && XL_TOK == MLAP_XTOK, "workspace sizing and kernels disagree");
constexpr int RIDER_XCOLS = 192;     // columns of a row of the rider's group sums: wk's 128, then w_proj's 64

// Fixed-order sums over the hidden axis (xlinear_fixed.h).  Column slabs: 0 .. q_lora/128 - 1 of w_dq, then four
// slabs of w_dkv_kr's latent part and one half slab (64 columns) of its rope part.
// With a rider (mlap_kernels.h) there is one slab more, wk's 128 columns, and the rope slab's upper half is w_proj.
__global__ __launch_bounds__(64 * XL_WAVES) void mlap_xlinear_kernel(const MlapParams p, const int nslabs, const int ngroups, const MlapRider rd)
{
    __shared__ __attribute__((aligned(16))) uint8_t smem[XL_LDS];
    const int slab = blockIdx.x % nslabs;
    const int g = (blockIdx.x / nslabs) % ngroups;
    const int t0 = (blockIdx.x / nslabs / ngroups) * XL_TOK;
    const int qslabs = p.q_lora / 128;
    const int nc = p.q_lora + MLAP_KV + MLAP_ROPE;
    const bool isq = slab < qslabs;
    XlSlab sl;
    if (slab == qslabs + 5) {
        sl.w = reinterpret_cast<const uint8_t *>(rd.wk);
        sl.pitch = 256;
        sl.wbytes = 256;
        sl.out = rd.xpart + (size_t)g * p.T * RIDER_XCOLS;
        sl.out_pitch = RIDER_XCOLS;
    } else {
        sl.w = isq ? reinterpret_cast<const uint8_t *>(p.w_dq) + slab * 256 : reinterpret_cast<const uint8_t *>(p.w_dkvkr) + (slab - qslabs) * 256;
        sl.pitch = (isq ? p.q_lora : MLAP_KV + MLAP_ROPE) * 2;
        sl.wbytes = (!isq && slab - qslabs == 4) ? 128 : 256;
        sl.out = p.xpart + (size_t)g * p.T * nc + slab * 128;
        sl.out_pitch = nc;
        if (sl.wbytes == 128 && rd.w_proj != nullptr) {
            sl.wbytes = 256;
            sl.w_hi = reinterpret_cast<const uint8_t *>(rd.w_proj);
            sl.pitch_hi = 128;
            sl.out_hi = rd.xpart + (size_t)g * p.T * RIDER_XCOLS + 128;
            sl.out_pitch_hi = RIDER_XCOLS;
        }
    }
    xl_body(sl, p.x, p.T, p.h, g, t0, smem);
}

// ---------------------------------------------------------------------------------------------
// Prefill form of the first launch: the same product on the matrix cores (xlinear_mfma.h), for MLAP_MFMA_MIN_TOKENS tokens and more
// when the caller has not asked for the fixed-order sums.  workgroup = (slab of 128 columns of [w_dq | w_dkv_kr],
// one of nsplit ranges of the hidden axis, 128 tokens); the 64 rope columns are a narrow slab of their own.
static_assert(XM_KC == MLAP_XBLOCK, "the workspace is sized in chunks of the hidden axis");

// Further workgroups take sums in their fixed order (xlinear_fixed.h, the matrix-core form of the
// sequential sums), 64 columns each: the rope columns of w_dkv_kr at every size -- the reference's acceptance rule allows
// the rotated key no outlier at all (deepseekv32_mla_prolog_quant.py:688: atol 1e-4, rtol 2^-7 per element, ratio 0), and
// a sum that lands next to a bf16 rounding boundary in another order moves a small rotated value by more than that --
// and, in the fused prolog, the indexer prolog's wk and w_proj.  They are short and follow the long workgroups of the
// other slabs, so they fill the launch's last round; two workgroups fit a compute unit.  (1000 tokens: 69 us here and 79
// in a launch of the indexer's own before they shared it.)  Up to 64 tokens all workgroups run at once and these are the longer
// ones beside another workgroup, so they start first (fused prolog, 32 tokens: 37.4 us per pass, at the end of the launch 39.3;
// 200 tokens 84.4, at the end 70.3).
// TB: at most 32 * TB tokens (xm_small_body), 0 for tiles of 128 tokens x 128 columns (xm_body), XM_BIG for 128 x 256 (xb_body).
constexpr int XM_BIG = 8;
template <int TB> constexpr int XM_FORM_LDS = TB == 0 ? XM_LDS : (TB == XM_BIG ? XB_LDS : XMS_LDS<TB == 1 ? 1 : 2>);
template <int TB> constexpr int XM_KERNEL_LDS = XM_FORM_LDS<TB> > XF_LDS ? XM_FORM_LDS<TB> : XF_LDS;
static_assert(2 * XM_KERNEL_LDS<0> <= 160 * 1024 && 2 * XM_KERNEL_LDS<2> <= 160 * 1024 && 2 * XM_KERNEL_LDS<XM_BIG> <= 160 * 1024, "two workgroups share a compute unit");
template <int TB>
__global__ __launch_bounds__(256, 2) void mlap_xlinear_mfma_kernel(const MlapParams p, const int nslabs, const int nsplit, const int own_wgs,
                                                                const XfGrid fg, const LipParams lip)
{
    __shared__ __attribute__((aligned(16))) uint8_t smem[XM_KERNEL_LDS<TB>];
    // Up to 128 tokens the fixed-order sums, the longer chains, start first and the launch is one round (65 to 128 tokens, last / first:
    // fused prolog, 72 tokens 48.1 / 46.9 us per pass, 100 52.3 / 50.4, 128 54.6 / 52.8, MLA prolog alone 128 52.4 / 50.4); beyond, where
    // they fill more than the first places, they come last (first: 160 tokens 62.6 / 63.5, 300 90.3 / 96.1, 1000 187.9 / 203.3).
    constexpr bool FIXED_FIRST = TB != XM_BIG;
    const int nfixed = (int)gridDim.x - own_wgs;                   // a multiple of eight, as own_wgs: the XCDs go round alike
    const int fixed = (int)blockIdx.x - (FIXED_FIRST ? 0 : own_wgs), bid = (int)blockIdx.x - (FIXED_FIRST ? nfixed : 0);
    if (FIXED_FIRST ? fixed < nfixed : fixed >= 0) {
        const XfJob j = xf_job(fixed, fg, p.T);
        if (j.g < 0) return;
        XlSlab sl;
        if (j.set == 0) {
            const int nc = p.q_lora + MLAP_KV + MLAP_ROPE;
            sl.w = reinterpret_cast<const uint8_t *>(p.w_dkvkr) + MLAP_KV * 2;
            sl.pitch = (MLAP_KV + MLAP_ROPE) * 2;
            sl.wbytes = MLAP_ROPE * 2;
            sl.out = p.xpart + (size_t)j.g * p.T * nc + p.q_lora + MLAP_KV;
            sl.out_pitch = nc;
        } else {
            sl = lip_xf_slab(lip, j.set - 1, j.g);
        }
        xf_body(sl, p.x, p.T, p.h, j.g, j.t0, fg.run, smem);
        return;
    }
    if constexpr (TB == XM_BIG) {
        // every XCD takes a run of the jobs in the order (range of h, token tile, slab): a range's weights and the hidden
        // states of a tile or two cross into its L2 once, chunk by chunk, as the run's workgroups walk the range together
        const int ttiles = (p.T + XB_TOK - 1) / XB_TOK;
        const int idx = (bid & 7) * (own_wgs >> 3) + (bid >> 3);
        if (idx >= nslabs * ttiles * nsplit) return;
        const int slab = idx % nslabs, sp = (idx / nslabs) / ttiles, t0 = ((idx / nslabs) % ttiles) * XB_TOK;
        const int qslabs = p.q_lora / XB_COLS;
        const int nc = p.q_lora + MLAP_KV + MLAP_ROPE;
        XmSlab sl;
        sl.w = slab < qslabs ? reinterpret_cast<const uint8_t *>(p.w_dq) + slab * (2 * XB_COLS)
                             : reinterpret_cast<const uint8_t *>(p.w_dkvkr) + (slab - qslabs) * (2 * XB_COLS);
        sl.pitch = (slab < qslabs ? p.q_lora : MLAP_KV + MLAP_ROPE) * 2;
        sl.pieces = 2 * XB_COLS / 16;
        sl.out = p.xpart + (size_t)sp * p.T * nc + slab * XB_COLS;
        sl.out_pitch = nc;
        const int nchunks = p.h / XM_KC;
        xb_body(sl, p.x, p.T, p.h, t0, (int)((long long)sp * nchunks / nsplit), (int)((long long)(sp + 1) * nchunks / nsplit), smem);
        return;
    } else {
    // Workgroups go round the eight XCDs, each with an L2 of its own, and the working set (hidden states + weights)
    // is several times one L2: the jobs of a slab (its ranges of h x token tiles) all run on XCD slab % 8, so a slab's
    // weights cross into one L2 only and every XCD reads the hidden states once for its two or so slabs.  The slabs
    // left over when their number is no multiple of eight are dealt out job by job.
    const int per_slab = nsplit * ((p.T + XM_TOK - 1) / XM_TOK);
    const int xcd = bid & 7, j = bid >> 3;
    const int full = nslabs >> 3;
    int slab, rem;
    if (j < full * per_slab) {
        slab = xcd + 8 * (j / per_slab);
        rem = j % per_slab;
    } else {
        const int e = (j - full * per_slab) * 8 + xcd;
        if (e >= (nslabs & 7) * per_slab) return;      // the whole workgroup leaves, before any barrier
        slab = 8 * full + e / per_slab;
        rem = e % per_slab;
    }
    const int sp = rem % nsplit;
    const int t0 = (rem / nsplit) * XM_TOK;
    const int qslabs = p.q_lora / 128;
    const int nc = p.q_lora + MLAP_KV + MLAP_ROPE;
    const bool isq = slab < qslabs;
    XmSlab sl;
    sl.w = isq ? reinterpret_cast<const uint8_t *>(p.w_dq) + slab * 256 : reinterpret_cast<const uint8_t *>(p.w_dkvkr) + (slab - qslabs) * 256;
    sl.pitch = (isq ? p.q_lora : MLAP_KV + MLAP_ROPE) * 2;
    sl.pieces = 16;                // (the narrow one, the rope columns, is not among them)
    sl.out = p.xpart + (size_t)sp * p.T * nc + slab * 128;
    sl.out_pitch = nc;
    const int nchunks = p.h / XM_KC;
    const int c_begin = (int)((long long)sp * nchunks / nsplit), c_end = (int)((long long)(sp + 1) * nchunks / nsplit);
    if constexpr (TB == 0) xm_body(sl, p.x, p.T, p.h, t0, c_begin, c_end, smem);
    else xm_small_body<TB>(sl, p.x, p.T, p.h, c_begin, c_end, smem);
    }
}

// ---------------------------------------------------------------------------------------------
constexpr int MID_WAVES = MLAP_MAX_QLORA / 128;   // 12

// sum over the wave's 128 values of rn(rn(v*v) * coef) as a balanced tree over neighbours
__device__ __forceinline__ float slab_square_sum(const float v0, const float v1, const float coef)
{
    return pair_tree_sum(__fmul_rn(__fmul_rn(v0, v0), coef), __fmul_rn(__fmul_rn(v1, v1), coef));
}

// Up to PROLOG_SMALL_TOKENS tokens the latents occupy 2 T compute units for the length of a few memory latencies, and the memory
// idles.  Further workgroups of the launch, one per head, ask for the first rows of the head's projection weights, which the last
// launch, bound by drawing weights, then finds in the L2 of the XCD it reads them on (workgroups go round the XCDs in both
// launches, prolog_small_head).  The values are dropped.  512 rows are what arrives before the latents are done: fused prolog, 0 /
// 256 / 512 / 768 rows: 8 tokens 34.1 / 33.2 / 32.4 / 32.1 us per pass, 16: 35.3 / 34.3 / 33.4 / 33.6, 32: 38.1 / 37.2 / 36.5 / 36.6;
// MLA prolog alone, 0 / 512: 8 tokens 27.9 / 27.4, 32: 31.1 / 29.9.  Into the L2 of another XCD, so that only the memory-side cache
// helps, 8 tokens gain 0.3 us instead of 1.7.  (The launch for more than 32 tokens has two workgroups per compute unit to hide the
// same latencies, and gained nothing at 48 and 200.)
constexpr int MLAP_AHEAD_ROWS = 512;
__device__ __forceinline__ void mlap_ask_ahead(const MlapParams &p, const int wg)
{
    if (wg < 0 || wg >= p.n_heads) return;
    const int8_t *src = p.w_uqqr + (size_t)prolog_small_head(wg, p.n_heads) * MLAP_QHEAD;
    constexpr int PIECES = MLAP_QHEAD / 64, N = MLAP_AHEAD_ROWS * PIECES / (64 * MID_WAVES);      // 64 bytes per lane
    static_assert(N * 64 * MID_WAVES == MLAP_AHEAD_ROWS * PIECES && MLAP_AHEAD_ROWS <= MLAP_MIN_QLORA, "whole passes over rows that exist");
    int v[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int piece = 64 * MID_WAVES * i + (int)threadIdx.x, row = piece / PIECES;
        v[i] = *reinterpret_cast<const int *>(src + (size_t)row * p.n_heads * MLAP_QHEAD + 64 * (piece - PIECES * row));
    }
#pragma unroll
    for (int i = 0; i < N; ++i) asm volatile("" ::"v"(v[i]));
}
// workgroups of the latents' launch in front of those (a multiple of eight: the XCDs go round the same way)
__host__ __device__ inline int mid_own_wgs(const int T) { return (2 * T + 7) / 8 * 8; }

// Workgroup 2t: the query latent of token t (one wave per slab of 128 channels).  Workgroup 2t+1: its
// key latent (waves 0..3) and key rope part (wave 4).
// ngroups partial sums over the hidden axis per column, ngroups_rope for the 64 rope columns (which keep the fixed-order
// form's groups when the other columns come from the matrix cores).
__global__ __launch_bounds__(64 * MID_WAVES) void mlap_mid_kernel(const MlapParams p, const int ngroups_other, const int ngroups_rope)
{
    __shared__ float slabsum[MID_WAVES];
    __shared__ float slabmax[MID_WAVES];
    if ((int)blockIdx.x >= 2 * p.T) return mlap_ask_ahead(p, (int)blockIdx.x - mid_own_wgs(p.T));
    const int l = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int t = blockIdx.x >> 1;
    const bool kvtype = blockIdx.x & 1;
    const int qslabs = p.q_lora / 128;
    const int nc = p.q_lora + MLAP_KV + MLAP_ROPE;
    const int nslab = kvtype ? 4 : qslabs;                               // slabs under the norm
    const bool rope_wave = kvtype && w == 4;
    const bool active = w < nslab || rope_wave;
    const int ngroups = rope_wave ? ngroups_rope : ngroups_other;
    const int col = (kvtype ? p.q_lora : 0) + w * 128 + 2 * (rope_wave ? (l & 31) : l);

    // Everything the chain below needs from memory is requested before the first value is looked at: the
    // cache row, the norm weights, the rotation factors and the group sums, sixteen groups at a time
    // (taken one after the other, the fourteen group loads of a 7168-wide hidden axis alone were fourteen
    // memory latencies).
    const long long dst = kvtype ? p.cache_index[t] : -1;
    uint32_t gm = 0;
    if (w < nslab) gm = reinterpret_cast<const uint32_t *>(kvtype ? p.gamma_ckv : p.gamma_cq)[w * 64 + l];
    uint16_t cs0 = 0, cs1 = 0, sn0 = 0, sn1 = 0;
    if (rope_wave && l < 32) {
        cs0 = p.cos[(size_t)t * MLAP_ROPE + l];
        cs1 = p.cos[(size_t)t * MLAP_ROPE + 32 + l];
        sn0 = p.sin[(size_t)t * MLAP_ROPE + l];
        sn1 = p.sin[(size_t)t * MLAP_ROPE + 32 + l];
    }
    float v0 = 0.f, v1 = 0.f;
    if (active) {
        const float *src = p.xpart + (size_t)t * nc + col;
        for (int g0 = 0; g0 < ngroups; g0 += 16) {
            f32x2 v[16];
#pragma unroll
            for (int g = 0; g < 16; ++g)
                v[g] = *reinterpret_cast<const f32x2 *>(src + (size_t)(g0 + g < ngroups ? g0 + g : ngroups - 1) * p.T * nc);
#pragma unroll
            for (int g = 0; g < 16; ++g) {
                if (g0 + g < ngroups) {
                    v0 = __fadd_rn(v0, v[g][0]);
                    v1 = __fadd_rn(v1, v[g][1]);
                }
            }
        }
        v0 = bf16_round_f32(v0);
        v1 = bf16_round_f32(v1);
    }
    const bool dst_ok = dst >= 0 && dst < p.cache_rows;

    if (rope_wave) {
        // lane l < 32 holds channels 2l and 2l+1, which after the de-interleave are channels l and 32+l:
        // the two partners of one rotation
        if (l < 32) {
            const float c0 = bf16_bits_to_f32(cs0), c1 = bf16_bits_to_f32(cs1);
            const float s0 = bf16_bits_to_f32(sn0), s1 = bf16_bits_to_f32(sn1);
            const float r0 = __builtin_fmaf(v0, c0, (-v1) * s0);      // products exact: one rounding
            const float r1 = __builtin_fmaf(v1, c1, v0 * s1);
            if (dst_ok) {
                p.kr_cache[(size_t)dst * MLAP_ROPE + l] = (uint16_t)(pack_bf16x2(r0, 0.f) & 0xffffu);
                p.kr_cache[(size_t)dst * MLAP_ROPE + 32 + l] = (uint16_t)(pack_bf16x2(r1, 0.f) & 0xffffu);
            }
        }
    }
    const int n = kvtype ? MLAP_KV : p.q_lora;
    if (w < nslab) {
        const float ss = slab_square_sum(v0, v1, (float)(1.0 / (double)n));
        if (l == 0) slabsum[w] = ss;
    }
    __syncthreads();
    float y0 = 0.f, y1 = 0.f;
    if (w < nslab) {
        float s = 0.f;
        for (int j = 0; j < nslab; ++j) s = __fadd_rn(s, slabsum[j]);
        const float d = __builtin_sqrtf(__fadd_rn(s, kvtype ? p.eps_ckv : p.eps_cq));   // correctly rounded (__fsqrt_rn is the 1-ulp hardware root here)
        y0 = bf16_round_f32(__fmul_rn(__fdiv_rn(v0, d), __uint_as_float(gm << 16)));
        y1 = bf16_round_f32(__fmul_rn(__fdiv_rn(v1, d), __uint_as_float(gm & 0xffff0000u)));
        const float m = wave_max_f32(fmaxf(fabsf(y0), fabsf(y1)));
        if (l == 0) slabmax[w] = m;
    }
    __syncthreads();
    if (w < nslab) {
        float amax = slabmax[w];
        if (!kvtype)
            for (int j = 0; j < nslab; ++j) amax = fmaxf(amax, slabmax[j]);
        float deq;
        const uint16_t q = quant_pair_amax(y0, y1, amax, deq);
        if (!kvtype) {
            reinterpret_cast<uint16_t *>(p.q_norm + (size_t)t * p.q_lora)[w * 64 + l] = q;
            if (w == 0 && l == 0) p.q_norm_scale[t] = deq;
        } else if (dst_ok) {
            reinterpret_cast<uint16_t *>(p.kv_cache + (size_t)dst * MLAP_KV)[w * 64 + l] = q;
            if (l == 0) p.k_scale_cache[(size_t)dst * 4 + w] = deq;
        }
    }
}

// The same at prefill sizes, a wave per token and latent (waves 2t: the query latent, 2t + 1: the key latent and key rope):
// no barriers, and the slabs' loads and reductions run side by side in one wave.  (The form above, a workgroup of twelve
// waves per latent that waits for memory once and meets twice, is all latency once the chip has run out of room for more
// workgroups: 1000 tokens 22.0 us.  As long as 512 of them have room it is the faster one: 64 tokens 5.4 us and 9.4, 256: 8.0 and 9.0;
// fused prolog, 64 tokens 43.2 us per pass and 47.1, 128: 54.0 and 57.2, 256: 70.6 and 72.3, but 300: 97.8 and 96.1.)
constexpr int MIDP_WAVES = 4;
constexpr int MIDP_MIN_TOKENS = 257;

// NS slabs of 128 columns at src (lane: columns 2l, 2l + 1 of each): the partial sums added ascending, rounded to bf16
template <int NS>
__device__ __forceinline__ void mid_sum_slabs(const float *src, const int ngroups, const size_t gstride, float (&v)[NS][2])
{
    constexpr int FLY = NS > 4 ? 3 : 8;                // groups in flight
#pragma unroll
    for (int j = 0; j < NS; ++j) v[j][0] = v[j][1] = 0.f;
    for (int g0 = 0; g0 < ngroups; g0 += FLY) {
        f32x2 x[FLY][NS];
#pragma unroll
        for (int g = 0; g < FLY; ++g)
#pragma unroll
            for (int j = 0; j < NS; ++j)
                x[g][j] = *reinterpret_cast<const f32x2 *>(src + (size_t)(g0 + g < ngroups ? g0 + g : ngroups - 1) * gstride + 128 * j);
#pragma unroll
        for (int g = 0; g < FLY; ++g)
            if (g0 + g < ngroups) {
#pragma unroll
                for (int j = 0; j < NS; ++j) {
                    v[j][0] = __fadd_rn(v[j][0], x[g][j][0]);
                    v[j][1] = __fadd_rn(v[j][1], x[g][j][1]);
                }
            }
    }
#pragma unroll
    for (int j = 0; j < NS; ++j) {
        v[j][0] = bf16_round_f32(v[j][0]);
        v[j][1] = bf16_round_f32(v[j][1]);
    }
}
// RMS norm over the NS slabs in place; amax: largest magnitude of each slab
template <int NS>
__device__ __forceinline__ void mid_norm_slabs(float (&v)[NS][2], const uint16_t *gamma, const float eps, const int l, float (&amax)[NS])
{
    constexpr float coef = (float)(1.0 / (double)(NS * 128));
    uint32_t gm[NS];
#pragma unroll
    for (int j = 0; j < NS; ++j) gm[j] = reinterpret_cast<const uint32_t *>(gamma)[64 * j + l];
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < NS; ++j) s = __fadd_rn(s, slab_square_sum(v[j][0], v[j][1], coef));
    const float d = __builtin_sqrtf(__fadd_rn(s, eps));          // correctly rounded
#pragma unroll
    for (int j = 0; j < NS; ++j) {
        v[j][0] = bf16_round_f32(__fmul_rn(__fdiv_rn(v[j][0], d), __uint_as_float(gm[j] << 16)));
        v[j][1] = bf16_round_f32(__fmul_rn(__fdiv_rn(v[j][1], d), __uint_as_float(gm[j] & 0xffff0000u)));
        amax[j] = wave_max_f32(fmaxf(fabsf(v[j][0]), fabsf(v[j][1])));
    }
}

template <int QS>
__global__ __launch_bounds__(64 * MIDP_WAVES) void mlap_mid_prefill_kernel(const MlapParams p, const int ngroups, const int ngroups_rope)
{
    const int l = threadIdx.x & 63;
    const int job = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * MIDP_WAVES + (threadIdx.x >> 6)));
    const int t = job >> 1;
    if (t >= p.T) return;
    const int nc = QS * 128 + MLAP_KV + MLAP_ROPE;
    const size_t gstride = (size_t)p.T * nc;
    const float *row = p.xpart + (size_t)t * nc + 2 * l;
    if ((job & 1) == 0) {
        float v[QS][2], amax[QS];
        mid_sum_slabs<QS>(row, ngroups, gstride, v);
        mid_norm_slabs<QS>(v, p.gamma_cq, p.eps_cq, l, amax);
        float m = amax[0];
#pragma unroll
        for (int j = 1; j < QS; ++j) m = fmaxf(m, amax[j]);
        float deq;
#pragma unroll
        for (int j = 0; j < QS; ++j)
            reinterpret_cast<uint16_t *>(p.q_norm + (size_t)t * p.q_lora)[64 * j + l] = quant_pair_amax(v[j][0], v[j][1], m, deq);
        if (l == 0) p.q_norm_scale[t] = deq;
        return;
    }
    const long long dst = p.cache_index[t];
    const bool dst_ok = dst >= 0 && dst < p.cache_rows;
    float r[1][2], v[4][2], amax[4];
    mid_sum_slabs<1>(row + QS * 128 + MLAP_KV - 2 * (l & 32), ngroups_rope, gstride, r);         // lanes 32.. repeat lanes 0..
    mid_sum_slabs<4>(row + QS * 128, ngroups, gstride, v);
    mid_norm_slabs<4>(v, p.gamma_ckv, p.eps_ckv, l, amax);
    if (!dst_ok) return;
    if (l < 32) {
        // channels 2l, 2l + 1 become channels l, 32 + l: the two partners of one rotation
        const uint16_t *c = p.cos + (size_t)t * MLAP_ROPE + l, *s = p.sin + (size_t)t * MLAP_ROPE + l;
        const float r0 = __builtin_fmaf(r[0][0], bf16_bits_to_f32(c[0]), (-r[0][1]) * bf16_bits_to_f32(s[0]));      // products exact: one rounding
        const float r1 = __builtin_fmaf(r[0][1], bf16_bits_to_f32(c[32]), r[0][0] * bf16_bits_to_f32(s[32]));
        p.kr_cache[(size_t)dst * MLAP_ROPE + l] = (uint16_t)(pack_bf16x2(r0, 0.f) & 0xffffu);
        p.kr_cache[(size_t)dst * MLAP_ROPE + 32 + l] = (uint16_t)(pack_bf16x2(r1, 0.f) & 0xffffu);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        float deq;
        reinterpret_cast<uint16_t *>(p.kv_cache + (size_t)dst * MLAP_KV)[64 * j + l] = quant_pair_amax(v[j][0], v[j][1], amax[j], deq);
        if (l == 0) p.k_scale_cache[(size_t)dst * 4 + j] = deq;
    }
}

// ---------------------------------------------------------------------------------------------
// One workgroup (two waves, one half of a quarter tile each) walks the jobs blockIdx.x, + gridDim.x, ...:
// the tile of the next job is requested into the other buffer before the current one is consumed, so the
// weights stream without a gap between jobs.  The wave pair adds its accumulators through one of two
// parking areas, alternating, with one barrier per job.
template <int HS>
constexpr int qproj_lds_bytes()
{
    return 4 * HS * (32 * 128 + 1024) + 2 * LIN_RED_BYTES;
}

// Jobs [0, njobs_a) belong to projection pa, jobs [njobs_a, njobs) to pb (same q_norm and reduction axis: the rider's).
template <int HS>
__global__ __launch_bounds__(128) void qproj_kernel(const QProj pa, const int njobs_a, const QProj pb, const int njobs)
{
    constexpr int BUF = HS * (32 * 128 + 1024);
    constexpr int NREQ = HS * 5;                       // requests of one job per wave
    __shared__ __attribute__((aligned(16))) uint8_t smem[qproj_lds_bytes<HS>()];
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l = threadIdx.x & 63;
    uint8_t *bufs = smem + w * 2 * BUF;
    uint8_t *park = smem + 4 * BUF;
    int job = blockIdx.x;
    const auto issue = [&](uint8_t *region, const int j) {
        if (j < njobs_a) q_issue<HS>(pa, region, j, w);
        else q_issue<HS>(pb, region, j - njobs_a, w);
    };
    if (job < njobs) issue(bufs, job);
    for (int k = 0; job < njobs; job += gridDim.x, ++k) {
        const int next = job + gridDim.x;
        if (next < njobs) {
            issue(bufs + ((k + 1) & 1) * BUF, next);
            VM_WAIT(NREQ);
        } else {
            VM_WAIT(0);
        }
        i32x16 acc[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][r] = 0;
        const uint8_t *region = bufs + (k & 1) * BUF;
#pragma unroll
        for (int s = 0; s < HS; ++s) q_step<HS>(region, s, l, acc);
        uint8_t *pk = park + (k & 1) * LIN_RED_BYTES;
        if (w == 1) q_pair_park(pk, l, acc);
        __syncthreads();
        if (w == 0) {
            if (job < njobs_a) q_pair_store_from(pa, pk, job, l, acc);
            else q_pair_store_from(pb, pk, job - njobs_a, l, acc);
        }
    }
}

// TB: token blocks per tile (prolog_common.h).
template <int TB>
__global__ __launch_bounds__(256) void qproj_prefill_kernel(const QProj p, const int njobs)
{
    __shared__ __attribute__((aligned(16))) uint8_t lds[QPF_LDS];
    q_prefill_body<TB>(p, q_prefill_job_of((int)blockIdx.x, njobs), lds);
}

__global__ __launch_bounds__(512) void qproj_prefill256_kernel(const QProj p, const int njobs)
{
    __shared__ __attribute__((aligned(16))) uint8_t lds[QP2_LDS];
    q_prefill256_body(p, q_prefill_job_of((int)blockIdx.x, njobs), lds);
}

// ---------------------------------------------------------------------------------------------
// Last launch: prolog_finish.h.
__global__ __launch_bounds__(256) void mlap_finish_kernel(const MlapParams p)
{
    __shared__ __attribute__((aligned(16))) uint8_t lds[MLAP_FIN_LDS];
    mlap_finish_body(p, (int)blockIdx.x, lds);
}

}  // namespace

hipError_t mlap_launch_finish(const MlapParams &p, hipStream_t stream)
{
    if (mlap_fused_projection(p)) return prolog_prefill_launch(&p, nullptr, stream);
    hipLaunchKernelGGL(mlap_finish_kernel, dim3((unsigned)mlap_finish_wgs(p)), dim3(256), 0, stream, p);
    return hipGetLastError();
}

int mlap_finish_wgs(const MlapParams &p) { return p.n_heads * 2 * ((p.T + MLAP_XTOK - 1) / MLAP_XTOK); }

hipError_t mlap_launch_front(const MlapParams &p, hipStream_t stream, const MlapRider *rider, const LipParams *lip_rider)
{
    const int nblk = p.h / MLAP_XBLOCK;
    int ngroups = (nblk + MLAP_XGROUP - 1) / MLAP_XGROUP;
    const int ngroups_fixed = ngroups;
    const int nslabs = p.q_lora / 128 + 5;
    if (rider != nullptr && !mlap_takes_rider(p)) return hipErrorInvalidValue;
    if (lip_rider != nullptr && !mlap_takes_lip_rider(p)) return hipErrorInvalidValue;
    LipParams lip;
    std::memset(&lip, 0, sizeof lip);
    if (lip_rider != nullptr) lip = *lip_rider;
    const MlapRider rd = rider != nullptr ? *rider : MlapRider{nullptr, nullptr, nullptr, nullptr, nullptr, 0};
    if (mlap_prefill_forms(p)) {
        // prefill sizes: the sums over the hidden axis on the matrix cores, in ranges of the hidden axis (partial sums per token)
        const int nchunks = p.h / XM_KC;
        const int ttiles = (p.T + XM_TOK - 1) / XM_TOK;
        const int cus = cu_count();
        if (cus <= 0) return hipErrorNoDevice;
        // every slab but the last, the rope columns, which keep their fixed-order sums
        const bool big = p.T > XM_TOK;
        // As many ranges as make two workgroups of 128 x 128 or one of 128 x 256 per compute unit (the other half of each is for the
        // fixed-order sums), MLAP_XM_MAX_SPLITS = 14 at most: that many up to 256 tokens, so that a token's latents do not depend
        // on how many tokens the launch has.  Fewer ranges are longer fp32 chains, further from the 64-bit sums (relative error
        // over 2048 columns of 7168 products: 14 ranges 1.44e-7, 12 1.52e-7, 10 1.63e-7, 8 1.80e-7), and one int8 value of a
        // latent that falls the other way is 9 % of its token's indexer query.  They would leave the fixed-order sums more room
        // beside them: fused prolog, 14 / 12 ranges: 129 tokens 60.0 / 60.5 us per pass, 192: 71.1 / 67.5; 14 / 10: 256 76.9 / 71.4
        // (alone 61.1 / 62.5); 14 / 12: 100 52.4 / 53.1 (alone 49.9 / 47.4).  At 256 tokens the fourteen as two to a workgroup, one
        // after the other, take 84.0.
        // Up to 64 tokens two workgroups share a compute unit, and the fixed-order sums start first (one per compute unit, those
        // last, so a second round: 9 tokens 39.1, in this form 32.2; 32: 42.5, 36.4; 48: 47.3, 43.3; 64: 52.9, 44.8, the last launch
        // in tiles of 128 tokens; two ranges per workgroup: 9 tokens 33.5, 32: 37.0, 48: 47.1, 64: 52.5).
        const int mslabs = (nslabs - 1) / (big ? XB_COLS / 128 : 1);
        ngroups = big ? cus / (mslabs * ttiles) : 2 * cus / nslabs;
        ngroups = ngroups < 1 ? 1 : ngroups;
        ngroups = ngroups > MLAP_XM_MAX_SPLITS ? MLAP_XM_MAX_SPLITS : ngroups;
        ngroups = ngroups > nchunks ? nchunks : ngroups;
        const int per_slab = ngroups * ttiles;
        const int wgs = big ? 8 * ((mslabs * per_slab + 7) / 8) : 8 * ((mslabs >> 3) * per_slab + ((mslabs & 7) * per_slab + 7) / 8);   // the kernel's XCD-wise job order
        const int sets = 1 + (lip_rider != nullptr ? LIP_XF_SETS : 0);
        const XfGrid fg = {sets, ngroups_fixed, xf_run(sets * ngroups_fixed, p.T, 2 * cus - wgs)};
        const dim3 g((unsigned)(wgs + xf_jobs(fg, p.T)));
#define XM_LAUNCH(TBV) hipLaunchKernelGGL(mlap_xlinear_mfma_kernel<TBV>, g, dim3(256), 0, stream, p, mslabs, ngroups, wgs, fg, lip)
        if (p.T <= 32) XM_LAUNCH(1);
        else if (p.T <= 64) XM_LAUNCH(2);
        else if (big) XM_LAUNCH(XM_BIG);
        else XM_LAUNCH(0);
#undef XM_LAUNCH
    } else {
        const int tgroups = (p.T + MLAP_XTOK - 1) / MLAP_XTOK;
        const int xslabs = nslabs + (rider != nullptr ? 1 : 0);
        hipLaunchKernelGGL(mlap_xlinear_kernel, dim3((unsigned)(xslabs * ngroups * tgroups)), dim3(64 * XL_WAVES), 0, stream, p, xslabs, ngroups, rd);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (p.T >= MIDP_MIN_TOKENS) {
        const dim3 g((unsigned)((2 * p.T + MIDP_WAVES - 1) / MIDP_WAVES)), b(64 * MIDP_WAVES);
        switch (p.q_lora / 128) {
        case 4: hipLaunchKernelGGL(mlap_mid_prefill_kernel<4>, g, b, 0, stream, p, ngroups, ngroups_fixed); break;
        case 8: hipLaunchKernelGGL(mlap_mid_prefill_kernel<8>, g, b, 0, stream, p, ngroups, ngroups_fixed); break;
        case 12: hipLaunchKernelGGL(mlap_mid_prefill_kernel<12>, g, b, 0, stream, p, ngroups, ngroups_fixed); break;
        default: return hipErrorInvalidValue;
        }
    } else {
        const bool ahead = mlap_fused_projection(p) && p.T <= PROLOG_SMALL_TOKENS;
        const dim3 g((unsigned)(ahead ? mid_own_wgs(p.T) + p.n_heads : 2 * p.T));
        hipLaunchKernelGGL(mlap_mid_kernel, g, dim3(64 * MID_WAVES), 0, stream, p, ngroups, ngroups_fixed);
    }
    e = hipGetLastError();
    if (e != hipSuccess || mlap_fused_projection(p)) return e;
    const QProj qp = {p.q_norm, p.w_uqqr, p.qpart, p.T, p.q_lora, p.n_heads * MLAP_QHEAD / 128, p.q_norm_scale, p.w_qb_scale};
    if (mlap_qsplits(p) == 1) {
        if (p.q_lora % (32 * QPF_STEPS)) return hipErrorInvalidValue;
        const int cus = cu_count();
        if (cus <= 0) return hipErrorNoDevice;
        const int njobs256 = q_prefill256_jobs(qp);
        if (4 * njobs256 >= 3 * cus) {                 // enough 256 x 256 tiles to fill the chip
            hipLaunchKernelGGL(qproj_prefill256_kernel, dim3((unsigned)njobs256), dim3(512), 0, stream, qp, njobs256);
            return hipGetLastError();
        }
        const int njobs = q_prefill_jobs(qp);
        const dim3 g((unsigned)njobs), b(256);
        if (q_prefill_token_blocks(p.T) == 2) hipLaunchKernelGGL(qproj_prefill_kernel<2>, g, b, 0, stream, qp, njobs);
        else hipLaunchKernelGGL(qproj_prefill_kernel<4>, g, b, 0, stream, qp, njobs);
        return hipGetLastError();
    }
    const int qjobs_a = qp.nslabs * QPROJ_KSPLIT * ((p.T + 31) / 32);
    const QProj qr = {p.q_norm, rd.w_qb, rd.qpart, p.T, p.q_lora, rd.q_slabs, p.q_norm_scale, nullptr};
    const int qjobs = qjobs_a + qr.nslabs * QPROJ_KSPLIT * ((p.T + 31) / 32);
    // as many workgroups as fit at once (by their LDS), every one with the same number of jobs where possible
    const int steps = p.q_lora / QPROJ_KSPLIT / 32;
    const int lds = steps == 12 ? qproj_lds_bytes<6>() : (steps == 8 ? qproj_lds_bytes<4>() : qproj_lds_bytes<2>());
    const int cus = cu_count();
    if (cus <= 0) return hipErrorNoDevice;
    const int slots = cus * (160 * 1024 / lds);
    const int rounds = (qjobs + slots - 1) / slots;
    const dim3 qgrid((unsigned)((qjobs + rounds - 1) / rounds));
    switch (steps) {
    case 4: hipLaunchKernelGGL(qproj_kernel<2>, qgrid, dim3(128), 0, stream, qp, qjobs_a, qr, qjobs); break;
    case 8: hipLaunchKernelGGL(qproj_kernel<4>, qgrid, dim3(128), 0, stream, qp, qjobs_a, qr, qjobs); break;
    case 12: hipLaunchKernelGGL(qproj_kernel<6>, qgrid, dim3(128), 0, stream, qp, qjobs_a, qr, qjobs); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t mlap_launch(const MlapParams &p, hipStream_t stream)
{
    hipError_t e = mlap_launch_front(p, stream);
    if (e != hipSuccess) return e;
    return mlap_launch_finish(p, stream);
}

}  // namespace pto
