// The last launch of both prologs for more than 32 tokens, projection included: a head's int8 up-projection is finished where it is
// made -- de-quantised out of the accumulators, rotated, and taken through the product with w_uk (attention query) or the
// Hadamard matrix and quantised (indexer query) -- instead of going to memory as bf16 for a launch of its own.
// Included by prolog_fused.hip after prolog_finish.h.
//
// Both bodies are one workgroup of four waves per (head, tile of tokens), two workgroups to a compute unit, or of eight per (two
// heads, tile).  The projection walks the whole reduction axis in chunks of 64 rows (LDS-DMA, v_mfma_i32_32x32x32_i8 as in
// prolog_common.h), the weights in a ring of three chunks, the tokens in two buffers.  The token tiles of a head run on one XCD,
// which reads its weights once.
// Measured with parts left out (4096 tokens, attention query, one / two heads to a workgroup): in all 297 / 274 us, chunk loop 141 / 133,
// of it requests and LDS reads 97 / 73; stores of q_nope 80 (6.7 TB/s), the rest of what follows the loop 78.  The parts add up: all
// workgroups are in the same one at a time, and workgroups of either query taken in turn, or half of them started 30 us
// late, change nothing at 4096 tokens and cost 8 % at 1000.  In the loop the matrix cores are busy 64 % of the clocks, at the
// 1.77 GHz that is left then.
// LDS-DMA out of the L2 runs at 31-36 TB/s where every cache line it touches is taken whole and at half of that in half lines:
// a workgroup of 256 tokens and one head has room for 64 bytes of a token row at a time only, the others take 128.
// As two launches with bf16 between them, as before, 1000 tokens took 281 us per pass, now 177 to 195; 4096: 906 and 652 to 700.
#pragma once
#include "prolog_finish.h"

#pragma clang fp contract(off)

namespace pto {
namespace {

constexpr int PF_KC = 64;                              // rows of the reduction axis per chunk
// Tokens in LDS, XC chunks of the reduction axis per request: rows of 128 bytes with 16-byte piece q of row t at
// q ^ ((t >> 1) & 7), or of 64 with q at q ^ ((t >> 2) & 3).
template <int XC> constexpr int PF_XPITCH = XC * PF_KC;
template <int XC> __device__ __forceinline__ int pf_xswizzle(const int t) { return XC == 2 ? (t >> 1) & 7 : (t >> 2) & 3; }

// The N token requests of a wave per XC chunks: 1 KiB each, request r of the tile the rows from r * 1024 / PF_XPITCH on
template <int XC, int N>
struct PfTokens {
    const int8_t *src[N];
    __device__ __forceinline__ PfTokens(const int8_t *q_norm, const int q_lora, const int T, const int t0, const int r0, const int l)
    {
        constexpr int PIECES = PF_XPITCH<XC> / 16;
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const int tl = (64 / PIECES) * (r0 + j) + l / PIECES;
            const int t = t0 + tl < T ? t0 + tl : T - 1;              // rows past the end repeat the last token
            src[j] = q_norm + (size_t)t * q_lora + 16 * ((l % PIECES) ^ pf_xswizzle<XC>(tl));
        }
    }
    __device__ __forceinline__ void request(const int s, const uint32_t dst) const
    {
#pragma unroll
        for (int j = 0; j < N; ++j) dma16(src[j] + s * PF_XPITCH<XC>, dst + 1024 * j);
    }
};

// ------------------------------------------------------------------------------------------------ attention query
// Wave (wc, wt) of the 4 * HB holds columns 96*wc .. +95 of the HB heads' 192 each x TB blocks of 32 tokens (3 * TB accumulators).
// Row r of a chunk of weights lies at 192 * HB * r, its 32-byte block b at b ^ ((r >> 2) & 1), two heads: b ^ ((r >> 1) & 3): the
// eight consecutive rows of a transposing read then fall on different banks.
// Then the rope channels meet in LDS as rows, are rotated and leave; then the tile's 128 nope channels become an operand
// [head][token][256 bytes] in LDS, 16-byte piece q at q ^ (t & 15), with the channels of every 16 in the order the halves of a wave
// want them (0-3 8-11 | 4-7 12-15); each wave takes 128 output columns of a head with its part of w_uk in registers:
// lane n's columns are 4n .. 4n+3, so a row leaves as 256 contiguous bytes.
template <int TB> constexpr int PFA_TOK = 64 * TB;
template <int XC, int TB> constexpr int PFA_X = PFA_TOK<TB> * PF_XPITCH<XC>;
template <int HB> constexpr int PFA_WPITCH = HB * MLAP_QHEAD;
template <int HB> constexpr int PFA_W = PF_KC * PFA_WPITCH<HB>;
constexpr int PFA_RPITCH = 144;                        // bytes between rope rows
template <int TB, int HB> constexpr int PFA_Q = HB * PFA_TOK<TB> * MLAP_NOPE * 2;
template <int XC, int TB, int HB> constexpr int PFA_LOOP_LDS = 2 * PFA_X<XC, TB> + 3 * PFA_W<HB>;
template <int XC, int TB, int HB> constexpr int PFA_LDS = PFA_LOOP_LDS<XC, TB, HB> > PFA_Q<TB, HB> ? PFA_LOOP_LDS<XC, TB, HB> : PFA_Q<TB, HB>;
static_assert(PFA_RPITCH <= MLAP_NOPE * 2, "the rope rows fit where the nope operand goes");

// Lane (row, e) of the rope rows at `rows` rotates pairs 4e .. 4e+3 of token t (channels 2j, 2j+1 are the partners j, 32 + j) and
// stores them; rows of tokens past the end are read and dropped.
__device__ __forceinline__ void pfa_rotate_rows(const MlapParams &p, const uint8_t *rows, const int row, const int t, const int head, const int e)
{
    const size_t tt = t < p.T ? t : p.T - 1;
    const u32x4 x = *reinterpret_cast<const u32x4 *>(rows + row * PFA_RPITCH + 16 * e);
    const u32x2 c0 = *reinterpret_cast<const u32x2_a2 *>(p.cos + tt * MLAP_ROPE + 4 * e), c1 = *reinterpret_cast<const u32x2_a2 *>(p.cos + tt * MLAP_ROPE + 32 + 4 * e);
    const u32x2 s0 = *reinterpret_cast<const u32x2_a2 *>(p.sin + tt * MLAP_ROPE + 4 * e), s1 = *reinterpret_cast<const u32x2_a2 *>(p.sin + tt * MLAP_ROPE + 32 + 4 * e);
    float r0[4], r1[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        auto at = [&](const u32x2 &q) { return __uint_as_float((j & 1) ? q[j >> 1] & 0xffff0000u : q[j >> 1] << 16); };
        const float v0 = __uint_as_float(x[j] << 16), v1 = __uint_as_float(x[j] & 0xffff0000u);
        r0[j] = __builtin_fmaf(v0, at(c0), (-v1) * at(s0));                   // products exact: one rounding
        r1[j] = __builtin_fmaf(v1, at(c1), v0 * at(s1));
    }
    if (t < p.T) {
        uint16_t *out = p.q_rope + (tt * p.n_heads + head) * MLAP_ROPE + 4 * e;
        *reinterpret_cast<u32x2_a2 *>(out) = u32x2{pack_bf16x2(r0[0], r0[1]), pack_bf16x2(r0[2], r0[3])};
        *reinterpret_cast<u32x2_a2 *>(out + 32) = u32x2{pack_bf16x2(r1[0], r1[1]), pack_bf16x2(r1[2], r1[3])};
    }
}

template <int XC, int TB, int HB>
__device__ __forceinline__ void mlap_prefill_body(const MlapParams &p, const int job, uint8_t *lds)
{
    const int l = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int half = l >> 5;
    const int wc = w & (2 * HB - 1), wt = w / (2 * HB);
    const int ncols = p.n_heads * MLAP_QHEAD;
    const int ttiles = (p.T + PFA_TOK<TB> - 1) / PFA_TOK<TB>;
    const int head0 = (job / ttiles) * HB;             // (their number is even)
    const int t0 = (job % ttiles) * PFA_TOK<TB>;
    const uint32_t base = (uint32_t)(uintptr_t)(lds_byte_t *)lds;
    auto token = [&](const int tl) { return t0 + tl < p.T ? t0 + tl : p.T - 1; };
    float ts[TB];
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) ts[tb] = p.q_norm_scale[token(32 * (TB * wt + tb) + (l & 31))];

    i32x16 acc[TB][3];
#pragma unroll
    for (int tb = 0; tb < TB; ++tb)
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[tb][i][r] = 0;
    {
        constexpr int XR = XC * TB / HB, WR = 3;
        constexpr int PPR = PFA_WPITCH<HB> / 16;     // 16-byte pieces of a weight row
        const PfTokens<XC, XR> xt(p.q_norm, p.q_lora, p.T, t0, XR * w, l);
        const int8_t *wsrc[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const int piece = 64 * (3 * w + j) + l, row = piece / PPR, pos = piece % PPR;
            wsrc[j] = p.w_uqqr + (size_t)row * ncols + head0 * MLAP_QHEAD + 16 * (pos ^ (2 * (HB == 1 ? (row >> 2) & 1 : (row >> 1) & 3)));
        }
        const size_t wstep = (size_t)PF_KC * ncols;
        uint32_t aoff[3];
#pragma unroll
        for (int i = 0; i < 3; ++i)
            aoff[i] = 2 * PFA_X<XC, TB> + (16 * half + ((l & 15) >> 1)) * PFA_WPITCH<HB> + 32 * ((3 * wc + i) ^ (HB == 1 ? (l >> 3) & 1 : (l >> 2) & 3)) + 16 * ((l >> 4) & 1) + 8 * (l & 1);
        const uint32_t boff = (32 * TB * wt + (l & 31)) * PF_XPITCH<XC>;
        typedef int v2i __attribute__((ext_vector_type(2)));
        staged_chunks<XC, XR, WR>(
            p.q_lora / PF_KC, [&](const int s, const int b) { xt.request(s, base + b * PFA_X<XC, TB> + 1024 * XR * w); },
            [&](const int c, const int slot) {
#pragma unroll
                for (int j = 0; j < 3; ++j) dma16(wsrc[j] + c * wstep, base + 2 * PFA_X<XC, TB> + slot * PFA_W<HB> + 1024 * (3 * w + j));
            },
            [&](const int odd, const int xb, const int slot) {
                const uint8_t *wp = lds + slot * PFA_W<HB>, *xp = lds + xb * PFA_X<XC, TB> + boff;
#pragma unroll
                for (int s = 0; s < PF_KC / 32; ++s) {
                    i32x4 a[3];
#pragma unroll
                    for (int i = 0; i < 3; ++i) {
                        const uint8_t *ap = wp + aoff[i] + s * 32 * PFA_WPITCH<HB>;
                        const v2i lo = __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) v2i *)(lds_byte_t *)ap);
                        const v2i hi = __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) v2i *)(lds_byte_t *)(ap + 8 * PFA_WPITCH<HB>));
                        a[i] = i32x4{lo[0], lo[1], hi[0], hi[1]};
                    }
#pragma unroll
                    for (int tb = 0; tb < TB; ++tb) {
                        const i32x4 b = *reinterpret_cast<const i32x4 *>(xp + tb * 32 * PF_XPITCH<XC> + 16 * ((4 * odd + 2 * s + half) ^ pf_xswizzle<XC>(l & 31)));
#pragma unroll
                        for (int i = 0; i < 3; ++i) acc[tb][i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[i], b, acc[tb][i], 0, 0, 0);
                    }
                }
            });
    }
    // registers 4*rg .. 4*rg+3 of product i: columns 96*wc + 32*i + 8*rg + 4*half .. +3 (of the head: 96*part) of token l % 32 of the block
    const int hh = wc >> 1, part = wc & 1;
    u32x2 pk[TB][3][4];
    {
        const float *cs = p.w_qb_scale + (head0 + hh) * MLAP_QHEAD + 96 * part + 4 * half;
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int rg = 0; rg < 4; ++rg) {
                const f32x4 c = *reinterpret_cast<const f32x4 *>(cs + 32 * i + 8 * rg);
#pragma unroll
                for (int tb = 0; tb < TB; ++tb) {
                    float f[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) f[j] = __fmul_rn(__fmul_rn((float)acc[tb][i][4 * rg + j], ts[tb]), c[j]);
                    pk[tb][i][rg] = u32x2{pack_bf16x2(f[0], f[1]), pack_bf16x2(f[2], f[3])};
                }
            }
    }
    {
        if (part == 1) {
#pragma unroll
            for (int tb = 0; tb < TB; ++tb)
#pragma unroll
                for (int i = 1; i < 3; ++i)
#pragma unroll
                    for (int rg = 0; rg < 4; ++rg)
                        *reinterpret_cast<u32x2 *>(lds + (PFA_TOK<TB> * hh + 32 * (TB * wt + tb) + (l & 31)) * PFA_RPITCH + 2 * (32 * (i - 1) + 8 * rg + 4 * half)) = pk[tb][i][rg];
        }
        __syncthreads();
        // lane (row, e) rotates pairs 4e .. 4e+3 (channels 2j, 2j+1 are the partners j, 32 + j), eight tokens at a time
        const int e = l & 7;
#pragma unroll
        for (int k = 0; k < 2 * TB; ++k) {
            const int row = 8 * (2 * TB * w + k) + (l >> 3);                                         // (a wave's rows are all of one head)
            pfa_rotate_rows(p, lds, row, t0 + row - PFA_TOK<TB> * (w >> 2), head0 + (w >> 2), e);
        }
        __syncthreads();
    }
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) {
        const int tl = 32 * (TB * wt + tb) + (l & 31);
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            if (part == 1 && i > 0) break;
            const int blk = 3 * part + i;                // 32 nope channels
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const u32x4 o = {pk[tb][i][2 * k][0], pk[tb][i][2 * k][1], pk[tb][i][2 * k + 1][0], pk[tb][i][2 * k + 1][1]};
                *reinterpret_cast<u32x4 *>(lds + (PFA_TOK<TB> * hh + tl) * 256 + 16 * ((2 * (2 * blk + k) + half) ^ (l & 15))) = o;
            }
        }
    }
    // w_uk of head w / 4, columns 128*(w % 4) + 4n .. +3, every row: rows 16*ks + 4*half + {0..3, 8..11} are this half's part of step ks
    const int head = head0 + (w >> 2), col = 128 * (w & 3) + 4 * (l & 31);
    bf16x8 wf[MLAP_NOPE / 16][4];
    {
        const uint16_t *src = p.w_uk + (size_t)head * MLAP_NOPE * MLAP_KV + (size_t)(4 * half) * MLAP_KV + col;
#pragma unroll
        for (int ks = 0; ks < MLAP_NOPE / 16; ++ks) {
            u32x2 row[8];
#pragma unroll
            for (int r = 0; r < 8; ++r) row[r] = *reinterpret_cast<const u32x2 *>(src + (size_t)(16 * ks + (r & 3) + 8 * (r >> 2)) * MLAP_KV);
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                u32x4 f;
#pragma unroll
                for (int d = 0; d < 4; ++d)
                    f[d] = __builtin_amdgcn_perm(row[2 * d + 1][c >> 1], row[2 * d][c >> 1], (c & 1) ? 0x07060302u : 0x05040100u);
                wf[ks][c] = __builtin_bit_cast(bf16x8, f);
            }
        }
    }
    __syncthreads();                                   // the operand of the second product is complete
    uint16_t *dst = p.q_nope + (size_t)head * MLAP_KV + col;
    const uint8_t *operand = lds + (w >> 2) * (PFA_TOK<TB> * 256);
#pragma unroll 1
    for (int blk = 0; blk < 2 * TB; ++blk) {
        const int tb0 = t0 + 32 * blk;
        if (tb0 >= p.T) break;                         // uniform
        f32x16 c[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) c[j][r] = 0.f;
#pragma unroll
        for (int ks = 0; ks < MLAP_NOPE / 16; ++ks) {
            const bf16x8 a = *reinterpret_cast<const bf16x8 *>(operand + (32 * blk + (l & 31)) * 256 + 16 * ((2 * ks + half) ^ (l & 15)));
#pragma unroll
            for (int j = 0; j < 4; ++j) c[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, wf[ks][j], c[j], 0, 0, 0);
        }
        // lane n holds columns 4n .. 4n+3 of tokens 8*(r/4) + 4*half + r%4
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int t = tb0 + 8 * (r >> 2) + 4 * half + (r & 3);
            if (t < p.T) *reinterpret_cast<u32x2_a2 *>(dst + (size_t)t * p.n_heads * MLAP_KV) = u32x2{pack_bf16x2(c[0][r], c[1][r]), pack_bf16x2(c[2][r], c[3][r])};
        }
    }
}

// ------------------------------------------------------------------------------------------------- indexer query
// A wave holds all 128 columns of its head x TB blocks of 32 tokens, so the rotation partners (channels i and i + 32) are in
// one lane and the rotated row is the Hadamard product's operand as it stands in the registers (the k-order of the transposing
// read is the accumulators' row order).  Weights: [head][64][128] per chunk, as q_build_a_tr reads them.  The matrix is
// requested once the chunk buffers are free: row r at 256 * r, 16-byte piece q at q ^ 4*(r & 3).
// FIXED (one tile of at most 64 tokens, the first two waves' blocks): the rotated rows meet in LDS and all four waves take the
// Hadamard sums in their fixed order, a block of 32 rows at a time.  (Fused prolog, 33
// tokens: 40.7 us per pass, 48: 42.4, 63: 43.7; in the cores' own order, which the interface does not allow below 64 tokens, 40.5,
// 42.4 and 43.2.)
template <int TB> constexpr int PFI_TOK = 128 * TB;
template <int XC, int TB> constexpr int PFI_X = PFI_TOK<TB> * PF_XPITCH<XC>;
constexpr int PFI_W = PF_KC * LIP_DIM;
constexpr int PFI_HAD = LIP_DIM * LIP_DIM * 2;
template <int XC, int TB, int HB> constexpr int PFI_LOOP_LDS = 2 * PFI_X<XC, TB> + 3 * HB * PFI_W;
constexpr int PFI_FIXED_TOK = 64;
constexpr int PFI_FIXED_LDS = PFI_HAD + PFI_FIXED_TOK * HB_PITCH * 2 + HB_SCRATCH;
template <int HB> constexpr int PFI_OUT_LDS = PFI_HAD + 4 * HB * 32 * QFP_OPITCH;
template <int HB> constexpr int PFI_FIN_LDS = PFI_FIXED_LDS > PFI_OUT_LDS<HB> ? PFI_FIXED_LDS : PFI_OUT_LDS<HB>;
template <int XC, int TB, int HB> constexpr int PFI_LDS = PFI_LOOP_LDS<XC, TB, HB> > PFI_FIN_LDS<HB> ? PFI_LOOP_LDS<XC, TB, HB> : PFI_FIN_LDS<HB>;

template <int XC, int TB, int HB, bool FIXED>
__device__ __forceinline__ void lip_prefill_body(const LipParams &p, const int job, uint8_t *lds)
{
    const int l = threadIdx.x & 63;
    const int w8 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int w = w8 & 3, hh = w8 >> 2;                // wave of the head's four
    const int half = l >> 5;
    const int ncols = p.n_heads * LIP_DIM;
    const int ttiles = (p.T + PFI_TOK<TB> - 1) / PFI_TOK<TB>;
    const bool exists = (job / ttiles) * HB + hh < p.n_heads;      // (of an odd number of heads the last workgroups take one twice)
    const int head = (job / ttiles) * HB + (exists ? hh : 0);
    const int t0 = (job % ttiles) * PFI_TOK<TB>;
    const uint32_t base = (uint32_t)(uintptr_t)(lds_byte_t *)lds;
    auto token = [&](const int tl) { return t0 + tl < p.T ? t0 + tl : p.T - 1; };

    i32x16 acc[TB][4];
#pragma unroll
    for (int tb = 0; tb < TB; ++tb)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[tb][i][r] = 0;
    {
        constexpr int XR = 2 * XC * TB / HB;
        const PfTokens<XC, XR> xt(p.q_norm, p.q_lora, p.T, t0, XR * w8, l);
        const int8_t *wsrc[2];
#pragma unroll
        for (int j = 0; j < 2; ++j)
            wsrc[j] = p.w_qb + (size_t)(8 * (2 * w + j) + (l >> 3)) * ncols + head * LIP_DIM + 16 * ((l & 7) ^ q_tr_piece_swizzle(l >> 3));
        const size_t wstep = (size_t)PF_KC * ncols;
        const uint32_t boff = (32 * TB * w + (l & 31)) * PF_XPITCH<XC>;
        staged_chunks<XC, XR, 2>(
            p.q_lora / PF_KC, [&](const int s, const int b) { xt.request(s, base + b * PFI_X<XC, TB> + 1024 * XR * w8); },
            [&](const int c, const int slot) {
#pragma unroll
                for (int j = 0; j < 2; ++j) dma16(wsrc[j] + c * wstep, base + 2 * PFI_X<XC, TB> + (slot * HB + hh) * PFI_W + 1024 * (2 * w + j));
            },
            [&](const int odd, const int xb, const int slot) {
                const uint8_t *wp = lds + 2 * PFI_X<XC, TB> + (slot * HB + hh) * PFI_W, *xp = lds + xb * PFI_X<XC, TB> + boff;
#pragma unroll
                for (int s = 0; s < PF_KC / 32; ++s) {
                    i32x4 a[4];
                    q_build_a_tr(wp, s, l, a);
#pragma unroll
                    for (int tb = 0; tb < TB; ++tb) {
                        const i32x4 b = *reinterpret_cast<const i32x4 *>(xp + tb * 32 * PF_XPITCH<XC> + 16 * ((4 * odd + 2 * s + half) ^ pf_xswizzle<XC>(l & 31)));
#pragma unroll
                        for (int i = 0; i < 4; ++i) acc[tb][i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[i], b, acc[tb][i], 0, 0, 0);
                    }
                }
            });
    }
    {
        const uint16_t *src = p.hq + (size_t)(4 * (8 / HB * w8) + (l >> 4)) * LIP_DIM + 8 * ((l & 15) ^ (4 * ((l >> 4) & 3)));
#pragma unroll 1
        for (int j = 0; j < 8 / HB; ++j) dma16(src + (size_t)4 * j * LIP_DIM, base + 1024 * (8 / HB * w8 + j));
    }
    const float *cs = p.w_qb_scale + head * LIP_DIM + 4 * half;
    bf16x8 bq[TB][LIP_DIM / 16];
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) {
        const size_t tt = token(32 * (TB * w + tb) + (l & 31));
        const float ts = p.q_norm_scale[tt];
        float v[4][16];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int rg = 0; rg < 4; ++rg) {
                const f32x4 c = *reinterpret_cast<const f32x4 *>(cs + 32 * i + 8 * rg);
#pragma unroll
                for (int j = 0; j < 4; ++j) v[i][4 * rg + j] = bf16_round_f32(__fmul_rn(__fmul_rn((float)acc[tb][i][4 * rg + j], ts), c[j]));
            }
#pragma unroll
        for (int rg = 0; rg < 4; ++rg) {
            const uint16_t *cp = p.cos + tt * LIP_ROPE + 8 * rg + 4 * half, *sp = p.sin + tt * LIP_ROPE + 8 * rg + 4 * half;
            const u32x2 c0 = *reinterpret_cast<const u32x2 *>(cp), c1 = *reinterpret_cast<const u32x2 *>(cp + 32);
            const u32x2 s0 = *reinterpret_cast<const u32x2 *>(sp), s1 = *reinterpret_cast<const u32x2 *>(sp + 32);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                auto at = [&](const u32x2 &q) { return __uint_as_float((j & 1) ? q[j >> 1] & 0xffff0000u : q[j >> 1] << 16); };
                const float v0 = v[0][4 * rg + j], v1 = v[1][4 * rg + j];
                v[0][4 * rg + j] = __builtin_fmaf(v0, at(c0), (-v1) * at(s0));        // products exact: one rounding (below)
                v[1][4 * rg + j] = __builtin_fmaf(v1, at(c1), v0 * at(s1));
            }
        }
#pragma unroll
        for (int ks = 0; ks < LIP_DIM / 16; ++ks) {
            u32x4 f;
#pragma unroll
            for (int d = 0; d < 4; ++d) f[d] = pack_bf16x2(v[ks >> 1][8 * (ks & 1) + 2 * d], v[ks >> 1][8 * (ks & 1) + 2 * d + 1]);
            bq[tb][ks] = __builtin_bit_cast(bf16x8, f);
        }
    }
    if constexpr (FIXED) {
        static_assert(TB == 1 && HB == 1 && PFI_FIXED_TOK >= LIP_MFMA_MIN_TOKENS, "one tile of two blocks");
        uint16_t *rows = reinterpret_cast<uint16_t *>(lds + PFI_HAD);
        if (32 * w < PFI_FIXED_TOK) {
            // dword d of bq[0][ks]: channels 16*ks + 8*(d / 2) + 4*half + 2*(d % 2), +1 of row 32*w + l % 32
#pragma unroll
            for (int ks = 0; ks < LIP_DIM / 16; ++ks) {
                const u32x4 f = __builtin_bit_cast(u32x4, bq[0][ks]);
                uint16_t *dst = rows + (32 * w + (l & 31)) * HB_PITCH + 16 * ks + 4 * half;
                *reinterpret_cast<u32x2 *>(dst) = u32x2{f[0], f[1]};
                *reinterpret_cast<u32x2 *>(dst + 8) = u32x2{f[2], f[3]};
            }
        }
        VM_WAIT(0);
        __syncthreads();                               // the rotated rows are complete, the matrix is staged
#pragma unroll 1
        for (int r0 = 0; r0 < p.T; r0 += 32) {
            if (r0) __syncthreads();                   // the last block's rows have left
            lip_fixed_rows(rows + r0 * HB_PITCH, reinterpret_cast<const uint16_t *>(lds), lds + PFI_HAD + PFI_FIXED_TOK * HB_PITCH * 2,
                           p.q_int8 + (size_t)r0 * p.n_heads * LIP_DIM, p.q_scale + (size_t)r0 * p.n_heads, p.n_heads, head, p.T - r0, w, l);
        }
        return;
    }
    VM_WAIT(0);
    __syncthreads();                                   // the matrix is staged
    uint8_t *mine = lds + PFI_HAD + w8 * (32 * QFP_OPITCH);
    const int arow = 4 * half + ((l & 15) >> 2);
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) {
        f32x16 c[4];
#pragma unroll
        for (int cb = 0; cb < 4; ++cb)
#pragma unroll
            for (int r = 0; r < 16; ++r) c[cb][r] = 0.f;
#pragma unroll
        for (int ks = 0; ks < LIP_DIM / 16; ++ks)
#pragma unroll
            for (int cb = 0; cb < 4; ++cb) {
                const int piece = 4 * cb + 2 * ((l >> 4) & 1) + ((l & 3) >> 1);
                const uint16_t *ap = reinterpret_cast<const uint16_t *>(lds + (16 * ks + arow) * 256 + 16 * (piece ^ (4 * ((l & 15) >> 2))) + 8 * (l & 1));
                const s16x4 a0 = lds_read_tr16(ap), a1 = lds_read_tr16(ap + 8 * 128);
                const s16x8 a = __builtin_shufflevector(a0, a1, 0, 1, 2, 3, 4, 5, 6, 7);
                c[cb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), bq[tb][ks], c[cb], 0, 0, 0);
            }
        const int tb0 = t0 + 32 * (TB * w + tb);
        const float deq = lip_quant_rows(c, mine, l);
        if (exists && l < 32 && tb0 + l < p.T) p.q_scale[(size_t)(tb0 + l) * p.n_heads + head] = (uint16_t)(pack_f16x2(deq, 0.f) & 0xffffu);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int r = 8 * k + (l >> 3);
            const u32x4 v = *reinterpret_cast<const u32x4 *>(mine + r * QFP_OPITCH + 16 * (l & 7));
            if (exists && tb0 + r < p.T) *reinterpret_cast<u32x4 *>(p.q_int8 + ((size_t)(tb0 + r) * p.n_heads + head) * LIP_DIM + 16 * (l & 7)) = v;
        }
    }
}

}  // namespace
}  // namespace pto
