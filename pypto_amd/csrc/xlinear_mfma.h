// Sums over the hidden axis on the matrix cores, for 9 tokens and more: x [T, h] bf16 times a slab of up
// to 128 columns of a row-major bf16 weight matrix, as partial sums over a range of the hidden axis.  Shared by the
// MLA prolog (w_dq, w_dkv_kr) and the lightning-indexer prolog (wk, w_proj); included after prolog_common.h.
//
// All products are exact in fp32 (bf16 x bf16); the sums are taken in the cores' own order, so the results may
// differ from the fixed-order sums of the decode kernels in the last bit.
//   workgroup = (slab, range of the hidden axis, 128 tokens), four waves: wave (wc, wt) holds columns
//   64*wc .. +63 x tokens 64*wt .. +63 as four 32x32 accumulators of
//   O^T[column][token] = sum_k W^T[column][k] x^T[k][token]
//   A = W^T: the slab's rows are row-major [k][columns], so the operand is read from LDS with the transposing
//   ds_read_b64_tr_b16; B = x^T: lane (token, half) holds 8 consecutive hidden states of its token.
//   Chunks of 64 hidden rows travel by LDS-DMA into two buffers (16 KiB of the slab + 16 KiB of hidden states
//   each), the next chunk under the products of the current one.  16-byte piece q of slab row r sits at piece q ^ 4*(r & 3),
//   piece q of token row t at q ^ ((t >> 1) & 7): the four rows of a transposing read and the 32 token rows of an
//   operand read then spread over all banks.  A slab narrower than 128 columns (8 * pieces) is staged unswizzled
//   by the lanes whose pieces exist; the columns past its end hold whatever the buffer held and are not stored.
#pragma once
#include "prolog_common.h"

namespace pto {
namespace {

constexpr int XM_TOK = 128;                      // tokens per workgroup
constexpr int XM_KC = 64;                        // hidden rows per chunk
constexpr int XM_W_BYTES = XM_KC * 256;          // slab rows are staged 256 bytes apart
constexpr int XM_X_BYTES = XM_TOK * XM_KC * 2;
constexpr int XM_BUF = XM_W_BYTES + XM_X_BYTES;
constexpr int XM_LDS = 2 * XM_BUF;
constexpr int XM_SPITCH = 272;                   // bytes between the rows of a wave's output staging area (32 tokens x 64 columns fp32)

struct XmSlab {
    const uint8_t *w;     // column 0 of the slab in row 0 of the weight matrix
    int pitch;            // bytes between rows of the weight matrix
    int pieces;           // 16-byte pieces of a row that belong to the slab: 16, or fewer for a narrow one
    float *out;           // partial sums of this range: out[t * out_pitch + column of the slab]
    int out_pitch;
};

// chunks [c_begin, c_end) of the hidden axis, tokens t0 .. t0 + 127 (rows past T - 1 repeat it and are not stored)
__device__ __forceinline__ void xm_body(const XmSlab &sl, const uint16_t *x, const int T, const int h, const int t0, const int c_begin,
                                        const int c_end, uint8_t *smem)
{
    const int l = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wc = w & 1, wt = w >> 1;
    const bool narrow = sl.pieces < 16;
    const bool idle = sl.pieces <= 8 && wc == 1;                   // no column of this wave's half exists
    const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_byte_t *)smem;

    // this wave's eight requests of a chunk: four of the slab (four rows each), four of the hidden states (eight
    // token rows each).  Their addresses are made once, for chunk 0; a chunk further on is a uniform number of bytes
    // further on (the loop then spends two additions per request instead of rebuilding the addresses).
    const int wrow = l >> 4, wpos = l & 15;
    const uint32_t woff = (uint32_t)(wrow * sl.pitch + 16 * (narrow ? (wpos < sl.pieces ? wpos : 0) : (wpos ^ (4 * wrow))));
    const uint64_t wmask = narrow ? ((1ull << sl.pieces) - 1) * 0x0001000100010001ull : ~0ull;
    const int xrow = l >> 3, xpos = l & 7;
    const uint8_t *wreq[4], *xreq[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int req = 4 * w + j;
        wreq[j] = sl.w + (size_t)(4 * req) * sl.pitch + woff;
        const int tl = 8 * req + xrow;                              // token row inside the workgroup's 128
        int t = t0 + tl;
        t = t < T ? t : T - 1;
        xreq[j] = reinterpret_cast<const uint8_t *>(x) + (size_t)t * h * 2 + 16 * (xpos ^ ((tl >> 1) & 7));
    }
    const size_t wstep = (size_t)XM_KC * sl.pitch;
    auto request_chunk = [&](const int c, const int buf) {
        const uint32_t dst = lds0 + (uint32_t)(buf * XM_BUF);
#pragma unroll
        for (int j = 0; j < 4; ++j) dma16_lanes(wreq[j] + (size_t)c * wstep, dst + 1024u * (4 * w + j), wmask);
#pragma unroll
        for (int j = 0; j < 4; ++j) dma16(xreq[j] + (size_t)c * (XM_KC * 2), dst + XM_W_BYTES + 1024u * (4 * w + j));
    };

    f32x16 acc[2][2];
#pragma unroll
    for (int cb = 0; cb < 2; ++cb)
#pragma unroll
        for (int tb = 0; tb < 2; ++tb)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[cb][tb][r] = 0.f;

    // per-lane read offsets inside a buffer
    // A: row 16*ks + 8*(l>>5) + (l&15)>>2 (+4), column 64*wc + 32*cb + 16*((l>>4)&1) + 4*(l&3)
    const int arow = 8 * (l >> 5) + ((l & 15) >> 2);
    const int aswz = narrow ? 0 : 4 * ((l & 15) >> 2);
    uint32_t aoff[2];
#pragma unroll
    for (int cb = 0; cb < 2; ++cb) {
        const int piece = 8 * wc + 4 * cb + 2 * ((l >> 4) & 1) + ((l & 3) >> 1);
        aoff[cb] = (uint32_t)(arow * 256 + 16 * (piece ^ aswz) + 8 * (l & 1));
    }
    // B: token row 64*wt + 32*tb + (l&31), piece 2*ks + (l>>5)
    const int brow = 64 * wt + (l & 31);
    const int bswz = (brow >> 1) & 7;
    // the next chunk is requested into the other buffer before the current one is waited for; two workgroups share a
    // compute unit, so eight waves keep requests in flight (the rate of LDS-DMA grows with the waves that issue it)
    if (c_begin < c_end) request_chunk(c_begin, 0);
    int buf = 0;
#pragma unroll 1
    for (int c = c_begin; c < c_end; ++c) {
        if (c + 1 < c_end) {
            request_chunk(c + 1, buf ^ 1);
            VM_WAIT(8);
        } else {
            VM_WAIT(0);
        }
        __syncthreads();                                           // every wave's part of chunk c has landed
        const uint8_t *wb = smem + buf * XM_BUF;
        const uint8_t *xb = wb + XM_W_BYTES;
        if (!idle) {
#pragma unroll
            for (int ks = 0; ks < XM_KC / 16; ++ks) {
                bf16x8 a[2], b[2];
#pragma unroll
                for (int cb = 0; cb < 2; ++cb) {
                    const uint16_t *ap = reinterpret_cast<const uint16_t *>(wb + aoff[cb] + 16 * ks * 256);
                    const s16x4 lo = lds_read_tr16(ap), hi = lds_read_tr16(ap + 4 * 128);
                    a[cb] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
                }
#pragma unroll
                for (int tb = 0; tb < 2; ++tb)
                    b[tb] = *reinterpret_cast<const bf16x8 *>(xb + (brow + 32 * tb) * 128 + 16 * ((2 * ks + (l >> 5)) ^ bswz));
#pragma unroll
                for (int cb = 0; cb < 2; ++cb)
#pragma unroll
                    for (int tb = 0; tb < 2; ++tb)
                        acc[cb][tb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[cb], b[tb], acc[cb][tb], 0, 0, 0);
            }
        }
        buf ^= 1;
        __syncthreads();                                           // the buffer may be requested into again
    }
    // accumulator register r of lane (token, half) is column 8*(r/4) + 4*half + r%4 of its 32-column block: 16-byte
    // fragments of 32 different rows per store; they leave through a staging area of the wave's own (the chunk
    // buffers are free past the loop's last barrier) as whole 256-byte row segments instead
    static_assert(4 * 32 * XM_SPITCH <= XM_LDS, "the staging areas reuse the chunk buffers");
    if (!idle) {
        uint8_t *stg = smem + w * (32 * XM_SPITCH);
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) {
            uint8_t *row = stg + (l & 31) * XM_SPITCH + 16 * (l >> 5);
#pragma unroll
            for (int cb = 0; cb < 2; ++cb)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const f32x4 v = {acc[cb][tb][4 * q], acc[cb][tb][4 * q + 1], acc[cb][tb][4 * q + 2], acc[cb][tb][4 * q + 3]};
                    *reinterpret_cast<f32x4 *>(row + 128 * cb + 32 * q) = v;
                }
            // the wave reads back what it wrote itself: LDS operations of a wave stay in order
            const int col = 64 * wc + 4 * (l & 15);
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const int r = 4 * k + (l >> 4);
                const f32x4 v = *reinterpret_cast<const f32x4 *>(stg + r * XM_SPITCH + 16 * (l & 15));
                const int t = t0 + 64 * wt + 32 * tb + r;
                if (t < T && col < 8 * sl.pieces) *reinterpret_cast<f32x4 *>(sl.out + (size_t)t * sl.out_pitch + col) = v;
            }
        }
    }
}

// ---------------------------------------------------------------------------------------------
// The same for more tokens: tiles of 128 tokens x 256 columns, wave w columns 64*w .. +63 of all the tokens (eight accumulators),
// so a byte of LDS-DMA serves a third more products.  The tokens travel 64 hidden rows -- a whole cache line -- at a time into two
// buffers, the slab 32 rows at a time into a ring of three: asked for 64 bytes of a row at a time, the second half of a line while
// the first is on its way, hidden states come at 16 bytes per clock and compute unit, however many chunks are ahead and whether
// they lie in the L2 or not (tiles of 256 tokens x 128 columns, as before: 4096 tokens alone 157 us, requests alone 153, products
// alone 89; now 132 and 122, out of the L2 59: bound by the latency of the first miss of every line).  Half of a compute unit's
// LDS: the other half is for the fixed-order sums, which keep the matrix cores busy and move next to nothing.
// Fused prolog with both, before / now: 200 tokens 71.9 / 68.8 us per pass, 400 100.7 / 94.0, 1000 192.2 / 185.7, 4096 689 / 658.
constexpr int XB_TOK = 128;
constexpr int XB_COLS = 256;
constexpr int XB_KC = 32;                        // hidden rows per chunk of the slab; the tokens take two chunks at a time
constexpr int XB_W_BYTES = XB_KC * XB_COLS * 2;
constexpr int XB_X_BYTES = XB_TOK * 2 * XB_KC * 2;
constexpr int XB_LDS = 2 * XB_X_BYTES + 3 * XB_W_BYTES;                      // 81 920 bytes

// hidden rows [2 * XB_KC * c_begin, 2 * XB_KC * c_end), tokens t0 .. t0 + 127; sl.w, sl.out: column 0 of the 256
__device__ __forceinline__ void xb_body(const XmSlab &sl, const uint16_t *x, const int T, const int h, const int t0, const int c_begin,
                                        const int c_end, uint8_t *smem)
{
    const int l = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int half = l >> 5;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_byte_t *)smem;
    // a wave's four requests of a chunk of the slab (two rows of 512 bytes each; 16-byte piece q of row r at q ^ 4*(r & 3)) and four
    // of the tokens (eight rows of 128 bytes; piece q of token row t at q ^ ((t >> 1) & 7))
    const uint8_t *wreq[4], *xreq[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int row = 2 * (4 * w + j) + half;
        wreq[j] = sl.w + (size_t)(2 * XB_KC * c_begin + row) * sl.pitch + 16 * ((l & 31) ^ (4 * (row & 3)));
        const int tl = 8 * (4 * w + j) + (l >> 3);
        const int t = t0 + tl < T ? t0 + tl : T - 1;
        xreq[j] = reinterpret_cast<const uint8_t *>(x) + ((size_t)t * h + 2 * XB_KC * c_begin) * 2 + 16 * ((l & 7) ^ ((tl >> 1) & 7));
    }
    const size_t wstep = (size_t)XB_KC * sl.pitch;
    f32x16 acc[2][4];
#pragma unroll
    for (int cb = 0; cb < 2; ++cb)
#pragma unroll
        for (int tb = 0; tb < 4; ++tb)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[cb][tb][r] = 0.f;
    // A: row 16*ks + 8*half + (l&15)>>2 (+4), column 64*w + 32*cb + 16*((l>>4)&1) + 4*(l&3)
    uint32_t aoff[2];
#pragma unroll
    for (int cb = 0; cb < 2; ++cb) {
        const int piece = 8 * w + 4 * cb + 2 * ((l >> 4) & 1) + ((l & 3) >> 1);
        aoff[cb] = (uint32_t)(2 * XB_X_BYTES + (8 * half + ((l & 15) >> 2)) * (2 * XB_COLS) + 16 * (piece ^ (4 * ((l & 15) >> 2))) + 8 * (l & 1));
    }
    const uint32_t boff = (l & 31) * (4 * XB_KC);
    const int bswz = (l >> 1) & 7;
    staged_chunks<2, 4, 4>(
        2 * (c_end - c_begin),
        [&](const int s, const int b) {
#pragma unroll
            for (int j = 0; j < 4; ++j) dma16(xreq[j] + (size_t)s * (4 * XB_KC), lds0 + b * XB_X_BYTES + 1024u * (4 * w + j));
        },
        [&](const int c, const int slot) {
#pragma unroll
            for (int j = 0; j < 4; ++j) dma16(wreq[j] + c * wstep, lds0 + 2 * XB_X_BYTES + slot * XB_W_BYTES + 1024u * (4 * w + j));
        },
        [&](const int odd, const int xb, const int slot) {
            const uint8_t *wp = smem + slot * XB_W_BYTES, *xp = smem + xb * XB_X_BYTES + boff;
#pragma unroll
            for (int ks = 0; ks < XB_KC / 16; ++ks) {
                bf16x8 a[2];
#pragma unroll
                for (int cb = 0; cb < 2; ++cb) {
                    const uint16_t *ap = reinterpret_cast<const uint16_t *>(wp + aoff[cb] + 16 * ks * (2 * XB_COLS));
                    const s16x4 lo = lds_read_tr16(ap), hi = lds_read_tr16(ap + 4 * XB_COLS);
                    a[cb] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
                }
#pragma unroll
                for (int tb = 0; tb < 4; ++tb) {
                    const bf16x8 b = *reinterpret_cast<const bf16x8 *>(xp + 32 * tb * (4 * XB_KC) + 16 * ((4 * odd + 2 * ks + half) ^ bswz));
#pragma unroll
                    for (int cb = 0; cb < 2; ++cb) acc[cb][tb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[cb], b, acc[cb][tb], 0, 0, 0);
                }
            }
        });
    static_assert(4 * 32 * XM_SPITCH <= XB_LDS, "the staging areas reuse the chunk buffers");
    uint8_t *stg = smem + w * (32 * XM_SPITCH);
#pragma unroll
    for (int tb = 0; tb < 4; ++tb) {
        uint8_t *row = stg + (l & 31) * XM_SPITCH + 16 * half;
#pragma unroll
        for (int cb = 0; cb < 2; ++cb)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const f32x4 v = {acc[cb][tb][4 * q], acc[cb][tb][4 * q + 1], acc[cb][tb][4 * q + 2], acc[cb][tb][4 * q + 3]};
                *reinterpret_cast<f32x4 *>(row + 128 * cb + 32 * q) = v;
            }
        // the wave reads back what it wrote itself: LDS operations of a wave stay in order
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int r = 4 * k + (l >> 4);
            const f32x4 v = *reinterpret_cast<const f32x4 *>(stg + r * XM_SPITCH + 16 * (l & 15));
            const int t = t0 + 32 * tb + r;
            if (t < T) *reinterpret_cast<f32x4 *>(sl.out + (size_t)t * sl.out_pitch + 64 * w + 4 * (l & 15)) = v;
        }
    }
}

// ---------------------------------------------------------------------------------------------
// The same for at most 32 * TB tokens (TB = 1 or 2), where the slab's weights are nearly all a workgroup reads.  The staged tokens
// are the launch's own (the form above stages 128 rows whatever T is), so two chunk buffers, the next chunk requested when the last
// one is consumed, are a third of a compute unit's LDS and all workgroups of a launch run at once.  (With a ring of seven chunks and
// one workgroup per compute unit the last workgroups were a second round.  More chunks on their way are slower all the same: they
// are in the way of the fixed-order sums' requests, which the launch ends with.  Fused prolog, 2 / 3 / 4 chunk buffers: 9 tokens
// 32.2 / 32.9 / 33.3 us per pass, 32: 36.4 / 37.0 / 37.6; MLA prolog alone, 2 / 3: 32 tokens 30.4 / 31.1, 64: 40.1 / 40.6; only the
// fused prolog at 64 goes the other way, 44.8 / 44.6.)
// Wave w takes token block w % TB and, of the slab's four blocks of 32 columns, the TB blocks from TB * (w / TB) on.
template <int TB> constexpr int XMS_CHUNK = XM_W_BYTES + TB * 32 * XM_KC * 2;
template <int TB> constexpr int XMS_LDS = 2 * XMS_CHUNK<TB>;                 // 40 960, 49 152 bytes

template <int TB>
__device__ __forceinline__ void xm_small_body(const XmSlab &sl, const uint16_t *x, const int T, const int h, const int c_begin, const int c_end,
                                              uint8_t *smem)
{
    static_assert(TB == 1 || TB == 2, "token blocks");
    constexpr int CHUNK = XMS_CHUNK<TB>;
    const int l = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int tb = w % TB, cb0 = TB * (w / TB);
    const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_byte_t *)smem;
    const int wrow = l >> 4, wpos = l & 15, xrow = l >> 3, xpos = l & 7;
    const uint8_t *wreq = sl.w + (size_t)(16 * w + wrow) * sl.pitch + 16 * (wpos ^ (4 * wrow));
    const uint8_t *xreq[TB];
#pragma unroll
    for (int j = 0; j < TB; ++j) {
        const int tl = 8 * (TB * w + j) + xrow;
        xreq[j] = reinterpret_cast<const uint8_t *>(x) + (size_t)(tl < T ? tl : T - 1) * h * 2 + 16 * (xpos ^ ((tl >> 1) & 7));
    }
    auto request_chunk = [&](const int c, const int buf) {
        const uint32_t dst = lds0 + (uint32_t)(buf * CHUNK);
#pragma unroll
        for (int j = 0; j < 4; ++j) dma16(wreq + ((size_t)c * XM_KC + 4 * j) * sl.pitch, dst + 1024u * (4 * w + j));
#pragma unroll
        for (int j = 0; j < TB; ++j) dma16(xreq[j] + (size_t)c * (XM_KC * 2), dst + XM_W_BYTES + 1024u * (TB * w + j));
    };
    f32x16 acc[TB];
#pragma unroll
    for (int i = 0; i < TB; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][r] = 0.f;
    const int arow = 8 * (l >> 5) + ((l & 15) >> 2), aswz = 4 * ((l & 15) >> 2);
    uint32_t aoff[TB];
#pragma unroll
    for (int i = 0; i < TB; ++i) aoff[i] = (uint32_t)(arow * 256 + 16 * ((4 * (cb0 + i) + 2 * ((l >> 4) & 1) + ((l & 3) >> 1)) ^ aswz) + 8 * (l & 1));
    const int brow = 32 * tb + (l & 31), bswz = (brow >> 1) & 7;
    if (c_begin < c_end) request_chunk(c_begin, 0);
    int buf = 0;
#pragma unroll 1
    for (int c = c_begin; c < c_end; ++c) {
        VM_WAIT(0);
        __syncthreads();                               // every wave's part of chunk c has landed; every wave is done with chunk c - 1
        if (c + 1 < c_end) request_chunk(c + 1, buf ^ 1);
        const uint8_t *wb = smem + buf * CHUNK;
        const uint8_t *xb = wb + XM_W_BYTES;
#pragma unroll
        for (int ks = 0; ks < XM_KC / 16; ++ks) {
            const bf16x8 b = *reinterpret_cast<const bf16x8 *>(xb + brow * 128 + 16 * ((2 * ks + (l >> 5)) ^ bswz));
#pragma unroll
            for (int i = 0; i < TB; ++i) {
                const uint16_t *ap = reinterpret_cast<const uint16_t *>(wb + aoff[i] + 16 * ks * 256);
                const s16x4 lo = lds_read_tr16(ap), hi = lds_read_tr16(ap + 4 * 128);
                const bf16x8 a = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
                acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc[i], 0, 0, 0);
            }
        }
        buf ^= 1;
    }
    __syncthreads();                                   // every wave is done with the last chunk: the buffers become staging areas
    // 32 tokens x 32 * TB columns per wave leave as whole row segments (as above)
    constexpr int SPITCH = 128 * TB + 16;
    static_assert(4 * 32 * SPITCH <= XMS_LDS<TB>, "the staging areas reuse the chunk buffers");
    uint8_t *stg = smem + w * (32 * SPITCH);
#pragma unroll
    for (int i = 0; i < TB; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const f32x4 v = {acc[i][4 * q], acc[i][4 * q + 1], acc[i][4 * q + 2], acc[i][4 * q + 3]};
            *reinterpret_cast<f32x4 *>(stg + (l & 31) * SPITCH + 16 * (l >> 5) + 128 * i + 32 * q) = v;
        }
    // the wave reads back what it wrote itself: LDS operations of a wave stay in order
    constexpr int LPR = 8 * TB, RPI = 64 / LPR;        // lanes per row, rows per store
#pragma unroll
    for (int k = 0; k < 32 / RPI; ++k) {
        const int r = RPI * k + l / LPR;
        const f32x4 v = *reinterpret_cast<const f32x4 *>(stg + r * SPITCH + 16 * (l % LPR));
        const int t = 32 * tb + r;
        if (t < T) *reinterpret_cast<f32x4 *>(sl.out + (size_t)t * sl.out_pitch + 32 * cb0 + 4 * (l % LPR)) = v;
    }
}

}  // namespace
}  // namespace pto
