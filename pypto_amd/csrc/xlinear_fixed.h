// Fixed-order sums over the hidden axis, one group of eight blocks of 64 rows per workgroup: x [T, h] bf16 times a
// slab of columns of a row-major bf16 weight matrix.  Two forms: xl_body on the vector ALU, 8 tokens per workgroup (the
// MLA prolog's fixed-order launches), and xf_body on the matrix cores, tiles of 32 tokens (the rope columns and the indexer
// prolog's wk and w_proj from 9 tokens on in the fused operator, from 64 on alone); included after prolog_common.h.
//
// Every product of two bf16 values is exact in fp32; a block is summed ascending from 0.0 by fp32 FMAs, the
// workgroup's eight block sums (one per wave) meet in LDS and are added ascending into the group sum, which is all
// that reaches memory: out[t * out_pitch + column].  The caller adds the group sums ascending.
//   workgroup = (slab, group of 512 hidden rows, 8 tokens), eight waves; wave w takes block 8*group + w: the block
//   of the slab travels to the wave's LDS region by LDS-DMA, behind its hidden states, which are widened to fp32 there
//   meanwhile; the product loop takes sixteen rows at a time as they arrive, weights per lane (columns 2l, 2l+1) and hidden
//   states as broadcasts (launch at 8 tokens 12.2 us with all rows waited for, now 11.3).
#pragma once
#include "prolog_common.h"

#pragma clang fp contract(off)

namespace pto {
namespace {

constexpr int XL_BLOCK = 64;                                           // rows per block
constexpr int XL_GROUP = 8;                                            // blocks per group
constexpr int XL_TOK = 8;                                              // tokens per workgroup
constexpr int XL_WAVES = XL_GROUP;                                     // one block per wave
constexpr int XL_W_BYTES = XL_BLOCK * 256;                             // a block of one slab: 64 rows x 256 bytes
constexpr int XL_X_BYTES = XL_TOK * XL_BLOCK * 4;                      // the hidden states as fp32
constexpr int XL_REGION = XL_W_BYTES + XL_X_BYTES + XL_TOK * XL_BLOCK * 2;   // + as they come
constexpr int XL_LDS = XL_WAVES * XL_REGION;

struct XlSlab {
    const uint8_t *w;     // column 0 of the slab in row 0 of the weight matrix
    int pitch;            // bytes between rows of the weight matrix
    int wbytes;           // bytes of a row that belong to the slab: 16, 32, 64, 128 or 256
    float *out;           // group sums of this group: out[t * out_pitch + column of the slab]
    int out_pitch;
    // xl_body only: a 256-byte slab may be two 128-byte halves of different matrices.  With w_hi set (wbytes = 256),
    // bytes 128..255 of a staged row are bytes 0..127 of w_hi's row, and columns 64..127 go to out_hi[t * out_pitch_hi + column - 64].
    const uint8_t *w_hi = nullptr;
    int pitch_hi = 0;
    float *out_hi = nullptr;
    int out_pitch_hi = 0;
};

// group g of the hidden axis, tokens t0 .. t0 + 7 (rows past T - 1 repeat it and are not stored)
__device__ __forceinline__ void xl_body(const XlSlab &sl, const uint16_t *x, const int T, const int h, const int g, const int t0, uint8_t *smem)
{
    const int l = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nblk = h / XL_BLOCK;
    const int wbytes = sl.wbytes;

    uint8_t *region = smem + w * XL_REGION;
    float *xs = reinterpret_cast<float *>(region + XL_W_BYTES);         // [8][64]
    const int c = g * XL_GROUP + w;                                       // this wave's block
    const int nb = nblk - g * XL_GROUP < XL_GROUP ? nblk - g * XL_GROUP : XL_GROUP;
    float a0[XL_TOK], a1[XL_TOK];
#pragma unroll
    for (int t = 0; t < XL_TOK; ++t) a0[t] = a1[t] = 0.f;

    if (w < nb) {
        const int k0 = c * XL_BLOCK;
        const uint32_t wdst = (uint32_t)(uintptr_t)(lds_byte_t *)region;
        {   // the hidden states first: lane l hidden states k0 + 8*(l%8) .. +7 of token t0 + l/8
            const int t = t0 + (l >> 3);
            dma16(x + (size_t)(t < T ? t : T - 1) * h + k0 + 8 * (l & 7), wdst + XL_W_BYTES + XL_X_BYTES);
        }
        {   // rows of wbytes bytes: wbytes/16 lanes per row
            const int lpr = wbytes >> 4;
            const int rpi = 64 / lpr;                                     // rows per request
            const bool hi = sl.w_hi != nullptr && (l & 15) >= 8;          // this lane's piece belongs to the second matrix
            const size_t pitch = hi ? sl.pitch_hi : sl.pitch;
            const uint8_t *src = (hi ? sl.w_hi - 128 : sl.w) + (size_t)(k0 + l / lpr) * pitch + 16 * (l % lpr);
#pragma unroll 1
            for (int i = 0; i < XL_BLOCK / rpi; ++i) dma16(src + (size_t)i * rpi * pitch, wdst + 1024 * i);
        }
        if (wbytes == 256) VM_WAIT(16);                                   // everything but the sixteen requests of the weights
        else VM_WAIT(0);
        asm volatile("" ::: "memory");
        {
            const u32x4 xr = *reinterpret_cast<const u32x4 *>(region + XL_W_BYTES + XL_X_BYTES + 16 * l);
            float *dst = xs + 8 * l;
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const f32x4 v = {__uint_as_float(xr[2 * q] << 16), __uint_as_float(xr[2 * q] & 0xffff0000u),
                                 __uint_as_float(xr[2 * q + 1] << 16), __uint_as_float(xr[2 * q + 1] & 0xffff0000u)};
                *reinterpret_cast<f32x4 *>(dst + 4 * q) = v;
            }
        }
        const int rowdw = wbytes >> 2;
        const uint32_t *wl = reinterpret_cast<const uint32_t *>(region) + (l & (rowdw - 1));   // lanes past the slab's width repeat earlier ones
        // Sixteen rows at a time, as they arrive (a whole slab's requests are of four rows each): the multiply-adds of a block
        // take as long as half of the launch's bytes.
        auto rows16 = [&](const int first) __attribute__((always_inline)) {
            asm volatile("" ::: "memory");
#pragma unroll 2
            for (int kk = first; kk < first + 16; kk += 4) {
                f32x4 xv[XL_TOK];
#pragma unroll
                for (int t = 0; t < XL_TOK; ++t) xv[t] = *reinterpret_cast<const f32x4 *>(xs + t * XL_BLOCK + kk);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const uint32_t wv = wl[(kk + j) * rowdw];
                    const float w0 = __uint_as_float(wv << 16), w1 = __uint_as_float(wv & 0xffff0000u);
#pragma unroll
                    for (int t = 0; t < XL_TOK; ++t) {
                        a0[t] = __builtin_fmaf(xv[t][j], w0, a0[t]);
                        a1[t] = __builtin_fmaf(xv[t][j], w1, a1[t]);
                    }
                }
            }
        };
        VM_WAIT(12);                                                      // (narrower slabs have arrived)
        rows16(0);
        VM_WAIT(8);
        rows16(16);
        VM_WAIT(4);
        rows16(32);
        VM_WAIT(0);
        rows16(48);
        // block sums into this wave's own (consumed) region: [8 tokens][128 columns]
        float *bs = reinterpret_cast<float *>(region);
#pragma unroll
        for (int t = 0; t < XL_TOK; ++t) {
            f32x2 v = {a0[t], a1[t]};
            *reinterpret_cast<f32x2 *>(bs + t * 128 + 2 * l) = v;
        }
    }
    __syncthreads();
    // group sum: thread (token = w, columns 2l, 2l+1) chains the block sums in ascending order
    {
        const int t = t0 + w;
        const int width = wbytes >> 1;                                    // columns of the slab
        if (t < T && 2 * l < width) {
            float s0 = 0.f, s1 = 0.f;
            for (int i = 0; i < nb; ++i) {
                const f32x2 v = *reinterpret_cast<const f32x2 *>(reinterpret_cast<const float *>(smem + i * XL_REGION) + w * 128 + 2 * l);
                s0 = __fadd_rn(s0, v[0]);
                s1 = __fadd_rn(s1, v[1]);
            }
            f32x2 v = {s0, s1};
            float *dst = sl.out + (size_t)t * sl.out_pitch + 2 * l;
            if (sl.w_hi != nullptr && l >= 32) dst = sl.out_hi + (size_t)t * sl.out_pitch_hi + 2 * l - 64;
            *reinterpret_cast<f32x2 *>(dst) = v;
        }
    }
}

// ---------------------------------------------------------------------------------------------
// The same sums for larger token counts on the matrix cores: v_mfma_f32_32x32x1_2b_f32 multiplies one hidden row at a
// time, so each of its results is one product (exact: both factors are bf16 values) added to the accumulator with one
// rounding -- an fp32 FMA -- and a chain of them is the sequential sum of the form above, bit for bit, whatever order
// the cores have inside an instruction of more rows.  (Subnormal products and sums, signed zeros included: checked
// against fmaf chains.)
//   workgroup = (slab of up to 64 columns, group of 512 hidden rows, a run of tiles of 32 tokens), four waves; wave w takes
//   blocks 2w and 2w + 1 of the group as the two independent products of the instruction (lanes 0..31 supply block 2w, lanes
//   32..63 block 2w + 1).  Row i of the first operand is column 2i (accumulator 0) or 2i + 1 (accumulator 1) of the slab: one
//   dword per lane and hidden row feeds both, and all 64 of a block stay in registers for every tile.  A tile's hidden
//   states are asked for as whole cache lines under the products of the tile before (a lane reading its own token's 128 bytes
//   piece by piece takes 64 lines at a time, more than the waves of a compute unit find in its first cache again).  The
//   eight block sums meet in LDS and are chained ascending into the group sum.
// Bound: the matrix cores' fp32 rate: 64 clocks per instruction, 139 TFLOP/s reached by a bare loop; 4.8 us per tile and SIMD at
// the clock that random operands leave.  256 columns x 4096 tokens x 7168 rows alone 162 us with the weights in LDS for one tile,
// now 148 (112 TFLOP/s).  The multiply-add form of the vector ALU this replaced (hidden states broadcast through DPP) ran at a
// quarter of the matrix cores' rate.
constexpr int XF_TOK = 32;                                               // tokens per tile; a workgroup takes a run of tiles
constexpr int XF_COLS = 64;                                              // columns per workgroup, at most
constexpr int XF_WAVES = 4;
constexpr int XF_TOK_PITCH = XF_COLS * 4 + 16;                           // bytes between token rows of a block sum
constexpr int XF_SUMS = XF_TOK * XF_TOK_PITCH;
constexpr int XF_LDS = XL_GROUP * XF_SUMS;                               // 69 632 bytes
static_assert(XL_GROUP == 2 * XF_WAVES, "two blocks per wave");

__host__ __device__ inline int xf_token_tiles(const int T) { return (T + XF_TOK - 1) / XF_TOK; }

// The jobs of a launch: sets of columns x groups x runs of token tiles.  Workgroups go round the eight XCDs; the sets of one
// (group, run) are consecutive workgroups of one XCD, so its hidden states cross into that L2 once.
struct XfGrid {
    int nsets, ngroups, run;      // run: token tiles of a workgroup
};
__host__ __device__ inline int xf_jobs(const XfGrid &f, const int T)
{
    return 8 * f.nsets * ((f.ngroups * ((xf_token_tiles(T) + f.run - 1) / f.run) + 7) / 8);
}
// Token tiles of a workgroup where `cols` sets x groups share `free` places for workgroups beside the launch's other ones: two
// where they make a single round and one more than a round and a third (fused prolog, 1 / 2 tiles: 130 tokens, a round in
// either case, 58.3 / 63.1 us per pass, 200: 72.9 / 69.1, 256: 76.3 / 72.5, 400, two of them 1.5 rounds, 95.4 / 106.3; the
// indexer prolog alone 400, one 1.07 rounds, 36.2 / 39.0, 512, 1.31 rounds, 39.3 / 41.3); beyond that two from 20 tiles on, for
// which a workgroup keeps its weights (1 / 2: 1000 tokens 189.2 / 185.1, 1300 248.7 / 245.5, 4096 681.8 / 674.7).
inline int xf_run(const int cols, const int T, const int free)
{
    const int tiles = xf_token_tiles(T);
    if ((tiles + 1) / 2 * cols <= free) return 3 * tiles * cols > 4 * free ? 2 : 1;
    return tiles < 20 ? 1 : 2;
}
struct XfJob {
    int set, g, t0;       // g < 0: padding of the job count
};
__device__ __forceinline__ XfJob xf_job(const int j, const XfGrid &f, const int T)
{
    const int q = j >> 3;
    const int c = (q / f.nsets) * 8 + (j & 7);
    XfJob r;
    r.set = q % f.nsets;
    r.g = c < f.ngroups * ((xf_token_tiles(T) + f.run - 1) / f.run) ? c % f.ngroups : -1;
    r.t0 = (c / f.ngroups) * f.run * XF_TOK;
    return r;
}

// group g of the hidden axis, `run` tiles of 32 tokens from t0 on (rows past T - 1 repeat it and are not stored); sl.wbytes <= 128
__device__ __forceinline__ void xf_body(const XlSlab &sl, const uint16_t *x, const int T, const int h, const int g, const int t0, const int run,
                                        uint8_t *smem)
{
    typedef __attribute__((ext_vector_type(32))) float f32x32;
    const int l = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int half = l >> 5, i = l & 31;
    const int nblk = h / XL_BLOCK;
    const int nb = nblk - g * XL_GROUP < XL_GROUP ? nblk - g * XL_GROUP : XL_GROUP;
    const int wbytes = sl.wbytes;
    const int tend = t0 + run * XF_TOK < T ? t0 + run * XF_TOK : T;
    // a group's last wave may have one block only: both halves then work on it, and the second result is dropped; a wave
    // without a block works on the group's first
    const bool active = 2 * w < nb;
    const int blk = active ? (half && 2 * w + 1 < nb ? 2 * w + 1 : 2 * w) : 0;
    // the block's weights, a dword (columns 2i, 2i + 1) per row, and the hidden states of the tile's token
    uint32_t wv[XL_BLOCK];
    {
        const uint8_t *row = sl.w + (size_t)g * (XL_GROUP * XL_BLOCK) * sl.pitch;         // (uniform)
        const uint32_t off = (uint32_t)(blk * XL_BLOCK * sl.pitch + (4 * i < wbytes ? 4 * i : 0));
#pragma unroll
        for (int k = 0; k < XL_BLOCK; ++k) wv[k] = *reinterpret_cast<const uint32_t *>(row + (size_t)k * sl.pitch + off);
    }
    // The hidden states: whole 128-byte rows of a block per eight lanes, put in order (a lane its token's) through the wave's own
    // part of the LDS.
    u32x4 xv[XL_BLOCK / 8], xn[XL_BLOCK / 8];
    uint8_t *mine = smem + 2 * w * XF_SUMS;
    const int blk1 = active && 2 * w + 1 < nb ? 2 * w + 1 : (active ? 2 * w : 0), blk0 = active ? 2 * w : 0;
    auto load_x = [&](const int tile0) {
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int tl = tile0 + 8 * (q & 3) + (l >> 3), t = tl < T ? tl : T - 1;
            xn[q] = *reinterpret_cast<const u32x4 *>(x + (size_t)t * h + (g * XL_GROUP + (q < 4 ? blk0 : blk1)) * XL_BLOCK + 8 * (l & 7));
        }
    };
    auto order_x = [&]() {
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int row = 8 * q + (l >> 3);
            *reinterpret_cast<u32x4 *>(mine + row * 128 + 16 * ((l & 7) ^ ((row >> 1) & 7))) = xn[q];
        }
#pragma unroll
        for (int q = 0; q < 8; ++q) xv[q] = *reinterpret_cast<const u32x4 *>(mine + l * 128 + 16 * (q ^ ((l >> 1) & 7)));
    };
    load_x(t0);
    order_x();
#pragma unroll 1
    for (int tile0 = t0; tile0 < tend; tile0 += XF_TOK) {
        if (tile0 + XF_TOK < tend) load_x(tile0 + XF_TOK);
        f32x32 a0, a1;
#pragma unroll
        for (int r = 0; r < 32; ++r) a0[r] = a1[r] = 0.f;
#pragma unroll
        for (int k = 0; k < XL_BLOCK; ++k) {
            asm volatile("" : "+v"(wv[k]));                              // (widened here, not in front of the loop: registers)
            const uint32_t xw = xv[k >> 3][(k >> 1) & 3];
            const float xf = __uint_as_float((k & 1) ? xw & 0xffff0000u : xw << 16);
            a0 = __builtin_amdgcn_mfma_f32_32x32x1f32(__uint_as_float(wv[k] << 16), xf, a0, 0, 0, 0);
            a1 = __builtin_amdgcn_mfma_f32_32x32x1f32(__uint_as_float(wv[k] & 0xffff0000u), xf, a1, 0, 0, 0);
            if (k % 4 == 3) __builtin_amdgcn_sched_barrier(0);           // (widened factors of a few rows at a time)
        }
        if (active) {
            // register 16*b + 4*q + j of lane (token, half) is row 8*q + 4*half + j of block b's product
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                uint8_t *row = smem + (2 * w + b) * XF_SUMS + i * XF_TOK_PITCH + 32 * half;
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        const int r = 16 * b + 4 * q + 2 * e;
                        const f32x4 v = {a0[r], a1[r], a0[r + 1], a1[r + 1]};
                        *reinterpret_cast<f32x4 *>(row + 64 * q + 16 * e) = v;
                    }
            }
        }
        __syncthreads();
        {   // thread (token, eight columns) chains the block sums in ascending order
            const int tl = threadIdx.x >> 3, c8 = 8 * (threadIdx.x & 7);
            const int t = tile0 + tl;
            if (t < T && 2 * c8 < wbytes) {
                float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
                for (int b = 0; b < nb; ++b) {
                    const f32x4 *src = reinterpret_cast<const f32x4 *>(smem + b * XF_SUMS + tl * XF_TOK_PITCH + 4 * c8);
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        const f32x4 v = src[e];
#pragma unroll
                        for (int j = 0; j < 4; ++j) s[4 * e + j] = __fadd_rn(s[4 * e + j], v[j]);
                    }
                }
                f32x4 *dst = reinterpret_cast<f32x4 *>(sl.out + (size_t)t * sl.out_pitch + c8);
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const f32x4 v = {s[4 * e], s[4 * e + 1], s[4 * e + 2], s[4 * e + 3]};
                    dst[e] = v;
                }
            }
        }
        if (tile0 + XF_TOK >= tend) break;
        __syncthreads();                                                 // the sums have been read
        order_x();
    }
}

}  // namespace
}  // namespace pto
