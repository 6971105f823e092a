// The last launch of both prologs for at most 32 tokens: a head's projection and everything that follows it, as in
// prolog_prefill.h, in the form that fits a decode batch, where the weights -- 67 MB of them -- are all there is to wait for.
// One workgroup of four waves per head and compute unit.  The launch's tokens lie in LDS whole; everything else of the LDS is a
// ring of requests that never runs dry: chunks of 64 rows of the head's projection and, behind them without a gap, its w_uk,
// sixteen rows at a time.  Bound: memory, 54 MB in 10 us behind the first 2 (another 13 MB are in the L2: mlap_ask_ahead).  With
// every chunk out of the L2 (timing only) an attention workgroup takes 8.1 us at 8 tokens and 9.0 at 32 instead of 13; with one
// chunk between barriers, six blocks of columns as 2, 2, 1, 1 over the waves and 60 KiB on their way it took 9.6 and 10.8 (fused
// prolog 8 tokens 32.6 us per pass, now 32.4, 16: 33.7 and 33.4, 32: 37.1 and 36.5).  (8 tokens as two launches with partial sums in between: 6 us
// more.)
// Included by prolog_fused.hip after prolog_prefill.h.
#pragma once
#include "prolog_prefill.h"

#pragma clang fp contract(off)

namespace pto {
namespace {

constexpr int PS_TOK = MLAP_MAX_QLORA * PROLOG_SMALL_TOKENS;        // the tokens: row t at q_lora * t, 16-byte piece q at q ^ (t & 15)
static_assert(PROLOG_SMALL_TOKENS == 32, "one block of tokens");

// at most n requests of this wave outstanding, n a constant after unrolling
__device__ __forceinline__ void ps_wait(const int n)
{
    switch (n) {
    case 8: VM_WAIT(8); break;
    case 10: VM_WAIT(10); break;
    case 12: VM_WAIT(12); break;
    case 13: VM_WAIT(13); break;
    case 14: VM_WAIT(14); break;
    case 15: VM_WAIT(15); break;
    case 16: VM_WAIT(16); break;
    case 18: VM_WAIT(18); break;
    case 20: VM_WAIT(20); break;
    default: VM_WAIT(0); break;
    }
}

// requests the tokens' rows 0 .. T - 1, a wave's share; rows from T on hold whatever was there, and so do their results
__device__ __forceinline__ void ps_request_tokens(const int8_t *q_norm, const int q_lora, const int T, const uint32_t dst, const int w, const int l)
{
    const int ppr = q_lora / 16, last = T * ppr - 1;
#pragma unroll 1
    for (int r = w; r * 64 <= last; r += 4) {
        int g = 64 * r + l;
        g = g < last ? g : last;
        const int row = g / ppr, pos = g - row * ppr;
        dma16(q_norm + (size_t)row * q_lora + 16 * (pos ^ (row & 15)), dst + 1024 * r);
    }
}
// the tokens' operand of contraction step ks (32 rows of the reduction axis)
__device__ __forceinline__ i32x4 ps_token_operand(const uint8_t *tok, const int q_lora, const int ks, const int l)
{
    return *reinterpret_cast<const i32x4 *>(tok + (l & 31) * q_lora + 16 * ((2 * ks + (l >> 5)) ^ (l & 15)));
}

// ------------------------------------------------------------------------------------------------ attention query
// Of the head's six blocks of 32 projected columns wave w makes w and, out of every second chunk, 4 + w % 2 (the rope channels: the
// waves' sums are whole numbers and are added at the end).  Of the product with w_uk each wave makes 128 columns, out of rows it has requested itself: that part of the ring needs no barriers.
constexpr int PSA_CHUNK = PF_KC * MLAP_QHEAD;          // 64 rows of 192 bytes of the projection
constexpr int PSA_CHUNKS = 8;
constexpr int PSA_STEP = 16 * 1024;                    // 16 rows of w_uk: [wave][16][256 bytes]
constexpr int PSA_STEPS = 6;
constexpr int PSA_RING = PS_TOK;
static_assert(PSA_CHUNKS * PSA_CHUNK == PSA_STEPS * PSA_STEP, "both go round the same ring");
static_assert(MLAP_MIN_QLORA % (PF_KC * PSA_CHUNKS) == 0, "w_uk starts at the ring's start");
constexpr int PSA_Q = PSA_RING + PSA_CHUNKS * PSA_CHUNK;   // nope channels [token][256 bytes], 16-byte piece q at q ^ (t & 15)
constexpr int PSA_SC = PSA_Q + PROLOG_SMALL_TOKENS * MLAP_NOPE * 2;    // per wave: scales of the tokens, of its two blocks' columns
constexpr int PSA_LDS = PSA_SC + 4 * 512;
constexpr int PSA_SPITCH = 272;                        // bytes between the rows of a wave's output staging area
// once the projection is made the tokens' place holds the rope rows and the staging areas
static_assert(32 * PFA_RPITCH + 4 * 32 * PSA_SPITCH <= PS_TOK, "staging fits");
constexpr int PSA_HALF = 16 * 1024;                    // and, before the staging areas, two waves' sums of the rope channels, 4 KB each
static_assert(PSA_HALF >= 32 * PFA_RPITCH && PSA_HALF + 2 * 4096 <= PS_TOK, "behind the rope rows");
static_assert(PSA_LDS <= 160 * 1024, "one workgroup fits a compute unit");

__device__ __forceinline__ void mlap_small_body(const MlapParams &p, const int head, uint8_t *lds)
{
    const int l = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int half = l >> 5;
    const int ncols = p.n_heads * MLAP_QHEAD;
    const int nch = p.q_lora / PF_KC;                  // 8, 16 or 24
    const uint32_t base = (uint32_t)(uintptr_t)(lds_byte_t *)lds;

    const int8_t *wsrc[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const int piece = 64 * (3 * w + j) + l, row = piece / 12, pos = piece % 12;
        wsrc[j] = p.w_uqqr + (size_t)row * ncols + head * MLAP_QHEAD + 16 * (pos ^ (2 * ((row >> 2) & 1)));
    }
    // w_uk: rows 4j + l/16 of a chunk's sixteen, this wave's 128 columns; 16-byte piece q of row r at q ^ 4*(r & 3)
    const uint16_t *usrc = p.w_uk + ((size_t)head * MLAP_NOPE + (l >> 4)) * MLAP_KV + 128 * w + 8 * ((l & 15) ^ (4 * (l >> 4)));
    auto request_w = [&](const int c) {
#pragma unroll
        for (int j = 0; j < 3; ++j)
            dma16(wsrc[j] + (size_t)c * PF_KC * ncols, base + PSA_RING + (c % PSA_CHUNKS) * PSA_CHUNK + 1024 * (3 * w + j));
    };
    auto request_u = [&](const int ks) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            dma16(usrc + (size_t)(16 * ks + 4 * j) * MLAP_KV, base + PSA_RING + (ks % PSA_STEPS) * PSA_STEP + 4096 * w + 1024 * j);
    };
    const int tl = l & 31;
    // (the scales too as requests: a load that the compiler tracks would wait for the whole ring)
    dma4(p.q_norm_scale + (tl < p.T ? tl : p.T - 1), base + PSA_SC + 512 * w);
    dma4(p.w_qb_scale + head * MLAP_QHEAD + 32 * (half && w < 2 ? w + 4 : w) + tl, base + PSA_SC + 512 * w + 256);
    ps_request_tokens(p.q_norm, p.q_lora, p.T, base, w, l);
#pragma unroll
    for (int c = 0; c < PSA_CHUNKS; ++c) request_w(c);

    i32x16 acc[2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][r] = 0;
    uint32_t aoff[2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
        aoff[i] = PSA_RING + (16 * half + ((l & 15) >> 1)) * MLAP_QHEAD + 32 * ((i ? 4 + (w & 1) : w) ^ ((l >> 3) & 1)) + 16 * ((l >> 4) & 1) + 8 * (l & 1);
    typedef int v2i __attribute__((ext_vector_type(2)));
    auto operand = [&](const int i, const int slot, const int s) {
        const uint8_t *ap = lds + slot * PSA_CHUNK + aoff[i] + s * 32 * MLAP_QHEAD;
        const v2i lo = __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) v2i *)(lds_byte_t *)ap);
        const v2i hi = __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) v2i *)(lds_byte_t *)(ap + 8 * MLAP_QHEAD));
        return i32x4{lo[0], lo[1], hi[0], hi[1]};
    };
    // chunks c and c + 1 (c even), for the rope block c + w / 2
    auto products = [&](const int c) {
        const int slot = c % PSA_CHUNKS;
        i32x4 b[4], a[4], ar[2];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            b[s] = ps_token_operand(lds, p.q_lora, 2 * c + s, l);
            a[s] = operand(0, slot + (s >> 1), s & 1);
        }
#pragma unroll
        for (int s = 0; s < 2; ++s) ar[s] = operand(1, slot + (w >> 1), s);
#pragma unroll
        for (int s = 0; s < 4; ++s) acc[0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[s], b[s], acc[0], 0, 0, 0);
#pragma unroll
        for (int s = 0; s < 2; ++s) acc[1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(ar[s], w >> 1 ? b[2 + s] : b[s], acc[1], 0, 0, 0);
    };
    // Two chunks between barriers.  Those of the next two turns, 12 requests, may be outstanding when they are waited for (at the
    // start three turns'); the two behind them take the places of the last turn's.
    VM_WAIT(18);
    __syncthreads();
    products(0);
    int c = 2;
#pragma unroll 1
    for (; c <= nch - PSA_CHUNKS; c += 2) {
        VM_WAIT(12);
        __syncthreads();                               // chunks c, c + 1 have landed for every wave; every wave is done with c - 1
        request_w(c + PSA_CHUNKS - 2);
        request_w(c + PSA_CHUNKS - 1);
        products(c);
    }
    // the last six chunks: as 24, 48, 72 KiB of the ring become free, one, three, four of w_uk's 16 KiB steps follow
    VM_WAIT(12);
    __syncthreads();
    request_u(0);
    products(c);
    VM_WAIT(10);
    __syncthreads();
    request_u(1);
    request_u(2);
    products(c + 2);
    VM_WAIT(12);
    __syncthreads();
    request_u(3);
    products(c + 4);
    __syncthreads();                                   // every wave is done with the projection's chunks and the tokens
    request_u(4);
    request_u(5);
    if (w >= 2) {
#pragma unroll
        for (int rg = 0; rg < 4; ++rg)
            *reinterpret_cast<i32x4 *>(lds + PSA_HALF + 4096 * (w - 2) + 1024 * rg + 16 * l) = i32x4{acc[1][4 * rg], acc[1][4 * rg + 1], acc[1][4 * rg + 2], acc[1][4 * rg + 3]};
    }
    // registers 4*rg .. 4*rg+3 of a block: columns 8*rg + 4*half .. +3 of token l % 32
    const float *sc_lds = reinterpret_cast<const float *>(lds + PSA_SC + 512 * w);
    const float ts = sc_lds[tl];
    auto dequantise = [&](const i32x16 &x, const int i, const int rg) {
        const f32x4 sc = *reinterpret_cast<const f32x4 *>(sc_lds + 64 + 32 * i + 4 * half + 8 * rg);
        float f[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) f[j] = __fmul_rn(__fmul_rn((float)x[4 * rg + j], ts), sc[j]);
        return u32x2{pack_bf16x2(f[0], f[1]), pack_bf16x2(f[2], f[3])};
    };
#pragma unroll
    for (int rg = 0; rg < 4; ++rg)
        *reinterpret_cast<u32x2 *>(lds + PSA_Q + tl * 256 + 16 * ((4 * w + rg) ^ (l & 15)) + 8 * half) = dequantise(acc[0], 0, rg);
    __syncthreads();                                   // the nope operand and the other waves' sums of the rope channels are complete
    if (w < 2) {
#pragma unroll
        for (int rg = 0; rg < 4; ++rg) {
            const i32x4 other = *reinterpret_cast<const i32x4 *>(lds + PSA_HALF + 4096 * w + 1024 * rg + 16 * l);
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[1][4 * rg + j] += other[j];
            *reinterpret_cast<u32x2 *>(lds + tl * PFA_RPITCH + 2 * (32 * w + 8 * rg + 4 * half)) = dequantise(acc[1], 1, rg);
        }
    }
    __syncthreads();                                   // the rope rows are complete, their sums read
    f32x16 o[4];
#pragma unroll
    for (int cb = 0; cb < 4; ++cb)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[cb][r] = 0.f;
    const uint32_t uoff = PSA_RING + 4096 * w + (8 * half + ((l & 15) >> 2)) * 256 + 8 * (l & 1);
#pragma unroll
    for (int ks = 0; ks < MLAP_NOPE / 16; ++ks) {
        // steps ks + 1 .. ks + 4, at first ks + 5, are outstanding; the place of the step before this one is this wave's to fill again
        if (ks == 0) VM_WAIT(20);
        else if (ks <= 3) VM_WAIT(16);
        else if (ks == 4) VM_WAIT(12);
        else if (ks == 5) VM_WAIT(8);
        else if (ks == 6) VM_WAIT(4);
        else VM_WAIT(0);
        asm volatile("" ::: "memory");
        if (ks >= 1 && ks + PSA_STEPS - 1 < MLAP_NOPE / 16) request_u(ks + PSA_STEPS - 1);
        const bf16x8 b = *reinterpret_cast<const bf16x8 *>(lds + PSA_Q + tl * 256 + 16 * ((2 * ks + half) ^ (l & 15)));
#pragma unroll
        for (int cb = 0; cb < 4; ++cb) {
            const int piece = 4 * cb + 2 * ((l >> 4) & 1) + ((l & 3) >> 1);
            const uint16_t *ap = reinterpret_cast<const uint16_t *>(lds + (ks % PSA_STEPS) * PSA_STEP + uoff + 16 * (piece ^ (4 * ((l & 15) >> 2))));
            const s16x4 lo = lds_read_tr16(ap), hi = lds_read_tr16(ap + 4 * 128);
            const s16x8 a = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
            o[cb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), b, o[cb], 0, 0, 0);
        }
        __builtin_amdgcn_s_waitcnt(0xC07F);            // lgkmcnt(0): the slot has been read
        asm volatile("" ::: "memory");
    }
    // lane (token, half) holds columns 8*(r/4) + 4*half + r%4 of each block: out through the staging area as 256-byte pieces of rows
    uint8_t *stg = lds + 32 * PFA_RPITCH + w * (32 * PSA_SPITCH);
#pragma unroll
    for (int cb = 0; cb < 4; ++cb)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const u32x2 v = {pack_bf16x2(o[cb][4 * q], o[cb][4 * q + 1]), pack_bf16x2(o[cb][4 * q + 2], o[cb][4 * q + 3])};
            *reinterpret_cast<u32x2 *>(stg + tl * PSA_SPITCH + 2 * (32 * cb + 8 * q + 4 * half)) = v;
        }
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const int t = 4 * k + (l >> 4);
        if (4 * k >= p.T) break;
        const u32x4 v = *reinterpret_cast<const u32x4 *>(stg + t * PSA_SPITCH + 16 * (l & 15));
        if (t < p.T) *reinterpret_cast<u32x4_a2 *>(p.q_nope + ((size_t)t * p.n_heads + head) * MLAP_KV + 128 * w + 8 * (l & 15)) = v;
    }
    pfa_rotate_rows(p, lds, 8 * w + (l >> 3), 8 * w + (l >> 3), head, l & 7);
}

// ------------------------------------------------------------------------------------------------- indexer query
// Wave w projects columns 32*w .. +31; the rows then meet in LDS as bf16, a wave per row rotates them, and the Hadamard sums
// are taken in their fixed order by all four waves (lip_fixed_rows).
constexpr int PSI_SLOT = PF_KC * LIP_DIM;
constexpr int PSI_SLOTS = 8;
constexpr int PSI_ROT = PROLOG_SMALL_TOKENS / 4;       // rows that a wave rotates
constexpr int PSI_HAD = PS_TOK;                        // the matrix, row r at 256 * r, 16-byte piece q at q ^ 4*(r & 3)
constexpr int PSI_RING = PSI_HAD + LIP_DIM * LIP_DIM * 2;
constexpr int PSI_LDS = PSI_RING + PSI_SLOTS * PSI_SLOT;
constexpr int PSI_SCRATCH = PSI_RING + 32 * HB_PITCH * 2;     // behind the rows, in the ring's place
static_assert(PSI_SCRATCH + HB_SCRATCH <= PSI_LDS, "the rows fit the ring's place");
static_assert(PSI_LDS <= 160 * 1024, "one workgroup fits a compute unit");

__device__ __forceinline__ void lip_small_body(const LipParams &p, const int head, uint8_t *lds)
{
    const int l = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int half = l >> 5;
    const int ncols = p.n_heads * LIP_DIM;
    const int nch = p.q_lora / PF_KC;
    const uint32_t base = (uint32_t)(uintptr_t)(lds_byte_t *)lds;
    const int8_t *wsrc[2];
#pragma unroll
    for (int j = 0; j < 2; ++j)
        wsrc[j] = p.w_qb + (size_t)(8 * (2 * w + j) + (l >> 3)) * ncols + head * LIP_DIM + 16 * ((l & 7) ^ q_tr_piece_swizzle(l >> 3));
    auto request_w = [&](const int c, const int slot) {
#pragma unroll
        for (int j = 0; j < 2; ++j) dma16(wsrc[j] + (size_t)c * PF_KC * ncols, base + PSI_RING + slot * PSI_SLOT + 1024 * (2 * w + j));
    };
    // (the loads that the compiler tracks come first: the waits below count the requests behind them)
    const int tl = l & 31;
    const float ts = p.q_norm_scale[tl < p.T ? tl : p.T - 1];
    f32x4 sc[4];
#pragma unroll
    for (int rg = 0; rg < 4; ++rg) sc[rg] = *reinterpret_cast<const f32x4 *>(p.w_qb_scale + head * LIP_DIM + 32 * w + 8 * rg + 4 * half);
    uint32_t rc[PSI_ROT], rs[PSI_ROT];                 // rotation factors of tokens w, w + 4, ..
#pragma unroll
    for (int k = 0; k < PSI_ROT; ++k) {
        const int t = w + 4 * k < p.T ? w + 4 * k : p.T - 1;
        rc[k] = rope_coef(p.cos, t, l);
        rs[k] = rope_coef(p.sin, t, l);
    }
    asm volatile("" ::: "memory");
    ps_request_tokens(p.q_norm, p.q_lora, p.T, base, w, l);
#pragma unroll
    for (int c = 0; c < PSI_SLOTS - 1; ++c) request_w(c, c);
    i32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0;
    auto products = [&](const int c, const int slot) {
#pragma unroll
        for (int s = 0; s < PF_KC / 32; ++s)
            acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(q_build_a_tr_one(lds + PSI_RING + slot * PSI_SLOT, s, l, w),
                                                        ps_token_operand(lds, p.q_lora, 2 * c + s, l), acc, 0, 0, 0);
    };
    int c = 0, slot = 0;
#pragma unroll 1
    for (; c + PSI_SLOTS - 1 <= nch - 1; ++c) {
        VM_WAIT(2 * (PSI_SLOTS - 2));                  // everything but the six chunks behind this one
        __syncthreads();
        request_w(c + PSI_SLOTS - 1, slot == 0 ? PSI_SLOTS - 1 : slot - 1);
        products(c, slot);
        slot = slot == PSI_SLOTS - 1 ? 0 : slot + 1;
    }
    {   // the matrix, behind the last chunk's requests
        const uint16_t *src = p.hq + (size_t)(32 * w + (l >> 4)) * LIP_DIM + 8 * ((l & 15) ^ (4 * (l >> 4)));
#pragma unroll 1
        for (int j = 0; j < 8; ++j) dma16(src + (size_t)4 * j * LIP_DIM, base + PSI_HAD + 1024 * (8 * w + j));
    }
#pragma unroll
    for (int j = 0; j < PSI_SLOTS - 1; ++j, ++c) {     // c = nch - 7 + j: 6 - j chunks and the matrix behind it
        ps_wait(2 * (PSI_SLOTS - 2 - j) + 8);
        __syncthreads();
        products(c, slot);
        slot = slot == PSI_SLOTS - 1 ? 0 : slot + 1;
    }
    VM_WAIT(0);
    __syncthreads();                                   // the matrix is there; every wave is done with the ring
    uint16_t *abf = reinterpret_cast<uint16_t *>(lds + PSI_RING);
    {
#pragma unroll
        for (int rg = 0; rg < 4; ++rg) {
            float f[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) f[j] = __fmul_rn(__fmul_rn((float)acc[4 * rg + j], ts), sc[rg][j]);
            *reinterpret_cast<u32x2 *>(abf + tl * HB_PITCH + 32 * w + 8 * rg + 4 * half) = u32x2{pack_bf16x2(f[0], f[1]), pack_bf16x2(f[2], f[3])};
        }
    }
    __syncthreads();                                   // the rows are complete
    const uint16_t *hmat = reinterpret_cast<const uint16_t *>(lds + PSI_HAD);
#pragma unroll
    for (int k0 = 0; k0 < PSI_ROT; k0 += 4) {          // (rows from T on are rotated along and dropped)
        if (4 * k0 >= p.T) break;
        uint32_t raw[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) raw[k] = *reinterpret_cast<const uint32_t *>(abf + (w + 4 * (k0 + k)) * HB_PITCH + 2 * l);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            float v0 = __uint_as_float(raw[k] << 16), v1 = __uint_as_float(raw[k] & 0xffff0000u);
            rope_pair(v0, v1, rc[k0 + k], rs[k0 + k], l);
            *reinterpret_cast<uint32_t *>(abf + (w + 4 * (k0 + k)) * HB_PITCH + 2 * l) = pack_bf16x2(v0, v1);
        }
    }
    __syncthreads();                                   // the rotated rows are complete
    lip_fixed_rows(abf, hmat, lds + PSI_SCRATCH, p.q_int8, p.q_scale, p.n_heads, head, p.T, w, l);
}

}  // namespace
}  // namespace pto
