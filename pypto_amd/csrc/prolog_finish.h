// What follows the projections of the two prologs (query rows: rope, Hadamard / absorb product, quantisation; key row and head
// weights of the indexer) as device functions over an LDS pool, so that the same code runs as a launch of its own and, for the
// fused operator, side by side in one launch.
// Included by lip_kernels.hip, mlap_kernels.hip and prolog_fused.hip after prolog_common.h.
#pragma once
#include "lip_kernels.h"
#include "mlap_kernels.h"
#include "prolog_common.h"

#pragma clang fp contract(off)

namespace pto {
namespace {

// the de-quantised int8 projection for columns col, col + 1 of token t, as bf16-valued floats: the unsplit form left
// them that way; the split form's partial sums are added and de-quantised here
__device__ __forceinline__ void q_value2(const int32_t *part, const int splits, const int T, const int t, const int ncols, const int col,
                                         const float ts, const float cs0, const float cs1, float &v0, float &v1)
{
    if (splits == 1) {
        const uint32_t v = *reinterpret_cast<const uint32_t *>(reinterpret_cast<const uint16_t *>(part) + (size_t)t * ncols + col);
        v0 = __uint_as_float(v << 16);
        v1 = __uint_as_float(v & 0xffff0000u);
        return;
    }
    int s0 = 0, s1 = 0;
#pragma unroll
    for (int kq = 0; kq < QPROJ_KSPLIT; ++kq) {
        const int2 v = *reinterpret_cast<const int2 *>(part + ((size_t)kq * T + t) * ncols + col);
        s0 += v.x;
        s1 += v.y;
    }
    v0 = bf16_round_f32(__fmul_rn(__fmul_rn((float)s0, ts), cs0));
    v1 = bf16_round_f32(__fmul_rn(__fmul_rn((float)s1, ts), cs1));
}

// ------------------------------------------------------------------------------ indexer prolog
// rope on channels 0..63 (lanes 0..31 hold channels 2l, 2l+1); the rotation partner of channel i is
// i+32 (negated) for i < 32 and i-32 otherwise: lane l ^ 16.  Results rounded to bf16.
__device__ __forceinline__ void rope_pair(float &v0, float &v1, const uint32_t c, const uint32_t s, const int l)
{
    const float p0 = xor16_f32(v0, l);
    const float p1 = xor16_f32(v1, l);
    if (l < 32) {
        const float sg = l < 16 ? -1.0f : 1.0f;
        // both products are exact, so the fused form rounds once, like product + product
        const float r0 = __builtin_fmaf(v0, __uint_as_float(c << 16), (sg * p0) * __uint_as_float(s << 16));
        const float r1 = __builtin_fmaf(v1, __uint_as_float(c & 0xffff0000u), (sg * p1) * __uint_as_float(s & 0xffff0000u));
        v0 = bf16_round_f32(r0);
        v1 = bf16_round_f32(r1);
    }
}
// the cos / sin pair of lane l (channels 2l, 2l+1 of token t); lanes 32..63 read lane l-32's, unused
__device__ __forceinline__ uint32_t rope_coef(const uint16_t *tab, const int t, const int l)
{
    return reinterpret_cast<const uint32_t *>(tab + (size_t)t * LIP_ROPE)[l & 31];
}

// y[j] = sum_i a[i] * H[i][j], i ascending; lane l computes columns 2l and 2l+1.  a: this wave's 128
// floats in LDS, hmat: the matrix in LDS as it is in memory (bf16, row-major; widened on the way into the
// registers, which costs two instructions per row and halves the workgroup's LDS).  Chunks of 16 rows are read
// one chunk ahead of the multiply-adds that consume them.
struct HadChunk {
    f32x4 a[4];
    f32x2 h[16];
};
__device__ __forceinline__ void had_load(HadChunk &c, const float *a, const uint16_t *hmat, const int l, const int i0)
{
#pragma unroll
    for (int u = 0; u < 4; ++u) c.a[u] = *reinterpret_cast<const f32x4 *>(a + i0 + 4 * u);
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        const uint32_t x = *reinterpret_cast<const uint32_t *>(hmat + (i0 + u) * LIP_DIM + 2 * l);
        c.h[u][0] = __uint_as_float(x << 16);
        c.h[u][1] = __uint_as_float(x & 0xffff0000u);
    }
}
__device__ __forceinline__ void had_fma(const HadChunk &c, float &o0, float &o1)
{
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        o0 = __builtin_fmaf(c.a[u >> 2][u & 3], c.h[u][0], o0);
        o1 = __builtin_fmaf(c.a[u >> 2][u & 3], c.h[u][1], o1);
    }
}
__device__ __forceinline__ void hadamard_pair(const float *a, const uint16_t *hmat, const int l, float &y0, float &y1)
{
    float o0 = 0.f, o1 = 0.f;
    HadChunk c0, c1;
    had_load(c0, a, hmat, l, 0);
#pragma unroll 1
    for (int i = 0; i < LIP_DIM; i += 32) {
        had_load(c1, a, hmat, l, i + 16);
        had_fma(c0, o0, o1);
        had_load(c0, a, hmat, l, i + 32 < LIP_DIM ? i + 32 : 0);
        had_fma(c1, o0, o1);
    }
    y0 = bf16_round_f32(o0);
    y1 = bf16_round_f32(o1);
}

// symmetric int8 quantisation of the wave's 128 values; returns the packed byte pair and the fp16 scale
__device__ __forceinline__ uint16_t quant_pair(const float y0, const float y1, uint16_t &scale_f16)
{
    const float amax = wave_max_f32(fmaxf(fabsf(y0), fabsf(y1)));
    float deq;
    const uint16_t q = quant_pair_amax(y0, y1, amax, deq);
    scale_f16 = (uint16_t)(pack_f16x2(deq, 0.f) & 0xffffu);
    return q;
}

constexpr int FIN_WAVES = 8;

// the 128x128 bf16 matrix into LDS, as it is (2048 pieces of 16 bytes over the workgroup's waves)
template <int WAVES>
__device__ __forceinline__ void stage_matrix(uint16_t *dst, const uint16_t *src)
{
    const u32x4 *s = reinterpret_cast<const u32x4 *>(src);
    u32x4 *d = reinterpret_cast<u32x4 *>(dst);
    constexpr int NT = 64 * WAVES;
#pragma unroll
    for (int i = 0; i < 2048 / NT; ++i) d[i * NT + threadIdx.x] = s[i * NT + threadIdx.x];
}

// a key row from its sums over the hidden axis (lane l: channels 2l, 2l+1): layer norm, rope, Hadamard product with the
// matrix in LDS (a: this wave's 128 floats of LDS), quantisation, scatter to cache row dst (skipped if out of range)
__device__ __forceinline__ void lip_key_row(const LipParams &p, const uint16_t *hmat, float *a, float v0, float v1, const uint32_t rc,
                                            const uint32_t rs, const uint32_t gm, const uint32_t bt, const long long dst, const int l)
{
    const float mean = __fmul_rn(pair_tree_sum(v0, v1), 1.0f / LIP_DIM);
    const float d0 = __fsub_rn(v0, mean), d1 = __fsub_rn(v1, mean);
    const float var = __fmul_rn(pair_tree_sum(__fmul_rn(d0, d0), __fmul_rn(d1, d1)), 1.0f / LIP_DIM);
    const float sd = __builtin_sqrtf(__fadd_rn(var, p.eps));   // correctly rounded (__fsqrt_rn is the 1-ulp hardware root here)
    v0 = bf16_round_f32(__fadd_rn(__fmul_rn(__fdiv_rn(d0, sd), __uint_as_float(gm << 16)), __uint_as_float(bt << 16)));
    v1 = bf16_round_f32(__fadd_rn(__fmul_rn(__fdiv_rn(d1, sd), __uint_as_float(gm & 0xffff0000u)), __uint_as_float(bt & 0xffff0000u)));
    rope_pair(v0, v1, rc, rs, l);
    f32x2 av = {v0, v1};
    *reinterpret_cast<f32x2 *>(&a[2 * l]) = av;
    float y0, y1;
    hadamard_pair(a, hmat, l, y0, y1);                 // the same wave wrote a: LDS operations of a wave stay in order
    uint16_t sc;
    const uint16_t q = quant_pair(y0, y1, sc);
    if (dst >= 0 && dst < p.cache_rows) {
        reinterpret_cast<uint16_t *>(p.k_cache + (size_t)dst * LIP_DIM)[l] = q;
        if (l == 0) p.k_cache_scale[dst] = sc;
    }
}
// head weight l of token t from its sum over the hidden axis
__device__ __forceinline__ void lip_weight(const LipParams &p, const int t, const int l, float v)
{
    v = __fmul_rn(__fmul_rn(bf16_round_f32(v), p.w_mul0), p.w_mul1);
    p.weights[(size_t)t * p.n_heads + l] = (uint16_t)(pack_f16x2(v, 0.f) & 0xffffu);
}

// Workgroups [0, q_wgs): FIN_WAVES query rows (token, head) each, one per wave.
// Workgroups [q_wgs, q_wgs + T): one token each -- waves add the groups of block sums over the hidden
// axis (two groups of eight blocks per wave and round), then wave 0 finishes the key row and wave 1 the
// weights row.
constexpr int LIP_FIN_LDS = LIP_DIM * LIP_DIM * 2 + FIN_WAVES * LIP_DIM * 4 + LIP_MAX_XGROUPS * LIP_XCOLS * 4;   // 55 296 bytes

// The work of workgroup wg of the second launch (64 * FIN_WAVES threads), in LIP_FIN_LDS bytes of LDS at lds.
__device__ __forceinline__ void lip_finish_body(const LipParams &p, const int q_wgs, const int wg, uint8_t *lds)
{
    uint16_t *hmat = reinterpret_cast<uint16_t *>(lds);
    float(*arow)[LIP_DIM] = reinterpret_cast<float(*)[LIP_DIM]>(lds + LIP_DIM * LIP_DIM * 2);
    float(*gsum)[LIP_XCOLS] = reinterpret_cast<float(*)[LIP_XCOLS]>(lds + LIP_DIM * LIP_DIM * 2 + FIN_WAVES * LIP_DIM * 4);
    const int l = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ncols = p.n_heads * LIP_DIM;

    if (wg < q_wgs) {
        stage_matrix<FIN_WAVES>(hmat, p.hq);
        const int row = wg * FIN_WAVES + w;            // (token, head)
        const bool live = row < p.T * p.n_heads;
        const int t = live ? row / p.n_heads : 0;
        const int head = live ? row % p.n_heads : 0;
        const int col = head * LIP_DIM + 2 * l;
        const float ts = p.q_norm_scale[t];
        const f32x2 cs = *reinterpret_cast<const f32x2 *>(p.w_qb_scale + col);
        const uint32_t rc = rope_coef(p.cos, t, l), rs = rope_coef(p.sin, t, l);
        float v0, v1;
        q_value2(p.qpart, qproj_splits(p.T), p.T, t, ncols, col, ts, cs[0], cs[1], v0, v1);
        rope_pair(v0, v1, rc, rs, l);
        f32x2 av = {v0, v1};
        *reinterpret_cast<f32x2 *>(&arow[w][2 * l]) = av;
        __syncthreads();
        float y0, y1;
        hadamard_pair(arow[w], hmat, l, y0, y1);
        uint16_t sc;
        const uint16_t q = quant_pair(y0, y1, sc);
        if (live) {
            reinterpret_cast<uint16_t *>(p.q_int8 + (size_t)row * LIP_DIM)[l] = q;
            if (l == 0) p.q_scale[row] = sc;
        }
        return;
    }

    const int t = wg - q_wgs;
    const bool group_rows = lip_x_group_rows(p);       // the rows are group sums already
    const int nblk = group_rows ? 0 : lip_xrows(p);
    const int ngroups = group_rows ? lip_xrows(p) : (nblk + LIP_XGROUP - 1) / LIP_XGROUP;
    stage_matrix<FIN_WAVES>(hmat, p.hk);
    const bool pl = l < p.n_heads;
    // everything wave 0 needs later is requested now
    const uint32_t rc = rope_coef(p.cos, t, l), rs = rope_coef(p.sin, t, l);
    const uint32_t gm = reinterpret_cast<const uint32_t *>(p.gamma)[l];
    const uint32_t bt = reinterpret_cast<const uint32_t *>(p.beta)[l];
    const long long dst = p.k_cache_index[t];
    if (group_rows) {
        for (int g = w; g < ngroups; g += FIN_WAVES) {
            const float *r = p.xpart + ((size_t)g * p.T + t) * LIP_XCOLS;
            *reinterpret_cast<f32x2 *>(&gsum[g][2 * l]) = *reinterpret_cast<const f32x2 *>(r + 2 * l);
            gsum[g][LIP_DIM + l] = r[LIP_DIM + (pl ? l : 0)];
        }
    }
    for (int g0 = w; g0 < ngroups && !group_rows; g0 += 2 * FIN_WAVES) {
        f32x2 kv[2][LIP_XGROUP];
        float wv[2][LIP_XGROUP];
        int nb[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int g = g0 + u * FIN_WAVES;
            const int left = nblk - g * LIP_XGROUP;
            nb[u] = left < 0 ? 0 : (left < LIP_XGROUP ? left : LIP_XGROUP);
            const float *src = p.xpart + ((size_t)(nb[u] ? g : 0) * LIP_XGROUP * p.T + t) * LIP_XCOLS;
#pragma unroll
            for (int i = 0; i < LIP_XGROUP; ++i) {
                const float *r = src + (size_t)(i < nb[u] ? i : 0) * p.T * LIP_XCOLS;
                kv[u][i] = *reinterpret_cast<const f32x2 *>(r + 2 * l);
                wv[u][i] = r[LIP_DIM + (pl ? l : 0)];
            }
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            if (nb[u] == 0) continue;
            float s0 = 0.f, s1 = 0.f, s2 = 0.f;
#pragma unroll
            for (int i = 0; i < LIP_XGROUP; ++i) {
                if (i < nb[u]) {
                    s0 = __fadd_rn(s0, kv[u][i][0]);
                    s1 = __fadd_rn(s1, kv[u][i][1]);
                    s2 = __fadd_rn(s2, wv[u][i]);
                }
            }
            const int g = g0 + u * FIN_WAVES;
            f32x2 sv = {s0, s1};
            *reinterpret_cast<f32x2 *>(&gsum[g][2 * l]) = sv;
            gsum[g][LIP_DIM + l] = s2;
        }
    }
    __syncthreads();
    if (w == 0) {
        float v0 = 0.f, v1 = 0.f;
        for (int g = 0; g < ngroups; ++g) {
            const f32x2 v = *reinterpret_cast<const f32x2 *>(&gsum[g][2 * l]);
            v0 = __fadd_rn(v0, v[0]);
            v1 = __fadd_rn(v1, v[1]);
        }
        lip_key_row(p, hmat, arow[0], v0, v1, rc, rs, gm, bt, dst, l);
    } else if (w == 1 && pl) {
        float v = 0.f;
        for (int g = 0; g < ngroups; ++g) v = __fadd_rn(v, gsum[g][LIP_DIM + l]);
        lip_weight(p, t, l, v);
    }
}

// The key rows and weights where the queries are finished by their projection's launch: a workgroup of four or eight waves takes as many tokens, one per wave (the
// matrix is staged once for all of them instead of once per token, and the rows are finished side by side instead of
// by one wave per workgroup).  A wave adds its token's partial rows in registers, in the order of the form they come
// in: group sums ascending, or blocks / ranges ascending into groups of eight and the groups ascending.
template <int WAVES> constexpr int LIP_FINT_LDS = LIP_DIM * LIP_DIM * 2 + WAVES * LIP_DIM * 4;

template <int WAVES>
__device__ __forceinline__ void lip_finish_tokens_prefill_body(const LipParams &p, const int wg, uint8_t *lds)
{
    uint16_t *hmat = reinterpret_cast<uint16_t *>(lds);
    float(*arow)[LIP_DIM] = reinterpret_cast<float(*)[LIP_DIM]>(lds + LIP_DIM * LIP_DIM * 2);
    const int l = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int t = wg * WAVES + w;
    const bool live = t < p.T;
    const int tt = live ? t : p.T - 1;
    stage_matrix<WAVES>(hmat, p.hk);
    const bool pl = l < p.n_heads;
    const uint32_t rc = rope_coef(p.cos, tt, l), rs = rope_coef(p.sin, tt, l);
    const uint32_t gm = reinterpret_cast<const uint32_t *>(p.gamma)[l];
    const uint32_t bt = reinterpret_cast<const uint32_t *>(p.beta)[l];
    const long long dst = live ? p.k_cache_index[tt] : -1;
    const bool group_rows = lip_x_group_rows(p);
    const int nrows = lip_xrows(p);
    const float *src = p.xpart + (size_t)tt * LIP_XCOLS;
    const size_t rstride = (size_t)p.T * LIP_XCOLS;
    float v0 = 0.f, v1 = 0.f, v2 = 0.f;
    for (int g0 = 0; g0 < nrows; g0 += LIP_XGROUP) {
        f32x2 kv[LIP_XGROUP];
        float wv[LIP_XGROUP];
        const int nb = nrows - g0 < LIP_XGROUP ? nrows - g0 : LIP_XGROUP;
#pragma unroll
        for (int i = 0; i < LIP_XGROUP; ++i) {
            const float *r = src + (size_t)(g0 + (i < nb ? i : 0)) * rstride;
            kv[i] = *reinterpret_cast<const f32x2 *>(r + 2 * l);
            wv[i] = r[LIP_DIM + (pl ? l : 0)];
        }
        if (group_rows) {
#pragma unroll
            for (int i = 0; i < LIP_XGROUP; ++i) {
                if (i < nb) {
                    v0 = __fadd_rn(v0, kv[i][0]);
                    v1 = __fadd_rn(v1, kv[i][1]);
                    v2 = __fadd_rn(v2, wv[i]);
                }
            }
        } else {
            float s0 = 0.f, s1 = 0.f, s2 = 0.f;
#pragma unroll
            for (int i = 0; i < LIP_XGROUP; ++i) {
                if (i < nb) {
                    s0 = __fadd_rn(s0, kv[i][0]);
                    s1 = __fadd_rn(s1, kv[i][1]);
                    s2 = __fadd_rn(s2, wv[i]);
                }
            }
            v0 = __fadd_rn(v0, s0);
            v1 = __fadd_rn(v1, s1);
            v2 = __fadd_rn(v2, s2);
        }
    }
    __syncthreads();                                   // the matrix is staged
    lip_key_row(p, hmat, arow[w], v0, v1, rc, rs, gm, bt, dst, l);
    if (pl && live) lip_weight(p, t, l, v2);
}


// A block of 32 query rows out of the Hadamard product (lane (row, half) holds channels 32*cb + 8*(r/4) + 4*half + r%4 of its
// row): rounded to bf16, quantised per row and left as int8 rows QFP_OPITCH bytes apart in the wave's staging area, from where
// they leave as whole 16-byte pieces.  Returns the row's de-quantisation scale.
constexpr int QFP_OPITCH = 144;
__device__ __forceinline__ float lip_quant_rows(f32x16 (&c)[4], uint8_t *mine, const int l)
{
    float amax = 0.f;
#pragma unroll
    for (int cb = 0; cb < 4; ++cb)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            c[cb][r] = bf16_round_f32(c[cb][r]);
            amax = fmaxf(amax, fabsf(c[cb][r]));
        }
    {
        const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(amax), __float_as_uint(amax), false, false);
        amax = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
    }
    float s = 0.f, deq = 0.f;
    if (amax > 0.f) {
        s = __fdiv_rn(127.0f, amax);
        deq = __fdiv_rn(1.0f, s);
    }
    uint8_t *orow = mine + (l & 31) * QFP_OPITCH + 4 * (l >> 5);
#pragma unroll
    for (int cb = 0; cb < 4; ++cb)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            uint32_t v = 0;
#pragma unroll
            for (int j = 0; j < 4; ++j) v |= (uint32_t)((int)rintf(__fmul_rn(c[cb][4 * g + j], s)) & 0xff) << (8 * j);
            *reinterpret_cast<uint32_t *>(orow + 32 * cb + 8 * g) = v;
        }
    return deq;
}

// The same from the Hadamard product's operands, with its sums in their fixed order: 32 rows of rotated query channels (bf16,
// HB_PITCH elements apart) times the matrix (row r at 256 * r bytes, 16-byte piece q at q ^ 4*(r & 3)), both in LDS, by a workgroup
// of four waves; the first T rows leave for rows 0 .. T - 1 of q_int8 and q_scale at head `head`.  v_mfma_f32_4x4x1_16b_f32
// multiplies one row of the matrix at a time, so each of its results is one exact product added with one rounding (as in
// xlinear_fixed.h) and a chain of 128 is the sequential sum.  Its sixteen blocks are 64 columns of the matrix (wave w: 64*(w & 1)
// ..) and all take the same four rows: one register holds 16 channels of them, block k's lanes channel k, which the instruction
// broadcasts.  A wave makes four rows up to 8 tokens, eight up to 16, else sixteen, as that many chains side by side.
// Bound: the matrix cores' fp32 rate, 15 clocks per link and chain.  With the sums, by clock stamps: 8 tokens 2.2 us, 16: 2.7, 32: 3.9
// (v_mfma_f32_16x16x1_4b_f32, whose chains are of 16 rows: 4.0 at any number of tokens); on the vector ALU, a wave per row, the
// fused prolog took 9 us longer at 32 tokens.
constexpr int HB_PITCH = LIP_DIM + 8;
constexpr int HB_SCRATCH = 32 * HB_PITCH * 2;
template <int G, int K>
__device__ __forceinline__ void had_links(f32x4 (&c)[G], const float (&a)[G][LIP_DIM / 16], const int kk, const u32x2 (&h)[4])
{
    const uint32_t hw = h[K >> 2][(K >> 1) & 1];
    const float hv = __uint_as_float((K & 1) ? hw & 0xffff0000u : hw << 16);
#pragma unroll
    for (int g = 0; g < G; ++g) c[g] = __builtin_amdgcn_mfma_f32_4x4x1f32(a[g][kk], hv, c[g], 4, K, 0);
    if constexpr (K < 15) had_links<G, K + 1>(c, a, kk, h);
}
// rows 4*G*(w / 2) .. +4*G-1, columns 64*(w & 1) .. +63 of the product, rounded to bf16, into out (HB_PITCH elements a row)
template <int G>
__device__ __forceinline__ void had_fixed_sums(const uint16_t *rows, const uint16_t *hmat, uint16_t *out, const int w, const int l)
{
    const int i = l & 15, q = l >> 4, row0 = 4 * G * (w >> 1);
    f32x4 c[G];
    float a[G][LIP_DIM / 16];
#pragma unroll
    for (int g = 0; g < G; ++g) {
        c[g] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < LIP_DIM / 16; ++kk) a[g][kk] = bf16_bits_to_f32(rows[(row0 + 4 * g + (l & 3)) * HB_PITCH + 16 * kk + (l >> 2)]);
    }
    // a transposing read leaves lane i of sixteen column i of four rows
    const uint16_t *hp = hmat + (i >> 2) * LIP_DIM + 8 * ((8 * (w & 1) + 2 * q + ((i & 3) >> 1)) ^ (4 * (i >> 2))) + 4 * (i & 1);
#pragma unroll
    for (int kk = 0; kk < LIP_DIM / 16; ++kk) {
        u32x2 h[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) h[j] = __builtin_bit_cast(u32x2, lds_read_tr16(hp + (16 * kk + 4 * j) * LIP_DIM));
        had_links<G, 0>(c, a, kk, h);
    }
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            out[(row0 + 4 * g + r) * HB_PITCH + 64 * (w & 1) + l] = (uint16_t)(pack_bf16x2(c[g][r], 0.f) & 0xffffu);
}
// scratch: HB_SCRATCH bytes that nothing else of the workgroup uses.  The rows and the matrix have to be complete (barrier).
__device__ __forceinline__ void lip_fixed_rows(const uint16_t *rows, const uint16_t *hmat, uint8_t *scratch, int8_t *q_int8, uint16_t *q_scale,
                                               const int n_heads, const int head, const int T, const int w, const int l)
{
    uint16_t *out = reinterpret_cast<uint16_t *>(scratch);
    if (T <= 8) had_fixed_sums<1>(rows, hmat, out, w, l);
    else if (T <= 16) had_fixed_sums<2>(rows, hmat, out, w, l);
    else had_fixed_sums<4>(rows, hmat, out, w, l);
    __syncthreads();                                   // the product's rows are complete
    if (8 * w >= T) return;
    // eight lanes a row, sixteen columns each
    const int row = 8 * w + (l >> 3);
    const uint16_t *src = out + row * HB_PITCH + 16 * (l & 7);
    const u32x4 d[2] = {*reinterpret_cast<const u32x4 *>(src), *reinterpret_cast<const u32x4 *>(src + 8)};
    float v[16], amax = 0.f;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        const uint32_t x = d[e >> 3][(e & 7) >> 1];
        v[e] = __uint_as_float((e & 1) ? x & 0xffff0000u : x << 16);
        amax = fmaxf(amax, fabsf(v[e]));
    }
    amax = fmaxf(amax, dpp_f32<DPP_XOR1>(amax));
    amax = fmaxf(amax, dpp_f32<DPP_XOR2>(amax));
    amax = fmaxf(amax, dpp_f32<DPP_HALF_MIRROR>(amax));
    float s = 0.f, deq = 0.f;
    if (amax > 0.f) {
        s = __fdiv_rn(127.0f, amax);
        deq = __fdiv_rn(1.0f, s);
    }
    u32x4 o;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        uint32_t x = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) x |= (uint32_t)((int)rintf(__fmul_rn(v[4 * g + j], s)) & 0xff) << (8 * j);
        o[g] = x;
    }
    if (row < T) {
        *reinterpret_cast<u32x4 *>(q_int8 + ((size_t)row * n_heads + head) * LIP_DIM + 16 * (l & 7)) = o;
        if ((l & 7) == 0) q_scale[(size_t)row * n_heads + head] = (uint16_t)(pack_f16x2(deq, 0.f) & 0xffffu);
    }
}

// ---------------------------------------------------------------------------------- MLA prolog
constexpr int FIN_W_BYTES = MLAP_NOPE * 64 * 2;    // a wave's slice of w_uk[head]: 128 rows x 64 columns bf16
constexpr int MLAP_FIN_LDS = 4 * FIN_W_BYTES + MLAP_XTOK * MLAP_NOPE * 4;   // 69 632 bytes

// The MLA prolog's last stage with every sum in its fixed order (absorb_exact; otherwise the projection's launch finishes its heads
// itself: prolog_small.h, prolog_prefill.h).  Workgroup (head, half of the 512 output columns, block of 8 tokens); wave w
// owns output columns colbase + 64w + l.
// The work of workgroup wg of the last launch (256 threads), in MLAP_FIN_LDS bytes of LDS at lds.
// workgroup barriers mlap_finish_body passes (every thread, unconditionally): a launch whose workgroups hold more
// than this body's 256 threads lets the surplus waves pass as many and leave
constexpr int MLAP_FIN_BARRIERS = 1;
__device__ __forceinline__ void mlap_finish_body(const MlapParams &p, const int wg, uint8_t *lds)
{
    uint8_t *wsl = lds;
    float(*arow)[MLAP_NOPE] = reinterpret_cast<float(*)[MLAP_NOPE]>(lds + 4 * FIN_W_BYTES);
    const int l = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int head = wg % p.n_heads;
    const int half = (wg / p.n_heads) & 1;
    const int t0 = (wg / p.n_heads / 2) * MLAP_XTOK;
    const int ncols = p.n_heads * MLAP_QHEAD;
    const int colbase = half * 256 + 64 * w;

    {   // this wave's slice: rows of 128 bytes, pitch 1024 bytes: 8 lanes per row, 8 rows per request
        const uint8_t *src = reinterpret_cast<const uint8_t *>(p.w_uk) + ((size_t)head * MLAP_NOPE + (l >> 3)) * (MLAP_KV * 2) +
                             colbase * 2 + 16 * (l & 7);
        const uint32_t dst = (uint32_t)(uintptr_t)(lds_byte_t *)(wsl + w * FIN_W_BYTES);
#pragma unroll 1
        for (int i = 0; i < MLAP_NOPE / 8; ++i) dma16(src + (size_t)i * 8 * MLAP_KV * 2, dst + 1024 * i);
    }
    // the head's query channels of tokens t0 + w and t0 + 4 + w: partial sums added, de-quantised, bf16
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int tl = 4 * u + w;
        const int t = t0 + tl;
        const int tt = t < p.T ? t : p.T - 1;
        const float ts = p.q_norm_scale[tt];
        // nope part: lane l -> channels 2l, 2l+1
        {
            const int col = head * MLAP_QHEAD + 2 * l;
            const f32x2 cs = *reinterpret_cast<const f32x2 *>(p.w_qb_scale + col);
            float av0, av1;
            q_value2(p.qpart, mlap_qsplits(p), p.T, tt, ncols, col, ts, cs[0], cs[1], av0, av1);
            const f32x2 av = {av0, av1};
            *reinterpret_cast<f32x2 *>(&arow[tl][2 * l]) = av;
        }
        // rope part (first half-workgroup only): lane l < 32 -> channels 2l, 2l+1 = rotation partners l, 32+l
        if (half == 0 && l < 32 && t < p.T) {
            const int col = head * MLAP_QHEAD + MLAP_NOPE + 2 * l;
            const f32x2 cs = *reinterpret_cast<const f32x2 *>(p.w_qb_scale + col);
            float v0, v1;
            q_value2(p.qpart, mlap_qsplits(p), p.T, t, ncols, col, ts, cs[0], cs[1], v0, v1);
            const float c0 = bf16_bits_to_f32(p.cos[(size_t)t * MLAP_ROPE + l]), c1 = bf16_bits_to_f32(p.cos[(size_t)t * MLAP_ROPE + 32 + l]);
            const float sn0 = bf16_bits_to_f32(p.sin[(size_t)t * MLAP_ROPE + l]), sn1 = bf16_bits_to_f32(p.sin[(size_t)t * MLAP_ROPE + 32 + l]);
            const float r0 = __builtin_fmaf(v0, c0, (-v1) * sn0);
            const float r1 = __builtin_fmaf(v1, c1, v0 * sn1);
            uint16_t *out = p.q_rope + ((size_t)t * p.n_heads + head) * MLAP_ROPE;
            out[l] = (uint16_t)(pack_bf16x2(r0, 0.f) & 0xffffu);
            out[32 + l] = (uint16_t)(pack_bf16x2(r1, 0.f) & 0xffffu);
        }
    }
    VM_WAIT(0);
    __syncthreads();                                   // (counted in MLAP_FIN_BARRIERS)

    // out[t][colbase + 64w + l] = sum_i a[t][i] * w_uk[head][i][col], i ascending; 8 tokens at once.
    // Chunks of four rows are read one chunk ahead of the multiply-adds that consume them.
    const uint16_t *wl = reinterpret_cast<const uint16_t *>(wsl + w * FIN_W_BYTES) + l;
    float acc[MLAP_XTOK];
#pragma unroll
    for (int t = 0; t < MLAP_XTOK; ++t) acc[t] = 0.f;
    struct Chunk {
        f32x4 a[MLAP_XTOK];
        uint16_t w[4];
    };
    auto load = [&](Chunk &c, const int i) {
#pragma unroll
        for (int t = 0; t < MLAP_XTOK; ++t) c.a[t] = *reinterpret_cast<const f32x4 *>(&arow[t][i]);
#pragma unroll
        for (int j = 0; j < 4; ++j) c.w[j] = wl[(i + j) * 64];
    };
    auto fma = [&](const Chunk &c) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float wv = bf16_bits_to_f32(c.w[j]);
#pragma unroll
            for (int t = 0; t < MLAP_XTOK; ++t) acc[t] = __builtin_fmaf(c.a[t][j], wv, acc[t]);
        }
    };
    Chunk c0, c1;
    load(c0, 0);
#pragma unroll 1
    for (int i = 0; i < MLAP_NOPE; i += 8) {
        load(c1, i + 4);
        fma(c0);
        load(c0, i + 8 < MLAP_NOPE ? i + 8 : 0);
        fma(c1);
    }
#pragma unroll
    for (int t = 0; t < MLAP_XTOK; ++t)
        if (t0 + t < p.T)
            p.q_nope[((size_t)(t0 + t) * p.n_heads + head) * MLAP_KV + colbase + l] = (uint16_t)(pack_bf16x2(acc[t], 0.f) & 0xffffu);
}

}  // namespace
}  // namespace pto
