// Lightning indexer (decode), gfx950 (MI355X): key scoring and top-k select.
//
// Semantics: lightning_indexer_decode_compute of the reference example
// (examples/models/deepseek_v32_exp/lightning_indexer_quant_impl.py:138-312), golden
// deepseekv32_lightning_indexer_quant.py:184-269:
//   x[h, j]  = fp16_rne(relu(q[h,:] . k[j,:]) / 2048)                int8 dot, exact in int32
//   score[j] = (sum_h w_scale[h] * x[h, j]) * k_scale[j]             fp32
// with the two orders the golden leaves to its libraries fixed as: head sum h ascending with the
// product rounded before the add (no fused multiply-add); select order (score descending, position
// ascending), -0.0 == +0.0.
//
// Kernels
//   li_score_kernel   w_scale[h] = fp16(q_scale * weight) if both fp16, else the fp32 product;
//                     one wave per run of 64-key pairs of blocks: the key rows travel from the paged
//                     cache into the wave's own LDS buffers by LDS-DMA (whole cache lines, two pairs
//                     ahead), v_mfma_i32_32x32x32_i8 with A = the token's 64 query heads (two 32-row
//                     operands resident in registers) and B = 32 key rows read from LDS in operand
//                     layout; a half-wave swap gives every lane all 64 heads of one key, summed in
//                     registers with the per-head factors in scalar registers; scores to a
//                     [T, max_seq] fp32 workspace, and one score of every 16 positions to a compact
//                     sample array behind it
//   li_select_kernel  one workgroup per query token, keys ordered by the strict word
//                     (score image << 32 | ~position): a histogram of up to 4096 sampled scores (the
//                     compact array the score kernel left) gives a pivot, one pass over the row
//                     compacts the keys above it (a row of up to 8192 keys skips both: all its keys are
//                     candidates), those are spread over 8192 buckets linear in the
//                     score and ordered inside buckets by counting; select_streaming (radix select
//                     over the row in memory + bitonic sort) is the capacity-free form it falls back to
#include <type_traits>

#include "common.h"
#include "li_kernels.h"
#include "pypto_amd_sfa.h"

// The head sum is defined as a rounded multiply followed by a rounded add.  __fmul_rn/__fadd_rn are
// plain operators to the compiler, so contraction is switched off for this whole file.  The pragma
// is honoured only when the file is compiled with -ffp-contract=on or off: hipcc's default, "fast",
// lets the backend fuse regardless.
#pragma clang fp contract(off)

namespace pto {
namespace {


// one scale or weight as it lies in memory, and its value: the conversion apart, so that several loads are on their way at once
__device__ __forceinline__ uint32_t load_raw(const void *p, const size_t i, const int dt)
{
    return dt == PTO_DT_FP32 ? static_cast<const uint32_t *>(p)[i] : static_cast<const uint16_t *>(p)[i];
}
__device__ __forceinline__ float raw_to_f32(const uint32_t raw, const int dt)
{
    if (dt == PTO_DT_FP32) return __uint_as_float(raw);
    return dt == PTO_DT_BF16 ? bf16_bits_to_f32((uint16_t)raw) : (float)__builtin_bit_cast(_Float16, (uint16_t)raw);
}

// n / d for n < 2^18 and inv = 1 / d to one unit in the last place: (n + 1/2) / d is no nearer to an integer than 1 / (2 d)
__device__ __forceinline__ int small_quotient(const int n, const float inv) { return (int)(((float)n + 0.5f) * inv); }

// order-preserving image of a score: larger score <=> larger key; -0.0 and +0.0 map to one key
__device__ __forceinline__ uint32_t score_key(const float x)
{
    uint32_t u = __float_as_uint(x);
    u = u == 0x80000000u ? 0u : u;
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// Wave-wide scan and reductions on DPP (no LDS traffic).  row_shr:n moves a value n lanes up inside
// its row of 16, row_bcast15/31 carry the last lane of a row / of the lower half-wave upward; lanes
// without a source keep the identity passed as the old value.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ uint32_t dpp_u32(const uint32_t identity, const uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_update_dpp((int)identity, (int)v, CTRL, ROW_MASK, 0xf, false);
}

// inclusive prefix sum over the 64 lanes
__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v)
{
    v += dpp_u32<0x111, 0xf>(0u, v);
    v += dpp_u32<0x112, 0xf>(0u, v);
    v += dpp_u32<0x114, 0xf>(0u, v);
    v += dpp_u32<0x118, 0xf>(0u, v);
    v += dpp_u32<0x142, 0xa>(0u, v);
    v += dpp_u32<0x143, 0xc>(0u, v);
    return v;
}

// the same within each row of sixteen lanes, and the minimum and maximum of a row in all of its lanes
__device__ __forceinline__ uint32_t row_incl_scan(uint32_t v)
{
    v += dpp_u32<0x111, 0xf>(0u, v);
    v += dpp_u32<0x112, 0xf>(0u, v);
    v += dpp_u32<0x114, 0xf>(0u, v);
    v += dpp_u32<0x118, 0xf>(0u, v);
    return v;
}

template <typename Op>
__device__ __forceinline__ float row_reduce(float v, Op op)
{
    v = op(v, __uint_as_float(dpp_u32<0x128, 0xf>(0u, __float_as_uint(v))));     // row_ror: 8, 4, 2, 1
    v = op(v, __uint_as_float(dpp_u32<0x124, 0xf>(0u, __float_as_uint(v))));
    v = op(v, __uint_as_float(dpp_u32<0x122, 0xf>(0u, __float_as_uint(v))));
    v = op(v, __uint_as_float(dpp_u32<0x121, 0xf>(0u, __float_as_uint(v))));
    return v;
}

template <typename Op>
__device__ __forceinline__ uint32_t wave_reduce_bits(uint32_t v, const uint32_t identity, Op op)
{
    v = op(v, dpp_u32<0x111, 0xf>(identity, v));
    v = op(v, dpp_u32<0x112, 0xf>(identity, v));
    v = op(v, dpp_u32<0x114, 0xf>(identity, v));
    v = op(v, dpp_u32<0x118, 0xf>(identity, v));
    v = op(v, dpp_u32<0x142, 0xa>(identity, v));
    v = op(v, dpp_u32<0x143, 0xc>(identity, v));
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);     // lane 63 holds the reduction of all lanes
}

__device__ __forceinline__ float wave_min(const float x)
{
    return __uint_as_float(wave_reduce_bits(__float_as_uint(x), 0x7f800000u, [](uint32_t a, uint32_t b) {
        return __float_as_uint(fminf(__uint_as_float(a), __uint_as_float(b)));
    }));
}

__device__ __forceinline__ float wave_max(const float x)
{
    return __uint_as_float(wave_reduce_bits(__float_as_uint(x), 0xff800000u, [](uint32_t a, uint32_t b) {
        return __float_as_uint(fmaxf(__uint_as_float(a), __uint_as_float(b)));
    }));
}

__device__ __forceinline__ uint32_t wave_max_u32(const uint32_t x)
{
    return wave_reduce_bits(x, 0u, [](uint32_t a, uint32_t b) { return a > b ? a : b; });
}

// fp32 product of one half of a packed fp16 pair with a wave-uniform fp32 factor, rounded once:
// v_fma_mix_f32 widens the fp16 operand on the fly.  The addend +0 turns a product of -0 into +0, which
// no later step can tell apart: the running sum starts at +0 and so never is -0 itself.
template <int HI>
__device__ __forceinline__ float mul_f16_f32(const uint32_t packed, const float w)
{
    float r;
    if (HI)
        asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(packed), "s"(w));
    else
        asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel:[0,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(packed), "s"(w));
    return r;
}

// the same with the factor in a vector register (read from LDS)
template <int HI>
__device__ __forceinline__ float mul_f16_f32_v(const uint32_t packed, const float w)
{
    float r;
    if (HI)
        asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(packed), "v"(w));
    else
        asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel:[0,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(packed), "v"(w));
    return r;
}

// sum + x * w for one half each of two packed fp16 pairs (the second wave-uniform), rounded once.  The product of two fp16
// values is exact in fp32, so this is the rounded multiply followed by the rounded add of the definition.
template <int HI>
__device__ __forceinline__ void fma_f16_pair(float &sum, const uint32_t x, const uint32_t w)
{
    if (HI)
        asm("v_fma_mix_f32 %0, %1, %2, %0 op_sel:[1,1,0] op_sel_hi:[1,1,0]" : "+v"(sum) : "v"(x), "s"(w));
    else
        asm("v_fma_mix_f32 %0, %1, %2, %0 op_sel:[0,0,0] op_sel_hi:[1,1,0]" : "+v"(sum) : "v"(x), "s"(w));
}

// x = fp16(relu(dot) / 2048) for two dots, packed.  The integer accumulators start at the bit pattern of 4.0f (DOT_ZERO, an
// operand the matrix instruction reads anyway), so that a sum's bits read as a float are 4 + dot * 2^-21 for dot >= 0 and
// 4 + dot * 2^-22 below: times 1024 less 4096 is dot / 2048 exactly, or something negative, without a conversion.  The pair is
// rounded once to fp16 (v_cvt_pk_f16_f32) and a packed integer max clears the negative ones.  (v_fma_mixlo/mixhi_f16, which
// write half a register, issue at half the rate: 9.2 clocks against 5.3.)
constexpr int DOT_ZERO = 0x40800000;
__device__ __forceinline__ uint32_t relu_fp16_pair(const int d0, const int d1)
{
    const uint32_t packed = pack_f16x2(__builtin_fmaf(__int_as_float(d0), 1024.f, -4096.f), __builtin_fmaf(__int_as_float(d1), 1024.f, -4096.f));
    // relu on the bit patterns: a negative fp16 (and -0) is a negative 16-bit integer
    typedef __attribute__((ext_vector_type(2))) short s16x2;
    const s16x2 zero = {0, 0};
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(s16x2, packed), zero));
}

// fp16(dot / 2048) for two dots, packed, sign kept
__device__ __forceinline__ uint32_t fp16_pair(const int d0, const int d1, const float scale)
{
    uint32_t packed;
    asm("v_fma_mixlo_f16 %0, %1, %2, 0" : "=v"(packed) : "v"((float)d0), "s"(scale));
    asm("v_fma_mixhi_f16 %0, %1, %2, 0" : "+v"(packed) : "v"((float)d1), "s"(scale));
    return packed;
}

// two heads of one key: ((x * q_scale) * k_scale, ReLU) * weight, every product rounded to fp16
__device__ __forceinline__ uint32_t dequant_relu_weight(const uint32_t x, const uint32_t qs, const uint32_t ks, const uint32_t w)
{
    typedef __attribute__((ext_vector_type(2))) short s16x2;
    f16x2 v = __builtin_bit_cast(f16x2, x) * __builtin_bit_cast(f16x2, qs);
    v = v * __builtin_bit_cast(f16x2, ks);
    const s16x2 zero = {0, 0};
    v = __builtin_bit_cast(f16x2, __builtin_elementwise_max(__builtin_bit_cast(s16x2, v), zero));
    return __builtin_bit_cast(uint32_t, v * __builtin_bit_cast(f16x2, w));
}

// Sample for the select: of every 16 consecutive positions that all lie inside the sequence, the score
// of one (picked by a hash of the group number) is also written to a compact array, so that the select
// kernel finds a sample of the row in a few contiguous cache lines instead of thousands of scattered ones.
__device__ __forceinline__ bool sample_lane(const int pos, const int cur)
{
    const uint32_t g = (uint32_t)pos >> 4;
    return (uint32_t)(pos & 15) == ((g * 2654435761u) >> 28) && (int)(16u * g + 15u) < cur;
}

constexpr int SC_PAIR_BYTES = 64 * LI_DIM;     // key rows of one staged pair of 32-key blocks
constexpr int SC_BUF_BYTES = SC_PAIR_BYTES + 256;   // + the 64 key scales (one dword per lane)

// One wave scores runs of 64 consecutive keys: two 32-key blocks X and Y per trip.
//   stage  key rows travel from the paged cache into the wave's own LDS buffers with
//          global_load_lds: consecutive lanes fetch consecutive 16-byte chunks, so every request is a
//          run of whole cache lines (loading the operand layout directly touches 32 lines with 32
//          bytes each per instruction and is bound by the address unit).  Chunk c of row r lands at
//          position c ^ ((r >> 1) & 7) of the row: the LDS serves sixteen lanes of an operand read at a time, two
//          rows of 128 bytes span its banks, so any sixteen rows meet every bank once (with c ^ (r & 7) rows
//          eight apart met in the same banks and every read took twice as long).  The
//          pair after the current one is in flight while the current one is scored.
//   MFMA   A = the token's 64 query heads as two 32-row operands (resident in registers), B = 32 key
//          rows read from LDS in operand layout; four accumulators per trip.  With the head
//          permutation below, lane (j, half) of block X's accumulators holds heads 32*half ..
//          32*half + 31 of key X_j, likewise for Y.
//   swap   after relu / scale / fp16 packing, v_permlane32_swap exchanges the upper half-wave of X's
//          registers with the lower half-wave of Y's: lane j < 32 then holds all 64 heads of key X_j
//          and lane 32 + j all 64 heads of key Y_j, the same head in the same register on every lane.
//   sum    every lane runs the sequential head sum h = 0..63 of its own key; the per-head factors are
//          wave-uniform and sit in scalar registers.
// At least two waves per SIMD: the 256 registers that leaves per lane are all architectural, so the
// matrix instructions accumulate in ordinary vector registers and the epilogue reads them directly.
// KDT = dtype code of the key scales: a compile-time choice keeps the scale load free of branches, so
// it stays in flight beside the staged rows.
// VAR = 1: the arithmetic of the reference's chained C++ operator (LightningIndexerTopkImpl,
// framework/src/operator/models/deepseek_v3.2_exp/lightning_indexer.cpp:149-197): fp16(dot/2048) is
// multiplied in fp16 by the head's query scale and by the key's scale before the ReLU, then in fp16 by
// the head's weight; the fp32 head sum (h ascending) is the score.  All three tensors are fp16 then.
// NT = query tokens of one sequence a wave scores per key pass (1 or 2): the reference scores all s1 tokens of
// a batch against a page in one matrix product (lightning_indexer_quant_impl.py:163-169, [S1*64, 128]); here
// a "unit" is a pair of consecutive tokens of a sequence (s1 is even), every staged
// key row and scale serves both, and their per-head factors sit in LDS instead of scalar registers.
// A workgroup of eight waves per compute unit, and nothing in front of the first requests that need not be there: as two workgroups of
// four the second one's sequence lengths came back behind the first one's key rows (7 us, and it ended as much later), the
// mapping took 2.3 us of divisions, and the queries, asked for behind two pairs of every wave, arrived behind 34 MB.  Kernel over
// rotating key caches, before / now: 4 tokens x 32 K keys 10.5 / 6.8 us, 32 x 8-64 K 36.9 / 31.1, 64 pairs of tokens x 4-32 K 44.8 / 40.5.
// (Pairs of a workgroup's runs drawn by whichever wave comes first, so that its waves end together instead of up to 8 us apart: +-0.
// Bound now: the first one by its bytes, 28.4 us with nothing but the requests and stores; the other by vector work and the
// products beside it, two waves to a SIMD.)
// HW: query scales and weights are fp16, so the per-head factors are fp16 values, their products with x exact and the head
// sum one instruction per head instead of two; the factors sit in scalar registers as packed pairs, for two tokens as well.
template <int KDT, int VAR = 0, int NT = 1, bool HW = false>
__global__ __launch_bounds__(64 * LI_SCORE_WAVES) __attribute__((amdgpu_waves_per_eu(2))) void li_score_kernel(const LiParams p)
{
    __shared__ __attribute__((aligned(16))) int8_t kstage[LI_SCORE_WAVES][2][SC_BUF_BYTES];
    __shared__ __attribute__((aligned(16))) float wsc_lds[NT > 1 && !HW ? LI_SCORE_WAVES : 1][NT][LI_HEADS];
    static_assert(SC_PAIR_BYTES == LI_HEADS * LI_DIM, "a token's query is staged where a pair of key blocks goes later");
    const int upb = p.S1 / NT;                       // units per sequence (two tokens to a unit: S1 is even)
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l = threadIdx.x & 63;
    const int j = l & 31;
    const int half = l >> 5;
    const int cap = p.maxblk * p.bs;
    auto clamped = [&](const int n) { return n < 0 ? 0 : (n > cap ? cap : n); };
    int unit, b, cur, key0, ppw;
    if (p.balanced) {
        // Balanced mapping: the launch has a fixed number of waves; every wave reads all sequence lengths, sizes the runs so that
        // the runs of all units just fill the launch, and takes the gw-th run.  Short and long sequences then cost the same number
        // of trips per wave and the whole pass is one round of resident waves.  The units of a sequence take the same run side by
        // side, mostly in one workgroup, so that its keys come from memory once: unit after unit, 4 x 2 tokens of 8 to 64 K keys took
        // 23.8 us instead of 21.7, 20 x 3 49.3 instead of 42.9, two tokens to a unit either way.  (Nothing is on its way
        // from memory meanwhile, so it is kept short: divisions by reciprocals, and for up to 64 sequences a single row of the table.)
        const int gw = blockIdx.x * LI_SCORE_WAVES + w;
        int found = -1, found_run = 0, found_len = 0;
        auto balance = [&](auto rows_tag) __attribute__((always_inline)) {
            constexpr int ROWS = decltype(rows_tag)::value;          // of 64 sequences each
            int len[ROWS], pairs[ROWS], total = 0;
#pragma unroll
            for (int i = 0; i < ROWS; ++i) {
                const int seq = l + 64 * i;
                len[i] = p.act[seq < p.B ? seq : p.B - 1];
            }
#pragma unroll
            for (int i = 0; i < ROWS; ++i) {
                len[i] = l + 64 * i < p.B ? clamped(len[i]) : 0;
                pairs[i] = (len[i] + 63) >> 6;
                total += pairs[i] * upb;
            }
            total = __builtin_amdgcn_readlane((int)wave_incl_scan((uint32_t)total), 63);
            // as few whole rounds as runs of the greatest length need (the launch has as many as the longest sequences would)
            int nwaves = p.round_waves;
            while (total > nwaves * LI_MAX_PAIRS_PER_WAVE && nwaves < (int)gridDim.x * LI_SCORE_WAVES) nwaves += p.round_waves;
            // the shortest run length whose runs fit the launch: every unit may waste one run on rounding
            ppw = (int)((float)(total + nwaves - 1) * __builtin_amdgcn_rcpf((float)nwaves));
            ppw = ppw < 1 ? 1 : (ppw > LI_MAX_PAIRS_PER_WAVE ? LI_MAX_PAIRS_PER_WAVE : ppw);
            for (;;) {
                const float inv_ppw = __builtin_amdgcn_rcpf((float)ppw);
                int base = 0;                 // runs of all sequences before row i of the table
#pragma unroll
                for (int i = 0; i < ROWS; ++i) {
                    const int runs = small_quotient(pairs[i] + ppw - 1, inv_ppw) * upb;
                    const int incl = (int)wave_incl_scan((uint32_t)runs);
                    const int run = gw - (base + incl - runs);
                    if (run >= 0 && run < runs) {
                        found = l + 64 * i;
                        found_run = run;
                        found_len = len[i];
                    }
                    base += __builtin_amdgcn_readlane(incl, 63);
                }
                if (base <= nwaves || ppw >= LI_MAX_PAIRS_PER_WAVE) break;
                ++ppw;
                found = -1;
            }
        };
        if (p.B <= 64) balance(std::integral_constant<int, 1>{});
        else balance(std::integral_constant<int, LI_MAX_BALANCED_SEQS / 64>{});
        const unsigned long long hit = __ballot(found >= 0);
        if (hit == 0ull) return;          // more waves than runs
        const int src = __ffsll((long long)hit) - 1;
        b = __builtin_amdgcn_readlane(found, src);
        cur = __builtin_amdgcn_readlane(found_len, src);
        const int of_seq = __builtin_amdgcn_readlane(found_run, src);
        const int run = upb == 1 ? of_seq : __builtin_amdgcn_readfirstlane(small_quotient(of_seq, __builtin_amdgcn_rcpf((float)upb)));
        unit = b * upb + of_seq - run * upb;
        key0 = run * (ppw * 64);
    } else {
        // runs of a fixed length, a sequence's units side by side here too and its waves next to the next one's (every unit in workgroups
        // of its own: 520 x 3 tokens of 1 to 4 K keys 240 us, of 3 to 4 K 252, 1200 x 4 of up to 1.5 K 409, now 157, 176 and 227; every
        // sequence in workgroups of its own 215, 261 and 267)
        ppw = p.ppw;
        const int gw = (int)blockIdx.x * LI_SCORE_WAVES + w;
        b = gw / p.seq_waves;
        if (b >= p.B) return;
        const int of_seq = gw - b * p.seq_waves;
        const int run = of_seq / upb;
        unit = b * upb + of_seq - run * upb;
        key0 = run * (ppw * 64);
        cur = clamped(p.act[b]);
    }
    const int t = b * p.S1 + (unit - b * upb) * NT;               // the unit's first token
    if (key0 >= cur) return;
    int npair = (cur - key0 + 63) >> 6;
    npair = npair > ppw ? ppw : npair;
    const int last_blk = ((cur + 31) >> 5) - 1;                  // last 32-key block holding a valid key

    // Per-head factors: lane l loads head l's (HW and VAR: lane i, 32 + i the packed pair of heads 2i and 2i + 1), in front of the
    // block table's entry, so that one wait serves them all.
    static_assert(!(VAR && NT > 1), "the fp16 variant scores one token per wave");
    typedef uint32_t u32_a2 __attribute__((aligned(2)));
    uint32_t raw_q[NT], raw_w[NT];
#pragma unroll
    for (int s = 0; s < NT; ++s) {
        const size_t ts = (size_t)(t + s);
        if (VAR || HW) {
            raw_q[s] = reinterpret_cast<const u32_a2 *>(static_cast<const uint16_t *>(p.q_scale) + ts * LI_HEADS)[j];
            raw_w[s] = reinterpret_cast<const u32_a2 *>(static_cast<const uint16_t *>(p.weight) + ts * LI_HEADS)[j];
        } else {
            raw_q[s] = load_raw(p.q_scale, ts * LI_HEADS + l, p.q_dt);
            raw_w[s] = load_raw(p.weight, ts * LI_HEADS + l, p.w_dt);
        }
    }

    // First cache row of every 32-key block of this wave's run, looked up once: lane i holds the row of
    // block i of the run (32 consecutive positions never straddle a page; a run has at most 64 blocks;
    // blocks past the end of the sequence repeat the last valid block).
    int run_row, page0, pb0;                  // (and the run's first page, in the table and in the cache)
    {
        int blk = (key0 >> 5) + l;
        blk = blk > last_blk ? last_blk : blk;
        const int pos0 = 32 * blk;
        const int page = pos0 / p.bs;
        int pb = p.bt[(size_t)b * p.maxblk + page];
        page0 = __builtin_amdgcn_readfirstlane(page);
        pb0 = __builtin_amdgcn_readfirstlane(pb);
        pb = pb < 0 ? 0 : (pb >= p.nblocks ? p.nblocks - 1 : pb);
        run_row = pb * p.bs + (pos0 - page * p.bs);
        asm volatile("" ::"v"(run_row));      // waited for here, not behind the requests below, which the compiler does not count
    }
    // Requests pair pr into buffer buf: per block four instructions of eight rows each.  Lane l owns
    // LDS slot l of an instruction's 1 KiB, i.e. row l/8 (of eight) and position l%8, and fetches chunk
    // (l%8) ^ (row/2 % 8) of that row; the instruction offset moves the cache address and the LDS address
    // alike.  A ninth instruction stages the dword holding the scale of the key whose sum this lane
    // will hold (X_j on the lower half-wave, Y_j on the upper).  Every load of the loop is written as
    // assembly: the compiler then tracks none of them, and the explicit waits of the trips decide
    // alone how long requests stay outstanding (two pairs ahead).
    const uint32_t lane_off = (uint32_t)((l >> 3) * LI_DIM + (((l & 7) ^ (l >> 4)) << 4));
    const uint32_t lane_off4 = lane_off ^ 64u;       // rows 8..15 and 24..31
    const uint32_t lds_base = (uint32_t)__builtin_amdgcn_readfirstlane(
        (int)(uint32_t)(uintptr_t)(__attribute__((address_space(3))) int8_t *)&kstage[w][0][0]);
    constexpr int KSZ = KDT == PTO_DT_FP32 ? 4 : 2;
    // two runs of 32 rows, at gx and gy, into 8 KiB of LDS
#define REQUEST_32_ROWS(HINT, G, DST)                                                              \
    asm volatile("s_mov_b32 m0, %3\n\t"                                                            \
                 "s_nop 0\n\t"                                                                     \
                 "global_load_lds_dwordx4 %0, %2" HINT "\n\t"                                      \
                 "global_load_lds_dwordx4 %1, %2 offset:1024" HINT "\n\t"                          \
                 "global_load_lds_dwordx4 %0, %2 offset:2048" HINT "\n\t"                          \
                 "global_load_lds_dwordx4 %1, %2 offset:3072" HINT                                 \
                 :: "v"(lane_off), "v"(lane_off4), "s"(G), "s"(DST) : "memory", "m0")
    auto request_rows = [&](const int8_t *gx, const int8_t *gy, const uint32_t dst, const bool once) {
        if (once) {
            REQUEST_32_ROWS(" nt", gx, dst);
            REQUEST_32_ROWS(" nt", gy, dst + 4096u);
        } else {
            REQUEST_32_ROWS("", gx, dst);
            REQUEST_32_ROWS("", gy, dst + 4096u);
        }
    };
#undef REQUEST_32_ROWS
    // Keys that one unit alone reads are asked for without being kept (32 sequences of 8 to 64 K keys 35.2 us, so 31.4); with
    // more units to a sequence the others find them in the caches (operator, 20 x 2 tokens of 5 to 60 K keys 35.9 us, not kept 39.7;
    // 18 x 3 of 20 to 130 K 84.1 and 95.9).  So do other sequences that begin with the same pages: up to 16 of them are asked
    // for the run's first page, in front of the queries and looked at with them, behind the first pair's requests (operator, 32
    // sequences, 16 / 64 / 256 common pages: not kept 45.0 / 45.8 / 42.8 us, so 43.0 / 41.3 / 36.6; no common page 44.0 either way.  Asked for
    // beside the sequence's own page, in front of all requests, that took 44.3; the first pair kept until the answer is there 44.6).
    constexpr int SHARERS = 16;
    const int sharers = p.B - 1 < SHARERS ? p.B - 1 : SHARERS;
    bool read_once = upb == 1;
    if (read_once) {
        const int seq = l >= sharers ? b : (b + 1 + l < p.B ? b + 1 + l : b + 1 + l - p.B);
        dma4(p.bt + (size_t)seq * p.maxblk + page0, lds_base + (uint32_t)(SC_BUF_BYTES + SC_PAIR_BYTES));       // where pair 1 has its scales
    }
    auto request_pair = [&](const int pr, const int buf) {
        const int rx = __builtin_amdgcn_readlane(run_row, 2 * pr), ry = __builtin_amdgcn_readlane(run_row, 2 * pr + 1);
        const uint32_t dst = lds_base + (uint32_t)(buf * SC_BUF_BYTES);
        request_rows(p.kcache + (size_t)rx * LI_DIM, p.kcache + (size_t)ry * LI_DIM, dst, read_once);
        // the aligned dword that holds this lane's scale
        const uintptr_t sa = (reinterpret_cast<uintptr_t>(p.k_scale) + ((size_t)(half ? ry : rx) + j) * KSZ) & ~(uintptr_t)3;
        asm volatile("s_mov_b32 m0, %1\n\t"
                     "s_nop 0\n\t"
                     "global_load_lds_dword %0, off"
                     :: "v"(sa), "s"(dst + (uint32_t)SC_PAIR_BYTES) : "memory", "m0");
    };

    // A operands.  Row i of operand 0 is head 32*((i>>2)&1) + 4*(i>>3) + (i&3), operand 1 adds 16:
    // with the 32x32 accumulator layout (row = 8*(r/4) + 4*half + r%4) lane (key, half) then holds
    // heads 32*half + r in register r of accumulator 0 and heads 32*half + 16 + r in accumulator 1.
    // The contraction runs over 16-byte chunks in the order 4*half + ks (ks = 0..3).
    // The queries travel through the pair buffers, in front of the first pairs: asked for behind them, as loads into registers,
    // they arrive when both pairs of every wave have, and no third pair is asked for meanwhile.
    i32x4 qa[NT][2][4];
    auto request_query = [&](const int s, const int buf) {
        const int8_t *q0 = p.q + (size_t)(t + s) * (LI_HEADS * LI_DIM);
        request_rows(q0, q0 + 32 * LI_DIM, lds_base + (uint32_t)(buf * SC_BUF_BYTES), false);
    };
    auto read_query = [&](auto s_tag, const int buf) {
        constexpr int s = decltype(s_tag)::value;
        asm volatile("" ::: "memory");
        const int head0 = 32 * ((j >> 2) & 1) + 4 * (j >> 3) + (j & 3);
        const int8_t *src = &kstage[w][buf][0];
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            qa[s][0][ks] = *reinterpret_cast<const i32x4 *>(src + head0 * LI_DIM + (((4 * half + ks) ^ ((head0 >> 1) & 7)) << 4));
            qa[s][1][ks] = *reinterpret_cast<const i32x4 *>(src + (head0 + 16) * LI_DIM + (((4 * half + ks) ^ ((head0 >> 1) & 7)) << 4));
        }
        if (s == 0 && read_once)
            read_once = __ballot(l < sharers && *reinterpret_cast<const int *>(&kstage[w][1][SC_PAIR_BYTES + 4 * l]) == pb0) == 0ull;
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0xC07F);                      // lgkmcnt(0): the buffer has been read
    };
    if (NT == 1) {
        request_query(0, 1);
        request_pair(0, 0);
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(9));
        read_query(std::integral_constant<int, 0>{}, 1);
    } else {
        request_query(0, 0);
        request_query(NT - 1, 1);
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(8));
        read_query(std::integral_constant<int, 0>{}, 0);
        request_pair(0, 0);
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(9));
        read_query(std::integral_constant<int, NT - 1>{}, 1);
    }
    if (npair > 1) request_pair(1, 1);

    // The factors, wave-uniform.  One token per wave, or fp16 ones: read back lane by lane they sit in scalar registers.  Two
    // tokens of other factors: they go to this wave's rows of wsc_lds and are read as broadcasts, four heads at a time, along
    // the head sum.  VAR = 1 keeps the fp16 query scales and weights of head pairs (2i, 2i+1) packed instead.
    float wsc[(VAR || HW || NT > 1) ? 1 : LI_HEADS];
    uint32_t wp[HW ? NT : 1][HW ? LI_HEADS / 2 : 1];             // HW: factors of heads 2i and 2i + 1
    uint32_t qs2[VAR ? LI_HEADS / 2 : 1], w2[VAR ? LI_HEADS / 2 : 1];
    if (VAR) {
#pragma unroll
        for (int h = 0; h < LI_HEADS / 2; ++h) {
            qs2[h] = (uint32_t)__builtin_amdgcn_readlane((int)raw_q[0], h);
            w2[h] = (uint32_t)__builtin_amdgcn_readlane((int)raw_w[0], h);
        }
    } else if (HW) {
#pragma unroll
        for (int s = 0; s < NT; ++s) {
            const f16x2 q2 = __builtin_bit_cast(f16x2, raw_q[s]), w2h = __builtin_bit_cast(f16x2, raw_w[s]);
            const uint32_t mine = pack_f16x2(__fmul_rn((float)q2[0], (float)w2h[0]), __fmul_rn((float)q2[1], (float)w2h[1]));
#pragma unroll
            for (int h = 0; h < LI_HEADS / 2; ++h) wp[s][h] = (uint32_t)__builtin_amdgcn_readlane((int)mine, h);
        }
    } else if (NT > 1) {
#pragma unroll
        for (int s = 0; s < NT; ++s) wsc_lds[w][s][l] = __fmul_rn(raw_to_f32(raw_q[s], p.q_dt), raw_to_f32(raw_w[s], p.w_dt));
    } else {
        const float mine = __fmul_rn(raw_to_f32(raw_q[0], p.q_dt), raw_to_f32(raw_w[0], p.w_dt));
#pragma unroll
        for (int h = 0; h < LI_HEADS; ++h) wsc[h] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, mine), h));
    }

    float *srow0 = p.scores + (size_t)t * p.score_stride;
    float *smp0 = p.sample + (size_t)t * (p.score_stride / LI_SAMPLE_GROUP);
    // 2^-11 as a run-time value, so that it sits in a scalar register (the mix instructions take no literal)
    const float scale = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(0x3a000000));
    // this lane's operand chunks of row j inside a staged block
    int koff[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) koff[ks] = j * LI_DIM + (((4 * half + ks) ^ ((j >> 1) & 7)) << 4);

    // One trip.  Requests and stores complete in the order they were made.  Behind this trip's pair there are the nine
    // requests of the following pair and the two stores per token (scores, sample) of each of the last two trips -- every
    // trip but the wave's last writes both -- and that many may be outstanding: a wait that counts the requests alone
    // holds a wave up until half of the pair it has only just asked for has landed too.  The trip's operands and scale
    // then move to registers, which frees the buffer for the pair two ahead, and the pair is scored.
    // (The wait itself orders nothing for the compiler: without the barrier in front of it a store of an earlier trip may move
    // behind it, and the wait would then pass with the trip's own requests still on their way.)
    auto wait_pair = [&](auto per_trip, const int pr) {
        constexpr int ST = decltype(per_trip)::value;
        asm volatile("" ::: "memory");
        if (pr + 1 < npair) {
            if (pr >= 2) __builtin_amdgcn_s_waitcnt(vmcnt_imm(9 + 2 * ST));
            else if (pr == 1) __builtin_amdgcn_s_waitcnt(vmcnt_imm(9 + ST));
            else __builtin_amdgcn_s_waitcnt(vmcnt_imm(9));
        } else {
            __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
        }
    };
    auto trip = [&](const int pr, const int buf) {
        const int8_t *src = &kstage[w][buf][0];
        i32x4 kx[4], ky[4];
        wait_pair(std::integral_constant<int, 2 * NT>{}, pr);
        asm volatile("" ::: "memory");
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            kx[ks] = *reinterpret_cast<const i32x4 *>(src + koff[ks]);
            ky[ks] = *reinterpret_cast<const i32x4 *>(src + 4096 + koff[ks]);
        }
        const uint32_t ksraw = *reinterpret_cast<const uint32_t *>(src + SC_PAIR_BYTES + 4 * l);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0xC07F);                      // lgkmcnt(0): the buffer has been read
        if (pr + 2 < npair) request_pair(pr + 2, buf);
        float ksc;
        uint32_t ks2 = 0;                                        // the key's fp16 scale twice (VAR = 1)
        if (KDT == PTO_DT_FP32) {
            ksc = __uint_as_float(ksraw);
        } else {
            // rows of a block are 32 consecutive scales, so the parity of the lane's element follows j
            const int rrow = __builtin_amdgcn_readlane(run_row, 2 * pr + 0);
            const int rrow1 = __builtin_amdgcn_readlane(run_row, 2 * pr + 1);
            const bool odd = ((reinterpret_cast<uintptr_t>(p.k_scale) + ((size_t)(half ? rrow1 : rrow) + j) * KSZ) & 2) != 0;
            const uint16_t hbits = (uint16_t)(odd ? ksraw >> 16 : ksraw);
            ksc = KDT == PTO_DT_BF16 ? bf16_bits_to_f32(hbits) : (float)__builtin_bit_cast(_Float16, hbits);
            ks2 = (uint32_t)hbits | ((uint32_t)hbits << 16);
        }
        // the staged pair serves every token of the unit
        auto score_token = [&](auto s_tag, float *srow, float *smp) {
            constexpr int s = decltype(s_tag)::value;
            i32x16 ax0, ax1, ay0, ay1;
#pragma unroll
            for (int r = 0; r < 16; ++r) ax0[r] = ax1[r] = ay0[r] = ay1[r] = VAR ? 0 : DOT_ZERO;
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) {
                ax0 = __builtin_amdgcn_mfma_i32_32x32x32_i8(qa[s][0][ks], kx[ks], ax0, 0, 0, 0);
                ax1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(qa[s][1][ks], kx[ks], ax1, 0, 0, 0);
                ay0 = __builtin_amdgcn_mfma_i32_32x32x32_i8(qa[s][0][ks], ky[ks], ay0, 0, 0, 0);
                ay1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(qa[s][1][ks], ky[ks], ay1, 0, 0, 0);
            }
            // lo[o][i] / hi[o][i]: heads 16*o + 2*i, +1 (lo) and 32 + 16*o + 2*i, +1 (hi) of this lane's key
            uint32_t lo[2][8], hi[2][8];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const uint32_t x0 = VAR ? fp16_pair(ax0[2 * i], ax0[2 * i + 1], scale) : relu_fp16_pair(ax0[2 * i], ax0[2 * i + 1]);
                const uint32_t y0 = VAR ? fp16_pair(ay0[2 * i], ay0[2 * i + 1], scale) : relu_fp16_pair(ay0[2 * i], ay0[2 * i + 1]);
                const uint32_t x1 = VAR ? fp16_pair(ax1[2 * i], ax1[2 * i + 1], scale) : relu_fp16_pair(ax1[2 * i], ax1[2 * i + 1]);
                const uint32_t y1 = VAR ? fp16_pair(ay1[2 * i], ay1[2 * i + 1], scale) : relu_fp16_pair(ay1[2 * i], ay1[2 * i + 1]);
                const auto s0 = __builtin_amdgcn_permlane32_swap(x0, y0, false, false);
                const auto s1 = __builtin_amdgcn_permlane32_swap(x1, y1, false, false);
                lo[0][i] = s0[0]; hi[0][i] = s0[1];
                lo[1][i] = s1[0]; hi[1][i] = s1[1];
            }
            float sum = 0.f;
            if (VAR) {
                const float one = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(0x3f800000));
#pragma unroll
                for (int o = 0; o < 2; ++o) {
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        const uint32_t v = dequant_relu_weight(lo[o][i], qs2[8 * o + i], ks2, w2[8 * o + i]);
                        sum = __fadd_rn(sum, mul_f16_f32<0>(v, one));
                        sum = __fadd_rn(sum, mul_f16_f32<1>(v, one));
                    }
                }
#pragma unroll
                for (int o = 0; o < 2; ++o) {
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        const uint32_t v = dequant_relu_weight(hi[o][i], qs2[16 + 8 * o + i], ks2, w2[16 + 8 * o + i]);
                        sum = __fadd_rn(sum, mul_f16_f32<0>(v, one));
                        sum = __fadd_rn(sum, mul_f16_f32<1>(v, one));
                    }
                }
                const int pos = key0 + 64 * pr + l;
                if (pos < cur) srow[pos] = sum;
                if (sample_lane(pos, cur)) smp[pos >> 4] = sum;
                return;
            }
            if (HW) {
#pragma unroll
                for (int q = 0; q < 32; ++q) {                       // heads ascending, two per register
                    const uint32_t x = q < 16 ? lo[q >> 3][q & 7] : hi[(q >> 3) & 1][q & 7];
                    fma_f16_pair<0>(sum, x, wp[s][q]);
                    fma_f16_pair<1>(sum, x, wp[s][q]);
                }
            } else if (NT > 1) {
                // heads ascending: lo[0][0..7], lo[1][0..7], hi[0][0..7], hi[1][0..7], two heads per register
                const f32x4 *wrow = reinterpret_cast<const f32x4 *>(&wsc_lds[w][s][0]);
#pragma unroll
                for (int q = 0; q < 16; ++q) {
                    const f32x4 w4 = wrow[q];                        // heads 4q .. 4q+3, the same address on every lane
                    const int o = (q >> 2) & 1, i = 2 * (q & 3);
                    const uint32_t x0 = q < 8 ? lo[o][i] : hi[o][i], x1 = q < 8 ? lo[o][i + 1] : hi[o][i + 1];
                    sum = __fadd_rn(sum, mul_f16_f32_v<0>(x0, w4[0]));
                    sum = __fadd_rn(sum, mul_f16_f32_v<1>(x0, w4[1]));
                    sum = __fadd_rn(sum, mul_f16_f32_v<0>(x1, w4[2]));
                    sum = __fadd_rn(sum, mul_f16_f32_v<1>(x1, w4[3]));
                }
            } else {
#pragma unroll
                for (int o = 0; o < 2; ++o) {
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        sum = __fadd_rn(sum, mul_f16_f32<0>(lo[o][i], wsc[16 * o + 2 * i]));
                        sum = __fadd_rn(sum, mul_f16_f32<1>(lo[o][i], wsc[16 * o + 2 * i + 1]));
                    }
                }
#pragma unroll
                for (int o = 0; o < 2; ++o) {
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        sum = __fadd_rn(sum, mul_f16_f32<0>(hi[o][i], wsc[32 + 16 * o + 2 * i]));
                        sum = __fadd_rn(sum, mul_f16_f32<1>(hi[o][i], wsc[32 + 16 * o + 2 * i + 1]));
                    }
                }
            }
            const int pos = key0 + 64 * pr + l;
            const float sc = __fmul_rn(sum, ksc);
            if (pos < cur) srow[pos] = sc;
            if (sample_lane(pos, cur)) smp[pos >> 4] = sc;
        };
        score_token(std::integral_constant<int, 0>{}, srow0, smp0);
        if (NT > 1)
            score_token(std::integral_constant<int, NT - 1>{}, srow0 + p.score_stride, smp0 + p.score_stride / LI_SAMPLE_GROUP);
    };
    for (int pr = 0; pr < npair; pr += 2) {
        trip(pr, 0);
        if (pr + 1 < npair) trip(pr + 1, 1);
    }
}

// ---------------------------------------------------------------------------------- select

constexpr int SEL_THREADS = 1024;
constexpr int SEL_WAVES = SEL_THREADS / 64;

// General select of one query token: every pass re-reads the score row (L2-resident) from memory.
// Slow (five passes over the row) but free of capacity assumptions; the fast kernel falls back to it.
// hist: >= 256 words, sortbuf: LI_MAX_SELECT entries, both in LDS.
__device__ void select_streaming(const LiParams &p, const int t, uint32_t *hist, unsigned long long *sortbuf)
{
    __shared__ uint32_t wave_gt[SEL_WAVES], wave_eq[SEL_WAVES];
    __shared__ uint32_t sh_prefix, sh_krem;

    const int b = t / p.S1;
    const int s = t - b * p.S1;
    const int tid = threadIdx.x;
    const int wv = tid >> 6;
    const int lane = tid & 63;
    int cur = p.act[b];
    const int cap = p.maxblk * p.bs;
    cur = cur < 0 ? 0 : (cur > cap ? cap : cur);
    int n = cur - (p.S1 - 1 - s);
    n = n < 0 ? 0 : n;
    const int k = p.k;
    const float *srow = p.scores + (size_t)t * p.score_stride;
    int32_t *out = p.topk_res + (size_t)t * k;

    // sort width: the next power of two that holds min(n, k) candidates
    const int nsel = n < k ? n : k;
    int width = 64;
    while (width < nsel) width <<= 1;
    for (int i = tid; i < width; i += SEL_THREADS) sortbuf[i] = 0ull;   // 0 sorts after every candidate

    if (n <= k) {
        __syncthreads();
        for (int i = tid; i < n; i += SEL_THREADS)
            sortbuf[i] = ((unsigned long long)score_key(srow[i]) << 32) | (uint32_t)(~(uint32_t)i);
    } else {
        // ---- radix select: after the passes, prefix = key of the k-th best and krem = how many
        // candidates with exactly that key are taken
        uint32_t prefix = 0, krem = (uint32_t)k;
        for (int pass = 0; pass < 4; ++pass) {
            const int shift = 24 - 8 * pass;
            for (int i = tid; i < 256; i += SEL_THREADS) hist[i] = 0;
            __syncthreads();
            const uint32_t himask = pass == 0 ? 0u : (0xffffffffu << (shift + 8));
            for (int i0 = 0; i0 < n; i0 += SEL_THREADS) {
                const int i = i0 + tid;
                bool active = false;
                uint32_t digit = 0;
                if (i < n) {
                    const uint32_t key = score_key(srow[i]);
                    active = (key & himask) == prefix;
                    digit = (key >> shift) & 0xffu;
                }
                // scores cluster: peel up to two digits shared by many lanes with one add each
                unsigned long long rem = __ballot(active);
#pragma unroll 1
                for (int peel = 0; peel < 2 && rem != 0ull; ++peel) {
                    const int first = __ffsll((long long)rem) - 1;
                    const uint32_t d = __shfl(digit, first);
                    const unsigned long long same = __ballot(active && digit == d) & rem;
                    if (__popcll(same) < 8) break;
                    if (lane == first) atomicAdd(&hist[d], (uint32_t)__popcll(same));
                    rem &= ~same;
                }
                if ((rem >> lane) & 1ull) atomicAdd(&hist[digit], 1u);
            }
            __syncthreads();
            if (tid < 64) {
                // bins in descending order: lane i owns bins 255-4i .. 252-4i
                uint32_t c[4];
                uint32_t tot = 0;
#pragma unroll
                for (int e = 0; e < 4; ++e) { c[e] = hist[255 - 4 * tid - e]; tot += c[e]; }
                uint32_t incl = tot;
#pragma unroll
                for (int off = 1; off < 64; off <<= 1) {
                    const uint32_t v = __shfl_up(incl, off);
                    if (lane >= off) incl += v;
                }
                uint32_t above = incl - tot;      // candidates in bins above this lane's four
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if (above < krem && krem <= above + c[e]) {
                        sh_prefix = prefix | ((uint32_t)(255 - 4 * tid - e) << shift);
                        sh_krem = krem - above;
                    }
                    above += c[e];
                }
            }
            __syncthreads();
            prefix = sh_prefix;
            krem = sh_krem;
            __syncthreads();
        }
        const uint32_t thr = prefix;
        const uint32_t n_gt = (uint32_t)k - krem;

        // ---- compaction in position order: wave wv owns positions [wv*seg, (wv+1)*seg)
        const int seg = ((n + SEL_WAVES - 1) / SEL_WAVES + 63) / 64 * 64;
        const int lo = wv * seg;
        int hi = lo + seg;
        hi = hi > n ? n : hi;
        uint32_t cgt = 0, ceq = 0;
        for (int i0 = lo; i0 < hi; i0 += 64) {
            const int i = i0 + lane;
            uint32_t key = 0;
            if (i < hi) key = score_key(srow[i]);
            cgt += (uint32_t)__popcll(__ballot(i < hi && key > thr));
            ceq += (uint32_t)__popcll(__ballot(i < hi && key == thr));
        }
        if (lane == 0) { wave_gt[wv] = cgt; wave_eq[wv] = ceq; }
        __syncthreads();
        uint32_t base_gt = 0, base_eq = 0;
        for (int i = 0; i < wv; ++i) { base_gt += wave_gt[i]; base_eq += wave_eq[i]; }
        const unsigned long long lt_mask = (1ull << lane) - 1ull;
        for (int i0 = lo; i0 < hi; i0 += 64) {
            const int i = i0 + lane;
            uint32_t key = 0;
            if (i < hi) key = score_key(srow[i]);
            const bool gt = i < hi && key > thr;
            const bool eq = i < hi && key == thr;
            const unsigned long long mgt = __ballot(gt), meq = __ballot(eq);
            const unsigned long long comp = ((unsigned long long)key << 32) | (uint32_t)(~(uint32_t)i);
            if (gt) sortbuf[base_gt + (uint32_t)__popcll(mgt & lt_mask)] = comp;
            if (eq) {
                const uint32_t rank = base_eq + (uint32_t)__popcll(meq & lt_mask);
                if (rank < krem) sortbuf[n_gt + rank] = comp;
            }
            base_gt += (uint32_t)__popcll(mgt);
            base_eq += (uint32_t)__popcll(meq);
        }
    }
    __syncthreads();

    // ---- bitonic sort, descending on (key, ~position): score descending, position ascending
    for (int size = 2; size <= width; size <<= 1) {
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            for (int i = tid; i < (width >> 1); i += SEL_THREADS) {
                const int pos = 2 * i - (i & (stride - 1));
                const unsigned long long a = sortbuf[pos], c = sortbuf[pos + stride];
                const bool desc = (pos & size) == 0;
                if ((a < c) == desc) { sortbuf[pos] = c; sortbuf[pos + stride] = a; }
            }
            __syncthreads();
        }
    }
    for (int i = tid; i < k; i += SEL_THREADS)
        out[i] = i < nsel ? (int32_t)(~(uint32_t)(sortbuf[i] & 0xffffffffull)) : -1;
}


// ------------------------------------------------------------------ register-resident select

// descending bitonic sort of width (power of two, 64..2048) 64-bit keys in LDS, 1024 threads.
// Thread tid owns positions 2*tid and 2*tid+1: strides 1..64 are done in registers and wave shuffles,
// only strides >= 128 go through LDS with a barrier.
__device__ __forceinline__ unsigned long long shfl_xor_u64(const unsigned long long v, const int mask)
{
    const uint32_t lo = (uint32_t)__shfl_xor((int)(uint32_t)v, mask);
    const uint32_t hi = (uint32_t)__shfl_xor((int)(uint32_t)(v >> 32), mask);
    return ((unsigned long long)hi << 32) | lo;
}

__device__ void bitonic_sort_desc(unsigned long long *buf, const int width, const int tid)
{
    const bool active = 2 * tid < width;
    unsigned long long e0 = 0ull, e1 = 0ull;
    if (active) { e0 = buf[2 * tid]; e1 = buf[2 * tid + 1]; }
    for (int size = 2; size <= width; size <<= 1) {
        const bool desc = ((2 * tid) & size) == 0;      // both positions of a thread share the direction bit (size >= 2)
        int stride = size >> 1;
        if (stride >= 128) {
            // cross-wave strides through LDS
            if (active) { buf[2 * tid] = e0; buf[2 * tid + 1] = e1; }
            __syncthreads();
            for (; stride >= 128; stride >>= 1) {
                for (int i = tid; i < (width >> 1); i += SEL_THREADS) {
                    const int pos = 2 * i - (i & (stride - 1));
                    const unsigned long long a = buf[pos], c = buf[pos + stride];
                    const bool d = (pos & size) == 0;
                    if ((a < c) == d) { buf[pos] = c; buf[pos + stride] = a; }
                }
                __syncthreads();
            }
            if (active) { e0 = buf[2 * tid]; e1 = buf[2 * tid + 1]; }
        }
        for (; stride >= 2; stride >>= 1) {
            // partner thread tid ^ (stride/2), same slot; the lower position keeps the max when descending
            const unsigned long long p0 = shfl_xor_u64(e0, stride >> 1);
            const unsigned long long p1 = shfl_xor_u64(e1, stride >> 1);
            const bool lower = ((2 * tid) & stride) == 0;
            const bool take_max = lower == desc;
            e0 = take_max ? (e0 > p0 ? e0 : p0) : (e0 < p0 ? e0 : p0);
            e1 = take_max ? (e1 > p1 ? e1 : p1) : (e1 < p1 ? e1 : p1);
        }
        {   // stride 1: the thread's own pair
            const unsigned long long hi = e0 > e1 ? e0 : e1, lo = e0 > e1 ? e1 : e0;
            e0 = desc ? hi : lo;
            e1 = desc ? lo : hi;
        }
    }
    if (active) { buf[2 * tid] = e0; buf[2 * tid + 1] = e1; }
    __syncthreads();
}

constexpr int SEL_SAMPLE = 4096;   // most keys sampled from a row
constexpr int SEL_CAP = 8192;      // candidates (keys above the pivot) the fast path holds in LDS
constexpr int SEL_STAGE = 4096;    // entries of the buckets down to the one holding the k-th best
constexpr int SEL_DIRECT = 8192;   // rows whose keys all go to the buckets
constexpr int SEL_COUNT_MAX = 128; // of those: most keys of a bucket that are ordered by counting

// the 64-bit word whose descending order is (score descending, position ascending); never zero
__device__ __forceinline__ unsigned long long order_word(const float score, const uint32_t pos)
{
    return ((unsigned long long)score_key(score) << 32) | (uint32_t)(~pos);
}

// score whose order-preserving image is key (the inverse of score_key)
__device__ __forceinline__ float key_score(const uint32_t key)
{
    return __uint_as_float((key & 0x80000000u) ? (key & 0x7fffffffu) : ~key);
}

constexpr int SEL_SBINS = 1024;    // bins of the sample histogram
constexpr int SEL_BUCKETS = 8192;  // buckets the candidates are spread over, eight per thread
constexpr int SEL_WAVE_CAP = SEL_CAP / SEL_WAVES;   // candidates one wave can compact
constexpr int SEL_CHUNK = 32 * SEL_THREADS;   // scores one trip of the row scan holds in registers

// One workgroup per query token: a distribution-adaptive bucket select.  Every key is ordered by the
// word (score image << 32) | ~position, a strict order, so ties need no special case.
//   1. up to 4096 scores are sampled: the score kernel left one score of every 16 positions (which of
//      the 16, a hash of the group number decides) in a compact array.  A histogram of the
//      sample over [sample min, sample max] gives the pivot: the lower edge of the bin in which the
//      sample reaches rank r = r0 + 6*sqrt(r0) + 8, r0 = k*S/n.  With overwhelming probability at
//      least k and at most SEL_CAP scores of the row lie at or above it;
//   2. one pass over the row (32 scores per thread in flight at once, requested before the sample is
//      looked at) compacts the keys at or above the pivot into a candidate list;
//   3. the candidates are spread over 8192 buckets linear in the score between the pivot and the
//      sample maximum, bucket 0 highest: bins follow the values instead of the float encoding, so
//      the counters see few collisions and buckets stay short whatever the scale of the scores;
//   4. a prefix sum over the bucket counts finds the bucket holding the k-th best key; the buckets
//      down to it are staged contiguously and each is ordered by counting (a key's rank = the number
//      of larger keys of its bucket).  Output slots below k are written straight to memory.
// Rows of up to SEL_DIRECT keys skip the first two: all their keys are candidates.
// A chain of short phases: what each costs is the latency of its loads or the vector work of sixteen waves on four SIMDs, so work
// that every wave would do alike is done by one (the pivot), or by a row of lanes (sums over the waves), and buckets are many
// and short.  Clocks at 32 K scores: sample and minimum 5.9 K, pivot 1.9, scan 3.7 (the row arrives at 14-20 bytes per clock),
// candidates 2.5, offsets 2.2, staging 1.7, ranking 3.5; 24.1 -> 21.3 K in all (pivot 5.1, ranking 4.7 before).
// If the pivot misjudges the row (fewer than k candidates, more than the list holds, or a bucket
// range too long to stage) the general streaming select runs instead.
__global__ __launch_bounds__(SEL_THREADS) void li_select_kernel(const LiParams p)
{
    __shared__ uint32_t cand[SEL_CAP];                 // positions
    __shared__ unsigned long long stage[SEL_STAGE];    // also the sort buffer of the other paths
    __shared__ uint16_t sbucket[SEL_STAGE];            // bucket of every staged entry
    __shared__ __attribute__((aligned(16))) uint32_t boff[SEL_BUCKETS + 4];   // counts, then first slots, of the buckets
    __shared__ uint32_t shist[SEL_SBINS];
    __shared__ uint32_t hist[256];                     // streaming path only
    __shared__ uint32_t wave_tot[SEL_WAVES], wave_sum[SEL_WAVES];
    __shared__ float wave_mn[SEL_WAVES], wave_mx[SEL_WAVES];
    __shared__ uint32_t sh_over, sh_pb, sh_tb, sh_stage;
    static_assert(SEL_BUCKETS == 8 * SEL_THREADS && SEL_WAVES == 16, "eight buckets per thread, a wave per lane of a row");

    const int t = blockIdx.x;
    const int b = t / p.S1;
    const int s = t - b * p.S1;
    const int tid = threadIdx.x;
    const int wv = tid >> 6;
    const int lane = tid & 63;
    int cur = p.act[b];
    const int cap = p.maxblk * p.bs;
    cur = cur < 0 ? 0 : (cur > cap ? cap : cur);
    int n = cur - (p.S1 - 1 - s);
    n = n < 0 ? 0 : n;
    const int k = p.k;
    const float *srow = p.scores + (size_t)t * p.score_stride;
    int32_t *out = p.topk_res + (size_t)t * k;

    // everything is selected; the tail of the output row is padding
    for (int i = n + tid; i < k; i += SEL_THREADS) out[i] = -1;
    if (n == 0) return;
    const int kk = n < k ? n : k;          // keys taken
    constexpr int CPT = SEL_WAVE_CAP / 64;
    unsigned long long ce[CPT];            // this lane's candidates, their buckets and places in them
    uint32_t cb[CPT], cslot[CPT];
    // the workgroup's minimum and maximum
    auto range_of = [&](const float mn, const float mx, float &lo, float &hi) __attribute__((always_inline)) {
        const float a = wave_min(mn), b2 = wave_max(mx);
        if (lane == 0) { wave_mn[wv] = a; wave_mx[wv] = b2; }
        __syncthreads();
        lo = row_reduce(wave_mn[lane & 15], [](float x, float y) { return fminf(x, y); });
        hi = row_reduce(wave_mx[lane & 15], [](float x, float y) { return fmaxf(x, y); });
    };
    auto to_bucket = [&](const int u, const float score, const uint32_t pos, const float lo, const float scale) __attribute__((always_inline)) {
        ce[u] = order_word(score, pos);
        const uint32_t lin = (uint32_t)fmaxf((key_score((uint32_t)(ce[u] >> 32)) - lo) * scale, 0.f);
        cb[u] = (uint32_t)SEL_BUCKETS - 1u - (lin < (uint32_t)SEL_BUCKETS ? lin : (uint32_t)SEL_BUCKETS - 1u);
        cslot[u] = atomicAdd(&boff[cb[u]], 1u);
    };
    auto no_candidates = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < CPT; ++u) {
            ce[u] = 0ull;
            cb[u] = (uint32_t)SEL_BUCKETS; // none
            cslot[u] = 0u;
        }
    };
    // ---- 4. bucket offsets (eight buckets per thread) and the bucket holding the k-th best key (sh_over: one of them is too long)
    auto offsets = [&]() {
        u32x4 *const mine = reinterpret_cast<u32x4 *>(boff) + 2 * tid;
        u32x4 c[2];
        c[0] = mine[0];
        c[1] = mine[1];
        const uint32_t tot = ((c[0][0] + c[0][1]) + (c[0][2] + c[0][3])) + ((c[1][0] + c[1][1]) + (c[1][2] + c[1][3]));
        const uint32_t incl = wave_incl_scan(tot);
        if (lane == 63) wave_sum[wv] = incl;
        __syncthreads();
        const uint32_t of_wave = wave_sum[lane & 15];
        uint32_t before = (uint32_t)__builtin_amdgcn_readlane((int)(row_incl_scan(of_wave) - of_wave), wv) + incl - tot;
        const bool here = before < (uint32_t)kk && (uint32_t)kk <= before + tot;
        uint32_t longest = 0u;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const uint32_t cnt = c[e >> 2][e & 3];
            c[e >> 2][e & 3] = before;
            if (before < (uint32_t)kk && longest < cnt) longest = cnt;
            if (here && before < (uint32_t)kk && (uint32_t)kk <= before + cnt) {
                sh_tb = (uint32_t)(8 * tid + e);
                sh_stage = before + cnt;
            }
            before += cnt;
        }
        mine[0] = c[0];
        mine[1] = c[1];
        if (tid == SEL_THREADS - 1) boff[SEL_BUCKETS] = before;
        if (longest > (uint32_t)SEL_COUNT_MAX) sh_over = 1u;
        __syncthreads();
    };
    // A short row, up to eight keys per thread: all of them go straight to the buckets, spread over their own range.  Where too
    // many fall together (equal scores, one far from the rest, an infinite one), or one is not a number, a row of which every key
    // is taken is sorted, and a longer one goes the way of the others.
    // (Rows of at most k keys always sorted beyond 512 keys and ordered by counting over the whole row up to there, as before,
    // two sequences of 450 keys took 24.3 us instead of 9.6, scores included, of 650 keys 18.5, of 1900 22.0 instead of 10.8.
    // By way of a pivot, two of 2200 keys take 13.5, as here 11.2, of 4096 15.0 and 12.1, of 8100 15.1 and 13.4.  A row that has to
    // leave pays for both ways: four of 8000 equal scores 57.3 by the pivot alone, 66.3 here, with every thousandth score 10^6 times
    // the others 43.4 and 52.2, of 1500 keys 22.0 and 23.4.  Scores crowd like that where one lies about eighty times as far out as the
    // others among 8000 keys, three hundred times among 2048.)
    auto sort_row = [&]() {
        int width = 64;
        while (width < n) width <<= 1;
        for (int i = tid; i < width; i += SEL_THREADS) stage[i] = i < n ? order_word(srow[i], (uint32_t)i) : 0ull;
        __syncthreads();
        bitonic_sort_desc(stage, width, tid);
        for (int i = tid; i < n; i += SEL_THREADS) out[i] = (int32_t)(~(uint32_t)stage[i]);
    };
    bool ordered = false;
    if (n <= SEL_DIRECT) {
        static_assert(LI_MAX_SELECT <= SEL_DIRECT && SEL_DIRECT <= CPT * SEL_THREADS, "a candidate's place for every key");
        float x[CPT];
        float mn = __builtin_inff(), mx = -__builtin_inff();
#pragma unroll
        for (int e = 0; e < CPT; ++e) {
            const int i = tid + e * SEL_THREADS;
            x[e] = e * SEL_THREADS < n ? srow[i < n ? i : 0] : 0.f;
        }
        for (int i = tid; i < SEL_BUCKETS / 4; i += SEL_THREADS) reinterpret_cast<u32x4 *>(boff)[i] = u32x4{0u, 0u, 0u, 0u};
        if (tid == 0) sh_over = 0u;
        bool odd = false;
#pragma unroll
        for (int e = 0; e < CPT; ++e)
            if (e * SEL_THREADS < n) {
                mn = fminf(mn, x[e]);
                mx = fmaxf(mx, x[e]);
                odd |= !(x[e] == x[e]);
            }
        float smin, smax;
        range_of(mn, mx, smin, smax);
        if (odd) sh_over = 1u;
        const float scale = smax - smin > 0.f ? (float)SEL_BUCKETS / (smax - smin) : 0.f;
        no_candidates();
#pragma unroll
        for (int e = 0; e < CPT; ++e)
            if (tid + e * SEL_THREADS < n) to_bucket(e, x[e], (uint32_t)(tid + e * SEL_THREADS), smin, scale);
        __syncthreads();
        offsets();
        ordered = sh_over == 0u;
        if (!ordered && n <= k) return sort_row();
        if (!ordered) __syncthreads();     // (everyone has seen it)
    }
    if (!ordered) {
        // ---- 1. sample: the loads go out first, then the first chunk of the row, so that one memory
        // latency covers both
        // (the score kernel left one score of every 16 positions in a compact array; a row longer than
        // 16 * SEL_SAMPLE takes every other one).  Rows with hardly any full group go the general way.
        const uint32_t s_full = (uint32_t)n / (uint32_t)LI_SAMPLE_GROUP;
        if (s_full < 64u) {
            select_streaming(p, t, hist, stage);                     // uniform: the whole workgroup goes
            return;
        }
        const uint32_t sstep = s_full > (uint32_t)SEL_SAMPLE ? 2u : 1u;
        const uint32_t S = s_full / sstep;
        constexpr int SPT = SEL_SAMPLE / SEL_THREADS;
        const float *smp = p.sample + (size_t)t * (p.score_stride / LI_SAMPLE_GROUP);
        float sx[SPT];
        bool sval[SPT];
#pragma unroll
        for (int e = 0; e < SPT; ++e) {
            const uint32_t i = (uint32_t)(tid + e * SEL_THREADS);
            sval[e] = i < S;
            sx[e] = smp[(sval[e] ? i : 0u) * sstep];
        }
        // the row as 16-byte vectors: thread tid holds vectors u*1024 + tid of a chunk.  The row buffer is
        // score_stride (a multiple of 32) long, so whole vectors stay inside it.
        const int last_vec = (int)(p.score_stride >> 2) - 1;
        auto load_chunk = [&](const int c0, f32x4 (&v)[8]) {
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int vi = (c0 >> 2) + u * SEL_THREADS + tid;
                v[u] = reinterpret_cast<const f32x4 *>(srow)[vi < last_vec ? vi : last_vec];
            }
        };
        f32x4 v[8], vn[8];
        load_chunk(0, v);
        const uint32_t r0 = ((uint32_t)k * S + (uint32_t)n - 1u) / (uint32_t)n;
        const uint32_t r = r0 + (uint32_t)(6.0f * __builtin_sqrtf((float)r0)) + 8u;

        no_candidates();
        for (int i = tid; i < SEL_SBINS; i += SEL_THREADS) shist[i] = 0u;
        for (int i = tid; i < SEL_BUCKETS / 4; i += SEL_THREADS) reinterpret_cast<u32x4 *>(boff)[i] = u32x4{0u, 0u, 0u, 0u};
        if (tid == 0) sh_over = 0u;
        float smin, smax;
        {
            float mn = __builtin_inff(), mx = -__builtin_inff();
#pragma unroll
            for (int e = 0; e < SPT; ++e)
                if (sval[e]) { mn = fminf(mn, sx[e]); mx = fmaxf(mx, sx[e]); }
            range_of(mn, mx, smin, smax);
        }
        float pivot = -__builtin_inff();       // candidates: score >= pivot
        float blo = smin;                      // lower edge of the lowest bucket
        if (r < S) {
            const float range = smax - smin;
            const float sscale = range > 0.f ? (float)SEL_SBINS / range : 0.f;
#pragma unroll
            for (int e = 0; e < SPT; ++e) {
                if (sval[e]) {
                    const uint32_t sb = (uint32_t)fmaxf((sx[e] - smin) * sscale, 0.f);
                    atomicAdd(&shist[sb < (uint32_t)SEL_SBINS ? sb : (uint32_t)SEL_SBINS - 1u], 1u);
                }
            }
            __syncthreads();
            // one wave scans the 1024 bins from the top (lane l owns the 16 bins below 1024 - 16*l): the bin in which the running
            // count reaches r.  (Every wave by itself, without the barrier: 2.2 thousand clocks of vector work instead of 0.9.)
            if (wv == 0) {
                const u32x4 *src = reinterpret_cast<const u32x4 *>(&shist[SEL_SBINS - 16 - 16 * lane]);
                uint32_t tot = 0;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const u32x4 x = src[q];
                    tot += (x[0] + x[1]) + (x[2] + x[3]);
                }
                const uint32_t before = wave_incl_scan(tot) - tot;
                // (found by exactly one lane: the sample holds S >= r scores); then the bin among its sixteen, a lane each
                const int at = __ffsll((long long)__ballot(before < r && r <= before + tot)) - 1;
                const uint32_t top = (uint32_t)(SEL_SBINS - 1 - 16 * at);
                const uint32_t cnt = shist[top - (uint32_t)(lane & 15)];
                const uint32_t incl = (uint32_t)__builtin_amdgcn_readlane((int)before, at) + row_incl_scan(cnt);
                const int in = __ffsll((long long)__ballot(incl - cnt < r && r <= incl)) - 1;
                if (lane == 0) sh_pb = top - (uint32_t)in;
            }
            __syncthreads();
            const uint32_t pb = sh_pb;
            pivot = smin + (float)pb * (range * (1.0f / (float)SEL_SBINS));
            blo = pivot;
        }
        // the buckets reach a quarter of the range past the sample maximum, so that the few scores above
        // it spread out too; anything beyond shares bucket 0
        const float bscale = smax - blo > 0.f ? (float)SEL_BUCKETS / (1.25f * (smax - blo)) : 0.f;

        // ---- 2. candidates.  Wave w compacts the positions of the candidates among its keys into its own region of the
        // list, cand[w*SEL_WAVE_CAP ...], so the waves share no counter.  A key costs a compare and an add-with-carry that
        // shifts the outcome into the lane's mask of its 32 keys; the few candidates (one key in twenty of a long row) are then
        // picked out of the masks, a candidate of every lane per trip, and their scores fetched again below (out of the L2).
        // (One LDS write per key, candidate or not, as before, took 14 to 17 of the kernel's 33 thousand clocks on 50 K keys.)
        // Wave-wide sums use DPP, not LDS.
        uint32_t wave_count = 0;               // candidates of this wave so far (uniform)
        auto scan_chunk = [&](const int c0, auto full_tag) {
            constexpr bool FULL = decltype(full_tag)::value;          // the whole chunk lies inside the row
            const int i_base = c0 + 4 * tid;
            uint32_t m = 0;                                           // key (u, c) is bit 31 - (4u + c)
#pragma unroll
            for (int u = 0; u < 8; ++u) {
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const int i = i_base + 4 * u * SEL_THREADS + c;
                    m = m + m + (((FULL || i < n) && v[u][c] >= pivot) ? 1u : 0u);
                }
            }
            const uint32_t mine = (uint32_t)__popc(m);
            const uint32_t incl = wave_incl_scan(mine);
            const uint32_t wave_n = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
            if (wave_count + wave_n > (uint32_t)SEL_WAVE_CAP) {       // region overflow: the streaming path will run
                if (lane == 0) sh_over = 1u;
                return;
            }
            uint32_t slot = (uint32_t)(wv * SEL_WAVE_CAP) + wave_count + incl - mine;
            wave_count += wave_n;
            while (m != 0u) {
                const uint32_t q = (uint32_t)__clz(m);                // 4u + c
                m &= 0x7fffffffu >> q;
                cand[slot++] = (uint32_t)i_base + ((q >> 2) * (4u * SEL_THREADS) + (q & 3u));
            }
        };
        for (int c0 = 0; c0 < n; c0 += SEL_CHUNK) {
            if (c0 + SEL_CHUNK < n) load_chunk(c0 + SEL_CHUNK, vn);
            if (c0 + SEL_CHUNK <= n) scan_chunk(c0, std::true_type{});
            else scan_chunk(c0, std::false_type{});
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = vn[u];
        }
        if (lane == 0) wave_tot[wv] = wave_count;

        // ---- 3. bucket of every candidate of the wave's own region (up to eight per lane) and its slot
        // inside the bucket
        uint32_t cpos[CPT];
        float csc[CPT];
#pragma unroll
        for (int u = 0; u < CPT; ++u) {
            const uint32_t j = (uint32_t)(u * 64 + lane);
            cpos[u] = j < wave_count ? cand[wv * SEL_WAVE_CAP + j] : 0u;
            csc[u] = (uint32_t)(u * 64) < wave_count ? srow[cpos[u]] : 0.f;             // (uniform: trips past the last are left out)
        }
#pragma unroll
        for (int u = 0; u < CPT; ++u)
            if ((uint32_t)(u * 64 + lane) < wave_count) to_bucket(u, csc[u], cpos[u], blo, bscale);
        __syncthreads();
        const uint32_t n_cand = (uint32_t)__builtin_amdgcn_readlane((int)row_incl_scan(wave_tot[lane & 15]), 15);
        if (sh_over != 0u || n_cand < (uint32_t)k) {
            select_streaming(p, t, hist, stage);                     // uniform: the whole workgroup goes
            return;
        }
        offsets();
    }

    const uint32_t tb = sh_tb;
    const uint32_t n_stage = sh_stage;
    if (n_stage > (uint32_t)SEL_STAGE) {
        select_streaming(p, t, hist, stage);
        return;
    }
#pragma unroll
    for (int u = 0; u < CPT; ++u) {
        if (cb[u] <= tb) {
            const uint32_t idx = boff[cb[u]] + cslot[u];
            stage[idx] = ce[u];
            sbucket[idx] = (uint16_t)cb[u];
        }
    }
    __syncthreads();
    // Order inside buckets by counting.  Neighbouring threads take neighbouring staged entries, which
    // mostly share a bucket, so the loop lengths of a wave agree and its LDS reads are broadcasts; a
    // thread's two entries are ranked side by side, four keys of each bucket per trip, to keep eight
    // reads in flight.  Entries past the first 2048 (the tail of the last bucket) take a second trip
    // that only the waves holding them make.
    for (uint32_t i0 = 0; i0 < n_stage; i0 += 2 * SEL_THREADS) {
        if (i0 + (uint32_t)(wv * 64) >= n_stage) break;          // wave-uniform: nothing staged for this wave
        unsigned long long e[2];
        uint32_t beg[2], len[2], rank[2];
        uint32_t maxlen = 0;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const uint32_t i = i0 + (uint32_t)(q * SEL_THREADS + tid);
            const bool ok = i < n_stage;
            e[q] = stage[ok ? i : 0u];
            const uint32_t bk = sbucket[ok ? i : 0u];
            beg[q] = boff[bk];
            len[q] = ok ? boff[bk + 1u] - beg[q] : 0u;
            rank[q] = 0u;
            maxlen = len[q] > maxlen ? len[q] : maxlen;
        }
        for (uint32_t j = 0; j < maxlen; j += 4) {
#pragma unroll
            for (int q = 0; q < 2; ++q) {
#pragma unroll
                for (uint32_t d = 0; d < 4; ++d) {
                    const bool in = j + d < len[q];
                    const unsigned long long x = stage[in ? beg[q] + j + d : 0u];
                    rank[q] += (in && x > e[q]) ? 1u : 0u;
                }
            }
        }
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const uint32_t fin = beg[q] + rank[q];
            if (i0 + (uint32_t)(q * SEL_THREADS + tid) < n_stage && fin < (uint32_t)kk) out[fin] = (int32_t)(~(uint32_t)e[q]);
        }
    }
}

}  // namespace

hipError_t li_launch(const LiParams &p, hipStream_t stream)
{
    const dim3 block(64 * LI_SCORE_WAVES);
    const int nt = p.nt;
    const dim3 grid((unsigned)p.score_wgs);
    const bool hw = p.q_dt == PTO_DT_FP16 && p.w_dt == PTO_DT_FP16;
#define LI_SCORE(KDT)                                                                                                      \
    do {                                                                                                                   \
        if (nt == 2) {                                                                                                     \
            if (hw) hipLaunchKernelGGL((li_score_kernel<KDT, 0, 2, true>), grid, block, 0, stream, p);                     \
            else hipLaunchKernelGGL((li_score_kernel<KDT, 0, 2, false>), grid, block, 0, stream, p);                       \
        } else {                                                                                                           \
            if (hw) hipLaunchKernelGGL((li_score_kernel<KDT, 0, 1, true>), grid, block, 0, stream, p);                     \
            else hipLaunchKernelGGL((li_score_kernel<KDT, 0, 1, false>), grid, block, 0, stream, p);                       \
        }                                                                                                                  \
    } while (0)
    if (p.variant == 1) hipLaunchKernelGGL((li_score_kernel<PTO_DT_FP16, 1>), grid, block, 0, stream, p);
    else if (p.k_dt == PTO_DT_FP32) LI_SCORE(PTO_DT_FP32);
    else if (p.k_dt == PTO_DT_FP16) LI_SCORE(PTO_DT_FP16);
    else LI_SCORE(PTO_DT_BF16);
#undef LI_SCORE
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(li_select_kernel, dim3((unsigned)p.T), dim3(SEL_THREADS), 0, stream, p);
    return hipGetLastError();
}

}  // namespace pto
