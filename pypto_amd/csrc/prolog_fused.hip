// MLA prolog + lightning-indexer prolog as one operator (mla_indexer_prolog_quant_d/_p of the reference,
// examples/models/deepseek_v32_exp/mla_indexer_prolog_quant_impl.py:141-256).  Three launches, the MLA prolog's with the
// indexer prolog's work in them:
//   sums over the hidden axis   up to 8 tokens wk as one more column slab, w_proj beside the rope columns of w_dkv_kr
//                        (MlapRider, 64 indexer heads); beyond, its fixed-order sums as further workgroups
//   latents              norms and quantisation
//   projections and everything behind them   a workgroup per head of either query (up to 32 tokens: prolog_small.h) or per head
//                        and tile of tokens (prolog_prefill.h), and workgroups for the indexer's key rows and weights
// With absorb_exact and fewer than 64 tokens the projections are a launch of their own (jobs of one kind), and the last one
// finishes both queries from their partial sums: the workgroups that finish the attention query (absorb product, 68 KB of LDS,
// four waves) and those that finish the indexer's query rows, key row and weights (54 KB, eight waves) do not depend on each
// other and fit a compute unit together.  Where the indexer prolog cannot ride (other than 64 indexer heads up to 8 tokens or
// with absorb_exact, w_proj rows that are no power of two of 16-byte pieces, sums over the hidden axis in the cores' order)
// its own launches follow.
#include <cstring>

#include "prolog_fused.h"
#include "prolog_prefill.h"
#include "prolog_small.h"
#include "lip_xjob.h"

namespace pto {
namespace {

constexpr int FUSED_FIN_LDS = MLAP_FIN_LDS > LIP_FIN_LDS ? MLAP_FIN_LDS : LIP_FIN_LDS;
static_assert(2 * FUSED_FIN_LDS <= 160 * 1024, "two workgroups of the last launch share a compute unit");

// Workgroups [0, mla_wgs): the MLA prolog's last launch (its 256 threads; the other four waves pass the body's
// barriers with them and leave).  The rest: the indexer prolog's second launch.
__global__ __launch_bounds__(64 * FIN_WAVES) void prolog_fused_finish_kernel(const MlapParams pm, const LipParams pl, const int mla_wgs,
                                                                             const int q_wgs)
{
    __shared__ __attribute__((aligned(16))) uint8_t lds[FUSED_FIN_LDS];
    if ((int)blockIdx.x < mla_wgs) {
        if (threadIdx.x >= 256) {
            for (int i = 0; i < MLAP_FIN_BARRIERS; ++i) __syncthreads();
            return;
        }
        mlap_finish_body(pm, (int)blockIdx.x, lds);
    } else {
        lip_finish_body(pl, q_wgs, (int)blockIdx.x - mla_wgs, lds);
    }
}

// Projections and last stages at prefill sizes (prolog_prefill.h): [0, mla_wgs) the attention query, then lip_wgs of the
// indexer query, then the indexer's key rows and weights, a token per wave.  64 * TB tokens per workgroup of a head of the
// attention query, 128 * LTB of the indexer's.
// HB: heads per workgroup of four waves each, which share the tokens.
// FIXED: the indexer query's Hadamard sums in their fixed order (fewer than LIP_MFMA_MIN_TOKENS tokens).
constexpr int pf_xc(const int ltb, const int hb) { return ltb == 1 || hb == 2 ? 2 : 1; }
template <int XC, int TB, int LTB, int HB>
constexpr int PF_LDS2 = PFA_LDS<XC, TB, HB> > PFI_LDS<pf_xc(LTB, HB), LTB, HB> ? PFA_LDS<XC, TB, HB> : PFI_LDS<pf_xc(LTB, HB), LTB, HB>;
template <int XC, int TB, int LTB, int HB>
constexpr int PF_LDS = PF_LDS2<XC, TB, LTB, HB> > LIP_FINT_LDS<4 * HB> ? PF_LDS2<XC, TB, LTB, HB> : LIP_FINT_LDS<4 * HB>;
template <int XC, int TB, int LTB, int HB, bool FIXED>
__global__ __launch_bounds__(256 * HB, 2) void prolog_prefill_kernel(const MlapParams pm, const LipParams pl, const int mla_wgs, const int lip_wgs)
{
    static_assert(2 / HB * PF_LDS<XC, TB, LTB, HB> <= 160 * 1024, "eight waves share a compute unit");
    __shared__ __attribute__((aligned(16))) uint8_t lds[PF_LDS<XC, TB, LTB, HB>];
    const int wg = (int)blockIdx.x;
    if (wg < mla_wgs) mlap_prefill_body<XC, TB, HB>(pm, q_prefill_job_of(wg, mla_wgs), lds);
    else if (wg < mla_wgs + lip_wgs) lip_prefill_body<pf_xc(LTB, HB), LTB, HB, FIXED>(pl, q_prefill_job_of(wg - mla_wgs, lip_wgs), lds);
    else lip_finish_tokens_prefill_body<4 * HB>(pl, wg - mla_wgs - lip_wgs, lds);
}

// The same for at most PROLOG_SMALL_TOKENS tokens (prolog_small.h), a workgroup per head.
constexpr int PS_LDS = PSA_LDS > PSI_LDS ? PSA_LDS : PSI_LDS;
static_assert(LIP_FINT_LDS<4> <= PS_LDS, "the token workgroups fit");
__global__ __launch_bounds__(256) void prolog_small_kernel(const MlapParams pm, const LipParams pl, const int mla_wgs, const int lip_wgs)
{
    __shared__ __attribute__((aligned(16))) uint8_t lds[PS_LDS];
    const int wg = (int)blockIdx.x;
    if (wg < mla_wgs) mlap_small_body(pm, prolog_small_head(wg, pm.n_heads), lds);
    else if (wg < mla_wgs + lip_wgs) lip_small_body(pl, wg - mla_wgs, lds);
    else lip_finish_tokens_prefill_body<4>(pl, wg - mla_wgs - lip_wgs, lds);
}

}  // namespace

hipError_t prolog_prefill_launch(const MlapParams *pm, const LipParams *pl, hipStream_t stream)
{
    const int T = pm ? pm->T : pl->T;
    MlapParams m;
    LipParams p;
    std::memset(&m, 0, sizeof m);
    std::memset(&p, 0, sizeof p);
    if (pm) m = *pm;
    if (pl) p = *pl;
    if (T <= PROLOG_SMALL_TOKENS) {
        const int mla = pm ? m.n_heads : 0, lip = pl ? p.n_heads : 0, tok = pl ? (T + 3) / 4 : 0;
        hipLaunchKernelGGL(prolog_small_kernel, dim3((unsigned)(mla + lip + tok)), dim3(256), 0, stream, m, p, mla, lip);
        return hipGetLastError();
    }
    // Up to 64 tokens the attention query's tiles have 64 (in tiles of 128, half and more of them padding: fused prolog 33 tokens 41.4
    // us per pass, now 40.6, 48: 43.3 and 42.4, 64: 44.6 and 43.6; MLA prolog alone 33: 35.9 and 34.1, 64: 39.9 and 38.7).
    // Tiles of 256 tokens from 257 on (tiles of 128, 307 tokens 91.5 us per pass, now 85.4, 384: 99.3 and 90.7, 600: 132.4 and 131.4,
    // 800: 165.0 and 160.5; 256 tokens the other way, 72.5 and 92.4: a tile per head leaves half of the chip's places empty) -- but where few
    // heads make workgroups for less than three quarters of the compute units, and the indexer's do not fill their places (tiles of
    // 256 / 128: MLA prolog alone, 16 heads, 300 tokens 63.3 / 50.9, 1000 86.2 / 76.0, 64 heads 512 76.2 / 64.6, 600 79.7 / 80.0; fused, 32
    // and 64 heads, 400 tokens 83.2 / 73.9, 769 113.6 / 120.0, 16 and 8 heads, 1000 tokens 114.5 / 104.2).
    const int cus = cu_count();
    if (cus <= 0) return hipErrorNoDevice;
    const int tiles128 = (T + 127) / 128, tiles256 = (T + 255) / 256;
    const int mla256 = pm ? m.n_heads * tiles256 : 0;
    const bool small = T <= 256 || (pm && 4 * mla256 < 3 * cus && mla256 + (pl ? p.n_heads * tiles128 : 0) <= 2 * cus);
    const int tiles = small ? tiles128 : tiles256;
    // Two heads to a workgroup of eight waves, which then reads each token once and as whole cache lines, from four tiles and 64 heads on,
    // where they are for six tenths of the compute units or more (one / two, on a fast card: 680 tokens 142.3 / 143.3 us per pass, 1000
    // 185.3 / 177.2, 1300 251.1 / 238.1, 1500 273.2 / 259.1, 2112 375.6 / 365.3, 4096 662.9 / 659.9; on a slow one: 1000 196.1 / 194.9, 1300
    // 265.9 / 258.8, 1500 288.5 / 276.8, 2112 397.1 / 399.2; 64 heads 1300 tokens 192.7 / 187.0, with 32 of the indexer 800 121.7 / 130.3; 16
    // heads 1000 126.6 / 140.6, 4096 396.0 / 399.7; 32 heads 1000 130.1 / 143.2, 3000 331.9 / 337.2).
    // The MLA prolog alone, with nothing behind them, takes them where their last round is six tenths full or more (one / two: 600
    // tokens 105.0 / 101.2, 1000 129.3 / 124.2, 1025 156.4 / 167.2, 1280 178.9 / 190.1, 1536 198.6 / 204.4, 1792 229.7 / 222.3, 2500 326.7 /
    // 331.3, 2816 359.5 / 351.5, 3500 420.4 / 428.5, 4096 492.4 / 466.6; 64 heads 1000 99.6 / 113.3, 1152 127.8 / 122.6, 2500 242 / 259).
    const int pairs = mla256 / 2, last_round = pairs % cus;
    const bool two = pl ? tiles >= 4 && m.n_heads >= 64 && 5 * pairs >= 3 * cus : pairs > 0 && (last_round == 0 || 5 * last_round >= 3 * cus);
    const int hb = pm && !small && two ? 2 : 1;
    const int mla_wgs = pm ? m.n_heads / hb * tiles : 0;
    // The indexer's half, whose workgroups are the shorter ones, is cut into tiles of 128 tokens up to six tiles of 256 of 64 heads (fused
    // prolog, tiles of 256 / 128: 1000 tokens 195.9 / 187.6 us per pass, 1300 252.3 / 243.9, 1500 271.3 / 265.7, 1800 315.8 / 322.2, 4096 652.3 /
    // 668.8; the indexer prolog alone 400: 45.3 / 36.4, 512: 46.2 / 37.5, 1536: 85.5 / 84.4, 2000: 107.0 / 110.3).
    const bool lip_small = small || (pl && 2 * p.n_heads * tiles <= 3 * cus);
    const int lip_wgs = pl ? (p.n_heads + hb - 1) / hb * (lip_small ? (T + 127) / 128 : tiles) : 0;
    const int tok_wgs = pl ? (T + 4 * hb - 1) / (4 * hb) : 0;
    const dim3 g((unsigned)(mla_wgs + lip_wgs + tok_wgs));
    auto run = [&](auto *kernel) { hipLaunchKernelGGL(kernel, g, dim3(256 * hb), 0, stream, m, p, mla_wgs, lip_wgs); };
    if (T < LIP_MFMA_MIN_TOKENS) run(prolog_prefill_kernel<2, 1, 1, 1, true>);
    else if (T <= PFA_TOK<1>) run(prolog_prefill_kernel<2, 1, 1, 1, false>);
    else if (small) run(prolog_prefill_kernel<2, 2, 1, 1, false>);
    else if (hb == 2 && lip_small) run(prolog_prefill_kernel<2, 4, 1, 2, false>);
    else if (hb == 2) run(prolog_prefill_kernel<2, 4, 2, 2, false>);
    else if (lip_small) run(prolog_prefill_kernel<1, 4, 1, 1, false>);
    else run(prolog_prefill_kernel<1, 4, 2, 1, false>);
    return hipGetLastError();
}

hipError_t prolog_fused_launch(const MlapParams &pm, const LipParams &pl, hipStream_t stream)
{
    // The fixed-order first launch: the indexer prolog's sums over the hidden axis are more column slabs of it and, with
    // absorb_exact, its int8 projection more jobs of the third (MlapRider).
    if (mlap_takes_rider(pm) && pl.T == pm.T && pl.h == pm.h && pl.q_lora == pm.q_lora && pl.x == pm.x && pl.q_norm == pm.q_norm &&
        pl.q_norm_scale == pm.q_norm_scale && pl.n_heads == 64) {
        const MlapRider rd = {pl.wk, pl.w_proj, pl.xpart, pl.w_qb, pl.qpart, pl.n_heads};
        hipError_t e = mlap_launch_front(pm, stream, &rd);
        if (e != hipSuccess) return e;
        LipParams pg = pl;
        pg.x_in_groups = 1;
        if (mlap_fused_projection(pm)) return prolog_prefill_launch(&pm, &pg, stream);
        const int mla_wgs = mlap_finish_wgs(pm);
        const int q_wgs = lip_finish_query_wgs(pg);
        hipLaunchKernelGGL(prolog_fused_finish_kernel, dim3((unsigned)(mla_wgs + q_wgs + pg.T)), dim3(64 * FIN_WAVES), 0, stream, pm, pg,
                           mla_wgs, q_wgs);
        return hipGetLastError();
    }
    // From 9 tokens on the MLA prolog's prefill forms take the indexer prolog's fixed-order sums along in the first launch, and
    // the last one makes and finishes both queries: three launches.  (On its own the indexer prolog keeps its two decode
    // launches below 64 tokens: 9 tokens 14.1 us per pass against 20.6 as the sums and this last launch, 32: 18.2 and 23.7.)
    const bool lip_rides = mlap_takes_lip_rider(pm) && pl.T == pm.T && pl.h == pm.h && pl.q_lora == pm.q_lora && pl.x == pm.x &&
                           pl.q_norm == pm.q_norm && pl.q_norm_scale == pm.q_norm_scale && !lip_x_on_matrix_cores(pl) &&
                           lip_x_group_width(pl) && pl.n_heads <= LIP_MAX_HEADS;
    LipParams px = pl;
    if (lip_rides) px.x_in_groups = 1;
    hipError_t e = mlap_launch_front(pm, stream, nullptr, lip_rides ? &px : nullptr);
    if (e != hipSuccess) return e;
    const bool joined = mlap_fused_projection(pm) && (lip_q_on_matrix_cores(px) || (lip_rides && px.T < LIP_MFMA_MIN_TOKENS));
    if (!joined || !lip_rides) {
        e = lip_launch_linear(px, stream);
        if (e != hipSuccess) return e;
    }
    if (joined) return prolog_prefill_launch(&pm, &px, stream);
    if (mlap_fused_projection(pm) || lip_q_on_matrix_cores(px)) {        // one half's last stage is part of its projection
        e = mlap_launch_finish(pm, stream);
        if (e != hipSuccess) return e;
        return lip_launch_finish(px, stream);
    }
    const int mla_wgs = mlap_finish_wgs(pm);
    const int q_wgs = lip_finish_query_wgs(px);
    hipLaunchKernelGGL(prolog_fused_finish_kernel, dim3((unsigned)(mla_wgs + q_wgs + px.T)), dim3(64 * FIN_WAVES), 0, stream, pm, px,
                       mla_wgs, q_wgs);
    return hipGetLastError();
}

}  // namespace pto
