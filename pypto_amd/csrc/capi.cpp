// C ABI of the library: argument validation, workspace sizing, launch heuristics.
// Declarations and the reference interfaces they stand in for: include/pypto_amd_sfa.h.
#include "pypto_amd_sfa.h"

#include <hip/hip_runtime.h>

#include <atomic>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <mutex>

#include "li_kernels.h"
#include "lip_kernels.h"
#include "prolog_fused.h"
#include "mlap_kernels.h"
#include "sfa_kernels.h"

// Scratch memory of pto_sfa_quant_launch_static: the partial results of the key splits live here
// instead of in a caller workspace.  One copy per GPU the library's code object is loaded on, held
// until the process ends.  In host code the name below is only a handle; the device address is asked
// for once per device (scratch_of) and that pointer is what the kernels get.
constexpr size_t SFA_STATIC_SCRATCH_BYTES = (size_t)40 << 20;
static __device__ __align__(256) unsigned char scratch[SFA_STATIC_SCRATCH_BYTES];

namespace {

thread_local char g_err[512] = "";

int fail(int code, const char *fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
    return code;
}

}  // namespace

namespace pto {
// compute units of the current device (one query per device ordinal, then cached)
int cu_count()
{
    constexpr int MAX_DEVICES = 64;
    static std::atomic<int> cached[MAX_DEVICES];
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    if (dev >= 0 && dev < MAX_DEVICES) {
        n = cached[dev].load(std::memory_order_relaxed);
        if (n > 0) return n;
    }
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) return 0;
    if (dev >= 0 && dev < MAX_DEVICES) cached[dev].store(n, std::memory_order_relaxed);
    return n;
}
}  // namespace pto

namespace {

using pto::cu_count;

// device address of this device's copy of the scratch array (NULL and *err set on failure)
void *scratch_of(int dev, hipError_t *err)
{
    constexpr int MAX_DEVICES = 64;
    static std::atomic<void *> ptrs[MAX_DEVICES];
    static std::mutex mu;
    *err = hipSuccess;
    if (dev < 0 || dev >= MAX_DEVICES) {
        *err = hipErrorInvalidDevice;
        return nullptr;
    }
    void *p = ptrs[dev].load(std::memory_order_acquire);
    if (p) return p;
    std::lock_guard<std::mutex> lock(mu);
    p = ptrs[dev].load(std::memory_order_relaxed);
    if (p) return p;
    void *addr = nullptr;
    *err = hipGetSymbolAddress(&addr, HIP_SYMBOL(scratch));     // the current device is dev (checked by the caller)
    if (*err != hipSuccess || !addr) {
        if (*err == hipSuccess) *err = hipErrorInvalidSymbol;
        return nullptr;
    }
    ptrs[dev].store(addr, std::memory_order_release);
    return addr;
}

struct SfaPlan {
    int head_groups;      // groups of 32 heads per workgroup: 1, 2 or 4
    int hgroups;          // workgroups that share a row's heads
    int nsplit;
    int whole_slots;      // rows 0 .. 8 * whole_slots - 1 are not split
    long long split_rows; // the others, or all of them
    bool part_f32;        // partial results in fp32 instead of fp16
    size_t scratch_bytes; // what a caller is asked for, for partial results: the launch uses as much or less
    size_t part_o_bytes;  // what the launch uses of it
    size_t part_ml_bytes;
    size_t predeq_bytes;  // the whole cache de-quantised once, behind the partial results (0: not worth it)
    size_t predeq_offset; // where in the workspace
};

constexpr size_t SFA_PREDEQ_MAX_BYTES = (size_t)64 << 20;

int sfa_check(const PtoSfaQuantArgs *a)
{
    if (!a) return fail(PTO_E_INVALID_ARG, "sfa: args is NULL");
    if (a->b < 1 || a->s1 < 1 || a->nq < 1) return fail(PTO_E_INVALID_ARG, "sfa: b, s1, nq must be >= 1");
    if (a->n_kv != 1) return fail(PTO_E_INVALID_ARG, "sfa: n_kv must be 1 (got %lld)", (long long)a->n_kv);
    if (a->topk < 1) return fail(PTO_E_INVALID_ARG, "sfa: topk must be >= 1");
    if (a->block_size < 1 || a->max_blocknum_perbatch < 1)
        return fail(PTO_E_INVALID_ARG, "sfa: block_size and max_blocknum_perbatch must be >= 1");
    if (a->kv_rows < 1) return fail(PTO_E_INVALID_ARG, "sfa: kv_rows must be >= 1");
    if (a->b > (1ll << 24) || a->s1 > (1ll << 24) || a->b * a->s1 > (1ll << 24) || a->nq > 65536 || a->topk > (1ll << 24) ||
        a->kv_rows > 0x7fffffffll || a->block_size > (1ll << 30) || a->max_blocknum_perbatch > (1ll << 30))
        return fail(PTO_E_INVALID_ARG, "sfa: shape out of the supported range");
    if (a->num_splits < 0) return fail(PTO_E_INVALID_ARG, "sfa: num_splits must be >= 0");
    if (!std::isfinite(a->softmax_scale)) return fail(PTO_E_INVALID_ARG, "sfa: softmax_scale is not finite");
    return PTO_OK;
}

// What dividing a call's rows over workgroups takes, in microseconds: what a launch pair over an int8 cache took over 1 to 128 rows x
// 16 to 128 heads x 1 to 64 splits (fitted to within 10 %; neighbouring choices differ by less).  The same figures serve the other
// cache formats and every number of keys.  A compute unit holds one workgroup; a round of them
// is as long as a split's tiles; starting, staging the query and the first tile and the merge launch are `fixed`, and
// the partial results cost with the number of workgroups that write them.  Fewer head groups per workgroup make
// a tile shorter, and the prologue, but the tiles of a row are de-quantised once per workgroup: that pays while the
// chip is not full (128 heads, 1 row: 22.0 us as 16 splits of four groups, 14.3 as 32 splits of one; 4 rows: 22.5, 20.0).
// Two groups are priced as the form of four waves they had when the bytes a caller is asked for were settled (1.58 a tile,
// where sfa_slice_kernel takes 1.1 to 1.45): up to 2048 keys that price chooses nothing, the second model below does.  Beyond,
// where it is not asked, the choice is within 6 % of the fastest division from 64 rows on (128 heads; 64 heads: from 16 on)
// and dear for fewer (4096 keys of an int8 cache, 128 heads: 1 row 19.0 where 32 splits of 64 heads take 16.1, 4 rows 27.1 and
// 22.9, 16 rows 36.7 and 33.0).
struct SfaPrices {
    long long rows, nq;
    int cus;
    int tiles;            // of the longest row
    bool f32;             // split rows leave fp32 partial results

    int shares(const int hg) const { return (int)((nq + 32 * hg - 1) / (32 * hg)); }
    int max_groups() const { return nq > 64 ? 4 : (nq > 32 ? 2 : 1); }
    size_t partial_bytes(const long long r, const int ns, const bool fp32 = false) const
    {
        return ns > 1 ? (size_t)r * ns * nq * (512 * (fp32 ? sizeof(float) : sizeof(uint16_t)) + 2 * sizeof(float)) : (size_t)0;
    }
    long long rounds(const long long wgs) const { return cus % 8 == 0 ? ((wgs + 7) / 8 + cus / 8 - 1) / (cus / 8) : (wgs + cus - 1) / cus; }
    int split_tiles(const int ns) const { return (tiles + ns - 1) / ns; }
    // of the split counts with equally long splits the smallest is the one to take: the one behind ns
    int next_splits(const int ns) const { return split_tiles(ns) > 1 ? (tiles + split_tiles(ns) - 2) / (split_tiles(ns) - 1) : tiles + 1; }

    double round_us(const int hg, const int ns) const { return split_tiles(ns) * (hg == 4 ? 1.75 : (hg == 2 ? 1.58 : 1.47)); }
    double tail_us(const int hg, const long long wgs, const int ns) const
    {
        if (ns == 1) return 6.0;
        const double fixed = hg == 4 ? 10.5 : (hg == 2 ? 9.5 : 9.3), per_wg = hg == 4 ? 0.045 : (hg == 2 ? 0.032 : 0.018);
        return fixed + per_wg * (double)wgs + (ns > 8 ? (hg == 1 ? 0.5 : 1.5) : 0.0);       // (more than eight splits: the wide merge)
    }
    // every row in ns splits, or `full` rounds of whole rows and the rows_b left over in ns splits
    double even(const int hg, const int ns) const
    {
        const long long wgs = rows * shares(hg) * ns;
        return (double)rounds(wgs) * round_us(hg, ns) + tail_us(hg, wgs, ns) +
               (f32 ? 0.25e-6 * (double)(partial_bytes(rows, ns, true) - partial_bytes(rows, ns)) : 0.0);
    }
    double mixed(const int hg, const int ns, const long long full, const long long rows_b) const
    {
        return (double)full * round_us(hg, 1) + round_us(hg, ns) + tail_us(hg, rows_b * shares(hg) * ns, ns);
    }

    // More than 32 heads: workgroups of 64 heads (sfa_slice_kernel).  Fitted to an int8 cache, 1 to 128 rows, top-k 2048,
    // 128 heads (measured: 32 rows 4 splits 32.3, 16 rows 8 splits 24.2, 4 rows 13 splits 18.4, 1 row 22 splits 14.0, against
    // 35.0, 28.6, 20.0 and 14.1 as four groups and one group of 32 heads; 36 to 64 rows alike; 128 rows 97.1 against 95.0).
    // A tile of whole rows takes 1.13 with 128 workgroups, 1.2 with 192 and 1.45 with 256 (top-k 1024, 96 rows: 44.9, as four groups
    // and two splits 49.4); partial results past one round's cost more (64 heads, 96 rows: 5 splits 58.8, 2 splits 51.8).
    // Against the fastest of every form and split count, two rows and more, top-k 1024 and 2048, both caches, the choice is within
    // 5 % in 104 of 108 shapes.  Where it is not: 128 rows of 128 heads over 1024 keys are priced 50.0 as two splits of four groups and
    // 52.4 as whole rows of this form, and take 57.4 and 54.3 (bf16 cache 58.3 and 50.6).  A single row's 32 splits are priced 14.5
    // and its 22 splits 14.1, and take 13.5 and 14.2.
    double slice_round_us(const int ns, const long long wgs) const           // (wgs of the launch: 256 and more fill the chip)
    {
        const int len = split_tiles(ns);
        const double full = wgs < cus ? (double)wgs / cus : 1.0;
        return ns == 1 ? (1.1 + 0.35 * full * full * full * full) * len : (0.59 + 0.0175 * len) * len;
    }
    double slice_tail_us(const long long r, const int ns) const
    {
        const double wgs = (double)(r * shares(2) * ns);
        return ns == 1 ? 6.0 : 13.2 + (ns > 8 ? 0.056 * wgs - 3.5 : 0.02 * wgs + (wgs > cus ? 0.03 * (wgs - cus) : 0.0));
    }
    double slice_even(const int ns) const
    {
        const long long wgs = rows * shares(2) * ns;
        const double n = (double)rounds(wgs);
        return n * slice_round_us(ns, wgs) + (n - 1.0) * 7.0 + slice_tail_us(rows, ns);     // (a further round starts and ends too)
    }
    double slice_mixed(const int ns, const long long full, const long long rows_b) const
    {
        return (double)full * (slice_round_us(1, cus) + 7.0) + slice_round_us(ns, cus) + slice_tail_us(rows_b, ns);
    }

    // of up to 2048 keys
    double of(const SfaPlan &pl) const
    {
        const bool slice = nq > 32 && pl.head_groups == 2;
        if (pl.whole_slots == 0) return slice ? slice_even(pl.nsplit) : even(pl.head_groups, pl.nsplit);
        const long long full = pl.whole_slots / (cus / 8 / shares(pl.head_groups)), rows_b = rows - 8ll * pl.whole_slots;
        return slice ? slice_mixed(pl.nsplit, full, rows_b) : mixed(pl.head_groups, pl.nsplit, full, rows_b);
    }
};

// The cheapest division by these prices of those whose partial results fit max_bytes (an explicit num_splits is taken as it is); with
// keep_whole of those that split no row.
SfaPlan sfa_divide(const PtoSfaQuantArgs *a, const SfaPrices &m, const size_t max_bytes, const bool keep_whole)
{
    SfaPlan pl{};
    const long long rows = m.rows;
    const int cus = m.cus, tiles = m.tiles, hg_max = m.max_groups();
    const bool f32 = m.f32;
    const int min_split = (int)((a->topk + pto::SFA_MAX_CHUNK - 1) / pto::SFA_MAX_CHUNK);
    const bool automatic = a->num_splits == 0 && min_split == 1;
    pl.head_groups = hg_max;
    int ns = a->num_splits;
    double best = -1.0;
    if (ns == 0) {
        for (int hg = hg_max; hg >= 1; hg /= 2)
            for (int s = min_split; s <= (keep_whole ? 1 : f32 ? (hg > 1 ? 1 : tiles < 8 ? tiles : 8) : tiles); s = m.next_splits(s)) {
                if (s > min_split && (m.partial_bytes(rows, s, f32) > max_bytes || rows * m.shares(hg) * s > 4ll * cus)) break;
                const double cost = m.even(hg, s);
                if (best < 0.0 || cost < best) {
                    best = cost;
                    ns = s;
                    pl.head_groups = hg;
                }
            }
    }
    ns = ns < min_split ? min_split : ns;
    ns = ns > tiles ? tiles : ns;
    ns = ns < 1 ? 1 : ns;
    pl.hgroups = m.shares(pl.head_groups);
    pl.nsplit = ns;
    pl.split_rows = rows;
    if (automatic && !f32 && !keep_whole && cus % 8 == 0) {
        // More rows than compute units: the full rounds of whole rows first, then the rows left over dealt out in
        // as many pieces as fill one more round (300 rows on 256 CUs: 32 whole rows per XCD, the other five or
        // six in five pieces each), where that beats the best uniform split above.
        const long long xcd_rows = (rows + 7) / 8;
        const long long per_round = cus / 8 / m.shares(hg_max);               // rows of an XCD that one round holds
        const long long full = per_round > 0 ? xcd_rows / per_round : 0;
        const long long rows_b = rows - 8 * full * per_round;                 // rows 8 * whole_slots and up
        if (full >= 1 && rows_b >= 1) {
            int sb = (int)(cus / (rows_b * m.shares(hg_max)));
            const int max_split = tiles / 4 > 0 ? tiles / 4 : 1;              // (a last round shorter than four tiles is all prologue)
            sb = sb > max_split ? max_split : sb;
            if (sb >= 2 && m.partial_bytes(rows_b, sb) <= max_bytes) {
                const double cost = m.mixed(hg_max, sb, full, rows_b);
                if (cost < best) {
                    best = cost;
                    pl.head_groups = hg_max;
                    pl.hgroups = m.shares(hg_max);
                    pl.nsplit = sb;
                    pl.whole_slots = (int)(full * per_round);
                    pl.split_rows = rows_b;
                }
            }
        }
    }
    pl.part_f32 = f32 && pl.nsplit > 1;
    pl.scratch_bytes = m.partial_bytes(pl.split_rows, pl.nsplit, f32);
    // Workgroups of 64 heads where they are the faster ones, within the bytes that a caller is asked for, which stay those of
    // the division above.
    if (a->nq > 32 && automatic) {
        const int sh = m.shares(2);
        if (pl.head_groups == 2) best = -1.0;             // (two groups of 32 heads: that is this form, at another price)
        auto take = [&](const double cost, const int s, const long long whole) {
            if (best >= 0.0 && cost >= best) return;
            best = cost;
            pl.nsplit = s;
            pl.head_groups = 2;
            pl.hgroups = sh;
            pl.whole_slots = (int)(whole / 8);
            pl.part_f32 = false;
            pl.split_rows = rows - whole;
        };
        for (int s = 1; s <= (f32 || keep_whole ? 1 : tiles); s = m.next_splits(s)) {
            if (s > 1 && (m.partial_bytes(rows, s) > pl.scratch_bytes || rows * sh * s > 4ll * cus)) break;
            take(m.slice_even(s), s, 0);
        }
        const long long per_round = cus / 8 / sh, full = per_round > 0 ? (rows + 7) / 8 / per_round : 0, rows_b = rows - 8 * full * per_round;
        if (!f32 && !keep_whole && cus % 8 == 0 && full >= 1 && rows_b >= 1) {            // full rounds of whole rows, the rows left over in pieces
            int s = (int)(cus / (rows_b * sh));
            s = s > tiles / 4 ? tiles / 4 : s;
            while (s >= 2 && m.partial_bytes(rows_b, s) > pl.scratch_bytes) --s;
            if (s >= 2) take(m.slice_mixed(s, full, rows_b), s, 8 * full * per_round);
        }
    }
    return pl;
}

// max_bytes: most bytes of partial results the caller can hold; the automatic choice (num_splits = 0) then takes the
// best split count among those that fit (an explicit count is the caller's own business)
SfaPlan sfa_plan(const PtoSfaQuantArgs *a, const size_t max_bytes = ~(size_t)0)
{
    const long long rows = a->b * a->s1;
    const int topk_tiles = (int)((a->topk + pto::SFA_KEY_TILE - 1) / pto::SFA_KEY_TILE);
    // (a size query on a host without a device plans for the 256 CUs of an MI355X; a launch there fails)
    const int cus = cu_count() > 0 ? cu_count() : 256;
    SfaPrices m = {rows, a->nq, cus, topk_tiles, false};
    const bool automatic = a->num_splits == 0 && a->topk <= pto::SFA_MAX_CHUNK;
    // A split row's partial results are fp16: one more rounding, to 11 bits, and a bf16 cache's values beyond 65504 become
    // infinite, where a whole row goes from its fp32 accumulators straight to bf16.  So the launches whose partials are fp16 are a
    // fixed set, and a launch outside of it that the model splits all the same leaves its partials in fp32.  The set: no
    // split shorter than four tiles, rows dealt to the XCDs whole (row t on XCD t % 8), costs in tiles -- 3 per round around whole
    // rows, 5.5 around split ones, the merge 1 and one per hundred partial rows.  (fp32 partials cost 0.25 us per MB they are
    // larger by; only workgroups of one head group leave them.  16 heads, whole rows against fp32 partials: 50 rows of 256 keys
    // 18.1 us and 14.7, 150 of 1024 58.7 and 52.3, 170 of 2048 109 and 88.6 -- as fp16 partials 12.8, 50.1 and 85.7.)
    auto half_partials = [&]() {
        const int sh = m.shares(m.max_groups()), max_split = topk_tiles / 4;
        if (cus % 8 != 0) return max_split > 1 && rows * sh < cus;
        const long long xcd_cus = cus / 8, xcd_rows = (rows + 7) / 8;
        auto xcd_rounds = [&](const int s) { return (double)((xcd_rows * sh * s + xcd_cus - 1) / xcd_cus); };
        const double whole = xcd_rounds(1) * (topk_tiles + 3.0);
        auto merge = [&](const long long r, const int s) { return 1.0 + 0.01 * (double)r * s * sh; };
        for (int s = 2; s <= max_split && m.partial_bytes(rows, s) <= max_bytes; ++s)
            if (xcd_rounds(s) * ((topk_tiles + s - 1) / s + 5.5) + merge(rows, s) < whole) return true;
        // full rounds of whole rows, and the rows left over in as many pieces as fill one more (below)
        const long long per_round = xcd_cus / sh, full = per_round > 0 ? xcd_rows / per_round : 0;
        const long long left = xcd_rows - full * per_round, rows_b = rows - 8 * full * per_round;
        if (full < 1 || left < 1 || rows_b < 1) return false;
        const int s = (int)(per_round / left < max_split ? per_round / left : max_split);
        return s >= 2 && m.partial_bytes(rows_b, s) <= max_bytes &&
               (double)full * (topk_tiles + 3.0) + (topk_tiles + s - 1) / s + 5.5 + merge(rows_b, s) < whole;
    };
    m.f32 = automatic && !half_partials();
    SfaPlan pl = sfa_divide(a, m, max_bytes, false);
    const size_t scratch_bytes = pl.scratch_bytes;
    // A row has no more keys than its pages hold, whatever topk is.
    const long long row_keys = a->max_blocknum_perbatch * a->block_size;
    if (automatic && row_keys < a->topk) m.tiles = (int)((row_keys + pto::SFA_KEY_TILE - 1) / pto::SFA_KEY_TILE);
    // The rows of a prefill chunk that begins less than a third of the most keys of a row into its sequence are of all lengths: more
    // of them than a round holds may stay whole and start longest first (sfa_last_first), and the launch ends evenly by itself (the
    // last round's rows in pieces / whole: 300 rows over 300 keys 41.7 / 33.6 us, 563 over 563 84.3 / 75.3; 800 over 1500, which
    // begin 700 keys into it, 237 / 256, 1100 over 2000 404 / 415).
    // The more rounds there are, the less the last one costs, and in pieces it costs the less the fewer its rows are.  Behind the first
    // round it has to be for 5/64 of a round per round before it, or 1/32 where most rows grow from short to long (128 heads, in pieces
    // / whole: top-k 2048, 530 over 562 72.8 / 64.7, 800 over 800 114.9 / 104.9, 518 over 646 74.9 / 77.8, 1030 over 1094 178.1 / 183.8;
    // top-k 512, 600 over 632 80.4 / 73.3, 518 over 582 63.4 / 67.5, 780 over 844 96.2 / 107.3, 1300 over 1300 189.0 / 211.9; 64 heads,
    // top-k 1024, 2060 over 2260 276 / 297).  From five rounds of up to 2048 keys on it is the order that counts (128 heads, 2060 over
    // 2060 555 / 545, 4100 over 4100 1552 / 1514).  Over 438 such chunks (64 and 128 heads, top-k 512 to 2048, 262 to 4200 rows) the
    // launch taken is 3.9 % faster than in pieces in the mean and 2.1 % slower at worst (3120 over 3120 1036 / 1058).
    // Of up to 32 heads, whose rows are the shorter ones, the less of a launch the last round is the fewer keys its rows may begin at
    // (in pieces / whole: 300 over 361 34.4 / 26.7 us, 563 over 676 62.1 / 61.5, 800 over 881 92.0 / 87.6, over 1121 122.3 / 127.4, 1100
    // over 1321 171.5 / 176.7, 1608 over 1930 341 / 352).
    const long long before = row_keys - a->s1, most = a->topk < row_keys ? a->topk : row_keys;
    const long long wgs = rows * m.shares(m.max_groups()), round = wgs / cus, left = wgs % cus;
    auto worth = [&]() {
        if (m.max_groups() == 1) return 8 * before * rows < 5 * most * cus;
        return round == 1 || 64 * left > 5 * round * cus || (a->topk >= pto::SFA_MAX_CHUNK && round >= 5 && 5 * before < most) ||
               (32 * left > round * cus && 4 * before < most && 5 * pto::sfa_full_rows(a->s1, a->topk, row_keys) < a->s1);
    };
    const bool ramp = automatic && wgs > cus && 3 * before < most && pto::sfa_last_first(a->b, a->s1, a->nq, a->topk, row_keys, cus) && worth();
    if (ramp) {
        pl = sfa_divide(a, m, max_bytes, true);
    } else if (m.tiles < topk_tiles) {
        // Priced by the keys of its pages a call may be divided another way than by topk.  It is taken where it holds no row's
        // partial results in fewer bits: whole rows stay whole, fp32 partial results fp32.  And it has to
        // be cheaper by what the prices are off by: nothing among up to eight splits of one form (24 rows of 64 heads over 384 keys,
        // 8 splits 17.2 us, 4 splits 14.7), 7 % beyond, where splits are priced too dear (2 rows of 128 heads over 896 keys, 16 splits
        // 12.5, 10 splits, 5 % cheaper by the prices, 13.6), unless half of the splits of 32 heads would be without a key (1 row of 16
        // heads over 896, 64 splits 12.1, 28 splits 10.7), 5 % for whole rows of 64 heads and an eighth for others (128 rows of 128 heads
        // over 384, 2 splits 34.7, whole 24.2; 128 rows of 16 heads over 256, 2 splits 21.2, whole, 10 % cheaper by the prices, 23.9).
        // More splits have to fit the bytes asked for and to be cheaper at all where the wide merge runs either way, by 1.5 % where only they
        // need it (64 heads: 5 rows over 768 keys, top-k 1024, 11 splits 14.2, 12 splits 13.4, 6 over 1792, top-k 2048, 13 splits 16.4, 14
        // splits 15.9; 12 rows over 1920, 8 splits 20.8, 10 splits, 1.8 % cheaper by the prices, 20.7, over 1408, 9 splits, 0.7 %, 18.7
        // and 19.0).
        // Over 903 pairs of divisions (1 to 500 rows, 16 to 128 heads, 128 to 1792 keys, all caches) the one taken is 5.4 % faster in
        // the mean than that of topk, and 4 % slower at worst; the cheaper one by the prices alone is 11 % slower at worst.
        const SfaPlan by_pages = sfa_divide(a, m, max_bytes, false);
        const double was = m.of(pl), gain = (was - m.of(by_pages)) / was;
        const bool few = pl.nsplit <= 8;
        bool better;
        if (by_pages.nsplit > pl.nsplit)
            better = pl.nsplit > 1 && gain > (few ? 0.015 : 0.0) &&
                     m.partial_bytes(by_pages.split_rows, by_pages.nsplit, by_pages.part_f32) <= scratch_bytes;
        else if (by_pages.nsplit == 1) better = gain > (few && by_pages.head_groups == 2 ? 0.05 : 0.125);
        else if (few && by_pages.head_groups == pl.head_groups) better = gain > 0.0;
        else better = gain > 0.07 || (by_pages.head_groups == 1 && pl.nsplit >= 2 * by_pages.nsplit);
        if (better && by_pages.whole_slots == 0 && (pl.whole_slots == 0 || by_pages.nsplit == 1) &&
            (by_pages.nsplit == 1 || by_pages.part_f32 == pl.part_f32))
            pl = by_pages;
    }
    pl.predeq_offset = (pl.scratch_bytes + 255) / 256 * 256;
    pl.scratch_bytes = scratch_bytes;                     // (asked for whatever the width of the block table)
    pl.part_o_bytes = pl.part_ml_bytes = 0;
    if (pl.nsplit > 1) {
        pl.part_ml_bytes = (size_t)pl.split_rows * pl.nsplit * a->nq * 2 * sizeof(float);
        pl.part_o_bytes = m.partial_bytes(pl.split_rows, pl.nsplit, pl.part_f32) - pl.part_ml_bytes;
    }
    // A launch that selects every cache row many times over (a prefill chunk: thousands of query rows over a few
    // thousand keys) de-quantises the cache once into the workspace and attends over the bf16 rows -- the same
    // bits, since the kernel's bf16-cache form reads exactly what its int8 form converts to, without the per-tile
    // conversion (8 % at 4096 query rows over 4096 keys).  Only for caches that fit a modest workspace.
    const size_t dq = (size_t)a->kv_rows * 512 * sizeof(uint16_t);
    pl.predeq_bytes = 0;
    if (rows * a->topk >= 8 * a->kv_rows && dq <= SFA_PREDEQ_MAX_BYTES && pl.predeq_offset + dq <= max_bytes) pl.predeq_bytes = dq;
    return pl;
}

size_t sfa_ws_bytes(const SfaPlan &pl)
{
    const size_t predeq = pl.predeq_bytes ? pl.predeq_offset + pl.predeq_bytes : 0;
    return predeq > pl.scratch_bytes ? predeq : pl.scratch_bytes;
}

constexpr int PACKED_ROW_BYTES = 656;     // 512 int8 | 64 bf16 | 4 fp32

// the packed-cache arguments seen as the three-array ones (the cache pointers are filled in by the caller)
PtoSfaQuantArgs unpacked_view(const PtoSaAntiquantArgs *a)
{
    PtoSfaQuantArgs q;
    std::memset(&q, 0, sizeof(q));
    q.query_nope = a->query_nope;
    q.query_rope = a->query_rope;
    q.key_nope_2d = a->nope_cache;
    q.key_rope_2d = a->nope_cache;
    q.k_nope_scales = a->nope_cache;
    q.topk_indices = a->topk_indices;
    q.block_table = a->block_table;
    q.kv_act_seqs = a->kv_act_seqs;
    q.attention_out = a->attention_out;
    q.workspace = a->workspace;
    q.workspace_bytes = a->workspace_bytes;
    q.b = a->b;
    q.s1 = a->s1;
    q.nq = a->nq;
    q.n_kv = a->n_kv;
    q.topk = a->topk;
    q.block_size = a->block_size;
    q.max_blocknum_perbatch = a->max_blocknum_perbatch;
    q.kv_rows = a->kv_rows;
    q.softmax_scale = a->softmax_scale;
    q.num_splits = a->num_splits;
    return q;
}

// checked arguments -> kernel parameters -> launch; the cache is given as three (base, row pitch) pairs
int sfa_enqueue(const PtoSfaQuantArgs *a, const int8_t *kn, int kn_pitch, const uint8_t *kr, int kr_pitch, const uint8_t *ksc,
                int ksc_pitch, void *hip_stream, bool kn_bf16 = false, const size_t plan_limit = ~(size_t)0)
{
    if (cu_count() <= 0) return fail(PTO_E_NO_DEVICE, "sfa: no usable device is current");
    const SfaPlan pl = sfa_plan(a, plan_limit);
    if (((long long)(a->b * a->s1) + 7) / 8 * 8 * pl.hgroups * pl.nsplit > 0x7ffffff0ll)     // (an upper bound of the grid)
        return fail(PTO_E_INVALID_ARG, "sfa: rows x head groups x key splits exceeds the largest launch");
    {
        const void *al16[] = {a->query_nope, a->query_rope, kn, kr, ksc, a->attention_out, a->workspace};
        for (const void *ptr : al16)
            if (reinterpret_cast<uintptr_t>(ptr) & 15)
                return fail(PTO_E_INVALID_ARG, "sfa: query, cache, output and workspace pointers must be 16-byte aligned");
        const void *al4[] = {a->topk_indices, a->block_table, a->kv_act_seqs};
        for (const void *ptr : al4)
            if (reinterpret_cast<uintptr_t>(ptr) & 3)
                return fail(PTO_E_INVALID_ARG, "sfa: index, block-table and length pointers must be 4-byte aligned");
    }
    const bool predeq = pl.predeq_bytes != 0 && !kn_bf16;
    const size_t need = predeq ? sfa_ws_bytes(pl) : pl.scratch_bytes;
    if (need > 0 && (!a->workspace || a->workspace_bytes < need))
        return fail(PTO_E_WORKSPACE, "sfa: workspace of %zu bytes required, %zu given", need, a->workspace ? a->workspace_bytes : (size_t)0);
    if (predeq) {
        uint16_t *dq = reinterpret_cast<uint16_t *>(static_cast<char *>(a->workspace) + pl.predeq_offset);
        hipError_t e = pto::sfa_dequant_cache(kn, kn_pitch, ksc, ksc_pitch, dq, a->kv_rows, static_cast<hipStream_t>(hip_stream));
        if (e != hipSuccess) return fail(PTO_E_LAUNCH, "sfa: launch failed: %s", hipGetErrorString(e));
        kn = reinterpret_cast<const int8_t *>(dq);
        kn_pitch = 1024;
        kn_bf16 = true;
    }

    pto::SfaParams p;
    p.q_nope = static_cast<const uint16_t *>(a->query_nope);
    p.q_rope = static_cast<const uint16_t *>(a->query_rope);
    p.kn = kn;
    p.kr = kr;
    p.ksc = ksc;
    p.kn_pitch = kn_pitch;
    p.kr_pitch = kr_pitch;
    p.ksc_pitch = ksc_pitch;
    p.kn_bf16 = kn_bf16 ? 1 : 0;
    p.topk_idx = a->topk_indices;
    p.bt = a->block_table;
    p.act = a->kv_act_seqs;
    p.out = static_cast<uint16_t *>(a->attention_out);
    p.part_o = a->workspace;
    p.part_ml = pl.part_ml_bytes > 0 ? reinterpret_cast<float *>(static_cast<char *>(a->workspace) + pl.part_o_bytes) : nullptr;
    p.kv_rows = a->kv_rows;
    p.T = (int)(a->b * a->s1);
    p.S1 = (int)a->s1;
    p.NQ = (int)a->nq;
    p.topk = (int)a->topk;
    p.bs = (int)a->block_size;
    p.maxblk = (int)a->max_blocknum_perbatch;
    p.nsplit = pl.nsplit;
    p.part_f32 = pl.part_f32 ? 1 : 0;
    p.whole_slots = pl.whole_slots;
    p.hgroups = pl.hgroups;
    p.head_groups = pl.head_groups;
    p.scale_log2 = a->softmax_scale * 1.4426950408889634f;
    hipError_t e = pto::sfa_launch(p, static_cast<hipStream_t>(hip_stream));
    if (e == hipErrorNoBinaryForGpu || e == hipErrorInvalidDeviceFunction)
        return fail(PTO_E_NO_DEVICE, "sfa: the library holds gfx950 code only: %s", hipGetErrorString(e));
    if (e != hipSuccess) return fail(PTO_E_LAUNCH, "sfa: launch failed: %s", hipGetErrorString(e));
    return PTO_OK;
}

constexpr long long LI_MAX_SEQ_HOST = pto::LI_MAX_SEQ;

int li_check(const PtoLiDecodeArgs *a)
{
    if (!a) return fail(PTO_E_INVALID_ARG, "li: args is NULL");
    if (a->t < 1 || a->b < 1 || a->t % a->b != 0) return fail(PTO_E_INVALID_ARG, "li: t must be a positive multiple of b");
    if (a->n_heads != 64 || a->head_dim != 128)
        return fail(PTO_E_INVALID_ARG, "li: n_heads must be 64 and head_dim 128 (got %lld, %lld)", (long long)a->n_heads,
                    (long long)a->head_dim);
    if (a->selected_count < 1 || a->selected_count > pto::LI_MAX_SELECT)
        return fail(PTO_E_INVALID_ARG, "li: selected_count must be in [1, %d]", pto::LI_MAX_SELECT);
    if (a->block_size < 32 || a->block_size % 32 != 0) return fail(PTO_E_INVALID_ARG, "li: block_size must be a multiple of 32");
    if (a->block_num < 1 || a->max_blocknum_perbatch < 1) return fail(PTO_E_INVALID_ARG, "li: block_num and max_blocknum_perbatch must be >= 1");
    if (a->max_blocknum_perbatch * a->block_size > pto::LI_MAX_SEQ)
        return fail(PTO_E_INVALID_ARG, "li: max_blocknum_perbatch * block_size exceeds %d", pto::LI_MAX_SEQ);
    if (a->t > (1ll << 20) || a->block_num > 0x7fffffffll || a->block_size > LI_MAX_SEQ_HOST || a->block_num * a->block_size > 0x7fffffffll)
        return fail(PTO_E_INVALID_ARG, "li: shape out of the supported range");
    if (a->t > 65535)
        return fail(PTO_E_INVALID_ARG, "li: at most 65535 query tokens per launch (got %lld)", (long long)a->t);
    if (a->arith_variant != 0 && a->arith_variant != 1) return fail(PTO_E_INVALID_ARG, "li: arith_variant must be 0 or 1");
    if (a->arith_variant == 1 &&
        (a->q_scale_dtype != PTO_DT_FP16 || a->k_scale_dtype != PTO_DT_FP16 || a->weight_dtype != PTO_DT_FP16))
        return fail(PTO_E_INVALID_ARG, "li: arith_variant 1 takes fp16 scales and weights");
    const int dts[3] = {a->q_scale_dtype, a->k_scale_dtype, a->weight_dtype};
    for (int d : dts)
        if (d != PTO_DT_FP16 && d != PTO_DT_FP32 && d != PTO_DT_BF16) return fail(PTO_E_INVALID_ARG, "li: unknown dtype code %d", d);
    return PTO_OK;
}

size_t li_ws_bytes(const PtoLiDecodeArgs *a)
{
    // score rows [t, max_blocknum_perbatch*block_size] fp32, then one sampled score per 16 positions
    const size_t stride = (size_t)a->max_blocknum_perbatch * a->block_size;
    return (size_t)a->t * (stride + stride / pto::LI_SAMPLE_GROUP) * sizeof(float);
}

int lip_check(const PtoLiPrologQuantArgs *a)
{
    if (!a) return fail(PTO_E_INVALID_ARG, "li_prolog: args is NULL");
    if (a->t < 1 || a->t > (1ll << 20)) return fail(PTO_E_INVALID_ARG, "li_prolog: t must be in [1, 2^20]");
    if (a->n_heads < 1 || a->n_heads > pto::LIP_MAX_HEADS)
        return fail(PTO_E_INVALID_ARG, "li_prolog: n_heads must be in [1, %d] (got %lld)", pto::LIP_MAX_HEADS, (long long)a->n_heads);
    static_assert(pto::LIP_MAX_QLORA == 1536, "the list below follows the kernel's instantiations");
    if (a->q_lora_rank != 512 && a->q_lora_rank != 1024 && a->q_lora_rank != 1536)
        return fail(PTO_E_INVALID_ARG, "li_prolog: q_lora_rank must be 512, 1024 or 1536 (got %lld)", (long long)a->q_lora_rank);
    const long long max_h = (long long)pto::LIP_MAX_XGROUPS * pto::LIP_XGROUP * pto::LIP_XBLOCK;
    if (a->h < pto::LIP_XBLOCK || a->h % pto::LIP_XBLOCK != 0 || a->h > max_h)
        return fail(PTO_E_INVALID_ARG, "li_prolog: h must be a positive multiple of %d, at most %lld (got %lld)", pto::LIP_XBLOCK,
                    max_h, (long long)a->h);
    if (a->cache_rows < 1 || a->cache_rows > 0x7fffffffll) return fail(PTO_E_INVALID_ARG, "li_prolog: cache_rows out of range");
    if (!std::isfinite(a->eps) || a->eps < 0) return fail(PTO_E_INVALID_ARG, "li_prolog: eps must be finite and >= 0");
    return PTO_OK;
}

// [4 partial int32 projections | block sums over the hidden axis]
size_t lip_qpart_bytes(const PtoLiPrologQuantArgs *a)
{
    return (size_t)pto::LIP_KSPLIT * a->t * a->n_heads * pto::LIP_DIM * sizeof(int32_t);
}
size_t lip_ws_bytes(const PtoLiPrologQuantArgs *a)
{
    return lip_qpart_bytes(a) + (size_t)(a->h / pto::LIP_XBLOCK) * a->t * pto::LIP_XCOLS * sizeof(float);
}

int mlap_check(const PtoMlaPrologQuantArgs *a)
{
    if (!a) return fail(PTO_E_INVALID_ARG, "mla_prolog: args is NULL");
    if (a->t < 1 || a->t > (1ll << 20)) return fail(PTO_E_INVALID_ARG, "mla_prolog: t must be in [1, 2^20]");
    if (a->n_heads < 2 || a->n_heads % 2 != 0 || a->n_heads > 1024)
        return fail(PTO_E_INVALID_ARG, "mla_prolog: n_heads must be even, in [2, 1024] (got %lld)", (long long)a->n_heads);
    if (a->q_lora_rank != 512 && a->q_lora_rank != 1024 && a->q_lora_rank != 1536)
        return fail(PTO_E_INVALID_ARG, "mla_prolog: q_lora_rank must be 512, 1024 or 1536 (got %lld)", (long long)a->q_lora_rank);
    const long long max_h = (long long)pto::MLAP_MAX_XGROUPS * pto::MLAP_XGROUP * pto::MLAP_XBLOCK;
    if (a->h < pto::MLAP_XBLOCK || a->h % pto::MLAP_XBLOCK != 0 || a->h > max_h)
        return fail(PTO_E_INVALID_ARG, "mla_prolog: h must be a positive multiple of %d, at most %lld (got %lld)", pto::MLAP_XBLOCK,
                    max_h, (long long)a->h);
    if (a->cache_rows < 1 || a->cache_rows > 0x7fffffffll) return fail(PTO_E_INVALID_ARG, "mla_prolog: cache_rows out of range");
    if (!std::isfinite(a->epsilon_cq) || a->epsilon_cq < 0 || !std::isfinite(a->epsilon_ckv) || a->epsilon_ckv < 0)
        return fail(PTO_E_INVALID_ARG, "mla_prolog: epsilons must be finite and >= 0");
    return PTO_OK;
}

// [group sums over the hidden axis | 4 partial int32 projections]
size_t mlap_xpart_bytes(const PtoMlaPrologQuantArgs *a)
{
    const size_t rows = (size_t)pto::mlap_xpart_rows((int)a->h, (int)a->t);
    const size_t bytes = rows * a->t * (a->q_lora_rank + pto::MLAP_KV + pto::MLAP_ROPE) * sizeof(float);
    return (bytes + 255) & ~(size_t)255;
}
size_t mlap_ws_bytes(const PtoMlaPrologQuantArgs *a)
{
    return mlap_xpart_bytes(a) + (size_t)pto::QPROJ_KSPLIT_HOST * a->t * a->n_heads * pto::MLAP_QHEAD * sizeof(int32_t);
}

}  // namespace

extern "C" {

const char *pto_last_error(void) { return g_err; }

const char *pto_version(void) { return "0.8.3"; }

int pto_abi_revision(void) { return PTO_ABI_REVISION; }

int pto_sfa_quant_workspace_bytes(const PtoSfaQuantArgs *a, size_t *bytes)
{
    if (!bytes) return fail(PTO_E_INVALID_ARG, "sfa: bytes is NULL");
    int rc = sfa_check(a);
    if (rc != PTO_OK) return rc;
    const SfaPlan pl = sfa_plan(a);
    *bytes = sfa_ws_bytes(pl);
    return PTO_OK;
}

int pto_sfa_quant_plan(const PtoSfaQuantArgs *a, PtoSfaPlan *plan)
{
    if (!plan) return fail(PTO_E_INVALID_ARG, "sfa: plan is NULL");
    int rc = sfa_check(a);
    if (rc != PTO_OK) return rc;
    const SfaPlan pl = sfa_plan(a);
    plan->heads_per_workgroup = 32 * pl.head_groups;
    plan->key_splits = pl.nsplit;
    plan->whole_rows = pl.nsplit > 1 ? 8 * (int64_t)pl.whole_slots : 0;
    plan->partial_element_bytes = pl.nsplit > 1 ? (pl.part_f32 ? 4 : 2) : 0;
    plan->partial_bytes = pl.part_o_bytes + pl.part_ml_bytes;
    return PTO_OK;
}

int pto_sfa_quant_launch(const PtoSfaQuantArgs *a, void *hip_stream)
{
    int rc = sfa_check(a);
    if (rc != PTO_OK) return rc;
    if (!a->query_nope || !a->query_rope || !a->key_nope_2d || !a->key_rope_2d || !a->k_nope_scales || !a->topk_indices ||
        !a->block_table || !a->kv_act_seqs || !a->attention_out)
        return fail(PTO_E_INVALID_ARG, "sfa: a tensor pointer is NULL");
    return sfa_enqueue(a, static_cast<const int8_t *>(a->key_nope_2d), 512, static_cast<const uint8_t *>(a->key_rope_2d), 128,
                       static_cast<const uint8_t *>(a->k_nope_scales), 16, hip_stream);
}

int pto_sfa_quant_launch_static(const PtoSfaQuantArgs *a, void *hip_stream)
{
    int rc = sfa_check(a);
    if (rc != PTO_OK) return rc;
    if (!a->query_nope || !a->query_rope || !a->key_nope_2d || !a->key_rope_2d || !a->k_nope_scales || !a->topk_indices ||
        !a->block_table || !a->kv_act_seqs || !a->attention_out)
        return fail(PTO_E_INVALID_ARG, "sfa: a tensor pointer is NULL");
    const SfaPlan pl = sfa_plan(a, SFA_STATIC_SCRATCH_BYTES);
    const size_t need = sfa_ws_bytes(pl);
    if (need > SFA_STATIC_SCRATCH_BYTES)
        return fail(PTO_E_WORKSPACE,
                    "sfa: the key splits of this shape need %zu bytes of scratch, the built-in array holds %zu; use "
                    "pto_sfa_quant_launch with a workspace, or fewer splits",
                    need, SFA_STATIC_SCRATCH_BYTES);
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return fail(PTO_E_NO_DEVICE, "sfa: no current device: %s", hipGetErrorString(e));
    void *ptr = scratch_of(dev, &e);
    if (!ptr) return fail(PTO_E_NO_DEVICE, "sfa: the scratch array has no address on device %d: %s", dev, hipGetErrorString(e));
    PtoSfaQuantArgs q = *a;
    q.workspace = ptr;
    q.workspace_bytes = SFA_STATIC_SCRATCH_BYTES;
    return sfa_enqueue(&q, static_cast<const int8_t *>(a->key_nope_2d), 512, static_cast<const uint8_t *>(a->key_rope_2d), 128,
                       static_cast<const uint8_t *>(a->k_nope_scales), 16, hip_stream, false, SFA_STATIC_SCRATCH_BYTES);
}

int pto_sfa_bf16kv_launch(const PtoSfaQuantArgs *a, void *hip_stream)
{
    int rc = sfa_check(a);
    if (rc != PTO_OK) return rc;
    if (!a->query_nope || !a->query_rope || !a->key_nope_2d || !a->key_rope_2d || !a->topk_indices || !a->block_table ||
        !a->kv_act_seqs || !a->attention_out)
        return fail(PTO_E_INVALID_ARG, "sfa: a tensor pointer is NULL");
    return sfa_enqueue(a, static_cast<const int8_t *>(a->key_nope_2d), 1024, static_cast<const uint8_t *>(a->key_rope_2d), 128,
                       static_cast<const uint8_t *>(a->key_nope_2d), 0, hip_stream, true);
}

int pto_sa_antiquant_workspace_bytes(const PtoSaAntiquantArgs *a, size_t *bytes)
{
    if (!a) return fail(PTO_E_INVALID_ARG, "sfa: args is NULL");
    const PtoSfaQuantArgs q = unpacked_view(a);
    return pto_sfa_quant_workspace_bytes(&q, bytes);
}

int pto_sa_antiquant_launch(const PtoSaAntiquantArgs *a, void *hip_stream)
{
    if (!a) return fail(PTO_E_INVALID_ARG, "sfa: args is NULL");
    const PtoSfaQuantArgs q = unpacked_view(a);
    int rc = sfa_check(&q);
    if (rc != PTO_OK) return rc;
    if (!a->query_nope || !a->query_rope || !a->nope_cache || !a->topk_indices || !a->block_table || !a->kv_act_seqs ||
        !a->attention_out)
        return fail(PTO_E_INVALID_ARG, "sfa: a tensor pointer is NULL");
    const uint8_t *base = static_cast<const uint8_t *>(a->nope_cache);
    return sfa_enqueue(&q, reinterpret_cast<const int8_t *>(base), PACKED_ROW_BYTES, base + 512, PACKED_ROW_BYTES, base + 640,
                       PACKED_ROW_BYTES, hip_stream);
}

int pto_li_decode_workspace_bytes(const PtoLiDecodeArgs *a, size_t *bytes)
{
    if (!bytes) return fail(PTO_E_INVALID_ARG, "li: bytes is NULL");
    int rc = li_check(a);
    if (rc != PTO_OK) return rc;
    *bytes = li_ws_bytes(a);
    return PTO_OK;
}

int pto_li_decode_launch(const PtoLiDecodeArgs *a, void *hip_stream)
{
    int rc = li_check(a);
    if (rc != PTO_OK) return rc;
    if (!a->idx_query || !a->idx_query_scale || !a->idx_key_cache || !a->idx_key_scale || !a->idx_weight || !a->act_seq_key ||
        !a->block_table || !a->topk_res)
        return fail(PTO_E_INVALID_ARG, "li: a tensor pointer is NULL");
    const size_t need = li_ws_bytes(a);
    if (!a->workspace || a->workspace_bytes < need)
        return fail(PTO_E_WORKSPACE, "li: workspace of %zu bytes required, %zu given", need, a->workspace ? a->workspace_bytes : (size_t)0);
    if (cu_count() <= 0) return fail(PTO_E_NO_DEVICE, "li: no usable device is current");
    {
        const void *al16[] = {a->idx_query, a->idx_key_cache, a->workspace};
        for (const void *ptr : al16)
            if (reinterpret_cast<uintptr_t>(ptr) & 15)
                return fail(PTO_E_INVALID_ARG, "li: query, key-cache and workspace pointers must be 16-byte aligned");
        const void *al4[] = {a->act_seq_key, a->block_table, a->topk_res};
        for (const void *ptr : al4)
            if (reinterpret_cast<uintptr_t>(ptr) & 3)
                return fail(PTO_E_INVALID_ARG, "li: length, block-table and result pointers must be 4-byte aligned");
        const void *sc[] = {a->idx_query_scale, a->idx_key_scale, a->idx_weight};
        const int sdt[] = {a->q_scale_dtype, a->k_scale_dtype, a->weight_dtype};
        for (int i = 0; i < 3; ++i)
            if (reinterpret_cast<uintptr_t>(sc[i]) & (sdt[i] == PTO_DT_FP32 ? 3 : 1))
                return fail(PTO_E_INVALID_ARG, "li: scale and weight pointers must be aligned to their element size");
    }

    pto::LiParams p;
    p.q = a->idx_query;
    p.q_scale = a->idx_query_scale;
    p.kcache = a->idx_key_cache;
    p.k_scale = a->idx_key_scale;
    p.weight = a->idx_weight;
    p.act = a->act_seq_key;
    p.bt = a->block_table;
    p.topk_res = a->topk_res;
    p.T = (int)a->t;
    p.B = (int)a->b;
    p.S1 = (int)(a->t / a->b);
    p.bs = (int)a->block_size;
    p.maxblk = (int)a->max_blocknum_perbatch;
    p.nblocks = (int)a->block_num;
    p.k = (int)a->selected_count;
    p.score_stride = (long long)a->max_blocknum_perbatch * a->block_size;
    p.scores = static_cast<float *>(a->workspace);
    p.sample = p.scores + (size_t)a->t * p.score_stride;
    p.q_dt = a->q_scale_dtype;
    p.k_dt = a->k_scale_dtype;
    p.w_dt = a->weight_dtype;
    p.variant = a->arith_variant;
    {   // A wave pays three dependent memory latencies before its first pair, so runs are made as long
        // as still leaves every SIMD two rounds of two waves; at most 32 pairs (2048 keys) per wave.
        // Two query tokens of a sequence share a wave's pass over a run of keys where they are an even number and the pass has
        // several rounds of work for every resident wave.  Below, and with a token left over, units of one token are the
        // faster ones: they read the same keys side by side anyway, and twice as many waves share the work more evenly (one / two
        // tokens to a unit: 20 x 2 tokens of 5 to 60 K keys 36.0 / 40.0 us, 40 x 4 of 2 to 16 K 39.0 / 39.3, 18 x 2 of 20 to 130 K
        // 65.5 / 65.0, 64 x 2 of 4 to 32 K 52.5 / 50.2, 18 x 4 of 20 to 130 K 104 / 99.6, but 18 x 3 84.0 / 100).
        int nt = 1;
        if (p.S1 % 2 == 0 && p.variant == 0) {
            const long long pairs2 = (long long)p.B * (p.S1 / 2) * ((p.score_stride + 63) / 64);
            if (pairs2 >= (long long)pto::LI_PAIR_MIN * cu_count() * pto::LI_SCORE_WAVES) nt = 2;
        }
        p.nt = nt;
        const long long units = (long long)p.B * (p.S1 / nt);    // token groups that share a key pass
        const long long pairs = units * ((p.score_stride + 63) / 64);
        long long ppw = pairs / ((long long)cu_count() * 4 * 4);
        p.ppw = (int)(ppw < 1 ? 1 : (ppw > pto::LI_MAX_PAIRS_PER_WAVE ? pto::LI_MAX_PAIRS_PER_WAVE : ppw));
        // With few units the kernel balances the runs itself from the actual lengths: one round of resident waves (a workgroup
        // per CU), more where the longest possible input would need them.  The kernel sizes the runs for as few whole rounds as
        // the actual lengths need (spread over all the launch's waves they left a few workgroups for a second round: 20 sequences
        // of 20 to 120 K keys, four tokens, 118 us, now 94).
        p.balanced = p.B <= pto::LI_MAX_BALANCED_SEQS && units <= pto::LI_MAX_BALANCED_UNITS;
        p.round_waves = cu_count() * pto::LI_SCORE_WAVES;
        const long long need = (pairs + pto::LI_MAX_PAIRS_PER_WAVE - 1) / pto::LI_MAX_PAIRS_PER_WAVE + 2 * units;
        const long long rounds = (need + p.round_waves - 1) / p.round_waves;
        const long long runs = (p.score_stride + p.ppw * 64 - 1) / (p.ppw * 64);
        p.seq_waves = (int)(p.S1 / nt * runs);
        p.score_wgs = (int)(p.balanced ? rounds * cu_count() : (p.B * (long long)p.seq_waves + pto::LI_SCORE_WAVES - 1) / pto::LI_SCORE_WAVES);
    }
    hipError_t e = pto::li_launch(p, static_cast<hipStream_t>(hip_stream));
    if (e != hipSuccess) return fail(PTO_E_LAUNCH, "li: launch failed: %s", hipGetErrorString(e));
    return PTO_OK;
}

int pto_li_prolog_quant_workspace_bytes(const PtoLiPrologQuantArgs *a, size_t *bytes)
{
    if (!bytes) return fail(PTO_E_INVALID_ARG, "li_prolog: bytes is NULL");
    int rc = lip_check(a);
    if (rc != PTO_OK) return rc;
    *bytes = lip_ws_bytes(a);
    return PTO_OK;
}

// checked arguments -> kernel parameters
static int lip_params(const PtoLiPrologQuantArgs *a, pto::LipParams &p)
{
    if (a && (a->sum_mode < 0 || a->sum_mode > 2)) return fail(PTO_E_INVALID_ARG, "li_prolog: sum_mode must be 0, 1 or 2");
    int rc = lip_check(a);
    if (rc != PTO_OK) return rc;
    if (!a->x || !a->q_norm || !a->q_norm_scale || !a->w_qb || !a->w_qb_scale || !a->wk || !a->w_proj || !a->ln_gamma_k ||
        !a->ln_beta_k || !a->cos_idx_rope || !a->sin_idx_rope || !a->hadamard_q || !a->hadamard_k || !a->k_cache ||
        !a->k_cache_scale || !a->k_cache_index || !a->q_int8 || !a->q_scale || !a->weights)
        return fail(PTO_E_INVALID_ARG, "li_prolog: a tensor pointer is NULL");
    const size_t need = lip_ws_bytes(a);
    if (!a->workspace || a->workspace_bytes < need)
        return fail(PTO_E_WORKSPACE, "li_prolog: workspace of %zu bytes required, %zu given", need,
                    a->workspace ? a->workspace_bytes : (size_t)0);
    const void *aligned[] = {a->x, a->q_norm, a->q_norm_scale, a->w_qb, a->w_qb_scale, a->wk, a->w_proj, a->ln_gamma_k, a->ln_beta_k,
                             a->cos_idx_rope, a->sin_idx_rope, a->hadamard_q, a->hadamard_k, a->k_cache, a->q_int8, a->workspace};
    for (const void *ptr : aligned)
        if (reinterpret_cast<uintptr_t>(ptr) & 15)
            return fail(PTO_E_INVALID_ARG, "li_prolog: tensor and workspace pointers must be 16-byte aligned");

    p.x = static_cast<const uint16_t *>(a->x);
    p.q_norm = a->q_norm;
    p.q_norm_scale = a->q_norm_scale;
    p.w_qb = a->w_qb;
    p.w_qb_scale = a->w_qb_scale;
    p.wk = static_cast<const uint16_t *>(a->wk);
    p.w_proj = static_cast<const uint16_t *>(a->w_proj);
    p.gamma = static_cast<const uint16_t *>(a->ln_gamma_k);
    p.beta = static_cast<const uint16_t *>(a->ln_beta_k);
    p.cos = static_cast<const uint16_t *>(a->cos_idx_rope);
    p.sin = static_cast<const uint16_t *>(a->sin_idx_rope);
    p.hq = static_cast<const uint16_t *>(a->hadamard_q);
    p.hk = static_cast<const uint16_t *>(a->hadamard_k);
    p.k_cache = a->k_cache;
    p.k_cache_scale = static_cast<uint16_t *>(a->k_cache_scale);
    p.k_cache_index = reinterpret_cast<const long long *>(a->k_cache_index);
    p.q_int8 = a->q_int8;
    p.q_scale = static_cast<uint16_t *>(a->q_scale);
    p.weights = static_cast<uint16_t *>(a->weights);
    p.qpart = static_cast<int32_t *>(a->workspace);
    p.xpart = reinterpret_cast<float *>(static_cast<char *>(a->workspace) + lip_qpart_bytes(a));
    p.cache_rows = a->cache_rows;
    p.T = (int)a->t;
    p.h = (int)a->h;
    p.q_lora = (int)a->q_lora_rank;
    p.n_heads = (int)a->n_heads;
    p.eps = a->eps;
    p.sum_mode = a->sum_mode;
    p.x_in_groups = 0;
    p.w_mul0 = (float)std::pow((double)a->n_heads, -0.5);
    p.w_mul1 = (float)std::pow((double)pto::LIP_DIM, -0.5);
    return PTO_OK;
}

int pto_li_prolog_quant_launch(const PtoLiPrologQuantArgs *a, void *hip_stream)
{
    pto::LipParams p;
    int rc = lip_params(a, p);
    if (rc != PTO_OK) return rc;
    hipError_t e = pto::lip_launch(p, static_cast<hipStream_t>(hip_stream));
    if (e != hipSuccess) return fail(PTO_E_LAUNCH, "li_prolog: launch failed: %s", hipGetErrorString(e));
    return PTO_OK;
}

int pto_mla_prolog_quant_workspace_bytes(const PtoMlaPrologQuantArgs *a, size_t *bytes)
{
    if (!bytes) return fail(PTO_E_INVALID_ARG, "mla_prolog: bytes is NULL");
    int rc = mlap_check(a);
    if (rc != PTO_OK) return rc;
    *bytes = mlap_ws_bytes(a);
    return PTO_OK;
}

// checked arguments -> kernel parameters
static int mlap_params(const PtoMlaPrologQuantArgs *a, pto::MlapParams &p)
{
    int rc = mlap_check(a);
    if (rc != PTO_OK) return rc;
    const void *ptrs[] = {a->token_x, a->w_dq, a->w_uq_qr, a->dequant_scale, a->w_uk, a->w_dkv_kr, a->gamma_cq, a->gamma_ckv,
                          a->cos, a->sin, a->cache_index, a->kv_cache, a->kr_cache, a->k_scale_cache, a->q_norm_out,
                          a->q_norm_scale_out, a->query_nope_out, a->query_rope_out};
    for (const void *ptr : ptrs)
        if (!ptr) return fail(PTO_E_INVALID_ARG, "mla_prolog: a tensor pointer is NULL");
    const size_t need = mlap_ws_bytes(a);
    if (!a->workspace || a->workspace_bytes < need)
        return fail(PTO_E_WORKSPACE, "mla_prolog: workspace of %zu bytes required, %zu given", need,
                    a->workspace ? a->workspace_bytes : (size_t)0);
    const void *aligned[] = {a->token_x, a->w_dq, a->w_uq_qr, a->dequant_scale, a->w_uk, a->w_dkv_kr, a->gamma_cq, a->gamma_ckv,
                             a->kv_cache, a->k_scale_cache, a->q_norm_out, a->workspace};
    for (const void *ptr : aligned)
        if (reinterpret_cast<uintptr_t>(ptr) & 15)
            return fail(PTO_E_INVALID_ARG, "mla_prolog: tensor and workspace pointers must be 16-byte aligned");

    p.x = static_cast<const uint16_t *>(a->token_x);
    p.w_dq = static_cast<const uint16_t *>(a->w_dq);
    p.w_uqqr = a->w_uq_qr;
    p.w_qb_scale = a->dequant_scale;
    p.w_uk = static_cast<const uint16_t *>(a->w_uk);
    p.w_dkvkr = static_cast<const uint16_t *>(a->w_dkv_kr);
    p.gamma_cq = static_cast<const uint16_t *>(a->gamma_cq);
    p.gamma_ckv = static_cast<const uint16_t *>(a->gamma_ckv);
    p.cos = static_cast<const uint16_t *>(a->cos);
    p.sin = static_cast<const uint16_t *>(a->sin);
    p.cache_index = reinterpret_cast<const long long *>(a->cache_index);
    p.kv_cache = a->kv_cache;
    p.kr_cache = static_cast<uint16_t *>(a->kr_cache);
    p.k_scale_cache = a->k_scale_cache;
    p.q_norm = a->q_norm_out;
    p.q_norm_scale = a->q_norm_scale_out;
    p.q_nope = static_cast<uint16_t *>(a->query_nope_out);
    p.q_rope = static_cast<uint16_t *>(a->query_rope_out);
    p.xpart = static_cast<float *>(a->workspace);
    p.qpart = reinterpret_cast<int32_t *>(static_cast<char *>(a->workspace) + mlap_xpart_bytes(a));
    p.cache_rows = a->cache_rows;
    p.T = (int)a->t;
    p.h = (int)a->h;
    p.q_lora = (int)a->q_lora_rank;
    p.n_heads = (int)a->n_heads;
    p.eps_cq = a->epsilon_cq;
    p.eps_ckv = a->epsilon_ckv;
    p.absorb_exact = a->absorb_exact ? 1 : 0;
    return PTO_OK;
}

int pto_mla_prolog_quant_launch(const PtoMlaPrologQuantArgs *a, void *hip_stream)
{
    pto::MlapParams p;
    int rc = mlap_params(a, p);
    if (rc != PTO_OK) return rc;
    hipError_t e = pto::mlap_launch(p, static_cast<hipStream_t>(hip_stream));
    if (e != hipSuccess) return fail(PTO_E_LAUNCH, "mla_prolog: launch failed: %s", hipGetErrorString(e));
    return PTO_OK;
}

// ---- both prologs as one operator: the query latent and its scale live in the common workspace

namespace {

struct FusedPlan {
    size_t q_norm_off, q_norm_scale_off, rest_off, total;
    PtoMlaPrologQuantArgs mla;
    PtoLiPrologQuantArgs idx;
};

// fills in what the two halves share and where the intermediates go (workspace base may be null: sizes only)
int fused_plan(const PtoMlaIndexerPrologQuantArgs *a, FusedPlan *pl)
{
    if (!a) return fail(PTO_E_INVALID_ARG, "mla_indexer_prolog: args is NULL");
    pl->mla = a->mla;
    pl->idx = a->indexer;
    pl->idx.x = a->mla.token_x;
    pl->idx.cos_idx_rope = a->mla.cos;
    pl->idx.sin_idx_rope = a->mla.sin;
    pl->idx.k_cache_index = a->mla.cache_index;
    pl->idx.t = a->mla.t;
    pl->idx.h = a->mla.h;
    pl->idx.q_lora_rank = a->mla.q_lora_rank;
    int rc = mlap_check(&pl->mla);
    if (rc != PTO_OK) return rc;
    rc = lip_check(&pl->idx);
    if (rc != PTO_OK) return rc;
    const size_t qn = ((size_t)a->mla.t * a->mla.q_lora_rank + 255) & ~(size_t)255;
    const size_t qs = ((size_t)a->mla.t * sizeof(float) + 255) & ~(size_t)255;
    const size_t w_mla = mlap_ws_bytes(&pl->mla), w_idx = lip_ws_bytes(&pl->idx);
    pl->q_norm_off = 0;
    pl->q_norm_scale_off = qn;
    pl->rest_off = qn + qs;
    // the partial sums of both halves are alive at once (the last launch finishes both), so each has its own area
    const size_t w_mla_pad = (w_mla + 255) & ~(size_t)255;
    pl->total = qn + qs + w_mla_pad + w_idx;
    char *base = static_cast<char *>(a->workspace);
    if (base) {
        int8_t *q_norm = a->mla.q_norm_out ? a->mla.q_norm_out : reinterpret_cast<int8_t *>(base + pl->q_norm_off);
        float *q_norm_scale = a->mla.q_norm_scale_out ? a->mla.q_norm_scale_out : reinterpret_cast<float *>(base + pl->q_norm_scale_off);
        pl->mla.q_norm_out = q_norm;
        pl->mla.q_norm_scale_out = q_norm_scale;
        pl->idx.q_norm = q_norm;
        pl->idx.q_norm_scale = q_norm_scale;
        pl->mla.workspace = base + pl->rest_off;
        pl->mla.workspace_bytes = w_mla;
        pl->idx.workspace = base + pl->rest_off + w_mla_pad;
        pl->idx.workspace_bytes = w_idx;
    }
    return PTO_OK;
}

}  // namespace

int pto_mla_indexer_prolog_quant_workspace_bytes(const PtoMlaIndexerPrologQuantArgs *a, size_t *bytes)
{
    if (!bytes) return fail(PTO_E_INVALID_ARG, "mla_indexer_prolog: bytes is NULL");
    FusedPlan pl;
    int rc = fused_plan(a, &pl);
    if (rc != PTO_OK) return rc;
    *bytes = pl.total;
    return PTO_OK;
}

int pto_mla_indexer_prolog_quant_launch(const PtoMlaIndexerPrologQuantArgs *a, void *hip_stream)
{
    FusedPlan pl;
    int rc = fused_plan(a, &pl);
    if (rc != PTO_OK) return rc;
    if (!a->workspace || a->workspace_bytes < pl.total)
        return fail(PTO_E_WORKSPACE, "mla_indexer_prolog: workspace of %zu bytes required, %zu given", pl.total,
                    a->workspace ? a->workspace_bytes : (size_t)0);
    if (reinterpret_cast<uintptr_t>(a->workspace) & 255)
        return fail(PTO_E_INVALID_ARG, "mla_indexer_prolog: the workspace must be 256-byte aligned");
    pto::MlapParams pm;
    pto::LipParams pi;
    rc = mlap_params(&pl.mla, pm);
    if (rc != PTO_OK) return rc;
    rc = lip_params(&pl.idx, pi);
    if (rc != PTO_OK) return rc;
    hipError_t e = pto::prolog_fused_launch(pm, pi, static_cast<hipStream_t>(hip_stream));
    if (e != hipSuccess) return fail(PTO_E_LAUNCH, "mla_indexer_prolog: launch failed: %s", hipGetErrorString(e));
    return PTO_OK;
}

}  // extern "C"
