// Launch parameters of the sparse-flash-attention kernels (internal to the library).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace pto {

constexpr int SFA_MAX_CHUNK = 2048;   // most keys one workgroup handles (row-translation table in LDS)
constexpr int SFA_KEY_TILE = 32;

struct SfaParams {
    const uint16_t *q_nope;   // [T*NQ, 512] bf16
    const uint16_t *q_rope;   // [T*NQ, 64]  bf16
    // The three parts of a cache row, each with its own base and row pitch in bytes: separate arrays
    // (pitches 512 / 128 / 16) or one packed array of 656-byte rows (512 int8 | 64 bf16 | 4 fp32).
    const int8_t *kn;         // 512 int8 latent values
    const uint8_t *kr;        // 64 bf16 rope values
    const uint8_t *ksc;       // 4 fp32 scales, one per 128 latent channels
    int kn_pitch, kr_pitch, ksc_pitch;
    int kn_bf16;              // the latent part is bf16 (1024 bytes, no scales) instead of int8
    const int32_t *topk_idx;  // [T, topk]
    const int32_t *bt;        // [B, maxblk]
    const int32_t *act;       // [B]
    uint16_t *out;            // [T*NQ, 512] bf16
    void *part_o;             // [split rows, nsplit, NQ, 512] fp16, or fp32 (part_f32): O / l of each key split (nsplit > 1)
    float *part_ml;           // [split rows, nsplit, NQ, 2]   reference max (log2 domain) and row sum of the split
    long long kv_rows;
    int T, S1, NQ, topk, bs, maxblk;
    int nsplit;               // key splits per query row, of the rows that are split
    int part_f32;             // (with one head group per workgroup and at most eight splits)
    int whole_slots;          // rows 0 .. 8 * whole_slots - 1 are not split (one workgroup per row and head group): the
                              // full rounds of a launch of more rows than compute units; 0 = every row is split alike
    int hgroups;              // workgroups' shares of the heads per query row (32 * head_groups heads each)
    int last_first;           // T - 1 where the rows of a launch of whole rows start with the last one, else 0 (sfa_last_first)
    int head_groups;          // groups of 32 heads per workgroup: 1, 4, or 2 (sfa_slice_kernel)
    int xcd_pieces;           // workgroups of split rows per XCD (set by sfa_launch)
    float scale_log2;         // softmax_scale * log2(e)
};

// Of s1 rows of a sequence, up to row_keys keys long, those that see topk keys: the others, before them, see one more each.
inline long long sfa_full_rows(const long long s1, const long long topk, const long long row_keys)
{
    const long long before = row_keys > s1 ? row_keys - s1 : 0, growing = (topk < row_keys ? topk : row_keys) - before;
    return growing < 0 ? s1 : (growing < s1 ? s1 - growing : 0);
}

// Whether a launch of whole rows starts with the last one.  Rows of a prefill chunk see the more keys the later they are: the longest
// first, it ends with short ones (one sequence, 128 heads, top-k 2048: 4096 rows over 4096 keys 1527 us, now 1496, 1000 over 1000 162.7
// and 158.7, 655 over 655 94.8 and 88.3).  But rows of full length that start together want the same things at the same time, and
// behind short ones of all lengths they do not.  With more than 32 heads the short rows stay in front (first to last / last to first)
// - where 45 % of the rows have full length and that is less than 2048 keys (128 heads: 2000 over 2000, top-k 512 266 / 300 us, 2500
//   over 2500, 1024 540 / 552; 64 heads: 1219 over 1219, 256 68 / 79, 512 94 / 104, 1024, 1219 over 1619 168 / 170.  Fewer of them: 1000
//   over 1000, 1024 160 / 156, 1500 over 2012, 1536 461 / 445; top-k 2048: 4096 over 5120 1876 / 1834);
// - where several sequences have a few hundred rows each and the launch ends with those of one (64 heads, top-k 2048: 8 x 128 rows
//   45.2 / 46.6, 4 x 1000 378 / 389; 128 heads: 64 x 16 that begin 300 keys into theirs 141.8 / 145.6; 2 x 300 56.9 / 54.7, 5 x 2000
//   2604 / 2540).
inline bool sfa_last_first(const long long b, const long long s1, const long long nq, const long long topk, const long long row_keys,
                           const int cus)
{
    if (s1 <= 8) return false;
    if (nq <= 32) return true;
    return (b <= 2 || s1 >= 4ll * cus) && (topk >= SFA_MAX_CHUNK || 20 * sfa_full_rows(s1, topk, row_keys) <= 9 * s1);
}

hipError_t sfa_launch(const SfaParams &p, hipStream_t stream);
// the int8 latent part of `rows` cache rows as bf16 [rows, 512] (what the attention kernel de-quantises them to)
hipError_t sfa_dequant_cache(const int8_t *kn, int kn_pitch, const uint8_t *ksc, int ksc_pitch, uint16_t *out, long long rows,
                             hipStream_t stream);

}  // namespace pto
