// Attention of 64 heads per workgroup of eight waves (included by sfa_kernels.hip).
//
// For launches of few rows: with 128 heads per workgroup only key splits fill the chip, and their partial results -- 33 MB
// written and read back at 32 rows -- cost as much as the key loop.  64 heads per workgroup halve them.  They also leave room for
// two waves per SIMD (242 registers), where one's vector work and LDS latency stand beside the other's products; four waves
// with one instruction stream per SIMD took 1.58 us per tile of 32 keys over 64 heads, these take 1.1 to 1.2.
//   scores: wave (kh, hq) multiplies the 16 keys of half kh with heads 16*hq .. +15 over all 576 channels
//           (v_mfma_f32_16x16x32_bf16: the accumulator's lane (head, quarter) holds four keys of one head), nothing to add up;
//   softmax: of those four scores, in place; the probabilities go round through LDS as the B operand of the second product;
//   values: wave w owns 64 value channels of all 64 heads; each transposed V operand serves two products.
// The products against V of tile n - 1 run beside the scores and the softmax of tile n: one barrier per tile, three tile buffers.
// Cache rows travel to registers two tiles ahead of their use, whole rows at a time, and are de-quantised on the way into LDS.
// Measured, steps with the merge launch: 32 rows of 128 heads over 2048 keys 34.8 -> 32.1 us, 40 rows of 64 heads over a bf16
// cache 34.8 -> 29.1, 128 rows of 64 heads 72 -> 62.  Bound by the vector units and by what a wave waits for: of 2580 clocks per
// tile the vector instructions take 1330 (de-quantisation 600), the products 1090, the LDS 1350; without the de-quantisation
// 2170, without either product 2490 to 2540.

constexpr int SL_PITCH = PITCH * 2;                       // bytes of a tile row: 512 latent and 64 rope channels as bf16, 16 spare
constexpr int SL_TILE = KT * SL_PITCH;
constexpr int SL_P = 3 * SL_TILE;                         // two buffers of P^T: [head half][k-step][lane] 16 bytes
constexpr int SL_P_BYTES = 4096;
constexpr int SL_MAX = SL_P + 2 * SL_P_BYTES;             // [key half][64 heads] fp32: maxima (and at the end the sums)
constexpr int SL_ALPHA = SL_MAX + 2 * 64 * 4;             // [64 heads] fp32: rescale factors (at the end 1 / sum)
constexpr int SL_FLAG = SL_ALPHA + 64 * 4;                // two words: the last tile whose maxima moved, by parity of the tile
constexpr int SL_PAGES = SL_FLAG + 16;                    // pages of the selected positions
constexpr int SL_POOL = SL_PAGES + SFA_MAX_CHUNK * 4;
constexpr int SL_QROPE = 64 * DN * 2;                     // query staging: 64 heads x 1024 bytes, then 64 x 128

// max and sum over the four lanes l, l ^ 16, l ^ 32, l ^ 48, in every one of them
__device__ __forceinline__ float across_quarters_max(const float x)
{
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    float lo, hi;
    both_halves(fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])), lo, hi);
    return fmaxf(lo, hi);
}
__device__ __forceinline__ float across_quarters_sum(const float x)
{
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    float lo, hi;
    both_halves(__uint_as_float(r[0]) + __uint_as_float(r[1]), lo, hi);
    return lo + hi;
}

// one dword of int8 times the scale: two dwords of bf16, each product rounded to fp32 and then to bf16
__device__ __forceinline__ u32x2 dequant_dword(const uint32_t r, const float sc)
{
    float f0, f1, f2, f3;
    asm("v_cvt_f32_i32_sdwa %0, sext(%1) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_0" : "=v"(f0) : "v"(r));
    asm("v_cvt_f32_i32_sdwa %0, sext(%1) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_1" : "=v"(f1) : "v"(r));
    asm("v_cvt_f32_i32_sdwa %0, sext(%1) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_2" : "=v"(f2) : "v"(r));
    asm("v_cvt_f32_i32_sdwa %0, sext(%1) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_3" : "=v"(f3) : "v"(r));
    return u32x2{pack_bf16x2(f0 * sc, f1 * sc), pack_bf16x2(f2 * sc, f3 * sc)};
}

template <bool QUANT>
__global__ __launch_bounds__(512) void sfa_slice_kernel(const SfaParams p)
{
    constexpr int NT = 512;
    __shared__ __attribute__((aligned(16))) uint8_t pool[SL_POOL];
    __shared__ int rows_lds[SFA_MAX_CHUNK];

    const int tid = threadIdx.x;
    const int l = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int half = l >> 5;
    const int col = l & 31;
    const int l16 = l & 15;
    const int quarter = l >> 4;
    const int hq = w & 3;                                  // scores: heads 16*hq .. +15 of the workgroup's 64,
    const int kh = w >> 2;                                 // the half kh of the tile's keys

    // workgroup -> (row, head share, key split): see sfa_decode_kernel
    const int xcd = blockIdx.x & 7;
    const int slot = blockIdx.x >> 3;
    const int wslots = p.whole_slots * p.hgroups;
    int t, within, nsplit;
    if (slot < wslots) {
        t = (slot / p.hgroups) * 8 + xcd;
        if (p.last_first != 0) t = t < p.T ? p.last_first - t : p.T;
        within = slot % p.hgroups;
        nsplit = 1;
    } else {
        const int per_row = p.hgroups * p.nsplit;
        const int piece = xcd * p.xcd_pieces + (slot - wslots);
        t = 8 * p.whole_slots + piece / per_row;
        within = piece % per_row;
        nsplit = p.nsplit;
    }
    if (t >= p.T) return;
    const int sp = within / p.hgroups;                     // the head shares of a split are neighbours: they gather the same rows
    const int hg = within - sp * p.hgroups;
    const int b = t / p.S1;
    const int s1i = t - b * p.S1;
    const int act_b = p.act[b];                            // asked for here, looked at behind the first requests
    auto split_keys = [&](const int n, int &kb, int &ke) {
        const int ntile = (n + KT - 1) / KT;
        const int tiles_per_split = (ntile + nsplit - 1) / nsplit;
        kb = sp * tiles_per_split * KT;
        ke = kb + tiles_per_split * KT;
        ke = ke > n ? n : ke;
    };

    const uint32_t pool_lds = (uint32_t)(uintptr_t)(lds_byte_t *)pool;

    // Positions of this split, then their pages, by LDS-DMA: a lane handles the entries it requested itself.  They are asked
    // for on the assumption that the row sees all topk keys, before the sequence's length has arrived, and again if it does
    // not (requests complete in order).  Keys past the last one stand in with the split's first.
    auto request_positions = [&](const int kb, const int nv) {
        for (int i0 = 0; i0 < nv; i0 += NT) {
            const int i = i0 + tid;
            dma4(p.topk_idx + (size_t)t * p.topk + kb + (i < nv ? i : 0), (uint32_t)(uintptr_t)(lds_byte_t *)(rows_lds + i0 + 64 * w));
        }
    };
    int kb_s, ke_s;
    split_keys(p.topk, kb_s, ke_s);
    if (ke_s > kb_s) request_positions(kb_s, ke_s - kb_s);
    // The workgroup's queries, staged through LDS in the tile buffers 0 and 1: wave w asks for heads 8w .. 8w+7, a head's
    // latent part per request, 16-byte chunk i of head j at i ^ (j & 15) so that the fragment reads touch every bank once.
    // Heads past the last one read it and are never stored.
    static_assert(SL_QROPE + 64 * DR * 2 <= 2 * SL_TILE, "the first tile goes to buffer 2");
    auto head_row = [&](const int j) {
        const int hd = hg * 64 + j;
        return (size_t)t * p.NQ + (hd < p.NQ ? hd : p.NQ - 1);
    };
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int j = 8 * w + i;
        dma16_base(p.q_nope + head_row(j) * DN, (uint32_t)(16 * (l ^ (j & 15))), pool_lds + j * (DN * 2));
    }
    dma16(p.q_rope + head_row(8 * w + (l >> 3)) * DR + 8 * ((l & 7) ^ (l >> 3)), pool_lds + SL_QROPE + w * 1024);

    int cur_seq = act_b - p.S1 + 1 + s1i;
    cur_seq = cur_seq < 0 ? 0 : (cur_seq > p.topk ? p.topk : cur_seq);
    int k_begin, k_end;
    split_keys(cur_seq, k_begin, k_end);
    const int n_valid = k_end > k_begin ? k_end - k_begin : 0;
    const int ntiles = (n_valid + KT - 1) / KT;
    if (k_begin != kb_s || n_valid != ke_s - kb_s) {       // uniform
        if (n_valid > 0) request_positions(k_begin, n_valid);
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
    } else {
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(9));          // the positions have landed, the queries may be on their way
    }
    asm volatile("" ::: "memory");
    // (rows beyond the requested ones, up to the end of the last tile, exist: requests come in whole waves, SFA_MAX_CHUNK a
    // multiple of the workgroup)
    {
        const int *pages = reinterpret_cast<const int *>(pool + SL_PAGES);
        static_assert(SFA_MAX_CHUNK % NT == 0, "whole requests");
        for (int i0 = 0; i0 < n_valid; i0 += NT) {
            const int blk0 = rows_lds[i0 + tid] / p.bs;
            const int blk = blk0 < 0 ? 0 : (blk0 >= p.maxblk ? p.maxblk - 1 : blk0);
            dma4(p.bt + (size_t)b * p.maxblk + blk, pool_lds + SL_PAGES + 4 * (i0 + 64 * w));
        }
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));          // (the queries too)
        asm volatile("" ::: "memory");
        for (int i0 = 0; i0 < n_valid; i0 += NT) {
            const int idx = rows_lds[i0 + tid];
            long long row = (long long)pages[i0 + tid] * p.bs + (idx - (idx / p.bs) * p.bs);
            row = row < 0 ? 0 : (row >= p.kv_rows ? p.kv_rows - 1 : row);
            rows_lds[i0 + tid] = (int)row;
        }
    }
    __syncthreads();

    // Gather: wave w takes keys 4w .. 4w+3 of every tile.  int8: two rows per load, a lane 16 channels; bf16: a row per load,
    // a lane 8 channels; the rope part of the four rows 8 bytes per lane.
    constexpr int NV = QUANT ? 2 : 4;
    struct Raw {
        u32x4 v[NV];
        float sc[QUANT ? 2 : 1];
        u32x2 rope;
    };
    Raw raw[2];                                            // tile n in raw[n & 1]
    const uint8_t *const kn_lane = reinterpret_cast<const uint8_t *>(p.kn) + (QUANT ? 16 * col : 16 * (2 * col + half));
    const uint8_t *const kr_lane = p.kr + 8 * (l & 15);
    const uint8_t *const ks_lane = QUANT ? p.ksc + 4 * (col >> 3) : nullptr;
    const int last_tile = ntiles - 1;
    auto gather_rows = [&](const int n, int (&row)[NV + 1]) __attribute__((always_inline)) {
        const int *rt = rows_lds + KT * (n < last_tile ? n : last_tile) + 4 * w;
#pragma unroll
        for (int i = 0; i < NV; ++i) row[i] = rt[QUANT ? 2 * i + half : i];
        row[NV] = rt[l >> 4];
    };
    auto gather = [&](Raw &r, const int (&row)[NV + 1]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            r.v[i] = *reinterpret_cast<const u32x4 *>(kn_lane + (uint64_t)(uint32_t)row[i] * (uint32_t)p.kn_pitch);
            if (QUANT) r.sc[i] = *reinterpret_cast<const float *>(ks_lane + (uint64_t)(uint32_t)row[i] * (uint32_t)p.ksc_pitch);
        }
        r.rope = *reinterpret_cast<const u32x2 *>(kr_lane + (uint64_t)(uint32_t)row[NV] * (uint32_t)p.kr_pitch);
    };
    // The tile's rows into LDS, in eight pieces of a dword per lane (int8) and one of the rope channels.  Of a row's 64 latent
    // pieces of eight channels the even ones come first, then the odd ones: a lane's sixteen channels are a piece of either
    // half, and lanes next to each other write next to each other.
    const uint32_t emit_off = QUANT ? (uint32_t)((4 * w + half) * SL_PITCH + 16 * col) : (uint32_t)(4 * w * SL_PITCH + 16 * l);
    const uint32_t emit_rope_off = (uint32_t)((4 * w + (l >> 4)) * SL_PITCH + DN * 2 + 8 * (l & 15));
    u32x4 dq;
    auto emit = [&](const Raw &r, const uint32_t tile, const int d) __attribute__((always_inline)) {
        if (d == 8) {
            *reinterpret_cast<u32x2 *>(pool + tile + emit_rope_off) = r.rope;
        } else if (QUANT) {
            const u32x2 x = dequant_dword(r.v[d >> 2][d & 3], r.sc[d >> 2]);
            if (d & 1) {
                dq[2] = x[0], dq[3] = x[1];
                *reinterpret_cast<u32x4 *>(pool + tile + emit_off + (2 * (d >> 2)) * SL_PITCH + 512 * ((d & 3) >> 1)) = dq;
            } else {
                dq[0] = x[0], dq[1] = x[1];
            }
        } else if (d & 1) {
            *reinterpret_cast<u32x4 *>(pool + tile + emit_off + (d >> 1) * SL_PITCH) = r.v[(d >> 1) % NV];
        }
    };

    f32x16 o[4];                                           // block 2*hb + d: heads 32*hb .., value channels 64w + 32d ..
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[i][r] = 0.f;
    float m_run = -INFINITY;                               // of head 16*hq + l16: reference maximum, log2 domain,
    float l_run = 0.f;                                     // and this lane's share of the sum of exp2(s - m_run)

    if (ntiles > 0) {                                      // uniform
        int row[NV + 1];
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            gather_rows(n, row);
            gather(raw[n], row);
        }
        // Q^T: of the latent part lane (head, quarter) holds the channels of the tile rows' 16-byte pieces 16*quarter + ks, of
        // the rope part channels 16*quarter + 8*ks .. +7
        bf16x8 qf[18];
#pragma unroll
        for (int ks = 0; ks < 16; ++ks)
            qf[ks] = *reinterpret_cast<const bf16x8 *>(pool + (16 * hq + l16) * (DN * 2) + 16 * ((32 * (quarter & 1) + 2 * ks + (quarter >> 1)) ^ l16));
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
            qf[16 + ks] = *reinterpret_cast<const bf16x8 *>(pool + SL_QROPE + (16 * hq + l16) * (DR * 2) + 16 * ((2 * quarter + ks) ^ (l16 & 7)));
        // Scores are scaled inside the exponent (one multiply-add per key).  That wants a positive scale: the sign of a negative
        // one moves into Q^T (exact), and a zero one becomes the smallest normal number, under which every finite score still
        // scales to an exponent that rounds to the same probabilities.
        float sc_log2 = p.scale_log2;
        if (sc_log2 < 0.f) {
            sc_log2 = -sc_log2;
#pragma unroll
            for (int i = 0; i < 18; ++i) {
                u32x4 v = __builtin_bit_cast(u32x4, qf[i]);
                v ^= 0x80008000u;
                qf[i] = __builtin_bit_cast(bf16x8, v);
            }
        }
        if (sc_log2 == 0.f) sc_log2 = 1.17549435e-38f;
        if (tid < 2) reinterpret_cast<int *>(pool + SL_FLAG)[tid] = -1;
#pragma unroll
        for (int d = 0; d < 9; ++d) emit(raw[0], 2 * SL_TILE, d);
        gather_rows(2, row);
        gather(raw[0], row);
        __syncthreads();

        // Score operand: row `a` of the wave's sixteen is key tile_row_of(16*kh + a); the accumulator then holds in lane
        // (head, quarter) the rows 4*quarter + r, the k-order of the second product's B operand.
        // (quarters 256 bytes apart: whichever sixteen lanes the LDS serves together, their rows alone decide the banks; with
        // quarters 16 bytes apart two in three of these reads took twice as long)
        const uint32_t kbase = (uint32_t)(tile_row_of(16 * kh + l16) * SL_PITCH + 256 * quarter);
        const uint32_t krope = (uint32_t)(tile_row_of(16 * kh + l16) * SL_PITCH + DN * 2 + 32 * quarter);
        const uint32_t vbase = (uint32_t)((half + 4 * ((l & 15) >> 2)) * SL_PITCH + 32 * ((l >> 4) & 1) + 8 * (l & 3) + 128 * w);
        const uint32_t pwrite = (uint32_t)(SL_P + (((hq >> 1) * 2 + kh) * 64 + 32 * (quarter & 1) + 16 * (hq & 1) + l16) * 16 + 8 * (quarter >> 1));
        int key_of[4];                                     // key of this lane's scores within the tile
#pragma unroll
        for (int e = 0; e < 4; ++e) key_of[e] = tile_row_of(16 * kh + 4 * quarter + e);

        bf16x8 vf[2][2], pf[2][2];
        f32x4 s;                                           // scores of the tile being multiplied
        float sv[4], mx = 0.f;                             // of the tile before it, and their maximum over the wave's keys
        float l_add = 0.f;                                 // that tile's probabilities, not yet in l_run
        auto load_v = [&](const uint32_t tile, const int kk, const int d) __attribute__((always_inline)) {
            const uint16_t *a0 = reinterpret_cast<const uint16_t *>(pool + tile + vbase + (16 * kk) * SL_PITCH + 64 * d);
            const s16x4 lo = lds_read_tr16(a0), hi = lds_read_tr16(a0 + SL_PITCH);       // (two rows on)
            vf[kk][d] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        };
        auto load_p = [&](const int pbuf, const int kk, const int hb) __attribute__((always_inline)) {
            pf[kk][hb] = *reinterpret_cast<const bf16x8 *>(pool + SL_P + pbuf * SL_P_BYTES + ((hb * 2 + kk) * 64 + l) * 16);
        };
        auto first_vp = [&](const uint32_t tile, const int pbuf) __attribute__((always_inline)) {
            load_v(tile, 0, 0), load_v(tile, 0, 1);
            load_p(pbuf, 0, 0), load_p(pbuf, 0, 1);
        };
        // Scores of the tile in buffer `cur`, whose first AHEAD operands are in fa (or on their way).
        constexpr int AHEAD = 6;
        bf16x8 fa[18];
        auto read_k = [&](const uint32_t cur, const int m) __attribute__((always_inline)) {
            fa[m] = *reinterpret_cast<const bf16x8 *>(pool + cur + (m < 16 ? kbase + 16 * m : krope + 16 * (m - 16)));
        };
        auto first_k = [&](const uint32_t cur) __attribute__((always_inline)) {
#pragma unroll
            for (int m = 0; m < AHEAD; ++m) read_k(cur, m);
        };
        auto scores = [&](const uint32_t cur) __attribute__((always_inline)) {
            f32x4 z = {};
            s = z;
#pragma unroll
            for (int m = 0; m < 18; ++m) {
                s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[m], qf[m], s, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                if (m + AHEAD < 18) read_k(cur, m + AHEAD);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        // The softmax of tile n.  The reference maximum follows the true one lazily: probabilities may reach
        // 2^RESCALE_TAU, which fp32 sums and bf16 P hold without loss.  A wave sees half of its heads' keys only; where one of
        // its scores passes that bound it raises the flag, and all waves take the tile's probabilities again (move_maxima)
        // once the barrier has made the flag seen.
        auto probabilities = [&](const int pbuf) __attribute__((always_inline)) {
            float e[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) e[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(sv[i], sc_log2, -m_run));
            const u32x2 pk = {pack_bf16x2(e[0], e[1]), pack_bf16x2(e[2], e[3])};
            *reinterpret_cast<u32x2 *>(pool + pwrite + pbuf * SL_P_BYTES) = pk;
            l_add = (e[0] + e[1]) + (e[2] + e[3]);
        };
        auto take_scores = [&](const int n) __attribute__((always_inline)) {
#pragma unroll
            for (int e = 0; e < 4; ++e) sv[e] = s[e];
            if ((n + 1) * KT > n_valid) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n * KT + key_of[e] >= n_valid) sv[e] = -INFINITY;
            }
            mx = fmaxf(fmaxf(sv[0], sv[1]), fmaxf(sv[2], sv[3]));
        };
        auto softmax = [&](const int n, const int pbuf) __attribute__((always_inline)) {
            take_scores(n);
            probabilities(pbuf);
            if (__any(mx * sc_log2 > m_run + RESCALE_TAU)) reinterpret_cast<int *>(pool + SL_FLAG)[pbuf] = n;
        };
        // Probabilities of the tile whose scores are in sv, with the maxima moved where they passed the bound (always, on the
        // first tile): two barriers, every wave takes part.
        auto move_maxima = [&](const int pbuf, const bool first) __attribute__((always_inline)) {
            mx = across_quarters_max(mx);
            if (l < 16) reinterpret_cast<float *>(pool + SL_MAX)[64 * kh + 16 * hq + l16] = mx;
            __syncthreads();
            mx = fmaxf(mx, reinterpret_cast<const float *>(pool + SL_MAX)[64 * (kh ^ 1) + 16 * hq + l16]) * sc_log2;
            const bool upd = mx > m_run + RESCALE_TAU;
            const float m_new = upd ? mx : m_run;
            const float alpha = upd ? __builtin_amdgcn_exp2f(m_run - m_new) : 1.0f;
            m_run = m_new;
            l_run *= alpha;
            if (kh == 0 && l < 16) reinterpret_cast<float *>(pool + SL_ALPHA)[16 * hq + l16] = alpha;
            probabilities(pbuf);
            __syncthreads();
            if (!first) {
#pragma unroll
                for (int hb = 0; hb < 2; ++hb) {
                    const float a = reinterpret_cast<const float *>(pool + SL_ALPHA)[32 * hb + col];
#pragma unroll
                    for (int d = 0; d < 2; ++d)
#pragma unroll
                        for (int e = 0; e < 16; ++e) o[2 * hb + d][e] *= a;
                }
            }
        };
        // O^T += V^T . P^T of the tile in buffer `prev`, P^T in buffer pbuf, whose first operands are read; NEXT: beside them the
        // tile of r goes into buffer `next` and the rows of tile n3 are asked for
        auto values = [&](auto next_tag, const int n3, const uint32_t prev, const uint32_t next, Raw &r, const int pbuf) __attribute__((always_inline)) {
            constexpr bool NEXT = decltype(next_tag)::value;
            int row[NV + 1];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int mp = 0; mp < 8; ++mp) {
                const int kk = mp >> 2, d = (mp >> 1) & 1, hb = mp & 1;
                o[2 * hb + d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[kk][d], pf[kk][hb], o[2 * hb + d], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                if (mp == 0) load_v(prev, 1, 0), load_p(pbuf, 1, 0);
                if (mp == 1) load_v(prev, 1, 1), load_p(pbuf, 1, 1);
                if (NEXT) {
                    emit(r, next, mp);
                    if (mp == 4) gather_rows(n3, row);
                    if (mp == 7) emit(r, next, 8), gather(r, row);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        // Every wave takes part in the tile's two halves of work in one of two orders: the waves of the keys' first half take the
        // scores of tile n first and then the products against V of tile n - 1, the others (the second wave of each SIMD) the
        // products first, so that one's LDS reads and vector work stand beside the other's products.
        auto moved_word = [&](const int pbuf) { return reinterpret_cast<const int *>(pool + SL_FLAG)[pbuf]; };
        uint32_t cur = 2 * SL_TILE, next = 0, prev = SL_TILE;                       // buffers of tiles n, n + 1, n - 1
        auto turn = [&](auto parity, const int n) __attribute__((always_inline)) {
            constexpr int PAR = decltype(parity)::value;                            // n & 1
            constexpr int pbuf = PAR ^ 1;                                           // of tile n - 1
            if (kh == 0) {
                first_k(cur);
                scores(cur);
            }
            const int moved = moved_word(pbuf);
            first_vp(prev, pbuf);
            if (__builtin_expect(__builtin_amdgcn_readfirstlane(moved) == n - 1, 0)) {      // rare
                move_maxima(pbuf, false);
                first_vp(prev, pbuf);
            }
            l_run += l_add;
            if (kh == 0) softmax(n, PAR);
            values(std::true_type{}, n + 3, prev, next, raw[PAR ^ 1], pbuf);
            if (kh == 1) {
                first_k(cur);
                scores(cur);
                softmax(n, PAR);
            }
            __syncthreads();
            const uint32_t third = prev;
            prev = cur;
            cur = next;
            next = third;
        };
        // the first tile: its maxima are moved at once
        first_k(cur);
        scores(cur);
#pragma unroll
        for (int d = 0; d < 9; ++d) emit(raw[1], next, d);
        gather_rows(3, row);
        gather(raw[1], row);
        take_scores(0);
        move_maxima(0, true);
        prev = cur;
        cur = next;
        next = SL_TILE;
        int n = 1;
        for (; n + 1 < ntiles; n += 2) {                   // (two to a trip without a way out between them: exits inside make
            turn(std::integral_constant<int, 1>{}, n);     // the compiler wait for every request)
            turn(std::integral_constant<int, 0>{}, n + 1);
        }
        if (n < ntiles) turn(std::integral_constant<int, 1>{}, n);
        // the products against V of the last tile
        const int pbuf = (ntiles & 1) ^ 1;
        if (__builtin_amdgcn_readfirstlane(moved_word(pbuf)) == ntiles - 1) move_maxima(pbuf, false);
        l_run += l_add;
        first_vp(prev, pbuf);
        values(std::false_type{}, 0, prev, 0, raw[0], pbuf);
    }

    // ---- epilogue.  1/l of every head through LDS; then the results, 64 heads x 1024 bytes, through the idle tile memory: 16-byte
    // piece i of head j at i ^ (j & 31), and out a head's row per store.
    l_run = across_quarters_sum(l_run);
    float *const sums = reinterpret_cast<float *>(pool + SL_MAX), *const il = reinterpret_cast<float *>(pool + SL_ALPHA);
    if (l < 16) sums[64 * kh + 16 * hq + l16] = l_run;
    __syncthreads();
    const size_t prow_base = ((size_t)(t - 8 * p.whole_slots) * nsplit + sp) * p.NQ;       // split rows only
    if (kh == 0 && l < 16) {
        const int hl = 16 * hq + l16;
        const float sum = sums[hl] + sums[64 + hl];
        il[hl] = sum > 0.f ? 1.0f / sum : 0.f;
        if (nsplit > 1 && hg * 64 + hl < p.NQ) {
            p.part_ml[(prow_base + hg * 64 + hl) * 2] = m_run;
            p.part_ml[(prow_base + hg * 64 + hl) * 2 + 1] = sum;
        }
    }
    __syncthreads();
    auto drain = [&](auto final_tag) {
        constexpr bool FINAL = decltype(final_tag)::value;
#pragma unroll
        for (int hb = 0; hb < 2; ++hb) {
            const float iv = il[32 * hb + col];
#pragma unroll
            for (int d = 0; d < 2; ++d)
#pragma unroll
                for (int q4 = 0; q4 < 4; ++q4) {
                    const f32x16 &a = o[2 * hb + d];
                    const float v0 = a[4 * q4] * iv, v1 = a[4 * q4 + 1] * iv, v2 = a[4 * q4 + 2] * iv, v3 = a[4 * q4 + 3] * iv;
                    const u32x2 pk = {FINAL ? pack_bf16x2(v0, v1) : pack_f16x2(v0, v1), FINAL ? pack_bf16x2(v2, v3) : pack_f16x2(v2, v3)};
                    const int piece = 16 * (w & 3) + 2 * (4 * d + q4) + (w >> 2);            // of the row, in channel order
                    *reinterpret_cast<u32x2 *>(pool + (32 * hb + col) * (DN * 2) + 16 * (piece ^ col) + 8 * half) = pk;
                }
        }
        __syncthreads();
        u32x4 v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = *reinterpret_cast<const u32x4 *>(pool + (8 * w + e) * (DN * 2) + 16 * (l ^ ((8 * w + e) & 31)));
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int head = hg * 64 + 8 * w + e;
            uint16_t *dst = FINAL ? p.out + ((size_t)t * p.NQ + head) * DN : static_cast<uint16_t *>(p.part_o) + (prow_base + head) * DN;
            if (head < p.NQ) *reinterpret_cast<u32x4 *>(dst + 8 * l) = v[e];
        }
    };
    if (nsplit == 1) drain(std::true_type{});
    else drain(std::false_type{});
}
