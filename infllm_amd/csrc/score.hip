// Column sums of the final attention probabilities of one linear stage
// (inf_llm/attention/dot_production_attention/torch_impl.py:27-28): the "local score"
// that InfLLM accumulates per token to choose representative keys
// (inf_llm/attention/context_manager.py:623-625).
//
// It needs the final log-sum-exp of every query, so it runs after the merge, or joins the partial ones itself, and
// recomputes Q.K^T.  Orientation: S[query, key] with keys in the MFMA column, so a lane owns one key (or two) and the
// column sum is a running per-lane scalar.  A workgroup of four waves owns 128 or 256 consecutive keys of one query
// head, 32 or 64 of them in a wave's registers (B operand) for the whole kernel, while the queries stream through
// LDS (A operand, shared by the waves).  Exactly one lane writes each (head, key) cell, so results are deterministic.
//
// key_sums is that loop: three workgroups a CU, queries from memory straight into LDS, positions in 32 bits.  It is in
// scores_kernel (a launch of scores, with or without the merge) and in block_end_kernel (what ends a block).  score_tile is
// the general form behind it (local_score_kernel): two workgroups a CU, queries by way of registers, any number of partial
// log-sum-exps, positions in 64 bits.
#include "carve.h"
#include "rank.h"
#include <algorithm>
#include <atomic>
#include <type_traits>

namespace {

template <int D>
constexpr int kQPad = D + 8;               // LDS row of Q (bf16 elements): 272 (144) bytes rotates the banks

struct ScoreMerge {
    MergeJob job;
    int32_t score_tiles;               // blockIdx.y below this scores, from there on merges
    float empty;                       // see key_sums
};
struct NoScoreMerge {};

// Workgroups are dispatched x fastest: all heads of one key tile, then the next tile.  The two tiles at either end of a masked key
// range see only part of the queries and finish early, so they go last: when the grid is a little more than what the chip holds
// at once, the workgroups that start late are then the short ones.  (None at the low end when the first query sees it.)  Where the
// queries are (nearly) as many as the keys, a tile's work falls from the first to the last instead: a CU that takes one of the
// first half and one of the second gets a long and a short one.
__device__ __forceinline__ int tile_of_slot(const infllm_score_args &a, int slot, int n_tiles) {
    if (a.mask == INFLLM_MASK_WINDOW && a.Lq >= (a.j_hi - a.j_lo) - (a.j_hi - a.j_lo) / 4)
        return slot < (n_tiles + 1) / 2 ? slot : n_tiles - 1 - (slot - (n_tiles + 1) / 2);
    if (a.mask == INFLLM_MASK_WINDOW && a.j_lo >= a.offset + a.Lq - a.window) return slot;
    if (n_tiles >= 6 && a.mask != INFLLM_MASK_NONE)
        return slot < n_tiles - 4 ? slot + 2 : slot == n_tiles - 4 ? 1 : slot == n_tiles - 3 ? n_tiles - 2 : slot == n_tiles - 2 ? 0 : n_tiles - 1;
    return slot;
}

// The general form, for partial log-sum-exps in any number and rings or rows that 32 bits do not address (the others:
// scores_kernel).  One workgroup of 256 threads: tile `slot` (in the order they are dispatched) of n_tiles of the keys, query
// head bx.  KS = 32-key halves per wave: 2 for long key ranges; 1 halves the work of a wave per query stage, which is what
// bounds the short launches that sit on the critical path between two blocks.  QS = queries per LDS stage: a short
// launch is a chain of stages that each wait for one global load (there is next to no arithmetic to hide it behind),
// so it takes stages of 128 queries and half as many of them.
template <int D, int KS, int QS>
__device__ __forceinline__ void score_tile(const infllm_score_args &a, const PartSets lps, int bx, int slot, int n_tiles, char *score_lds) {
    constexpr int kWaveKeys = 32 * KS, kKeysPerWg = 4 * kWaveKeys, kQStage = QS;
    bf16_t(*Qs)[kQStage][kQPad<D>] = (bf16_t(*)[kQStage][kQPad<D>])score_lds;                               // [2][QS][kQPad]
    float(*Ls)[kQStage] = (float(*)[kQStage])(score_lds + 2 * kQStage * kQPad<D> * sizeof(bf16_t));      // [2][QS]

    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int col = lane & 31, grp = lane >> 5;
    const int G = a.H / a.Hkv;
    // bx walks the kv heads first, then the query heads of a group: workgroups go to the 8 XCDs round-robin by
    // linear id, so with 8 (16, ...) kv heads the query heads that share a K tile sit behind the same L2 and that tile
    // leaves HBM once instead of once per query head
    const int b = bx / a.H, hx = bx % a.H, g = hx % a.Hkv, h = g * G + hx / a.Hkv;
    const int tile = tile_of_slot(a, slot, n_tiles);
    const int64_t jg = (a.j_lo / kWaveKeys + (int64_t)tile * 4) * kWaveKeys;         // first key of the workgroup
    const int64_t j0 = jg + (int64_t)wave * kWaveKeys;                               // first key of this wave
    const float scale = a.softmax_scale * 1.4426950408889634f;

    // ---- this wave's 64 keys as the B operand (lane = key column)
    bf16x8 kreg[KS][D / 16];
    bool jok[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        const int64_t j = j0 + ks * 32 + col;
        jok[ks] = j >= a.j_lo && j < a.j_hi;
        const bf16_t *krow = (const bf16_t *)a.d_k + (int64_t)b * a.k_sb + (int64_t)g * a.k_sh + (j % a.cap) * a.k_sl;
#pragma unroll
        for (int kk = 0; kk < D / 16; ++kk) {
            u32x4 raw = jok[ks] ? *(const u32x4 *)(krow + kk * 16 + grp * 8) : u32x4{0, 0, 0, 0};
            kreg[ks][kk] = __builtin_bit_cast(bf16x8, raw);
        }
    }

    // ---- query range: what the workgroup stages, and what this wave needs of it
    auto query_range = [&](int64_t jf, int64_t jl, int64_t &lo, int64_t &hi) {   // keys [jf, jl] -> queries [lo, hi)
        lo = 0;
        hi = a.Lq;
        jf = max(jf, a.j_lo);
        jl = min(jl, a.j_hi - 1);
        if (jl < jf) {
            hi = 0;
            return;
        }
        if (a.mask == INFLLM_MASK_WINDOW) {
            lo = max(lo, jf - a.offset);
            hi = min(hi, jl - a.offset + a.window);
        } else if (a.mask == INFLLM_MASK_COMPLEMENT) {
            lo = max(lo, jf - a.offset + a.window);
        }
    };
    int64_t g_lo, g_hi, w_lo, w_hi;
    query_range(jg, jg + kKeysPerWg - 1, g_lo, g_hi);
    query_range(j0, j0 + kWaveKeys - 1, w_lo, w_hi);
    const int st_lo = (int)(g_lo / kQStage), st_hi = g_hi > g_lo ? (int)((g_hi - 1) / kQStage) + 1 : st_lo;

    const bf16_t *qbase = (const bf16_t *)a.d_q + (int64_t)b * a.q_sb + (int64_t)h * a.q_sh;
    const float *lse = a.d_lse + ((int64_t)b * a.H + h) * a.Lq;
    constexpr int kChunks = D / 8, kLdRows = 256 / kChunks;        // chunks of a row, rows of Q a pass of the workgroup loads
    const int ld_chunk = tid % kChunks, ld_row = tid / kChunks;
    u32x4 qbuf[kQStage / kLdRows];
    float lbuf = 0.f;
    auto load_stage = [&](int s) {
        const int i0 = s * kQStage;
#pragma unroll
        for (int i = 0; i < kQStage / kLdRows; ++i) {
            const int qi = i0 + ld_row + kLdRows * i;
            qbuf[i] = qi < a.Lq ? *(const u32x4 *)(qbase + (int64_t)qi * a.q_sl + ld_chunk * 8) : u32x4{0, 0, 0, 0};
        }
        if (tid < kQStage) {
            if (i0 + tid >= a.Lq) {
                lbuf = INFINITY;                                                  // +inf => probability 0
            } else if (a.n_parts <= 0) {
                lbuf = lse[i0 + tid];
            } else {                                                              // join the stages' partial values here
                const int64_t rows = (int64_t)a.B * a.H * a.Lq;
                float m = -INFINITY, den = 0.f;
                for (int p0 = 0; p0 < a.n_parts; p0 += 8) {
                    float l8[8], m8 = -INFINITY;
#pragma unroll
                    for (int i = 0; i < 8; ++i) l8[i] = p0 + i < a.n_parts ? lse[lps.l(p0 + i, rows) + i0 + tid] : -INFINITY;
#pragma unroll
                    for (int i = 0; i < 8; ++i) m8 = fmaxf(m8, l8[i]);
                    if (m8 == -INFINITY) continue;
                    const float m_new = fmaxf(m, m8);
                    den *= __builtin_amdgcn_exp2f(m - m_new);
#pragma unroll
                    for (int i = 0; i < 8; ++i) den += __builtin_amdgcn_exp2f(l8[i] - m_new);
                    m = m_new;
                }
                lbuf = den > 0.f ? m + log2f(den) : INFINITY;
            }
        }
    };
    auto store_stage = [&](int buf) {
#pragma unroll
        for (int i = 0; i < kQStage / kLdRows; ++i) *(u32x4 *)&Qs[buf][ld_row + kLdRows * i][ld_chunk * 8] = qbuf[i];
        if (tid < kQStage) Ls[buf][tid] = lbuf;
    };

    float colsum[KS] = {};
    if (st_hi > st_lo) load_stage(st_lo);
    if (st_hi > st_lo) {
        store_stage(0);
        if (st_lo + 1 < st_hi) load_stage(st_lo + 1);
    }
    __syncthreads();
    for (int s = st_lo; s < st_hi; ++s) {
        const int cur = (s - st_lo) & 1;
        const int64_t i0 = (int64_t)s * kQStage;
        // does the wave see every (query, key) pair of this stage?
        bool fast = i0 >= w_lo && i0 + kQStage <= w_hi && i0 + kQStage <= a.Lq && j0 >= a.j_lo && j0 + kWaveKeys <= a.j_hi;
        if (a.mask == INFLLM_MASK_WINDOW)
            fast = fast && (i0 - (j0 + kWaveKeys - 1) + a.offset >= 0) && (i0 + kQStage - 1 - j0 + a.offset < a.window);
        if (a.mask == INFLLM_MASK_COMPLEMENT) fast = fast && (i0 - (j0 + kWaveKeys - 1) + a.offset >= a.window);
        // The sub-tiles of 32 queries are software pipelined: the MFMAs of sub-tile qs+1 are issued before the exponentials of
        // sub-tile qs, in ONE basic block, so that the scheduler can interleave them (an MFMA runs for 32 cycles in the
        // background of the VALU); with everything behind per-sub-tile branches the two kinds of work only ever alternated.
        // A stage with pairs that are masked takes the same form with a select behind every exponential: it costs a third more
        // than an unmasked one, where sub-tiles looked at one by one (and left out where nothing was visible) cost twice as
        // much - and the workgroups on the diagonal end a launch.  Together with two queries' log-sum-exps per trip to memory: the
        // operator over 512 queries x (4,608 + 2,624) keys 112.5 -> 106.8 us, a prompt of 131,072 tokens 29,520 -> 28,935.
        auto stage = [&](auto masked) {
            constexpr int kSub = kQStage / 32;
            constexpr bool kMasked = decltype(masked)::value;
            // the queries that see this lane's keys: q_first .. q_first + q_count - 1
            int q_first[KS];
            uint32_t q_count[KS];
            if constexpr (kMasked) {
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) {
                    const int64_t at = j0 + ks * 32 + col - a.offset;
                    const int64_t from = a.mask == INFLLM_MASK_WINDOW ? at : a.mask == INFLLM_MASK_COMPLEMENT ? at + a.window : 0;
                    const int64_t to = a.mask == INFLLM_MASK_WINDOW ? at + a.window : a.Lq;
                    q_first[ks] = (int)min(max(from, (int64_t)0), (int64_t)a.Lq);
                    q_count[ks] = (uint32_t)max((int)min(max(to, (int64_t)0), (int64_t)a.Lq) - q_first[ks], 0);
                }
            }
            f32x16 sacc[2][KS];
            f32x4 l4[2][4];
            auto issue = [&](int qs, int pb) {
                bf16x8 qa[D / 16];                              // A operand: lane = query row
                const bf16_t *qrow = &Qs[cur][qs * 32 + col][grp * 8];
#pragma unroll
                for (int kk = 0; kk < D / 16; ++kk) qa[kk] = *(const bf16x8 *)(qrow + kk * 16);
#pragma unroll
                for (int q4 = 0; q4 < 4; ++q4) l4[pb][q4] = *(const f32x4 *)&Ls[cur][qs * 32 + 8 * q4 + 4 * grp];
#pragma unroll
                for (int ks = 0; ks < KS; ++ks)
#pragma unroll
                    for (int r = 0; r < 16; ++r) sacc[pb][ks][r] = 0.f;
#pragma unroll
                for (int kk = 0; kk < D / 16; ++kk)
#pragma unroll
                    for (int ks = 0; ks < KS; ++ks)
                        sacc[pb][ks] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(qa[kk], kreg[ks][kk], sacc[pb][ks], 0, 0, 0);
            };
            issue(0, 0);
            __builtin_amdgcn_sched_barrier(0);                  // (the fences keep sub-tiles apart: registers)
#pragma unroll
            for (int qs = 0; qs < kSub; ++qs) {
                const int pb = qs & 1;
                if (qs + 1 < kSub) issue(qs + 1, pb ^ 1);
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) {
                    const int from = kMasked ? (int)i0 + qs * 32 + 4 * grp - q_first[ks] : 0;
                    float acc = 0.f;
#pragma unroll
                    for (int r = 0; r < 16; ++r) {              // query 8 * (r >> 2) + 4 * grp + (r & 3) of the sub-tile
                        const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[pb][ks][r], scale, -l4[pb][r >> 2][r & 3]));
                        if (kMasked) acc += (uint32_t)(from + 8 * (r >> 2) + (r & 3)) < q_count[ks] ? p : 0.f;
                        else acc += p;
                    }
                    colsum[ks] += acc;
                }
                if (qs + 1 < kSub) {
                    // one MFMA, then its share of the exponentials (16 * KS of each per sub-tile)
#pragma unroll
                    for (int i = 0; i < D / 16 * KS; ++i) {
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);      // MFMA
                        __builtin_amdgcn_sched_group_barrier(0x002, (kMasked ? 2 : 1) * 512 / D, 0);      // VALU
                        __builtin_amdgcn_sched_group_barrier(0x400, 256 / D, 0);      // transcendental
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        if (fast) stage(std::false_type{});
        else if (i0 < w_hi && i0 + kQStage > w_lo) stage(std::true_type{});                  // wave-uniform
        if (s + 1 < st_hi) {
            store_stage(cur ^ 1);
            if (s + 2 < st_hi) load_stage(s + 2);
        }
        __syncthreads();
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        const float tot = colsum[ks] + wave_xor32(colsum[ks]);
        const int64_t j = j0 + ks * 32 + col;
        if (grp == 0 && jok[ks]) {
            float *dst = a.d_score + (int64_t)b * a.score_sb + (int64_t)h * a.score_sh + (j % a.score_cap);
            *dst = a.accumulate ? *dst + tot : tot;
        }
    }
}

template <int D, int KS, int QS>
__global__ __launch_bounds__(256, 2) void local_score_kernel(infllm_score_args a) {
    extern __shared__ __attribute__((aligned(16))) char score_lds[];
    score_tile<D, KS, QS>(a, PartSets{a.n_parts, 0, 0}, blockIdx.x, blockIdx.y, gridDim.y, score_lds);
}

// What ends a block, in one launch: the scores of its keys, the merge of its partial outputs, the units that leave the window
// with it (their rows to their home, their representatives) and the next block's selection and page table.
//
// The next block waits for a chain of latencies in it that needs little of the chip: the block's share of the scores of the
// keys that leave -> the representatives of the units they make up (context_manager.py:268-277) -> the ranking.  The rest - the
// scores of the keys that stay, the merge, the units' rows - depends on none of it and fills the chip meanwhile.  So the
// carving workgroups (one per unit and head: 128 keys x 512 queries, half of them outside the window) come first in the grid;
// the one that is done last ranks.  As two launches, carving with the merge and the rest of the scores with the ranking, which
// can begin when the first has ended: 5 us a block of 512 queries x 4,096 keys x 32 heads more (17.2 + 28).  What the last one does
// is what the launch waits for, beside a chip full of other loads: it scores under one mean query (four took 18.6 us, the scores'
// last workgroup ends 3 to 10 us earlier), sees to nothing but its own stores, and counts with four lanes an entry: prompts of
// 131,072 tokens 27,610 -> 26,830 us, of 24,300 with 36 heads of 64 3,350 -> 3,200.
//
// A carving workgroup's steps are as short as they can be: everything it reads is requested at once; the unit's keys are in
// LDS (every wave needs them all), four sub-tiles of 32 queries a wave take turns with each of them; a sub-tile's column sums
// are added in the order of the queries, as score_tile adds them (the same bits); the picks by counting, all rows at once.
constexpr int kCarveMaxLq = 512, kCarveMaxUnit = 128;
struct BlockEnd {
    infllm_score_args s;               // the keys that stay
    MergeJob merge;                    // the block's partials (out NULL: merged before)
    int32_t n_carve, n_score, n_copy, n_early;     // workgroups of each kind (carve, score, early, copy), those that merge behind them
    int32_t cap, slot0, win;           // rows of the ring; that of the first key of the first scoring workgroup; the window
    // The keys that are scored first, then the others in ascending order: those of the block's own first queries, masked for some of them and
    // seen by all, are the longest.  They were the last but one, on the CUs that carve and score already, and the launch waited for
    // them (32.5 us behind the first workgroup's start, most others 25 to 29).  Prompts of 16,001 / 131,072 tokens, 32 heads of 128:
    // 2,613 -> 2,575 / 25,035 -> 24,602 us; 24,300 with 36 heads of 64, whose launch waits for the ranking: unchanged.
    int32_t first_tile;
    // units that leave
    const bf16_t *ring_k_raw;
    int64_t t0;                        // their first key, and its row
    int32_t unit_slot0, bs, n_units, repr_topk;
    bf16_t *rep_out;
    int64_t rep_sb, rep_su;
    CarveCopy cc;
    RankJob rank;
    int32_t ranks;                     // does the launch rank?
    uint32_t *ticket;                  // zero; the last of the carving workgroups to finish puts it back
};

// Column sums of the probabilities for 128 * KS consecutive keys of a query head, 32 * KS a wave and KS a lane (both halves of
// the wave get them).  The keys are those from position jg on, of which [lo, hi) count; key r of them lies in row slot + r of the
// ring, or a ring's length before.  A key is visible at distances [first, beyond) of a query.  JOIN: the log-sum-exps are
// joined from partial ones (at a.d_lse + lps), of all queries before the first stage; else they are finished (a.d_lse) and
// come with a stage's queries.  `empty` stands for the sum of a query whose partial ones are all empty: one that sees nothing, or
// whose logits are no numbers.  +infinity leaves those out; -infinity, what a finished sum holds then, makes the scores of all keys
// that such a query sees infinite or NaN.
//
// A wave's exponentials and MFMAs overlap (half a sub-tile of 32 queries apart), so the loop runs at the rate of the vector unit
// (768 cycles of a sub-tile of 32 queries x 64 keys); what is left is a launch of one or two rounds of workgroups whose first 5
// of 20 us are the wait for their keys.  So registers and LDS are kept to a third of a CU: all carving and scoring workgroups of
// 512 queries x 4,096 keys x 32 heads are in flight at once, one's wait beside another's loop.  The queries go from memory
// straight into LDS (64 rows a stage, three stages in turn, no registers on the way), and a wave's two accumulators are the halves
// of a sub-tile instead of two sub-tiles.  With half a CU each (score_tile, and carving workgroups with a loop of their own):
// prompts of 131,072 / 16,001 tokens 27,000 -> 26,000 / 2,816 -> 2,726 us, of 24,300 with 36 heads of 64 3,185 -> 3,136.
//
// QR queries a stage, NB stages in LDS; QG groups of four waves hold the same keys and share a stage's queries (see paired_waves).
constexpr int kQRows = 64;                             // queries of a stage
template <int D>
constexpr size_t kQBytes = (size_t)3 * kQRows * D * sizeof(bf16_t);
// A carving workgroup's stages: heads of 64 have room for 128 queries, of 32 keys a wave four steps instead of two, and the next block
// waits for them (prompt of 24,300 tokens, 36 heads: 3,105 -> 3,089 us; the scores' own stages, four steps as they are, 0.5 % slower
// with 128).  Heads of 128 have room for two stages of 96: 0.2 % slower, the scores' 2.8 %.
template <int D>
constexpr int kCarveRows = D == 64 ? 128 : 64;
template <int D>
constexpr int kCarveBufs = D == 64 ? 2 : 3;
template <int D>
constexpr size_t kCarveBytes = (size_t)kCarveBufs<D> * kCarveRows<D> * D * sizeof(bf16_t);

template <int D, int KS, bool JOIN, int QR = kQRows, int NB = 3, int QG = 1>
__device__ __forceinline__ void key_sums(const infllm_score_args &a, const PartSets lps, int b, int h, int64_t jg, int slot, int cap, int lo, int hi, int first,
                                         int beyond, float empty, char *lds, float (&sums)[KS]) {
    constexpr int kWaveKeys = 32 * KS, kRow = D * 2, kStage = QR * kRow;
    constexpr int kThreads = 256 * QG, kOwn = QR / QG;             // of a stage's queries those that are a group's
    const int tid = threadIdx.x, any_wave = __builtin_amdgcn_readfirstlane(tid >> 6), wave = any_wave & 3, group = any_wave >> 2;
    const int lane = tid & 63, col = lane & 31, grp = lane >> 5;
    b = __builtin_amdgcn_readfirstlane(b), h = __builtin_amdgcn_readfirstlane(h), slot = __builtin_amdgcn_readfirstlane(slot);
    lo = __builtin_amdgcn_readfirstlane(lo), hi = __builtin_amdgcn_readfirstlane(hi);
    const int g = __builtin_amdgcn_readfirstlane(h / (a.H / a.Hkv)), Lq = a.Lq;
    const float scale = a.softmax_scale * 1.4426950408889634f;
    float *Ls = (float *)(lds + NB * kStage);                       // JOIN: [Lq rounded up to a stage]; else [NB][QR]
    // a key's distance to query q is q + d - its place among the keys
    const int d = (int)min(max(a.offset - jg, (int64_t)-(1 << 29)), (int64_t)(1 << 29));
    // queries that see any of the keys, in stages
    const int q_lo = max(lo - d + first, 0), q_hi = (int)min((int64_t)hi - d - 1 + beyond, (int64_t)Lq);
    const int st_lo = q_lo / QR, st_hi = hi > lo && q_hi > q_lo ? (q_hi - 1) / QR + 1 : st_lo;

    // ---- queries into LDS: an instruction fills 1024 bytes; a wave the rows from 16 * wave on
    constexpr int kRowsPerLd = 1024 / kRow, kLd = QR / (4 * QG * kRowsPerLd);
    const bf16_t *qbase = (const bf16_t *)a.d_q + (int64_t)b * a.q_sb + (int64_t)h * a.q_sh;
    const float *lse = a.d_lse + ((int64_t)b * a.H + h) * Lq;
    const uint32_t q_lds = lds_address(lds) + any_wave * (kLd * 1024);
    auto load_stage = [&](int s, int buf) {
#pragma unroll
        for (int i = 0; i < kLd; ++i) {
            const int r = kRowsPerLd * (kLd * any_wave + i) + lane / (D / 8);                   // (rows behind the last query: the last one's, masked)
            const int q = min(s * QR + r, Lq - 1);
            load_to_lds16(qbase, (uint32_t)((int64_t)q * a.q_sl + ((lane & (D / 8 - 1)) ^ swz<D>(r)) * 8) * 2, q_lds + buf * kStage + i * 1024);
        }
        constexpr int kLse = QR / (4 * QG);
        if (!JOIN && lane < kLse)
            load_to_lds4(lse, (uint32_t)min(s * QR + any_wave * kLse + lane, Lq - 1) * 4, lds_address((char *)(Ls + buf * QR + any_wave * kLse)));
    };
    // ---- partial log-sum-exps of the first queries, two a thread.  What a wave requests comes back in order: they are joined while the keys
    //      are on their way (prompts of 24,300 tokens, 36 heads of 64, 2,859 -> 2,838 us, of 131,072 with 32 of 128 23,831 -> 23,705; waves in pairs, with up to 2,048 queries to join, are 0.8 % slower so).
    const int64_t all = (int64_t)a.B * a.H * Lq;
    float l8[2][8];
    auto ask_sums = [&](int i0) {
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int p = 0; p < 8; ++p) l8[e][p] = i0 + e * kThreads < Lq && p < a.n_parts ? lse[lps.l(p, all) + i0 + e * kThreads] : -INFINITY;
    };
    constexpr bool kSumsFirst = JOIN && QG == 1;
    if constexpr (kSumsFirst) {
        ask_sums(tid);
        asm volatile("" ::: "memory");
    }
    if (st_lo < st_hi) load_stage(st_lo, 0);

    // ---- this wave's keys as the B operand (lane = key column), by way of the stages that are not on their way yet: 32 keys of every wave
    //      at a time, whole rows in order.  (Keys that do not count: one that does again, its sums are not used.)  Straight into registers,
    //      by lanes that fetch their own key's pieces, they are 64 lines an instruction, and the 12 waves of a CU asked for 6 us: keys in
    //      registers 7.2 us behind the launch's start, 5.5 so.  Prompts of 16,001 / 131,072 tokens 2,521 -> 2,505 / 24,210 -> 23,937 us,
    //      operator over 512 x (4,608 + 2,624) keys 93.2 -> 92.2.
    constexpr int kKeyLds = 32 / QG / kRowsPerLd;
    static_assert((NB - 1) * kStage >= 128 * kRow && (KS == 1 || QG == 1), "room for 128 keys behind the first stage");
    const bf16_t *kbase = (const bf16_t *)a.d_k + (int64_t)b * a.k_sb + (int64_t)g * a.k_sh;
    const uint32_t k_lds = lds_address(lds) + kStage;
    auto ask_keys = [&](int ks) {
        if (hi > lo)
#pragma unroll
            for (int i = 0; i < kKeyLds; ++i) {
                const int r = kRowsPerLd * (kKeyLds * any_wave + i) + lane / (D / 8);
                int row = slot + min(max((r >> 5) * kWaveKeys + ks * 32 + (r & 31), lo), hi - 1);
                row = row < cap ? row : row - cap;
                load_to_lds16_at(kbase + (int64_t)row * a.k_sl + ((lane & (D / 8 - 1)) ^ swz<D>(r)) * 8, k_lds + (kKeyLds * any_wave + i) * 1024);
            }
    };
    bf16x8 kreg[KS][D / 16];
    auto take_keys = [&](int ks) {                                  // (a wave's rows are its own, or of it and the other group's)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if constexpr (QG > 1) asm volatile("s_barrier" ::: "memory");
        const uint32_t at = k_lds + (wave * 32 + col) * kRow + ((grp ^ swz<D>(col)) * 16);
#pragma unroll
        for (int kk = 0; kk < D / 16; ++kk) kreg[ks][kk] = __builtin_bit_cast(bf16x8, *(const __attribute__((address_space(3))) u32x4 *)(uintptr_t)(at ^ (kk * 32)));
#pragma unroll
        for (int kk = 0; kk < D / 16; ++kk) asm volatile("" : "+v"(kreg[ks][kk]));         // (read before the rows are overwritten)
    };
    ask_keys(0);
    take_keys(0);
    if constexpr (kSumsFirst) {                                     // (they have come; the compiler's wait for them belongs here)
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int p = 0; p < 8; ++p) asm volatile("" : "+v"(l8[e][p]));
    }
    if constexpr (KS > 1) ask_keys(1);
    // ---- joined log-sum-exps of all queries
    if constexpr (JOIN) {
        const int padded = (Lq + QR - 1) / QR * QR;
        for (int i0 = tid; i0 < padded; i0 += 2 * kThreads) {
            if (!kSumsFirst || i0 >= 2 * kThreads) ask_sums(i0);
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                float m8 = -INFINITY, den = 0.f;
#pragma unroll
                for (int p = 0; p < 8; ++p) m8 = fmaxf(m8, l8[e][p]);
                if (m8 != -INFINITY) {
#pragma unroll
                    for (int p = 0; p < 8; ++p) den += __builtin_amdgcn_exp2f(l8[e][p] - m8);
                }
                if (i0 + e * kThreads < padded) Ls[i0 + e * kThreads] = den > 0.f ? m8 + log2f(den) : empty;
            }
        }
    }
    if constexpr (KS > 1) take_keys(1);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");                 // the sums are there, and the keys' place is free
    if (NB > 2 && st_lo + 1 < st_hi) load_stage(st_lo + 1, 1);

    // (the keys' wait belongs here: in front of their first use, inside the loop, it would be one for the stages on their way)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int kk = 0; kk < D / 16; ++kk) asm volatile("" : "+v"(kreg[ks][kk]));
    const int w_first = wave * kWaveKeys;
    const int w_lo = max(lo, w_first), w_hi = min(hi, w_first + kWaveKeys);                   // the wave's keys that count
    const bool whole = w_lo == w_first && w_hi == w_first + kWaveKeys;
    float colsum[KS] = {};
    int buf = 0;
    for (int s = st_lo; s < st_hi; ++s) {
        // this wave's rows of the stage have landed (of three buffers, those of the next may be on their way), then everyone's; the
        // buffer that is requested next was read a stage ago
        if (NB > 2 && s + 1 < st_hi) asm volatile("s_waitcnt vmcnt(%0)" ::"i"(JOIN ? kLd : kLd + 1) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        asm volatile("s_barrier" ::: "memory");
        if (s + NB - 1 < st_hi) load_stage(s + NB - 1, buf == 0 ? NB - 1 : buf - 1);
        const int i0 = s * QR + group * kOwn;                   // this wave's first query of the stage
        auto stage = [&](auto masked) {
            constexpr bool kMasked = decltype(masked)::value;
            constexpr int kSteps = kOwn / 32 * KS;          // (sub-tile of 32 queries, 32 keys), keys first
            int q_first[KS];                                    // the queries that see this lane's keys: q_first .. q_first + q_count - 1
            uint32_t q_count[KS];
            if constexpr (kMasked) {
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) {
                    const int r = w_first + ks * 32 + col - d;
                    q_first[ks] = min(max(r + first, 0), Lq);
                    q_count[ks] = (uint32_t)max((int)min(max((int64_t)r + beyond, (int64_t)0), (int64_t)Lq) - q_first[ks], 0);
                }
            }
            f32x16 acc[2];
            bf16x8 qa[D / 16];                                  // A operand: lane = query row
            const uint32_t q_at = lds_address(lds) + buf * kStage + (group * kOwn + col) * kRow + ((grp ^ swz<D>(col)) * 16);
            auto issue = [&](int t) {
                const int qs = t / KS, ks = t % KS;
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[t & 1][r] = 0.f;
#pragma unroll
                for (int kk = 0; kk < D / 16; ++kk) {
                    if (ks == 0) qa[kk] = __builtin_bit_cast(bf16x8, *(const __attribute__((address_space(3))) u32x4 *)(uintptr_t)((q_at ^ (kk * 32)) + qs * 32 * kRow));
                    acc[t & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(qa[kk], kreg[ks][kk], acc[t & 1], 0, 0, 0);
                }
            };
            issue(0);
            __builtin_amdgcn_sched_barrier(0);                  // (the fences keep the steps apart: registers)
#pragma unroll
            for (int t = 0; t < kSteps; ++t) {
                const int qs = t / KS, ks = t % KS;
                if (t + 1 < kSteps) issue(t + 1);
                f32x4 l4[4];
#pragma unroll
                for (int q4 = 0; q4 < 4; ++q4) l4[q4] = *(const f32x4 *)&Ls[(JOIN ? i0 : buf * QR + group * kOwn) + qs * 32 + 8 * q4 + 4 * grp];
                const int from = kMasked ? i0 + qs * 32 + 4 * grp - q_first[ks] : 0;
                float sum = 0.f;
#pragma unroll
                for (int r = 0; r < 16; ++r) {                  // query 8 * (r >> 2) + 4 * grp + (r & 3) of the sub-tile
                    const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(acc[t & 1][r], scale, -l4[r >> 2][r & 3]));
                    if (kMasked) sum += (uint32_t)(from + 8 * (r >> 2) + (r & 3)) < q_count[ks] ? p : 0.f;
                    else sum += p;
                }
                colsum[ks] += sum;
                if (t + 1 < kSteps) {
#pragma unroll
                    for (int i = 0; i < D / 16; ++i) {
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);      // MFMA
                        __builtin_amdgcn_sched_group_barrier(0x002, (kMasked ? 2 : 1) * 512 / D, 0);      // VALU
                        __builtin_amdgcn_sched_group_barrier(0x400, 256 / D, 0);      // transcendental
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        // every pair is visible / some are (wave-uniform)
        if (whole && i0 + kOwn <= Lq && i0 + d - (w_first + kWaveKeys - 1) >= first && i0 + kOwn - 1 + d - w_first < beyond) stage(std::false_type{});
        else if (w_hi > w_lo && i0 + kOwn - 1 + d - w_lo >= first && i0 + d - (w_hi - 1) < beyond) stage(std::true_type{});
        buf = buf == NB - 1 ? 0 : buf + 1;
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) sums[ks] = colsum[ks] + wave_xor32(colsum[ks]);
    if constexpr (QG > 1) {                                     // the first group gets the sums of all, in the order of the queries
        float(*part)[4][KS][64] = (float(*)[4][KS][64])lds;
        __syncthreads();
        if (group > 0)
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) part[group - 1][wave][ks][lane] = sums[ks];
        __syncthreads();
#pragma unroll
        for (int o = 0; o < QG - 1; ++o)
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) sums[ks] += part[o][wave][ks][lane];
    }
}

// Heads of different kv heads next to each other, see score_tile.
__device__ __forceinline__ void head_of(const infllm_score_args &a, int bx, int &b, int &h) {
    b = bx / a.H;
    const int hx = bx - b * a.H, rest = hx / a.Hkv;
    h = (hx - rest * a.Hkv) * (a.H / a.Hkv) + rest;
}

// The scores of a launch whose log-sum-exps are finished: the form of the kernel that keeps three workgroups on a CU
// (operator over 512 queries x (4,608 + 2,624) keys 108.4 -> 102.9 us a pass, prompt of 16,001 tokens 2,745 -> 2,723).
//
// MERGE: the launch also carries the merge of the partial attention outputs, in workgroups behind the scoring ones, which join the
// partial log-sum-exps themselves, by the merge's own arithmetic (the operator, whose merge was a launch in front of this one:
// 101.0 -> 96.8 us).
struct ScoreForm {
    int ks, rows, bufs, groups;            // 32-key halves of a wave; queries of a stage, stages in LDS, groups of waves that share one
};
enum { kWide = 0, kNarrow = 1, kPaired = 2 };
constexpr ScoreForm kScoreForms[3] = {{2, 64, 3, 1}, {1, 64, 3, 1}, {1, 128, 2, 2}};
template <int D, int FORM, bool MERGE>
__global__ __launch_bounds__(256 * kScoreForms[FORM].groups, (D == 64 || FORM == kPaired ? 4 : 3)) void scores_kernel(infllm_score_args a, int slot0, int cap, int first, int beyond,
                                                                        std::conditional_t<MERGE, ScoreMerge, NoScoreMerge> sm) {
    extern __shared__ __attribute__((aligned(1024))) char score_lds[];
    constexpr ScoreForm F = kScoreForms[FORM];
    constexpr int KS = F.ks, kKeys = 128 * KS;
    int n_tiles = gridDim.y;
    PartSets lps{};
    float empty = 0.f;
    if constexpr (MERGE) {
        n_tiles = sm.score_tiles;
        if ((int)blockIdx.y >= n_tiles) {
            merge_piece<D>(sm.job, ((int64_t)((int)blockIdx.y - n_tiles) * gridDim.x + blockIdx.x) * (256 * F.groups) + threadIdx.x);
            return;
        }
        lps = sm.job.ps;
        empty = sm.empty;
    }
    int b, h;
    head_of(a, blockIdx.x, b, h);
    const int tile = tile_of_slot(a, blockIdx.y, n_tiles);
    const int64_t jg = a.j_lo / (32 * KS) * (32 * KS) + (int64_t)tile * kKeys;
    const int lo = (int)max(a.j_lo - jg, (int64_t)0), hi = (int)min(a.j_hi - jg, (int64_t)kKeys);
    float sums[KS];
    key_sums<D, KS, MERGE, F.rows, F.bufs, F.groups>(a, lps, b, h, jg, slot0 + tile * kKeys, cap, lo, hi, first, beyond, empty, score_lds, sums);
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        const int r = (threadIdx.x >> 6) * (32 * KS) + ks * 32 + lane;
        if (lane < 32 && r >= lo && r < hi && threadIdx.x < 256) {
            float *dst = a.d_score + (int64_t)b * a.score_sb + (int64_t)h * a.score_sh + (jg + r) % a.score_cap;
            *dst = a.accumulate ? *dst + sums[ks] : sums[ks];
        }
    }
}

// The representatives of a unit for one head: the unit's scores complete, the picks by counting - a row's place in the order is
// the number of rows in front of it -, all rows at once.
template <int D>
__device__ __forceinline__ void carve_unit(const BlockEnd &j, int h, int u, int b, char *lds) {
    const infllm_score_args &a = j.s;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, col = lane & 31, bs = j.bs;
    const int slot = j.unit_slot0 + u * bs;
    auto slot_of = [&](int r) {                                   // ring row of row r of the unit
        const int s = slot + r;
        return s < j.cap ? s : s - j.cap;
    };
    const int own_row = wave * 32 + col;
    const float track = own_row < bs ? a.d_score[(int64_t)b * a.score_sb + (int64_t)h * a.score_sh + slot_of(own_row)] : 0.f;
    float sum[1];
    key_sums<D, 1, true, kCarveRows<D>, kCarveBufs<D>>(a, j.merge.ps, b, h, j.t0 + (int64_t)u * bs, slot, j.cap, 0, bs, 0, j.win, INFINITY, lds, sum);
    __syncthreads();                                             // (the queries' place is free)
    uint64_t *rank_key = (uint64_t *)lds;
    int32_t *chosen = (int32_t *)(rank_key + kCarveMaxUnit);
    if (lane < 32) rank_key[own_row] = own_row < bs ? pick_key(track + sum[0], own_row) : 0;
    __syncthreads();
    {
        constexpr int kLanes = 256 / kCarveMaxUnit;              // lanes that count for a row
        const int r = tid / kLanes, p = tid % kLanes;
        const uint64_t own = rank_key[r];
        int before = 0;
#pragma unroll 16
        for (int i = 0; i < kCarveMaxUnit / kLanes; ++i) before += rank_key[i * kLanes + p] > own;
#pragma unroll
        for (int o = 1; o < kLanes; o <<= 1) before += __shfl_xor(before, o, 64);
        if (p == 0 && r < bs && before < j.repr_topk) chosen[before] = r;
    }
    __syncthreads();
    if (tid * 2 < D) {
        const bf16_t *raw = j.ring_k_raw + ((int64_t)b * a.Hkv + h / (a.H / a.Hkv)) * j.cap * D + tid * 2;
        float a0 = 0.f, a1 = 0.f;
#pragma unroll 4
        for (int i = 0; i < j.repr_topk; ++i) {
            const uint32_t w = *(const uint32_t *)(raw + (int64_t)slot_of(chosen[i]) * D);
            a0 += bf16_bits_to_f32(w & 0xffffu);
            a1 += bf16_bits_to_f32(w >> 16);
        }
        const float inv = 1.f / (float)j.repr_topk;
        // performed at the level of the memory hierarchy that all XCDs share: the workgroup that ranks reads it there
        __hip_atomic_store((uint32_t *)(j.rep_out + (int64_t)b * j.rep_sb + (int64_t)u * j.rep_su + (int64_t)h * D + tid * 2), pack_bf16x2(a0 * inv, a1 * inv),
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// Rows of representatives that the ranking takes, in 512s: 36 heads of 128, 40 of 64.  (Registers: heads of 64 with 32 keys a wave
// are three workgroups to a CU, which leaves 168 of them.)
template <int D>
constexpr int kRankCpl = D == 64 ? 5 : 9;

template <int D, int KS>
__global__ __launch_bounds__(256, (D == 64 ? 4 : 3)) void block_end_kernel(BlockEnd) {
    extern __shared__ __attribute__((aligned(1024))) char score_lds[];
    // The arguments where they lie, for each kind of workgroup anew.  (As the parameter they are loads that all kinds share, made in
    // front of the first branch and kept: 215 scalar registers were written to vector lanes and back on every workgroup's way.  Prompts of
    // 16,001 / 131,072 tokens 2,692 -> 2,624 / 25,698 -> 24,969 us, of 24,300 with 36 heads of 64 unchanged.)
    auto arguments = []() -> const BlockEnd & {
        auto *p = (const __attribute__((address_space(4))) char *)__builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" : "+s"(p));
        return *(const BlockEnd *)p;
    };
    touch_arguments<sizeof(BlockEnd)>();                          // (prompts of 16,001 / 131,072 tokens 0.7 / 0.4 %)
    int x = blockIdx.x;
    const int n_carve = arguments().n_carve;
    if (x < n_carve) {
        const BlockEnd &j = arguments();
        if (j.n_units > 0) {
            const int rest = x / j.s.H;
            carve_unit<D>(j, x - rest * j.s.H, rest % j.n_units, rest / j.n_units, score_lds);
            if (!j.ranks) return;
            // The representatives are the only thing that crosses workgroups, and their stores have been performed where every
            // XCD sees them before the ticket is drawn: no workgroup has to write its L2 back.
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            int &last = *(int *)(score_lds + kCarveMaxUnit * 16);
            if (threadIdx.x == 0) last = __hip_atomic_fetch_add(j.ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (uint32_t)j.n_carve - 1;
            __syncthreads();
            if (!last) return;
            __syncthreads();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
            if (threadIdx.x == 0) __hip_atomic_store(j.ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __builtin_amdgcn_s_setprio(3);                            // (the launch waits for it)
        rank_block<kRankCpl<D>>(j.rank, 0, j.rank.n_new, false, *(RankLds<kRankCpl<D>> *)score_lds);
        return;
    }
    x -= n_carve;
    const int n_score = arguments().n_score;
    if (x < n_score) {
        const BlockEnd &j = arguments();
        const infllm_score_args &a = j.s;
        constexpr int kKeys = 128 * KS;
        const int rows = a.B * a.H, nth = x / rows, tile = nth == 0 ? j.first_tile : nth - (nth <= j.first_tile);
        int b, h;
        head_of(a, x - nth * rows, b, h);
        const int64_t jg = a.j_lo / (32 * KS) * (32 * KS) + (int64_t)tile * kKeys;
        const int slot = j.slot0 + tile * kKeys;
        const int lo = (int)max(a.j_lo - jg, (int64_t)0), hi = (int)min(a.j_hi - jg, (int64_t)kKeys);
        float sums[KS];
        key_sums<D, KS, true>(a, j.merge.ps, b, h, jg, slot, j.cap, lo, hi, 0, j.win, INFINITY, score_lds, sums);
        const int lane = threadIdx.x & 63;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const int r = (threadIdx.x >> 6) * (32 * KS) + ks * 32 + lane, row = slot + r < j.cap ? slot + r : slot + r - j.cap;
            if (lane < 32 && r >= lo && r < hi) a.d_score[(int64_t)b * a.score_sb + (int64_t)h * a.score_sh + row] += sums[ks];
        }
        return;
    }
    x -= n_score;
    const BlockEnd &j = arguments();
    if (x < j.n_early) {                                          // the first: pages that depend on no selection; the others: the units
        const PageList &pages = j.rank.pages;                     // carved before, for the blocks behind the next
        if (x > 0) rank_block<kRankCpl<D>>(j.rank, x, j.rank.n_before, false, *(RankLds<kRankCpl<D>> *)score_lds);
        else
            for (int e = threadIdx.x, n = pages.n_pages - pages.n_unit_pages; e < n * pages.B; e += 256)
                write_page(pages, e / n, pages.n_unit_pages + e % n, nullptr, nullptr);
        return;
    }
    x -= j.n_early;
    if (x < j.n_copy) carve_copy<D>(j.cc, (int64_t)x * 256 + threadIdx.x);
    else merge_piece<D>(j.merge, (int64_t)(x - j.n_copy) * 256 + threadIdx.x);
}

}  // namespace

namespace {

int check_score_args(const infllm_score_args *a) {
    INFLLM_REQUIRE(a != nullptr, "local_score: null argument block");
    INFLLM_REQUIRE(a->d_q && a->d_k && a->d_lse && a->d_score, "local_score: null pointer");
    INFLLM_REQUIRE(a->B > 0 && a->H > 0 && a->Hkv > 0 && a->H % a->Hkv == 0 && a->Lq > 0,
                   "local_score: bad geometry B=%d H=%d Hkv=%d Lq=%d", a->B, a->H, a->Hkv, a->Lq);
    INFLLM_REQUIRE(a->cap > 0 && a->score_cap > 0 && a->j_lo >= 0, "local_score: bad ring sizes");
    INFLLM_REQUIRE(a->j_hi - a->j_lo <= a->cap && a->j_hi - a->j_lo <= a->score_cap,
                   "local_score: key range [%lld,%lld) exceeds the ring", (long long)a->j_lo, (long long)a->j_hi);
    INFLLM_REQUIRE(a->mask >= 0 && a->mask <= 2, "local_score: unknown mask %d", a->mask);
    INFLLM_REQUIRE(a->n_parts >= 0 && a->n_parts <= 1024, "local_score: %d partial log-sum-exps", a->n_parts);
    INFLLM_REQUIRE((a->q_sl % 8 | a->q_sh % 8 | a->q_sb % 8 | a->k_sl % 8 | a->k_sh % 8 | a->k_sb % 8) == 0,
                   "local_score: strides must be multiples of 8");
    INFLLM_REQUIRE(a->j_hi - a->j_lo <= (int64_t)65000 * 256, "local_score: key range of %lld rows exceeds one launch",
                   (long long)(a->j_hi - a->j_lo));
    return 0;
}

template <int D>
size_t score_lds_bytes(int qs) { return (size_t)(2 * qs * kQPad<D> * sizeof(bf16_t) + 2 * qs * sizeof(float)); }
constexpr int kScoreCus = 256;
constexpr int kMergedMaxLq = 2048;                     // 4 bytes of LDS per query whose log-sum-exps are joined in the launch
template <int D>
int score_lds_setup() {
    static std::atomic<bool> lds_set{false};           // dynamic LDS above 64 KiB must be enabled once per kernel
    if (!lds_set.load(std::memory_order_acquire)) {
        hipError_t e = hipFuncSetAttribute((const void *)local_score_kernel<D, 1, 128>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                           (int)score_lds_bytes<D>(128));
        if (e == hipSuccess)
            e = hipFuncSetAttribute((const void *)local_score_kernel<D, 2, 128>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    (int)score_lds_bytes<D>(128));
        if (e != hipSuccess) return infllm_fail(-2, "local_score: %s", hipGetErrorString(e));
        lds_set.store(true, std::memory_order_release);
    }
    return 0;
}

// Keys of a wave, in 32s.  64 keys halve what a workgroup reads of the queries per key, but a launch of fewer than two
// workgroups per CU is only as fast as one of them: it takes 32 keys a wave and twice the workgroups
// (1,999-token prompt: 172 -> 162 us; 16,001 tokens, whose first blocks see few keys: 3276 -> 3223).
inline bool wide_waves(const infllm_score_args &a) {
    return a.j_hi - a.j_lo > 1024 && (int64_t)a.B * a.H * (((a.j_hi - 1) / 64 - a.j_lo / 64 + 4) / 4) >= 2 * kScoreCus;
}

// What the forms of score.hip that keep positions in 32 bits take.  A query's distance to a key stays below 2^30 then (2^28 between the
// first ones, up to 2^28 queries, a range of keys below 2^24), so that a window of that or more may be cut to it.
constexpr int64_t kMaxRows = 1 << 30;
inline bool in_reach(const infllm_score_args &a) {
    const int64_t apart = a.mask == INFLLM_MASK_NONE ? 0 : a.offset - a.j_lo;
    return (a.cap < kMaxRows || a.j_hi < kMaxRows) && a.Lq < kMaxRows / 4 && a.q_sl >= 0 && a.q_sl < kMaxRows && a.Lq * a.q_sl < kMaxRows &&
           apart > -kMaxRows / 4 && apart < kMaxRows / 4;
}

// job: the log-sum-exps are to be joined (a.n_parts of them), and its merge goes along
template <int D, int FORM, bool MERGE>
int scores_launch(const infllm_score_args &a, const MergeJob *job, float empty, void *stream) {
    constexpr ScoreForm F = kScoreForms[FORM];
    constexpr int wave_keys = 32 * F.ks, threads = 256 * F.groups;
    constexpr size_t q_bytes = (size_t)F.bufs * F.rows * D * sizeof(bf16_t);
    const int gx = a.B * a.H;
    const int64_t tiles = (a.j_hi - 1) / wave_keys - a.j_lo / wave_keys + 1, window = std::min(std::max(a.window, -kMaxRows), kMaxRows);
    const int cap = (int)std::min(a.cap, kMaxRows), slot0 = (int)(a.j_lo % a.cap - a.j_lo % wave_keys);      // (below 0: rows that do not count)
    const int first = (int)(a.mask == INFLLM_MASK_WINDOW ? 0 : a.mask == INFLLM_MASK_COMPLEMENT ? window : -kMaxRows);
    const int beyond = (int)(a.mask == INFLLM_MASK_WINDOW ? std::max<int64_t>(window, 0) : kMaxRows);
    int rows = (int)((tiles + 3) / 4);
    const auto kern = scores_kernel<D, FORM, MERGE>;
    constexpr size_t most = q_bytes + (MERGE ? kMergedMaxLq : F.bufs * F.rows) * sizeof(float);
    if constexpr (most > 65536) {                       // dynamic LDS above 64 KiB must be enabled once per kernel
        static std::atomic<bool> lds_set{false};
        if (!lds_set.load(std::memory_order_acquire)) {
            const hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)most);
            if (e != hipSuccess) return infllm_fail(-2, "local_score: %s", hipGetErrorString(e));
            lds_set.store(true, std::memory_order_release);
        }
    }
    if constexpr (MERGE) {
        const ScoreMerge sm{*job, rows, empty};
        rows += (int)((((int64_t)job->B * job->H * job->Lq * (D / 8) + threads - 1) / threads + gx - 1) / gx);
        INFLLM_REQUIRE(rows <= 65535, "local_score: %d rows of workgroups", rows);
        hipLaunchKernelGGL(kern, dim3(gx, rows), dim3(threads), q_bytes + (size_t)(a.Lq + F.rows - 1) / F.rows * F.rows * sizeof(float), (hipStream_t)stream, a, slot0,
                           cap, first, beyond, sm);
    } else
        hipLaunchKernelGGL(kern, dim3(gx, rows), dim3(threads), q_bytes + F.bufs * F.rows * sizeof(float), (hipStream_t)stream, a, slot0, cap, first, beyond,
                           NoScoreMerge{});
    INFLLM_CHECK_LAUNCH("local_score");
    return 0;
}

// A narrow launch that the chip holds at once at two workgroups a CU (heads of 64: three) lasts as long as its longest workgroup, a
// chain of stages whose waits and pipeline ends weigh as much as their work: it takes twice the waves a workgroup and twice the
// queries a stage.  Beyond that the smaller workgroups fill up better, and few queries are no chain.  (Causal, 32 heads of 128: 500 /
// 1,000 / 1,998 queries 12.1 / 19.5 / 35.0 us, so 10.2 / 15.5 / 28.3; 2,700: 47.6 and 51.4; 200 queries x 2,000 keys 10.6 and 11.1; 36 heads of
// 64: 1,024 / 2,700 / 3,100 16.8 / 39.0 / 44.7 and 12.9 / 34.8 / 50.1; 8 heads of 128: 3,100 47.8 and 34.9.)
template <int D>
inline bool paired_waves(const infllm_score_args &a) {
    return a.Lq >= 256 && (int64_t)a.B * a.H * (((a.j_hi - 1) / 32 - a.j_lo / 32 + 4) / 4) <= (D == 64 ? 3 : 2) * kScoreCus;
}

template <int D, bool MERGE>
int scores_launch(const infllm_score_args &a, const MergeJob *job, float empty, void *stream) {
    if (wide_waves(a)) return scores_launch<D, kWide, MERGE>(a, job, empty, stream);
    if (paired_waves<D>(a)) return scores_launch<D, kPaired, MERGE>(a, job, empty, stream);
    return scores_launch<D, kNarrow, MERGE>(a, job, empty, stream);
}

template <int D>
int score_launch(const infllm_score_args *a, void *stream) {
    int rc = check_score_args(a);
    if (rc) return rc;
    if (a->j_hi <= a->j_lo) return 0;
    if (a->n_parts <= 0 && in_reach(*a)) return scores_launch<D, false>(*a, nullptr, 0.f, stream);
    rc = score_lds_setup<D>();
    if (rc) return rc;
    const bool wide = wide_waves(*a);
    const int64_t tiles = wide ? (a->j_hi - 1) / 64 - a->j_lo / 64 + 1 : (a->j_hi - 1) / 32 - a->j_lo / 32 + 1;
    const auto kern = wide ? local_score_kernel<D, 2, 128> : local_score_kernel<D, 1, 128>;
    hipLaunchKernelGGL(kern, dim3(a->B * a->H, (unsigned)((tiles + 3) / 4)), dim3(256), score_lds_bytes<D>(128), (hipStream_t)stream, *a);
    INFLLM_CHECK_LAUNCH("local_score");
    return 0;
}

template <int D>
int score_launch_merged(const infllm_score_args *a, const MergeJob *job, float empty, void *stream) {
    INFLLM_REQUIRE(a && job, "local_score_merged: null argument");
    INFLLM_REQUIRE(job->B == a->B && job->H == a->H && job->Lq == a->Lq && job->P >= 1 && job->P <= 8,
                   "local_score_merged: the merge does not belong to these queries");
    infllm_score_args sc = *a;
    sc.d_lse = job->lse_part;
    sc.n_parts = job->P;
    const int rc = check_score_args(&sc);
    if (rc) return rc;
    if (sc.j_hi - sc.j_lo <= 1024 || sc.Lq > kMergedMaxLq || !in_reach(sc)) return 1;
    return scores_launch<D, true>(sc, job, empty, stream);
}

}  // namespace

template <int D>
static int block_end_launch(BlockEnd &j, bool scores, hipStream_t st) {
    static_assert(kCarveBytes<D> >= kQBytes<D> && kCarveRows<D> >= kQRows && sizeof(RankLds<kRankCpl<D>>) <= kCarveBytes<D> && kCarveMaxUnit * 16 + 4 <= kCarveBytes<D>, "LDS of a workgroup");
    const infllm_score_args &a = j.s;
    const bool wide = scores && wide_waves(a);
    if (scores) {
        const int wave_keys = wide ? 64 : 32;
        const int64_t tiles = (a.j_hi - 1) / wave_keys - a.j_lo / wave_keys + 1;
        j.n_score = (int32_t)((tiles + 3) / 4 * a.B * a.H);
        j.slot0 = (int32_t)(a.j_lo % a.cap - a.j_lo % wave_keys);       // (below 0: rows that do not count)
        j.first_tile = (int32_t)std::max<int64_t>(0, std::min((a.offset - a.j_lo / wave_keys * wave_keys) / (4 * wave_keys), (tiles + 3) / 4 - 1));
    }
    const int64_t copies = (int64_t)2 * a.B * a.Hkv * j.n_units * j.bs * (D / 8), pieces = j.merge.out ? (int64_t)a.B * a.H * a.Lq * (D / 8) : 0;
    INFLLM_REQUIRE(copies < (1ll << 32), "block_end: copy too large");
    j.n_copy = (int32_t)((copies + 255) / 256);
    const int64_t wgs = (int64_t)j.n_carve + j.n_score + j.n_early + j.n_copy + (pieces + 255) / 256;
    INFLLM_REQUIRE(wgs < (1ll << 31), "block_end: grid too large");
    if (wgs == 0) return 0;
    const auto kern = wide ? block_end_kernel<D, 2> : block_end_kernel<D, 1>;
    hipLaunchKernelGGL(kern, dim3((unsigned)wgs), dim3(256), kCarveBytes<D> + (size_t)(a.Lq + kCarveRows<D> - 1) / kCarveRows<D> * kCarveRows<D> * sizeof(float), st, j);
    INFLLM_CHECK_LAUNCH("block_end");
    return 0;
}

// library-internal: does infllm_block_end take blocks of n queries with P partials and units of bs tokens?
bool infllm_block_end_takes(int32_t n, int32_t P, int32_t bs, bool units, bool ring_is_track) {
    return P <= 8 && n <= kMergedMaxLq && (!units || (n <= kCarveMaxLq && bs % 32 == 0 && bs <= kCarveMaxUnit && ring_is_track));
}

// ... and does it rank units by rows of C elements?
bool infllm_block_end_ranks(int32_t C, int32_t dim) { return C % 8 == 0 && C <= (dim == 64 ? kRankCpl<64> : kRankCpl<128>) * 512; }

// library-internal: the scores of the block's queries (`a`, whose d_lse / n_parts are set from the job's partials) for keys
// [a->j_lo, a->j_hi) unless that is empty, the merge of the job (out NULL: done before), scores and representatives of the n_units
// units of bs tokens from position t0 on, which leave the window behind the block, and their rows to their home (as
// infllm_repr_keys_carve lays them out); and, with rank, the selection of block rank->j0 and its scores of the rank->n_new units,
// and the scores of the first n_before of them under the n_rank - 1 blocks behind it.  (The units carved now get those with the next
// block: the workgroup that finishes last, which the launch waits for, scores for one block only.)
int infllm_block_end(const infllm_score_args *a, const MergeJob *job, const void *d_ring_k_raw, const void *d_ring_v, int64_t t0, int32_t bs, int32_t n_units,
                     int32_t repr_topk, void *d_rep_out, int64_t rep_sb, int64_t rep_su, void *d_out_k, void *d_out_v, int64_t out_sb, int64_t out_su,
                     int64_t out_sh, const RankJob *rank, int32_t n_rank, uint32_t *d_ticket, void *stream, int32_t dim) {
    INFLLM_REQUIRE(a && job, "block_end: null pointer");
    INFLLM_REQUIRE(dim == 128 || dim == 64, "block_end: head_dim %d", dim);
    INFLLM_REQUIRE(infllm_block_end_takes(a->Lq, job->P, bs, n_units > 0, a->cap == a->score_cap) && a->mask == INFLLM_MASK_WINDOW, "block_end: no kernel for this block");
    BlockEnd j{};
    j.s = *a;
    j.s.d_lse = job->lse_part;
    j.s.n_parts = job->P;
    const int rc = check_score_args(&j.s);
    if (rc) return rc;
    INFLLM_REQUIRE(job->B == a->B && job->H == a->H && job->Lq == a->Lq && job->P >= 1, "block_end: the merge does not belong to these queries");
    INFLLM_REQUIRE(a->accumulate && a->cap < (1ll << 30) && (int64_t)a->Lq * a->q_sl < (1ll << 30) && a->j_hi <= a->offset + a->Lq &&
                       a->j_lo >= a->offset - a->cap, "block_end: bad ring or strides");
    j.merge = *job;
    j.cap = (int32_t)a->cap;
    j.win = (int32_t)std::min<int64_t>(a->window, 1 << 30);
    if (n_units > 0) {
        INFLLM_REQUIRE(d_ring_k_raw && d_ring_v && d_rep_out && d_out_k && d_out_v, "block_end: null pointer");
        INFLLM_REQUIRE(repr_topk >= 1 && repr_topk <= bs && t0 >= 0 && (int64_t)n_units * bs <= a->cap, "block_end: bad sizes");
        INFLLM_REQUIRE(t0 + (int64_t)n_units * bs <= a->offset + 1, "block_end: the units reach into the block");
        INFLLM_REQUIRE((rep_sb | rep_su) % 2 == 0 && (out_sb | out_su | out_sh) % 8 == 0, "block_end: bad strides");
        INFLLM_REQUIRE((int64_t)a->H * n_units * a->B < (1ll << 30), "block_end: batch too large");
        j.n_carve = a->H * n_units * a->B;
        j.ring_k_raw = (const bf16_t *)d_ring_k_raw;
        j.t0 = t0; j.unit_slot0 = (int32_t)(t0 % a->cap); j.bs = bs; j.n_units = n_units; j.repr_topk = repr_topk;
        j.rep_out = (bf16_t *)d_rep_out; j.rep_sb = rep_sb; j.rep_su = rep_su;
        CarveCopy &cc = j.cc;
        cc.ring_a = (const bf16_t *)d_ring_k_raw; cc.ring_b = (const bf16_t *)d_ring_v;
        cc.out_a = (bf16_t *)d_out_k; cc.out_b = (bf16_t *)d_out_v;
        cc.ring_cap = j.cap; cc.slot0 = j.unit_slot0; cc.out_sb = out_sb; cc.out_su = out_su; cc.out_sh = out_sh;
        cc.Hkv = a->Hkv; cc.B = a->B; cc.n = n_units * bs; cc.unit_rows = bs;
    }
    if (rank) {
        INFLLM_REQUIRE(infllm_block_end_ranks(rank->C, dim) && n_rank >= 1 && rank->n_new <= 2 * kRankNew && rank->n_before <= rank->n_new && d_ticket, "block_end: no ranking for rows of %d elements", rank->C);
        INFLLM_REQUIRE(rank->n_list + rank->first_new + rank->n_new - rank->n_base <= kRankEntries, "block_end: too many units to rank");
        j.rank = *rank;
        j.ranks = 1;
        j.n_early = 1 + (rank->n_before > 0 ? n_rank - 1 : 0);
        j.ticket = d_ticket;
        j.n_carve = std::max(j.n_carve, 1);                       // (nothing carved: a workgroup that only ranks)
    }
    const bool scores = a->j_hi > a->j_lo;
    return dim == 128 ? block_end_launch<128>(j, scores, (hipStream_t)stream) : block_end_launch<64>(j, scores, (hipStream_t)stream);
}

extern "C" int infllm_local_score(const infllm_score_args *a, void *stream) { return score_launch<kD>(a, stream); }

// library-internal: the same for heads of 128 or 64
int infllm_local_score_dim(const infllm_score_args *a, int32_t dim, void *stream) {
    INFLLM_REQUIRE(dim == 128 || dim == 64, "local_score: head_dim %d", dim);
    return dim == 128 ? score_launch<128>(a, stream) : score_launch<64>(a, stream);
}

// library-internal: the local score of a block and the merge of its partial attention outputs in one launch.  The
// scores are taken against the joint log-sum-exp of the job's partials (a->d_lse and a->n_parts are set from the job);
// returns 1, with nothing launched, where the one-launch form does not apply (short key ranges).
int infllm_local_score_merged(const infllm_score_args *a, const MergeJob *job, void *stream, int32_t dim) {
    INFLLM_REQUIRE(dim == 128 || dim == 64, "local_score: head_dim %d", dim);
    return dim == 128 ? score_launch_merged<128>(a, job, INFINITY, stream) : score_launch_merged<64>(a, job, INFINITY, stream);
}

// ... for the operator: scores and the merge over two sets of partials (P1 + P2 <= 8), heads of 128
int infllm_merge_job(const uint16_t *d_o_part, const float *d_lse_part, int32_t P1, const uint16_t *d_o_part2, const float *d_lse_part2, int32_t P2, int32_t B,
                     int32_t H, int32_t Lq, void *d_out, int64_t o_sb, int64_t o_sh, int64_t o_sl, float *d_lse, MergeJob *job, int32_t dim);
extern "C" int infllm_local_score_merge_pair(const infllm_score_args *a, const uint16_t *d_o_part, const float *d_lse_part, int32_t P1, const uint16_t *d_o_part2,
                                             const float *d_lse_part2, int32_t P2, void *d_out, int64_t o_sb, int64_t o_sh, int64_t o_sl, float *d_lse, void *stream) {
    INFLLM_REQUIRE(a && d_out, "local_score_merge_pair: null pointer");
    if (P1 + P2 > 8 || a->j_hi <= a->j_lo) return 1;
    MergeJob job;
    const int rc = infllm_merge_job(d_o_part, d_lse_part, P1, d_o_part2, d_lse_part2, P2, a->B, a->H, a->Lq, d_out, o_sb, o_sh, o_sl, d_lse, &job, kD);
    return rc ? rc : score_launch_merged<kD>(a, &job, -INFINITY, stream);
}
