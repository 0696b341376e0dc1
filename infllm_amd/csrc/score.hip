// Column sums of the final attention probabilities of one linear stage
// (inf_llm/attention/dot_production_attention/torch_impl.py:27-28): the "local score"
// that InfLLM accumulates per token to choose representative keys
// (inf_llm/attention/context_manager.py:623-625).
//
// It needs the final log-sum-exp of every query, so it runs after the merge and
// recomputes Q.K^T.  Orientation: S[query, key] with keys in the MFMA column, so a lane
// owns one key and the column sum is a running per-lane scalar.  A workgroup owns 256
// consecutive keys of one query head: each of its 4 waves keeps 64 keys in registers
// (B operand) for the whole kernel, while tiles of 64 or 128 queries stream through LDS
// (A operand, shared by the 4 waves, double buffered).  Exactly one lane writes each
// (head, key) cell, so results are deterministic.
#include "carve.h"
#include "rank.h"
#include <algorithm>
#include <atomic>
#include <type_traits>

namespace {

template <int D>
constexpr int kQPad = D + 8;               // LDS row of Q (bf16 elements): 272 (144) bytes rotates the banks

// KS = 32-key halves per wave: 2 for long key ranges; 1 halves the work of a wave per query stage, which is what
// bounds the short launches that sit on the critical path between two blocks.  QS = queries per LDS stage: a short
// launch is a chain of stages that each wait for one global load (there is next to no arithmetic to hide it behind),
// so it takes stages of 128 queries and half as many of them.
//
// MERGE: the launch also carries the merge of the block's partial attention outputs: every scoring workgroup merges
// two (row, 8 dims) pieces per thread (merge_issue / merge_finish of common.h) while it waits for its keys.  The two
// kinds of work do not depend on each other - the scoring workgroups join the partial log-sum-exps themselves, by
// the merge's own arithmetic - and the merge is a handful of loads per thread that are in flight during a wait the
// workgroup has anyway: one launch instead of two on the chain from one block's selection to the next, and no
// workgroups of its own that would queue for the scoring workgroups' places.  In this form the joined log-sum-exps of
// ALL the launch's queries are put into LDS once, in the same wait, instead of stage by stage.
struct ScoreMerge {
    MergeJob job;
    int32_t score_tiles;               // blockIdx.y below this scores, from there on merges
};
// RANK: the launch also ranks the units for the next block (rank.h), in workgroups of their own that are dispatched first:
// a chain of latencies that needs next to nothing of the chip, and that the scores do not depend on
struct ScoreMergeRank : ScoreMerge {
    RankJob rank;
    int32_t rank_slots, n_rank;        // rows of the grid in front that rank; workgroups in them with something to do
};
struct NoScoreMerge {};
constexpr int kScore = 0, kScoreMerge = 1, kScoreMergeRank = 2;

template <int D, int KS, int QS, int WITH = kScore>
__global__ __launch_bounds__(256, 2) void local_score_kernel(
    infllm_score_args a, std::conditional_t<WITH == kScoreMergeRank, ScoreMergeRank, std::conditional_t<WITH == kScoreMerge, ScoreMerge, NoScoreMerge>> sm) {
    constexpr bool MERGE = WITH != kScore;
    constexpr int kWaveKeys = 32 * KS, kKeysPerWg = 4 * kWaveKeys, kQStage = QS;
    int n_tiles = gridDim.y, slot = blockIdx.y;
    PartSets lps{a.n_parts, 0, 0};
    extern __shared__ __attribute__((aligned(16))) char score_lds[];
    if constexpr (WITH == kScoreMergeRank) {
        slot -= sm.rank_slots;
        if (slot < 0) {
            const int x = (int)blockIdx.y * gridDim.x + blockIdx.x;
            if (x < sm.n_rank) rank_block<9>(sm.rank, x, *(RankLds *)score_lds);
            return;
        }
    }
    if constexpr (MERGE) {
        n_tiles = sm.score_tiles;
        if (slot >= n_tiles) {
            merge_piece<D>(sm.job, ((int64_t)(slot - n_tiles) * gridDim.x + blockIdx.x) * 256 + threadIdx.x);
            return;
        }
        lps = sm.job.ps;
    }
    bf16_t(*Qs)[kQStage][kQPad<D>] = (bf16_t(*)[kQStage][kQPad<D>])score_lds;                               // [2][QS][kQPad]
    float(*Ls)[kQStage] = (float(*)[kQStage])(score_lds + 2 * kQStage * kQPad<D> * sizeof(bf16_t));      // [2][QS]
    [[maybe_unused]] float *Lall = (float *)Ls;                                                        // MERGE: [Lq rounded up to QS]

    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int col = lane & 31, grp = lane >> 5;
    const int G = a.H / a.Hkv;
    // blockIdx.x walks the kv heads first, then the query heads of a group: workgroups go to the 8 XCDs round-robin by
    // linear id, so with 8 (16, ...) kv heads the query heads that share a K tile sit behind the same L2 and that tile
    // leaves HBM once instead of once per query head
    const int b = blockIdx.x / a.H, hx = blockIdx.x % a.H, g = hx % a.Hkv, h = g * G + hx / a.Hkv;
    // Workgroups are dispatched x fastest: all heads of one key tile, then the next tile.  The two tiles at either end
    // of a masked key range see only part of the queries and finish early, so they go last: when the grid is a little
    // more than what the chip holds at once, the workgroups that start late are then the short ones.
    // Where the queries are (nearly) as many as the keys, a tile's work falls from the first to the last instead: a CU that
    // takes one of the first half and one of the second gets a long and a short one.
    int tile = slot;
    if (a.mask == INFLLM_MASK_WINDOW && a.Lq >= (a.j_hi - a.j_lo) - (a.j_hi - a.j_lo) / 4)
        tile = slot < (n_tiles + 1) / 2 ? slot : n_tiles - 1 - (slot - (n_tiles + 1) / 2);
    else if (n_tiles >= 6 && a.mask != INFLLM_MASK_NONE)
        tile = slot < n_tiles - 4 ? slot + 2 : slot == n_tiles - 4 ? 1 : slot == n_tiles - 3 ? n_tiles - 2 : slot == n_tiles - 2 ? 0 : n_tiles - 1;
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
        if (!MERGE && tid < kQStage) {
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
        if (!MERGE && tid < kQStage) Ls[buf][tid] = lbuf;
    };

    float colsum[KS] = {};
    if (st_hi > st_lo) load_stage(st_lo);
    if constexpr (MERGE) {
        // joined log-sum-exps of every query of the launch (the per-stage join above for one group of 8 partials)
        const int64_t rows = (int64_t)a.B * a.H * a.Lq;
        const int lq_pad = (a.Lq + kQStage - 1) / kQStage * kQStage;
        for (int i0 = tid; i0 < lq_pad; i0 += 512) {                       // two queries a thread: one trip to memory for 512
            float l8[2][8];
#pragma unroll
            for (int e = 0; e < 2; ++e)
#pragma unroll
                for (int p = 0; p < 8; ++p) l8[e][p] = i0 + e * 256 < a.Lq && p < a.n_parts ? lse[lps.l(p, rows) + i0 + e * 256] : -INFINITY;
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                float m8 = -INFINITY, den = 0.f;
#pragma unroll
                for (int p = 0; p < 8; ++p) m8 = fmaxf(m8, l8[e][p]);
                if (m8 != -INFINITY) {
#pragma unroll
                    for (int p = 0; p < 8; ++p) den += __builtin_amdgcn_exp2f(l8[e][p] - m8);
                }
                if (i0 + e * 256 < lq_pad) Lall[i0 + e * 256] = den > 0.f ? m8 + log2f(den) : INFINITY;              // +inf => probability 0
            }
        }
    }
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
        // operator over 512 queries x (4,608 + 2,624) keys 112.5 -> 106.8 us, a prompt of 131,072 tokens 29,680 -> 28,930.
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
                for (int q4 = 0; q4 < 4; ++q4) l4[pb][q4] = *(const f32x4 *)(MERGE ? &Lall[i0 + qs * 32 + 8 * q4 + 4 * grp] : &Ls[cur][qs * 32 + 8 * q4 + 4 * grp]);
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
constexpr int kMergedMaxLq = 2048;                     // MERGE: 4 bytes of LDS per query of the launch
template <int D>
size_t score_lds_bytes_merged(int qs, int lq) { return (size_t)(2 * qs * kQPad<D> * sizeof(bf16_t) + (size_t)((lq + qs - 1) / qs * qs) * sizeof(float)); }

template <int D>
int score_lds_setup() {
    static std::atomic<bool> lds_set{false};           // dynamic LDS above 64 KiB must be enabled once per kernel
    if (!lds_set.load(std::memory_order_acquire)) {
        hipError_t e = hipFuncSetAttribute((const void *)local_score_kernel<D, 1, 128>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                           (int)score_lds_bytes<D>(128));
        if (e == hipSuccess)
            e = hipFuncSetAttribute((const void *)local_score_kernel<D, 2, 128>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    (int)score_lds_bytes<D>(128));
        for (const void *k : {(const void *)local_score_kernel<D, 2, 128, kScoreMerge>, (const void *)local_score_kernel<D, 2, 128, kScoreMergeRank>,
                              (const void *)local_score_kernel<D, 1, 128, kScoreMerge>, (const void *)local_score_kernel<D, 1, 128, kScoreMergeRank>})
            if (e == hipSuccess) e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)score_lds_bytes_merged<D>(128, kMergedMaxLq));
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

template <int D>
int score_launch(const infllm_score_args *a, void *stream) {
    int rc = check_score_args(a);
    if (rc) return rc;
    if (a->j_hi <= a->j_lo) return 0;
    rc = score_lds_setup<D>();
    if (rc) return rc;
    if (wide_waves(*a)) {
        const int64_t tiles = (a->j_hi - 1) / 64 - a->j_lo / 64 + 1;
        hipLaunchKernelGGL((local_score_kernel<D, 2, 128>), dim3(a->B * a->H, (unsigned)((tiles + 3) / 4)), dim3(256), score_lds_bytes<D>(128),
                           (hipStream_t)stream, *a, NoScoreMerge{});
    } else {
        const int64_t tiles = (a->j_hi - 1) / 32 - a->j_lo / 32 + 1;
        hipLaunchKernelGGL((local_score_kernel<D, 1, 128>), dim3(a->B * a->H, (unsigned)((tiles + 3) / 4)), dim3(256), score_lds_bytes<D>(128),
                           (hipStream_t)stream, *a, NoScoreMerge{});
    }
    INFLLM_CHECK_LAUNCH("local_score");
    return 0;
}

template <int D>
int score_launch_merged(const infllm_score_args *a, const MergeJob *job, void *stream, const RankJob *rank = nullptr, int n_rank = 0) {
    INFLLM_REQUIRE(a && job, "local_score_merged: null argument");
    INFLLM_REQUIRE(job->B == a->B && job->H == a->H && job->Lq == a->Lq && job->P >= 1 && job->P <= 8,
                   "local_score_merged: the merge does not belong to these queries");
    infllm_score_args sc = *a;
    sc.d_lse = job->lse_part;
    sc.n_parts = job->P;
    int rc = check_score_args(&sc);
    if (rc) return rc;
    if (sc.j_hi - sc.j_lo <= 1024 || sc.Lq > kMergedMaxLq) return 1;
    rc = score_lds_setup<D>();
    if (rc) return rc;
    const bool wide = wide_waves(sc);
    const int wave_keys = wide ? 64 : 32;
    const int64_t tiles = (sc.j_hi - 1) / wave_keys - sc.j_lo / wave_keys + 1;
    const int score_tiles = (int)((tiles + 3) / 4);
    const int64_t merge_wgs = ((int64_t)job->B * job->H * job->Lq * (D / 8) + 255) / 256;
    const int gx = sc.B * sc.H;
    const int merge_slots = job->out ? (int)((merge_wgs + gx - 1) / gx) : 0;      // (none: the job has been done by then)
    if (rank) {
        INFLLM_REQUIRE(rank->C <= 9 * 512 && rank->C % 8 == 0 && n_rank >= 1, "local_score_merged: no ranking for rows of %d elements", rank->C);
        ScoreMergeRank sm;
        sm.job = *job;
        sm.score_tiles = score_tiles;
        sm.rank = *rank;
        sm.n_rank = n_rank;
        sm.rank_slots = (n_rank + gx - 1) / gx;
        const auto kern = wide ? local_score_kernel<D, 2, 128, kScoreMergeRank> : local_score_kernel<D, 1, 128, kScoreMergeRank>;
        hipLaunchKernelGGL(kern, dim3(gx, (unsigned)(sm.rank_slots + score_tiles + merge_slots)), dim3(256), score_lds_bytes_merged<D>(128, sc.Lq),
                           (hipStream_t)stream, sc, sm);
        INFLLM_CHECK_LAUNCH("local_score_merged");
        return 0;
    }
    const auto kern = wide ? local_score_kernel<D, 2, 128, kScoreMerge> : local_score_kernel<D, 1, 128, kScoreMerge>;
    hipLaunchKernelGGL(kern, dim3(gx, (unsigned)(score_tiles + merge_slots)), dim3(256), score_lds_bytes_merged<D>(128, sc.Lq), (hipStream_t)stream, sc,
                       ScoreMerge{*job, score_tiles});
    INFLLM_CHECK_LAUNCH("local_score_merged");
    return 0;
}

// The keys that leave the window behind this block: the block's share of their scores, added to what the earlier blocks left
// in the track, and at once the representatives of the units they make up (context_manager.py:268-277) - what the next
// block's retrieval waits for, in one launch in front of the rest of the scores.  A chain of latencies with little work in
// it (a workgroup per unit and head: 128 keys x 512 queries, half of them outside the window), so each step is as short as
// it can be: a wave per sub-tile of 32 queries, whose rows are requested at once together with everything else the kernel
// reads; the unit's keys in LDS (every wave needs them all); a sub-tile's column sums added in the order of the queries, as
// local_score_kernel adds them (the same bits); the picks by counting, all rows at once.  The workgroups behind the heads'
// copy the units' rows to their home and merge the block's partial outputs: independent work for a chip that is half idle.
constexpr int kCarveMaxLq = 512, kCarveMaxUnit = 128;
struct CarveScore {
    infllm_score_args s;
    MergeJob merge;
    const bf16_t *ring_k_raw;
    int32_t slot0, cap, to_first;      // ring row of the first unit; dist of query 0 to the first unit's first key
    int32_t win, bs, n_units, repr_topk;
    bf16_t *rep_out;
    int64_t rep_sb, rep_su;
    CarveCopy cc;
};

template <int D>
__global__ __launch_bounds__(1024) void carve_score_kernel(CarveScore j) {
    constexpr int kChunks = D / 8;
    __shared__ __attribute__((aligned(16))) bf16_t keys[kCarveMaxUnit * D];        // chunk c of row r at c ^ (r mod kChunks)
    __shared__ float lse_sh[kCarveMaxLq];
    __shared__ float sums[kCarveMaxLq / 32][2][kCarveMaxUnit];
    __shared__ uint64_t rank_key[kCarveMaxUnit];
    __shared__ int32_t chosen[kCarveMaxUnit];
    const infllm_score_args &a = j.s;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, col = lane & 31, grp = lane >> 5;
    if ((int)blockIdx.x >= a.H) {
        const int x = (int)blockIdx.x - a.H;
        const int64_t wg = (int64_t)blockIdx.z * gridDim.y + blockIdx.y;
        if (x < j.cc.x_extra) carve_copy<D>(j.cc, (wg * j.cc.x_extra + x) * 1024 + tid);
        else merge_piece<D>(j.merge, (wg * ((int)gridDim.x - a.H - j.cc.x_extra) + (x - j.cc.x_extra)) * 1024 + tid);
        return;
    }
    const int h = blockIdx.x, u = blockIdx.y, b = blockIdx.z, g = h / (a.H / a.Hkv), bs = j.bs;
    const float scale = a.softmax_scale * 1.4426950408889634f;
    auto slot_of = [&](int r) {                                   // ring row of row r of the unit
        const int s = j.slot0 + u * bs + r;
        return s < j.cap ? s : s - j.cap;
    };
    // queries that see any of the unit's keys: i < n_q (they all lie behind the keys), one sub-tile of 32 a wave
    const int d_first = j.to_first - u * bs;                      // distance of query 0 to the unit's first key
    const int n_q = max(min(a.Lq, j.win + bs - 1 - d_first), 0), n_sub = (n_q + 31) / 32;
    const bool works = wave < n_sub;
    bf16x8 qa[D / 16];
    if (works) {
        const bf16_t *row = (const bf16_t *)a.d_q + (int64_t)b * a.q_sb + (int64_t)h * a.q_sh + (int64_t)min(wave * 32 + col, a.Lq - 1) * a.q_sl + grp * 8;
#pragma unroll
        for (int kk = 0; kk < D / 16; ++kk) qa[kk] = __builtin_bit_cast(bf16x8, *(const u32x4 *)(row + kk * 16));
    }
    constexpr int kLoads = kCarveMaxUnit * kChunks / 1024;
    u32x4 k_in[kLoads], raw_in[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
        const int r = (tid + i * 1024) / kChunks, c = tid % kChunks;
        if (r >= bs) continue;
        const int64_t at = (int64_t)slot_of(r);
        k_in[i] = *(const u32x4 *)((const bf16_t *)a.d_k + (int64_t)b * a.k_sb + (int64_t)g * a.k_sh + at * a.k_sl + c * 8);
        raw_in[i] = *(const u32x4 *)(j.ring_k_raw + (((int64_t)b * a.Hkv + g) * j.cap + at) * D + c * 8);
    }
    float track = 0.f;
    if (tid < bs) track = a.d_score[(int64_t)b * a.score_sb + (int64_t)h * a.score_sh + slot_of(tid)];
    if (tid < n_sub * 32) {                                      // joined log-sum-exps (local_score_kernel's join)
        const int64_t rows = (int64_t)a.B * a.H * a.Lq;
        const float *lse = a.d_lse + ((int64_t)b * a.H + h) * a.Lq;
        float l8[8], m8 = -INFINITY, den = 0.f;
#pragma unroll
        for (int p = 0; p < 8; ++p) l8[p] = tid < a.Lq && p < a.n_parts ? lse[j.merge.ps.l(p, rows) + tid] : -INFINITY;
#pragma unroll
        for (int p = 0; p < 8; ++p) m8 = fmaxf(m8, l8[p]);
        if (m8 != -INFINITY) {
#pragma unroll
            for (int p = 0; p < 8; ++p) den += __builtin_amdgcn_exp2f(l8[p] - m8);
        }
        lse_sh[tid] = den > 0.f ? m8 + log2f(den) : INFINITY;    // +inf => probability 0
    }
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
        const int r = (tid + i * 1024) / kChunks, c = tid % kChunks;
        if (r < bs) *(u32x4 *)&keys[(r * kChunks + (c ^ (r % kChunks))) * 8] = k_in[i];
    }
    __syncthreads();
    if (works) {
        f32x4 l4[4];
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) l4[q4] = *(const f32x4 *)&lse_sh[wave * 32 + 8 * q4 + 4 * grp];
        for (int kg = 0; kg < bs / 32; ++kg) {
            const bf16_t *krow = &keys[(kg * 32 + col) * D];
            f32x16 s;
#pragma unroll
            for (int r = 0; r < 16; ++r) s[r] = 0.f;
#pragma unroll
            for (int kk = 0; kk < D / 16; ++kk)
                s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(qa[kk], *(const bf16x8 *)(krow + ((kk * 2 + grp) ^ (col % kChunks)) * 8), s, 0, 0, 0);
            const int e0 = d_first + wave * 32 - kg * 32;        // distance of the sub-tile's first query to the group's first key
            float acc = 0.f;
            if (e0 - 31 >= 0 && e0 + 31 < j.win) {
#pragma unroll
                for (int r = 0; r < 16; ++r) acc += __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], scale, -l4[r >> 2][r & 3]));
            } else {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int dist = e0 - col + 8 * (r >> 2) + 4 * grp + (r & 3);
                    const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], scale, -l4[r >> 2][r & 3]));
                    acc += dist >= 0 && dist < j.win ? p : 0.f;
                }
            }
            sums[wave][grp][kg * 32 + col] = acc;
        }
    }
    __syncthreads();
    // ---- the representatives: row r's place in the order is the number of rows in front of it; the raw keys take the place
    //      of the rotated ones meanwhile
#pragma unroll
    for (int i = 0; i < kLoads; ++i)
        if ((tid + i * 1024) / kChunks < bs) *(u32x4 *)&keys[(tid + i * 1024) * 8] = raw_in[i];
    if (tid < kCarveMaxUnit) {
        uint64_t key = 0;
        if (tid < bs) {
            float lo = 0.f, hi = 0.f;
            if (n_sub == kCarveMaxLq / 32) {
#pragma unroll
                for (int st = 0; st < kCarveMaxLq / 32; ++st) lo += sums[st][0][tid], hi += sums[st][1][tid];
            } else {
#pragma unroll 4
                for (int st = 0; st < n_sub; ++st) lo += sums[st][0][tid], hi += sums[st][1][tid];
            }
            key = pick_key(track + (lo + hi), tid);
        }
        rank_key[tid] = key;
    }
    __syncthreads();
    {
        const int r = tid >> 3, p = tid & 7;
        const uint64_t own = rank_key[r];
        int before = 0;
#pragma unroll
        for (int i = 0; i < kCarveMaxUnit / 8; ++i) before += rank_key[i * 8 + p] > own;
#pragma unroll
        for (int o = 1; o < 8; o <<= 1) before += __shfl_xor(before, o, 64);
        if (p == 0 && r < bs && before < j.repr_topk) chosen[before] = r;
    }
    __syncthreads();
    if (tid * 2 >= D) return;
    float a0 = 0.f, a1 = 0.f;
    for (int i = 0; i < j.repr_topk; ++i) {
        const uint32_t w = *(const uint32_t *)&keys[chosen[i] * D + tid * 2];
        a0 += bf16_bits_to_f32(w & 0xffffu);
        a1 += bf16_bits_to_f32(w >> 16);
    }
    const float inv = 1.f / (float)j.repr_topk;
    *(uint32_t *)(j.rep_out + (int64_t)b * j.rep_sb + (int64_t)u * j.rep_su + (int64_t)h * D + tid * 2) = pack_bf16x2(a0 * inv, a1 * inv);
}

}  // namespace

// library-internal: scores and representatives of the n_units units of bs tokens from position t0 on, which leave the
// window behind the block of `a` (whose d_lse / n_parts are set from the job's partials), their rows to their home (as
// infllm_repr_keys_carve lays them out), and the job itself, the merge of the block's partials (job->out NULL: none).  Returns 1, with nothing
// launched, for units or blocks the kernel does not take.
int infllm_carve_score(const infllm_score_args *a, const MergeJob *job, const void *d_ring_k_raw, const void *d_ring_v, int64_t t0, int32_t bs, int32_t n_units,
                       int32_t repr_topk, void *d_rep_out, int64_t rep_sb, int64_t rep_su, void *d_out_k, void *d_out_v, int64_t out_sb, int64_t out_su,
                       int64_t out_sh, void *stream, int32_t dim) {
    INFLLM_REQUIRE(a && job && d_ring_k_raw && d_ring_v && d_rep_out && d_out_k && d_out_v, "carve_score: null pointer");
    INFLLM_REQUIRE(dim == 128 || dim == 64, "carve_score: head_dim %d", dim);
    if (n_units == 0) return 0;
    if (bs % 32 != 0 || bs > kCarveMaxUnit || a->Lq > kCarveMaxLq || job->P > 8 || a->mask != INFLLM_MASK_WINDOW || a->cap != a->score_cap) return 1;
    CarveScore j{};
    j.s = *a;
    j.s.d_lse = job->lse_part;
    j.s.n_parts = job->P;
    const int rc = check_score_args(&j.s);
    if (rc) return rc;
    INFLLM_REQUIRE(repr_topk >= 1 && repr_topk <= bs && n_units > 0 && t0 >= 0 && (int64_t)n_units * bs <= a->cap && n_units <= 65535 && a->B <= 65535,
                   "carve_score: bad sizes");
    INFLLM_REQUIRE(t0 + (int64_t)n_units * bs <= a->offset + 1, "carve_score: the units reach into the block");
    INFLLM_REQUIRE((rep_sb | rep_su) % 2 == 0 && (out_sb | out_su | out_sh) % 8 == 0, "carve_score: bad strides");
    INFLLM_REQUIRE(job->B == a->B && job->H == a->H && job->Lq == a->Lq && job->P >= 1, "carve_score: the merge does not belong to these queries");
    INFLLM_REQUIRE(a->cap < (1ll << 30), "carve_score: ring too large");
    j.merge = *job;
    j.ring_k_raw = (const bf16_t *)d_ring_k_raw;
    j.slot0 = (int32_t)(t0 % a->cap); j.cap = (int32_t)a->cap; j.bs = bs; j.n_units = n_units; j.repr_topk = repr_topk;
    j.to_first = (int32_t)std::min<int64_t>(a->offset - t0, 1 << 29);
    j.win = (int32_t)std::min<int64_t>(a->window, 1 << 28);
    j.rep_out = (bf16_t *)d_rep_out; j.rep_sb = rep_sb; j.rep_su = rep_su;
    CarveCopy &cc = j.cc;
    cc.ring_a = (const bf16_t *)d_ring_k_raw; cc.ring_b = (const bf16_t *)d_ring_v;
    cc.out_a = (bf16_t *)d_out_k; cc.out_b = (bf16_t *)d_out_v;
    cc.ring_cap = j.cap; cc.slot0 = j.slot0; cc.out_sb = out_sb; cc.out_su = out_su; cc.out_sh = out_sh;
    cc.Hkv = a->Hkv; cc.B = a->B; cc.n = n_units * bs; cc.unit_rows = bs;
    const int64_t per_x = (int64_t)n_units * a->B, elems = (int64_t)2 * a->B * a->Hkv * cc.n * (dim / 8), pieces = (int64_t)a->B * a->H * a->Lq * (dim / 8);
    INFLLM_REQUIRE(elems < (1ll << 32), "carve_score: copy too large");
    cc.x_extra = (int32_t)(((elems + 1023) / 1024 + per_x - 1) / per_x);
    const int32_t x_merge = job->out ? (int32_t)(((pieces + 1023) / 1024 + per_x - 1) / per_x) : 0;
    const dim3 grid(a->H + cc.x_extra + x_merge, n_units, a->B);
    if (dim == 128) hipLaunchKernelGGL(carve_score_kernel<128>, grid, dim3(1024), 0, (hipStream_t)stream, j);
    else hipLaunchKernelGGL(carve_score_kernel<64>, grid, dim3(1024), 0, (hipStream_t)stream, j);
    INFLLM_CHECK_LAUNCH("carve_score");
    return 0;
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
    return dim == 128 ? score_launch_merged<128>(a, job, stream) : score_launch_merged<64>(a, job, stream);
}
// ... and with the next block's ranking in n_rank workgroups
int infllm_local_score_merged_rank(const infllm_score_args *a, const MergeJob *job, const RankJob *rank, int32_t n_rank, void *stream, int32_t dim) {
    INFLLM_REQUIRE(rank && (dim == 128 || dim == 64), "local_score: bad ranking");
    return dim == 128 ? score_launch_merged<128>(a, job, stream, rank, n_rank) : score_launch_merged<64>(a, job, stream, rank, n_rank);
}
