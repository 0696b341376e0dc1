// The streaming memory with every unit resident in HBM: a whole append() call as launches that follow each other on the
// stream without the host in between (inf_llm/attention/context_manager.py:474-545, 614-679, 682-813).
//
// A block's selection decides which units its global stage reads.  When units live in host memory the host has to see the
// ids, run the residency policy and start copies (stream.hip).  When every unit has a home in HBM - 512 KiB per unit and
// layer at the reference geometry, of 288 GB - the selection only has to become addresses: the kernel that ranks the units
// writes the global stage's page table itself, and the host enqueues block after block.  The residency policy (which unit
// would sit in which of max_cached_block slots) no longer moves data; its bookkeeping follows the selections as they arrive
// in a pinned log.
//
// A call of several queries: prologue of all its tokens, mean queries, the k best of the units that exist for every
// block's mean query (one pass), the local stage of all blocks; then per block the global stage, and one launch for merge, local
// score, the units it carves (representatives, rows into their home) and the ranking for the next block.  A single query (a decode
// step): prologue with the units' scores, one streaming attention launch over window, units, sinks and remainder, and one that joins
// its splits and adds the probabilities to the window's score track - no second read of the window's keys.
#include <algorithm>
#include <atomic>
#include <chrono>
#include <vector>

#include "decode.h"
#include "rank.h"

int infllm_reduce_partials_blocks(const float *d_parts, int32_t B, int32_t n, int32_t exc, int32_t C, float *d_out, void *stream);
int infllm_attn_stage_blocked(const infllm_attn_args *a, int32_t exc, int64_t block_rows, void *stream, int32_t dim);
int infllm_attn_paged(const infllm_attn_args *a, const infllm_page *h_pages, void *stream, int32_t dim);
int infllm_inline_page_limit();
int infllm_merge_job(const uint16_t *d_o_part, const float *d_lse_part, int32_t P1, const uint16_t *d_o_part2, const float *d_lse_part2,
                     int32_t P2, int32_t B, int32_t H, int32_t Lq, void *d_out, int64_t o_sb, int64_t o_sh, int64_t o_sl, float *d_lse,
                     MergeJob *job, int32_t dim);
int infllm_attn_merge2(const uint16_t *d_o_part, const float *d_lse_part, int32_t P1, const uint16_t *d_o_part2, const float *d_lse_part2,
                       int32_t P2, int32_t B, int32_t H, int32_t Lq, void *d_out, int64_t o_sb, int64_t o_sh, int64_t o_sl, float *d_lse,
                       void *stream, int32_t dim);
int infllm_attn_merge_blocked(const uint16_t *d_o_part, const float *d_lse_part, int32_t P, int32_t B, int32_t H, int32_t n, int32_t exc, int64_t block_rows,
                              void *d_out, int64_t o_sb, int64_t o_sh, int64_t o_sl, float *d_lse, void *stream, int32_t dim);
int infllm_local_score_dim(const infllm_score_args *a, int32_t dim, void *stream);
int infllm_local_score_merged(const infllm_score_args *a, const MergeJob *job, void *stream, int32_t dim);
bool infllm_block_end_takes(int32_t n, int32_t P, int32_t bs, bool units, bool ring_is_track);
bool infllm_block_end_ranks(int32_t C, int32_t dim);
int infllm_block_end(const infllm_score_args *a, const MergeJob *job, const void *d_ring_k_raw, const void *d_ring_v, int64_t t0, int32_t bs, int32_t n_units,
                     int32_t repr_topk, void *d_rep_out, int64_t rep_sb, int64_t rep_su, void *d_out_k, void *d_out_v, int64_t out_sb, int64_t out_su,
                     int64_t out_sh, const RankJob *rank, int32_t n_rank, uint32_t *d_ticket, void *stream, int32_t dim);
int infllm_repr_keys_carve(const float *d_ring_score, const void *d_ring_k_raw, int64_t ring_cap, int32_t B, int32_t H, int32_t Hkv,
                           int64_t t0, int32_t bs, int32_t n_units, int32_t repr_topk, void *d_rep_out, int64_t rep_sb, int64_t rep_su,
                           int32_t *d_idx_out, const void *d_ring_v, void *d_out_k, void *d_out_v, int64_t out_sb, int64_t out_su,
                           int64_t out_sh, void *stream, int32_t dim);
int infllm_gather_rows_pair(const void *d_ring_a, void *d_out_a, const void *d_ring_b, void *d_out_b, int64_t ring_cap, int32_t B,
                            int32_t Hkv, int64_t t0, int32_t n, int32_t unit_rows, int64_t out_sb, int64_t out_su, int64_t out_sh,
                            void *stream, int32_t dim);
int infllm_step_scores(const void *d_reps, int64_t rep_stride, int32_t N, const infllm_ingest_args *in, int32_t dim, int32_t b, bool prologue, float *d_scores,
                       void *stream);
int infllm_key_splits(const infllm_layer_desc *d, int32_t n_queries, int32_t n_tiles);

namespace {

template <int CPL>
__global__ __launch_bounds__(256) void rank_kernel(RankJob jb) {
    __shared__ __attribute__((aligned(16))) RankLds<CPL> lds;
    rank_block<CPL>(jb, blockIdx.x, jb.n_new, true, lds);
}

// the page table of a block that attends every unit, where the attention's launch does not hold it
__global__ __launch_bounds__(256) void pages_kernel(PageList j) {
    const int p = blockIdx.x * 256 + threadIdx.x;
    if (p < j.n_pages) write_page(j, blockIdx.y, p, nullptr, j.chunk);
}

// The end of a decode step: output rows = the joined splits; the window's score track += the probabilities, from the
// logits that the attention launch left behind; and the number of the step in the host's log, where the attention that selected the
// units has left their ids.  Of a selection that launches of its own made (more units or longer rows than a step's scores take, one split) the
// ids are copied there too.
// grid (B * H, 1 + ceil(window / 1024)): y == 0 joins, the others score.  A handful of loads per thread and nothing else, so
// all of them are requested before the first is waited for (32 heads, 64 splits: 11.4 -> 6 us with the splits' rows as
// 16-byte pieces, one batch instead of a chain of four).
struct FinishJob {
    const _Float16 *o_part;
    const float *lse_part;
    int32_t P, B, H;
    bf16_t *out;
    int64_t o_sb, o_sh;
    const float *logits;                   // [B, H, logit_stride]
    int64_t logit_stride;
    float *score;                          // [B, H, ring_cap]
    int32_t ring_cap, slot0;               // ring row of the window's first key
    int32_t n;                             // keys of the window
    const int32_t *ids;                    // the selection [n_ids] (NULL: it is in the log already) and its log slot, a sequence number behind
                                           // them; log NULL: none
    int32_t *log;
    int32_t n_ids, seq;
};

template <int D>
__global__ __launch_bounds__(256) void decode_finish_kernel(FinishJob j) {
    constexpr int kPieces = D / 8, kGroups = 256 / kPieces, kMaxParts = 64, kMine = kMaxParts / kGroups;
    __shared__ float w_sh[kMaxParts];
    __shared__ __attribute__((aligned(16))) float part[kGroups][D];
    const int tid = threadIdx.x, lane = tid & 63, rh = blockIdx.x;
    const int64_t rows = (int64_t)j.B * j.H;
    const float l0 = lane < j.P ? j.lse_part[lane * rows + rh] : -INFINITY;
    // joint log-sum-exp: every wave for itself
    float e0 = 0.f, m = 0.f, den = 0.f;
    auto join = [&]() {
        m = l0;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
        e0 = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(l0 - m);
        den = e0;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) den += __shfl_xor(den, o, 64);
    };
    if (blockIdx.y > 0) {
        constexpr int kPer = 4;
        const int y0 = ((int)blockIdx.y - 1) * 1024;
        const float *logit = j.logits + (int64_t)rh * j.logit_stride;
        float *score = j.score + (int64_t)rh * j.ring_cap;
        float x[kPer], old[kPer];
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            const int k = y0 + i * 256 + tid;
            if (k >= j.n) continue;
            const int at = j.slot0 + k;
            x[i] = logit[k];
            old[i] = score[at < j.ring_cap ? at : at - j.ring_cap];
        }
        join();
        const float lse = den > 0.f ? m + log2f(den) : INFINITY;
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            const int k = y0 + i * 256 + tid, at = j.slot0 + k;
            if (k < j.n) score[at < j.ring_cap ? at : at - j.ring_cap] = old[i] + __builtin_amdgcn_exp2f(x[i] - lse);
        }
        return;
    }
    const int c = tid % kPieces, q = tid / kPieces;
    f16x8 o[kMine];
#pragma unroll
    for (int i = 0; i < kMine; ++i) {
        const int p = q + i * kGroups;
        o[i] = p < j.P ? *(const f16x8 *)(j.o_part + ((int64_t)p * rows + rh) * D + c * 8) : f16x8{0, 0, 0, 0, 0, 0, 0, 0};
    }
    // The log is the host's memory: stores there, and the fence behind them, were what the launch ended with.  Where the launch in front has
    // stored the ids there is nothing to wait for.  (One token behind 512K tokens 29.4 -> 28.0 us a pass.)
    const bool logs = rh == 0 && j.log;
    if (logs && !j.ids && tid == 0) __hip_atomic_store(j.log + j.n_ids, j.seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    if (logs && j.ids)
        for (int i = tid; i < j.n_ids; i += 256) __hip_atomic_store(j.log + i, j.ids[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    join();
    if (tid < 64) w_sh[lane] = e0;
    __syncthreads();
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < kMine; ++i) {
        const float w = w_sh[q + i * kGroups];
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] += (float)o[i][e] * w;
    }
    *(f32x4 *)&part[q][c * 8] = f32x4{acc[0], acc[1], acc[2], acc[3]};
    *(f32x4 *)&part[q][c * 8 + 4] = f32x4{acc[4], acc[5], acc[6], acc[7]};
    __syncthreads();
    if (tid < D / 2) {
        float lo = 0.f, hi = 0.f;
#pragma unroll
        for (int i = 0; i < kGroups; ++i) lo += part[i][2 * tid], hi += part[i][2 * tid + 1];
        const float inv = den > 0.f ? 1.f / den : 0.f;
        *(uint32_t *)(j.out + (int64_t)(rh / j.H) * j.o_sb + (int64_t)(rh % j.H) * j.o_sh + tid * 2) = pack_bf16x2(lo * inv, hi * inv);
    }
    if (logs && j.ids) {                                         // (written through to the host's memory: a fence would write the whole L2 back)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (tid == 0) __hip_atomic_store(j.log + j.n_ids, j.seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

struct Timer {
    std::vector<hipEvent_t> ev;
    std::vector<int> n_queries, n_keys;
    int used = 0, seen = 0;
};

struct Resident {
    infllm_resident_desc d;
    int64_t length = 0, cursor = 0;
    int32_t init_len = 0, n_units = 0;
    // selections whose bookkeeping is still to be done, oldest first: every unit of the first `all` (>= 0), or what log slot
    // `slot` holds once its sequence number is `seq`
    struct Entry {
        int32_t all, slot, seq;
    };
    std::vector<Entry> queue;
    size_t head = 0;
    int32_t next_seq = 0;
    int32_t slots_used = 0;
    int64_t hits = 0, misses = 0, evictions = 0, blocks = 0, ranked = 0;
    Timer timer[3];
    int timing_cap = 0, timing_stride = 1;
    hipStream_t last_stream = nullptr;
};

#define HIP_OK(call, what)                                                              \
    do {                                                                                \
        hipError_t e_ = (call);                                                         \
        if (e_ != hipSuccess) return infllm_fail(-2, "%s: %s", what, hipGetErrorString(e_)); \
    } while (0)

int timer_begin(Resident *R, int which, int n_queries, int n_keys, hipStream_t st) {
    Timer &t = R->timer[which];
    if (R->timing_cap <= 0 || t.used >= R->timing_cap || t.seen++ % R->timing_stride) return -1;
    const int i = t.used++;
    t.n_queries[i] = n_queries;
    t.n_keys[i] = n_keys;
    (void)hipEventRecord(t.ev[2 * i], st);
    return i;
}
void timer_end(Resident *R, int which, int i, hipStream_t st) {
    if (i >= 0) (void)hipEventRecord(R->timer[which].ev[2 * i + 1], st);
}

// ---- the residency bookkeeping of the selections that have arrived (wait: of all)
int drain(Resident *R, bool wait) {
    const infllm_resident_desc &d = R->d;
    const int stride = d.B * std::max(d.topk, 1) + 1;
    int32_t ids[64], slots[64], mu[64], ms[64];
    std::vector<int32_t> ev(d.max_cached);
    while (R->head < R->queue.size()) {
        const Resident::Entry &e = R->queue[R->head];
        int n = e.all;
        const int32_t *log = nullptr;
        if (e.all < 0) {
            log = d.h_log + (int64_t)e.slot * stride;
            const volatile int32_t *flag = log + stride - 1;
            if (*flag != e.seq) {
                if (!wait) break;
                HIP_OK(hipStreamSynchronize(R->last_stream), "resident: wait for a selection");
                if (*flag != e.seq) HIP_OK(hipDeviceSynchronize(), "resident: wait for a selection");      // (it was made on another stream)
                INFLLM_REQUIRE(*flag == e.seq, "resident: a selection did not arrive");
            }
            std::atomic_thread_fence(std::memory_order_acquire);
            n = d.topk;
            --R->slots_used;
        }
        for (int u = 0; u < d.B; ++u) {
            for (int i = 0; i < n; ++i) ids[i] = log ? log[(int64_t)u * d.topk + i] : i;
            int32_t n_ev = 0;
            const int m = infllm_cache_touch(d.h_caches[u], ids, n, slots, mu, ms, ev.data(), &n_ev);
            if (m < 0) return m;
            R->hits += n - m;
            R->misses += m;
            R->evictions += n_ev;
        }
        ++R->head;
    }
    if (R->head == R->queue.size()) {
        R->queue.clear();
        R->head = 0;
    }
    return 0;
}

// a log slot for a selection: waits for the oldest when all are on their way (the stream is that many blocks behind)
int take_slot(Resident *R, int32_t *slot, int32_t *seq) {
    if (R->slots_used >= R->d.log_slots) {
        int rc = drain(R, false);
        if (rc) return rc;
        if (R->slots_used >= R->d.log_slots) {
            rc = drain(R, true);
            if (rc) return rc;
        }
    }
    *seq = ++R->next_seq;
    *slot = (int32_t)((uint32_t)*seq % (uint32_t)R->d.log_slots);
    ++R->slots_used;
    R->queue.push_back(Resident::Entry{-1, *slot, *seq});
    return 0;
}

struct Carve {
    int32_t take, count;                   // init tokens peeled, units carved
};
// the state machine behind a block that ends at b1 (context_manager.py:614-679)
Carve carve_after(const infllm_resident_desc &d, int64_t cursor, int32_t init_len, int64_t b1) {
    int64_t live = b1 - cursor;
    Carve c{0, 0};
    if (init_len < d.n_init && live > d.n_local) {
        c.take = (int32_t)std::min<int64_t>(d.n_init - init_len, live - d.n_local);
        live -= c.take;
    }
    c.count = (int32_t)std::max<int64_t>((live - d.n_local) / d.block_size, 0);
    return c;
}

bf16_t *unit_home(const Resident *R, const infllm_resident_call *a, int unit) {
    const infllm_resident_desc &d = R->d;
    const int ch = unit / d.units_per_chunk;
    return (bf16_t *)(uintptr_t)a->h_chunks[ch] + (int64_t)(unit - ch * d.units_per_chunk) * d.B * 2 * d.Hkv * d.block_size * d.dim;
}

PageList page_list(const Resident *R, const infllm_resident_call *a, int n_sel, int64_t b1) {
    const infllm_resident_desc &d = R->d;
    PageList j{};
    j.out = d.d_pages;
    j.tiles_per_unit = (d.block_size + kTile - 1) / kTile;
    j.n_unit_pages = n_sel * j.tiles_per_unit;
    j.n_init_pages = (R->init_len + kTile - 1) / kTile;
    j.cursor = R->cursor;
    j.overflow_end = std::max(b1 - d.n_local, R->cursor);
    int over = 0;
    for (int64_t pos = j.cursor; pos < j.overflow_end; ++over)
        pos += std::min(std::min(j.overflow_end - pos, (int64_t)kTile), d.ring_cap - pos % d.ring_cap);
    j.n_pages = j.n_unit_pages + j.n_init_pages + over;
    j.Hkv = d.Hkv; j.bs = d.block_size; j.init_len = R->init_len; j.dim = d.dim;
    j.ring_cap = d.ring_cap; j.init_cap = d.init_cap;
    j.init_kv = (const bf16_t *)d.d_init_kv; j.ring_k = (const bf16_t *)d.d_ring_k_raw; j.ring_v = (const bf16_t *)d.d_ring_v;
    j.chunk = a->d_chunks; j.per_chunk = d.units_per_chunk; j.B = d.B; j.n_chunks = a->n_chunks;
    return j;
}

int launch_rank(Resident *R, const RankJob &jb, int n_wgs, hipStream_t st) {
    const int cpl = (jb.C + 511) / 512;
    INFLLM_REQUIRE(jb.C % 8 == 0 && cpl <= 16 && jb.n_new <= 2 * kRankNew && jb.n_list + jb.first_new + jb.n_new - jb.n_base <= kRankEntries,
                   "resident: no ranking for rows of %d elements, %d new units", jb.C, jb.n_new);
#define RANK(n) hipLaunchKernelGGL(rank_kernel<n>, dim3(n_wgs), dim3(256), 0, st, jb)
    if (cpl <= 1) RANK(1);
    else if (cpl <= 2) RANK(2);
    else if (cpl <= 4) RANK(4);
    else if (cpl <= 5) RANK(5);
    else if (cpl <= 8) RANK(8);
    else if (cpl <= 9) RANK(9);
    else RANK(16);
#undef RANK
    INFLLM_CHECK_LAUNCH("rank");
    return 0;
}

infllm_ingest_args ingest_args(const Resident *R, const infllm_resident_call *a, int64_t st, int n) {
    const infllm_resident_desc &d = R->d;
    infllm_ingest_args in{};
    in.d_q = (const bf16_t *)a->d_q + st * a->q_sl; in.d_k = (const bf16_t *)a->d_k + st * a->k_sl; in.d_v = (const bf16_t *)a->d_v + st * a->v_sl;
    in.q_sb = a->q_sb; in.q_sh = a->q_sh; in.q_sl = a->q_sl;
    in.k_sb = a->k_sb; in.k_sh = a->k_sh; in.k_sl = a->k_sl;
    in.v_sb = a->v_sb; in.v_sh = a->v_sh; in.v_sl = a->v_sl;
    in.B = d.B; in.H = d.H; in.Hkv = d.Hkv; in.n = n;
    in.pos0 = R->length; in.glb_pos = d.n_local - 1;
    in.d_inv_freq = d.d_inv_freq; in.distance_scale = d.distance_scale;
    in.d_ring_k_raw = d.d_ring_k_raw; in.d_ring_k_rot = d.d_ring_k_rot; in.d_ring_v = d.d_ring_v;
    in.d_ring_score = d.d_ring_score; in.ring_cap = d.ring_cap;
    in.d_q_loc = a->d_q_loc; in.d_q_glb = a->d_q_glb;
    return in;
}

// Init tokens that leave the window behind a block.
int carve_init(Resident *R, const Carve &c, hipStream_t st) {
    if (c.take <= 0) return 0;
    const infllm_resident_desc &d = R->d;
    INFLLM_REQUIRE(R->init_len + c.take <= d.init_cap, "resident: init overflow");
    bf16_t *ik = (bf16_t *)d.d_init_kv + (int64_t)R->init_len * d.dim;
    const int64_t sh = d.init_cap * d.dim, sb = 2 * (int64_t)d.Hkv * sh;
    const int rc = infllm_gather_rows_pair(d.d_ring_k_raw, ik, d.d_ring_v, ik + (int64_t)d.Hkv * sh, d.ring_cap, d.B, d.Hkv, R->cursor, c.take, c.take, sb, 0,
                                           sh, st, d.dim);
    if (rc) return rc;
    R->cursor += c.take;
    R->init_len += c.take;
    return 0;
}

// Units that one launch carves: those from position t0 on, at most n and of one chunk.  The state moves on behind them.
struct UnitRun {
    int32_t n = 0;
    int64_t t0 = 0;
    bf16_t *rep = nullptr, *home_k = nullptr, *home_v = nullptr;
};
int next_run(Resident *R, const infllm_resident_call *a, int n, UnitRun *run) {
    const infllm_resident_desc &d = R->d;
    *run = UnitRun{};
    if (n <= 0) return 0;
    const int unit = R->n_units;
    run->n = std::min(n, d.units_per_chunk - unit % d.units_per_chunk);
    INFLLM_REQUIRE(unit + run->n <= a->n_chunks * d.units_per_chunk && unit + run->n <= a->rep_rows, "resident: no room for unit %d", unit + run->n - 1);
    run->t0 = R->cursor;
    run->rep = (bf16_t *)a->d_reps + unit * a->rep_su;
    run->home_k = unit_home(R, a, unit);
    run->home_v = run->home_k + (int64_t)d.Hkv * d.block_size * d.dim;
    R->cursor += (int64_t)run->n * d.block_size;
    R->n_units += run->n;
    return 0;
}

// Init tokens and units that leave the window, with scores that are complete.
int carve(Resident *R, const infllm_resident_call *a, const Carve &c, hipStream_t st) {
    const infllm_resident_desc &d = R->d;
    int rc = carve_init(R, c, st);
    const int64_t unit_elems = (int64_t)d.Hkv * d.block_size * d.dim;
    UnitRun run;
    for (int done = 0; done < c.count && !rc; done += run.n) {
        rc = next_run(R, a, c.count - done, &run);
        if (rc) return rc;
        rc = infllm_repr_keys_carve(d.d_ring_score, d.d_ring_k_raw, d.ring_cap, d.B, d.H, d.Hkv, run.t0, d.block_size, run.n, d.repr_topk, run.rep, a->rep_sb,
                                    a->rep_su, nullptr, d.d_ring_v, run.home_k, run.home_v, 2 * unit_elems, (int64_t)d.B * 2 * unit_elems,
                                    (int64_t)d.block_size * d.dim, st, d.dim);
        if (rc > 0) return infllm_fail(-2, "resident: no carving kernel after the checks");
    }
    return rc;
}

// One query.  A step that selects takes the scores of all units, with the prologue, then the attention, which selects, then the end
// of the step; a step that attends all units has the prologue with the attention (two launches for three: 4 us of a prompt of 1,999
// tokens, whose last token is one).
int decode_step(Resident *R, const infllm_resident_call *a, int64_t st0, hipStream_t st) {
    const infllm_resident_desc &d = R->d;
    const int C = d.H * d.dim, N = R->n_units, B = d.B;
    const int64_t b0 = R->length, b1 = b0 + 1;
    const infllm_ingest_args in = ingest_args(R, a, st0, 1);
    const bool retrieve = N > d.topk;
    const int n_sel = std::min(N, d.topk);
    DecodeJob j{};
    j.q[0] = (const bf16_t *)a->d_q_loc; j.q[1] = (const bf16_t *)a->d_q_glb;
    j.q_sb = C; j.q_sh = d.dim;
    j.B = B; j.H = d.H; j.Hkv = d.Hkv;
    j.scale = d.softmax_scale;
    j.nsplit = (int32_t)std::min<int64_t>(64, a->part_rows / ((int64_t)B * d.H));
    FinishJob f{};
    int rc = 0;
    bool selects = false;                                        // the attention does, from scores
    if (retrieve) {
        int32_t slot = 0;
        rc = take_slot(R, &slot, &f.seq);
        if (rc) return rc;
        f.log = d.d_log + (int64_t)slot * (B * d.topk + 1);
        f.ids = d.d_ids; f.n_ids = B * d.topk;
        selects = j.nsplit >= 2;
        for (int u = 0; u < B && selects; ++u) {                  // the prologue rides with the first row's scores
            rc = infllm_step_scores((const bf16_t *)a->d_reps + (int64_t)u * a->rep_sb, a->rep_su, N, &in, d.dim, u, u == 0,
                                    a->d_unit_scores + (int64_t)u * a->unit_scores_sb, st);
            if (rc < 0) return rc;
            if (rc == 1) selects = false;                         // (of all rows or of none: it depends on their length and number)
        }
        if (!selects) {
            rc = infllm_ingest_dim(&in, d.dim, a->d_qbar, st);
            for (int u = 0; u < B && !rc; ++u) {
                const bf16_t *reps = (const bf16_t *)a->d_reps + (int64_t)u * a->rep_sb;
                float *scores = a->d_unit_scores + (int64_t)u * a->unit_scores_sb;
                rc = infllm_unit_scores(reps, a->rep_su, 0, N, C, a->d_qbar + (int64_t)u * C, scores, st);
                if (!rc) rc = infllm_topk(scores, N, d.topk, d.d_ids + (int64_t)u * d.topk, st);
            }
            if (rc) return rc;
        }
    } else
        R->queue.push_back(Resident::Entry{n_sel, 0, 0});
    const bool rides = !retrieve && B <= 32767;                  // the prologue with the attention (whose grid holds 65,535 batch rows)
    if (!retrieve && !rides) {
        rc = infllm_ingest_dim(&in, d.dim, nullptr, st);
        if (rc) return rc;
    }
    int64_t blocks = 0;
    auto seg = [&](const void *k, const void *v, int64_t sb, int64_t sh, int64_t rows, int q, int logit0) {
        j.seg[j.n_seg++] = DecodeSeg{(const bf16_t *)k, (const bf16_t *)v, sb, sh, sb, sh, (int32_t)rows, q, 0, nullptr, logit0};
        blocks += (rows + kDecodeBlock - 1) / kDecodeBlock;
    };
    const int64_t ring_sh = d.ring_cap * d.dim, ring_sb = d.Hkv * ring_sh;
    auto ring = [&](const void *k, int64_t lo, int64_t hi, int q, bool logits) {
        for (int64_t pos = lo; pos < hi;) {
            const int64_t row = pos % d.ring_cap, n = std::min(hi - pos, d.ring_cap - row);
            seg((const bf16_t *)k + row * d.dim, (const bf16_t *)d.d_ring_v + row * d.dim, ring_sb, ring_sh, n, q, logits ? (int)(pos - lo) : -1);
            pos += n;
        }
    };
    if (n_sel > 0) {
        DecodeSeg &sg = j.seg[j.n_seg++];
        sg = DecodeSeg{};
        sg.rows = d.block_size; sg.q = 1; sg.n_ids = n_sel; sg.ids = retrieve ? d.d_ids : nullptr; sg.logit0 = -1;
        blocks += (int64_t)n_sel * ((d.block_size + kDecodeBlock - 1) / kDecodeBlock);
        j.chunk = a->d_chunks; j.per_chunk = d.units_per_chunk;
        j.unit_sh = (int64_t)d.block_size * d.dim; j.unit_v_off = d.Hkv * j.unit_sh; j.row_elems = 2 * j.unit_v_off; j.unit_elems = B * j.row_elems;
    }
    if (R->init_len > 0) {
        const int64_t sh = d.init_cap * d.dim, sb = 2 * d.Hkv * sh;
        seg(d.d_init_kv, (const bf16_t *)d.d_init_kv + d.Hkv * sh, sb, sh, R->init_len, 1, -1);
    }
    ring(d.d_ring_k_raw, R->cursor, std::max(b1 - d.n_local, R->cursor), 1, false);
    const int64_t far_blocks = blocks, j_lo = std::max<int64_t>(0, b1 - d.n_local);
    const int far_segs = j.n_seg;
    j.new_logit = (int32_t)(b0 - j_lo);
    ring(d.d_ring_k_rot, j_lo, rides ? b0 : b1, 0, true);
    j.nsplit = infllm_decode_splits(B, d.H, d.Hkv, d.dim, blocks, j.nsplit, rides ? (int64_t)B * d.Hkv : 0, 0);
    j.o_part = a->d_o_part; j.lse_part = a->d_lse_part;
    j.logits = a->d_logits; j.logit_stride = d.n_local;
    if (selects) {
        j.nsplit = std::max(j.nsplit, 2);
        j.unit_scores = a->d_unit_scores; j.unit_scores_sb = a->unit_scores_sb;
        j.n_scores = N;
        j.lead_segs = far_segs;
        j.lead_splits = infllm_decode_lead_splits(j.nsplit, far_blocks, blocks - far_blocks);
        j.ids_out = d.d_ids;
        j.log = f.log;
        f.ids = nullptr;
    }
    rc = rides ? infllm_decode_memory_step(&j, &in, d.dim, st) : infllm_decode_attn(&j, d.dim, st);
    if (rc) return rc;
    f.o_part = (const _Float16 *)a->d_o_part; f.lse_part = a->d_lse_part;
    f.P = j.nsplit; f.B = B; f.H = d.H;
    f.out = (bf16_t *)a->d_out + st0 * a->o_sl; f.o_sb = a->o_sb; f.o_sh = a->o_sh;
    f.logits = a->d_logits; f.logit_stride = d.n_local;
    f.score = d.d_ring_score; f.ring_cap = (int32_t)d.ring_cap; f.slot0 = (int32_t)(j_lo % d.ring_cap); f.n = (int32_t)(b1 - j_lo);
    const dim3 grid(B * d.H, 1 + (f.n + 1023) / 1024);
    if (d.dim == 128) hipLaunchKernelGGL(decode_finish_kernel<128>, grid, dim3(256), 0, st, f);
    else hipLaunchKernelGGL(decode_finish_kernel<64>, grid, dim3(256), 0, st, f);
    INFLLM_CHECK_LAUNCH("decode_finish");
    rc = carve(R, a, carve_after(d, R->cursor, R->init_len, b1), st);
    if (rc) return rc;
    R->length = b1;
    ++R->blocks;
    return 0;
}

// Key splits of the global stage.  Heads of 128: a CU holds one workgroup, the host-driven path's rule (and its bits).  Heads
// of 64: it holds two, so the chip is full at twice as many workgroups, and a launch of a little more than that would start
// over for the few; a workgroup keeps four tiles or more.
int stage_splits(const infllm_resident_desc &d, int n_queries, int n_tiles) {
    if (d.dim == 64 && n_queries > 32) {
        const int wgs = (((n_queries + 31) / 32) * (d.H / d.Hkv) + 7) / 8 * d.Hkv * d.B;
        return std::max(1, std::min({2 * d.num_cus / wgs, n_tiles / 4, d.max_splits}));
    }
    infllm_layer_desc geo{};
    geo.B = d.B; geo.H = d.H; geo.Hkv = d.Hkv; geo.exc = d.exc; geo.max_splits = d.max_splits; geo.num_cus = d.num_cus;
    return infllm_key_splits(&geo, n_queries, n_tiles);
}

// n queries, worked off in execution blocks
int prompt_call(Resident *R, const infllm_resident_call *a, int64_t st0, int n, hipStream_t st) {
    const infllm_resident_desc &d = R->d;
    const int C = d.H * d.dim, B = d.B, exc = d.exc, n_blocks = (n + exc - 1) / exc, D = d.dim;
    const int64_t call_b0 = R->length, row_elems = D;
    INFLLM_REQUIRE(call_b0 + n - R->cursor <= d.ring_cap, "resident: a call of %d tokens at %lld does not fit the rings (%lld rows, carving cursor %lld)", n,
                   (long long)call_b0, (long long)d.ring_cap, (long long)R->cursor);
    infllm_ingest_args in = ingest_args(R, a, st0, n);
    // how many units there are when the call's last block selects
    int32_t units = R->n_units, init = R->init_len, last_sel = R->n_units;
    {
        int64_t cur = R->cursor;
        for (int i = 0; i < n_blocks; ++i) {
            last_sel = units;
            const Carve c = carve_after(d, cur, init, call_b0 + std::min((i + 1) * exc, n));
            cur += c.take + (int64_t)c.count * d.block_size;
            init += c.take;
            units += c.count;
        }
    }
    const bool retrieve = last_sel > d.topk;
    INFLLM_REQUIRE(units <= a->rep_rows && units <= a->n_chunks * d.units_per_chunk, "resident: no room for %d units", units);
    INFLLM_REQUIRE(!retrieve || (a->scores_cols >= units && a->d_call_scores), "resident: no room for the scores of %d units", units);
    in.d_qpart = retrieve ? a->d_qpart : nullptr;
    int rc = infllm_ingest_dim(&in, D, nullptr, st);
    if (rc) return rc;
    const int n0 = R->n_units, n_list = std::min(n0, d.topk);
    if (retrieve) {
        rc = infllm_reduce_partials_blocks(a->d_qpart, B, n, exc, C, a->d_qbar, st);
        if (rc) return rc;
        for (int u = 0; u < B && n0 > 0; ++u) {
            const bf16_t *reps = (const bf16_t *)a->d_reps + (int64_t)u * a->rep_sb;
            rc = infllm_score_topk_queries(reps, a->rep_su, n0, C, a->d_qbar + (int64_t)u * C, (int64_t)B * C, n_blocks, n_list,
                                           a->d_call_scores + (int64_t)u * a->scores_cols, (int64_t)B * a->scores_cols, a->d_base + (int64_t)u * d.topk,
                                           (int64_t)B * d.topk, st);
            for (int i = 0; i < n_blocks && rc == 1; ++i) {          // row lengths without that kernel: block by block
                float *sc = a->d_call_scores + ((int64_t)i * B + u) * a->scores_cols;
                int rc2 = infllm_unit_scores(reps, a->rep_su, 0, n0, C, a->d_qbar + ((int64_t)i * B + u) * C, sc, st);
                if (!rc2) rc2 = infllm_topk(sc, n0, n_list, a->d_base + ((int64_t)i * B + u) * d.topk, st);
                if (rc2) return rc2;
                if (i == n_blocks - 1) rc = 0;
            }
            if (rc) return rc;
        }
    }

    // ---- the local stage: `group` blocks per launch; the blocks' partials lie in regions that are used in turn.  The key
    //      splits are those of the host-driven path's launches of two blocks (a workgroup's queries, keys and splits do not
    //      depend on how many blocks share its launch), so that both paths give the same bits.
    const int group = std::max(1, std::min(d.group_blocks, n_blocks));
    const int64_t lo0 = std::max<int64_t>(0, call_b0 - d.n_local);
    infllm_layer_desc geo{};
    geo.B = B; geo.H = d.H; geo.Hkv = d.Hkv; geo.exc = exc; geo.max_splits = d.max_splits; geo.num_cus = d.num_cus;
    const int pair_n = std::min(n, 2 * exc);
    int nsplit = infllm_key_splits(&geo, pair_n, (int)((call_b0 + pair_n - lo0 + kTile - 1) / kTile));
    const int64_t rows_one = (int64_t)B * d.H * std::min(n, exc);
    while (nsplit > 1 && (int64_t)8 * B * d.H * exc / (nsplit * rows_one) < (n_blocks > 1 ? 4 : 1)) --nsplit;
    INFLLM_REQUIRE(a->part_rows / (nsplit * rows_one) >= group, "resident: partial rows do not fit");
    const int64_t block_rows = nsplit * rows_one;

    // the score launch of nq queries from the call's query q0 on, which see the keys [lo, hi)
    auto score_args = [&](int64_t q0, int nq, int64_t lo, int64_t hi) {
        infllm_score_args sc{};
        sc.d_q = (const bf16_t *)a->d_q_loc + q0 * row_elems;
        sc.q_sl = D; sc.q_sh = (int64_t)n * D; sc.q_sb = (int64_t)d.H * n * D;
        sc.B = B; sc.H = d.H; sc.Hkv = d.Hkv; sc.Lq = nq;
        sc.d_k = d.d_ring_k_rot;
        sc.k_sl = D; sc.k_sh = d.ring_cap * D; sc.k_sb = d.Hkv * d.ring_cap * D;
        sc.cap = d.ring_cap; sc.j_lo = lo; sc.j_hi = hi;
        sc.mask = INFLLM_MASK_WINDOW; sc.accumulate = 1; sc.offset = call_b0 + q0; sc.window = d.n_local;
        sc.d_lse = a->d_lse; sc.softmax_scale = d.softmax_scale;
        sc.d_score = d.d_ring_score; sc.score_sh = d.ring_cap; sc.score_sb = d.H * d.ring_cap; sc.score_cap = d.ring_cap;
        return sc;
    };
    int32_t j_done = -1;                          // the block whose page table is on the device
    int plain_end = 0;                            // blocks in front of this one are done
    int32_t scored = n0;                          // units that have scores under the mean queries of all blocks to come
    for (int i = 0; i < n_blocks; ++i) {
        const int nb = std::min(exc, n - i * exc);
        const int64_t b0 = call_b0 + (int64_t)i * exc, b1 = b0 + nb, lo = std::max<int64_t>(0, b0 - d.n_local);
        const int N = R->n_units;
        if (i % group == 0) {
            const int gn = std::min(group * exc, n - i * exc);
            infllm_attn_args at{};
            at.d_q = (const bf16_t *)a->d_q_loc + (int64_t)i * exc * row_elems;
            at.q_sl = D; at.q_sh = (int64_t)n * D; at.q_sb = (int64_t)d.H * n * D;
            at.B = B; at.H = d.H; at.Hkv = d.Hkv; at.Lq = gn;
            at.d_k = d.d_ring_k_rot; at.d_v = d.d_ring_v;
            at.k_sl = at.v_sl = D;
            at.k_sh = at.v_sh = d.ring_cap * D;
            at.k_sb = at.v_sb = d.Hkv * d.ring_cap * D;
            at.cap = d.ring_cap; at.j_lo = lo; at.j_hi = b0 + gn;
            at.mask = INFLLM_MASK_WINDOW; at.offset = b0; at.window = d.n_local;
            at.nsplit = nsplit;
            at.softmax_scale = d.softmax_scale;
            at.d_o_part = a->d_o_part; at.d_lse_part = a->d_lse_part;
            // Blocks that read nothing but the window and from which nothing leaves (a stream's first n_local tokens) have no
            // chain from one to the next: their partials are merged and their scores taken in one launch each for all of them
            // (eight blocks: 16 launches of some 20 us; 4,096 queries at once keep the chip full).
            int m = 0;
            for (; i + m < std::min(n_blocks, i + group); ++m) {
                const int64_t e1 = call_b0 + std::min((i + m + 1) * exc, n);
                const Carve c = carve_after(d, R->cursor, R->init_len, e1);
                if (c.take || c.count || page_list(R, a, std::min(N, d.topk), e1).n_pages) break;
            }
            const int q0 = i * exc, nq = std::min(m * exc, n - q0);
            // ... or both in one launch, where all blocks of this one are such and few enough for it: their partials are those of one
            // long block then (1,998 queries: the merge's 10 us)
            const bool whole = m >= 2 && nq == gn && gn <= 2048;
            const int ti = timer_begin(R, 0, gn, (int)(b0 + gn - lo), st);
            rc = infllm_attn_stage_blocked(&at, whole ? (gn + 31) / 32 * 32 : exc, whole ? (int64_t)nsplit * B * d.H * gn : block_rows, st, D);
            timer_end(R, 0, ti, st);
            if (rc) return rc;
            if (m >= 2) {
                bf16_t *out = (bf16_t *)a->d_out + (st0 + q0) * a->o_sl;
                const infllm_score_args sc = score_args(q0, nq, lo, b0 + nq);
                rc = 1;
                if (whole) {
                    MergeJob job;
                    rc = infllm_merge_job(a->d_o_part, a->d_lse_part, nsplit, nullptr, nullptr, 0, B, d.H, gn, out, a->o_sb, a->o_sh, a->o_sl, a->d_lse, &job, D);
                    if (!rc) rc = infllm_local_score_merged(&sc, &job, st, D);
                    if (rc < 0) return rc;
                }
                if (rc == 1) {
                    rc = infllm_attn_merge_blocked(a->d_o_part, a->d_lse_part, nsplit, B, d.H, nq, whole ? gn : exc, block_rows, out, a->o_sb, a->o_sh, a->o_sl,
                                                   a->d_lse, st, D);
                    if (!rc) rc = infllm_local_score_dim(&sc, D, st);
                    if (rc) return rc;
                }
                plain_end = i + m;
            }
        }
        if (i < plain_end) {
            R->queue.push_back(Resident::Entry{0, 0, 0});
            R->length = b1;
            ++R->blocks;
            continue;
        }
        const uint16_t *o_loc = a->d_o_part + (int64_t)(i % group) * block_rows * D;
        const float *lse_loc = a->d_lse_part + (int64_t)(i % group) * block_rows;

        // ---- the block's page table and global stage
        const int n_sel = std::min(N, d.topk);
        const PageList pl = page_list(R, a, n_sel, b1);
        INFLLM_REQUIRE(pl.n_pages <= d.max_pages, "resident: %d pages exceed the table (%d)", pl.n_pages, d.max_pages);
        const bool all_units = N <= d.topk;
        if (all_units) R->queue.push_back(Resident::Entry{N, 0, 0});
        // A block that attends every unit has its table from here, and the launch of the global stage takes one of up to 64 pages along
        // (a launch of its own for the table: 4.7 us; five of them in a prompt of 16,001 tokens: 2,729 us with, 2,708 without).
        infllm_page carried[kInlinePages];
        const bool carries = all_units && pl.n_pages > 0 && (int64_t)B * pl.n_pages <= kInlinePages;
        if (carries) {
            for (int u = 0; u < B; ++u)
                for (int p = 0; p < pl.n_pages; ++p) carried[u * pl.n_pages + p] = page_of(pl, u, p, nullptr, a->h_chunks);
        } else if (all_units && pl.n_pages > 0) {
            hipLaunchKernelGGL(pages_kernel, dim3((pl.n_pages + 255) / 256, B), dim3(256), 0, st, pl);
            INFLLM_CHECK_LAUNCH("pages");
        } else if (!all_units && j_done != i) {                   // the call's first block (the others' tables came with the previous block)
            int32_t slot = 0, seq = 0;
            rc = take_slot(R, &slot, &seq);
            if (rc) return rc;
            RankJob jb{};
            jb.reps = (const bf16_t *)a->d_reps; jb.rep_sb = a->rep_sb; jb.rep_su = a->rep_su;
            jb.qbars = a->d_qbar; jb.scores = a->d_call_scores; jb.cols = a->scores_cols; jb.base = a->d_base;
            jb.B = B; jb.C = C; jb.k = d.topk; jb.n_list = n_list; jb.n_base = n0; jb.first_new = scored; jb.n_new = N - scored; jb.j0 = jb.j_sel = i;
            jb.log = d.d_log + (int64_t)slot * (B * d.topk + 1); jb.seq = seq;
            jb.pages = pl;
            rc = launch_rank(R, jb, 1, st);
            if (rc) return rc;
        }
        int parts = nsplit, ns_g = 0;
        if (pl.n_pages > 0) {
            infllm_attn_args at{};
            at.d_q = (const bf16_t *)a->d_q_glb + (int64_t)i * exc * row_elems;
            at.q_sl = D; at.q_sh = (int64_t)n * D; at.q_sb = (int64_t)d.H * n * D;
            at.B = B; at.H = d.H; at.Hkv = d.Hkv; at.Lq = nb;
            at.cap = kTile;
            at.d_pages = d.d_pages; at.n_pages = pl.n_pages;
            at.softmax_scale = d.softmax_scale;
            ns_g = stage_splits(d, nb, pl.n_pages);
            if (D == 64) ns_g = std::min(ns_g, std::max(1, 8 - nsplit));              // (up to 8 partials are merged along with the scores)
            at.nsplit = ns_g;
            at.d_o_part = a->d_o_part2; at.d_lse_part = a->d_lse_part2;
            INFLLM_REQUIRE((int64_t)ns_g * B * d.H * nb <= a->part_rows2, "resident: global partial rows do not fit");
            const int tw = timer_begin(R, 2, nb, 0, st);          // (where the stream of the host-driven path waits for missed units)
            timer_end(R, 2, tw, st);
            const int ti = timer_begin(R, 1, nb, pl.n_pages * kTile, st);
            rc = infllm_attn_paged(&at, carries ? carried : nullptr, st, D);
            timer_end(R, 1, ti, st);
            if (rc) return rc;
            parts += ns_g;
        }
        // ---- what ends the block
        bf16_t *out = (bf16_t *)a->d_out + (st0 + (int64_t)i * exc) * a->o_sl;
        MergeJob job;
        rc = infllm_merge_job(o_loc, lse_loc, nsplit, ns_g ? a->d_o_part2 : nullptr, ns_g ? a->d_lse_part2 : nullptr, ns_g, B, d.H, nb, out, a->o_sb, a->o_sh,
                              a->o_sl, a->d_lse, &job, D);
        if (rc) return rc;
        infllm_score_args sc = score_args((int64_t)i * exc, nb, lo, b1);
        // Blocks with a kernel for it - long key ranges, up to eight partials, up to 512 queries and units of 32, 64, 96 or 128
        // tokens where units leave - end in one launch (infllm_block_end): scores, merge, the units that leave and the next
        // block's ranking.  The others' scores with the merge, carving and ranking are launches of their own.  (Prompts of 16,001 /
        // 131,072 tokens, 24,300 with 36 heads of 64: two launches, carving in front of the scores, 3,035 / 29,430 / 3,468 us, one
        // 2,882 / 28,140 / 3,400.)
        const Carve c = carve_after(d, R->cursor, R->init_len, b1);
        const bool early = b1 - lo > 1024 && infllm_block_end_takes(nb, parts, d.block_size, c.count > 0, true);
        UnitRun run;
        auto end_block = [&](const infllm_score_args &s, const RankJob *rank, int n_rank) {
            const int64_t unit_elems = (int64_t)d.Hkv * d.block_size * d.dim;
            return infllm_block_end(&s, &job, d.d_ring_k_raw, d.d_ring_v, run.t0, d.block_size, run.n, d.repr_topk, run.rep, a->rep_sb, a->rep_su, run.home_k,
                                    run.home_v, 2 * unit_elems, (int64_t)d.B * 2 * unit_elems, (int64_t)d.block_size * d.dim, rank, n_rank, a->d_ticket, st, D);
        };
        if (early) {
            rc = carve_init(R, c, st);
            if (!rc) rc = next_run(R, a, c.count, &run);
            for (int done = run.n; !rc && done < c.count; done += run.n) {      // (units of several chunks: all but the last chunk's ahead)
                infllm_score_args none = sc;
                none.j_lo = none.j_hi;
                rc = end_block(none, nullptr, 0);
                job.out = nullptr;                                               // merged along with the first of them
                if (!rc) rc = next_run(R, a, c.count - done, &run);
            }
            if (rc) return rc;
        } else {
            rc = parts <= 8 ? infllm_local_score_merged(&sc, &job, st, D) : 1;
            if (rc < 0) return rc;
            if (rc == 1) {
                rc = infllm_attn_merge2(o_loc, lse_loc, nsplit, ns_g ? a->d_o_part2 : nullptr, ns_g ? a->d_lse_part2 : nullptr, ns_g, B, d.H, nb, out,
                                        a->o_sb, a->o_sh, a->o_sl, a->d_lse, st, D);
                if (!rc) rc = infllm_local_score_dim(&sc, D, st);
                if (rc) return rc;
            }
            rc = carve(R, a, c, st);
            if (rc) return rc;
        }
        R->length = b1;
        ++R->blocks;
        // ---- the next block's selection and page table
        const int N1 = R->n_units;
        const bool rank = i + 1 < n_blocks && retrieve && (c.count > 0 || N1 > d.topk);
        RankJob jb{};
        if (rank) {
            const bool select = N1 > d.topk;
            jb.reps = (const bf16_t *)a->d_reps; jb.rep_sb = a->rep_sb; jb.rep_su = a->rep_su;
            jb.qbars = a->d_qbar; jb.scores = a->d_call_scores; jb.cols = a->scores_cols; jb.base = a->d_base;
            jb.B = B; jb.C = C; jb.k = d.topk; jb.n_list = n_list; jb.n_base = n0; jb.first_new = scored; jb.n_new = N1 - scored; jb.n_before = N - scored;
            jb.j0 = i + 1; jb.j_sel = select ? i + 1 : -1;
            if (select) {
                int32_t slot = 0, seq = 0;
                rc = take_slot(R, &slot, &seq);
                if (rc) return rc;
                jb.log = d.d_log + (int64_t)slot * (B * d.topk + 1); jb.seq = seq;
                jb.pages = page_list(R, a, d.topk, std::min(call_b0 + n, b1 + exc));
                INFLLM_REQUIRE(jb.pages.n_pages <= d.max_pages, "resident: %d pages exceed the table (%d)", jb.pages.n_pages, d.max_pages);
                j_done = i + 1;
                ++R->ranked;
            }
        }
        const int n_rank = jb.n_new > 0 ? n_blocks - (i + 1) : 1;
        bool ranked = !rank;
        if (early) {
            sc.j_lo = std::max(lo, R->cursor);
            const bool carry = rank && infllm_block_end_ranks(C, D);
            rc = end_block(sc, carry ? &jb : nullptr, n_rank);
            if (rc) return rc;
            if (carry) ranked = true, scored = N;
        }
        if (!ranked) {
            rc = launch_rank(R, jb, n_rank, st);
            if (rc) return rc;
            scored = N1;
        }
    }
    return 0;
}

}  // namespace

extern "C" int infllm_resident_fits(const infllm_resident_desc *d) {
    INFLLM_REQUIRE(d, "resident_fits: null descriptor");
    const int per_block = (d->exc + d->n_init + d->block_size - 1) / d->block_size + 1;
    const int per_call = (std::max(d->call_tokens, d->exc) + d->n_init + d->block_size - 1) / d->block_size + 1;
    return d->topk >= 1 && d->topk <= 64 && per_block <= kRankNew && d->topk + per_call <= kRankEntries && (d->H * d->dim) % 8 == 0 &&
                   d->H * d->dim <= 16 * 512 && (d->dim == 128 || d->dim == 64) && d->block_size <= 2048 &&
                   d->exc % 32 == 0
               ? 1
               : 0;
}

extern "C" int64_t infllm_resident_part_rows(const infllm_resident_desc *d) {
    if (!d || d->B <= 0 || d->H <= 0 || d->Hkv <= 0 || d->H % d->Hkv || d->exc <= 0) return infllm_fail(-1, "resident_part_rows: bad descriptor");
    int64_t rows = 0;
    for (int n = 1; n <= d->exc; ++n) rows = std::max<int64_t>(rows, (int64_t)stage_splits(*d, n, d->max_pages) * n);
    return rows * d->B * d->H;
}

extern "C" void *infllm_resident_create(const infllm_resident_desc *desc) {
    auto bad = [](const char *m) -> void * {
        infllm_fail(-1, "resident_create: %s", m);
        return nullptr;
    };
    if (!desc) return bad("null descriptor");
    const infllm_resident_desc &d = *desc;
    if (d.B <= 0 || d.H <= 0 || d.Hkv <= 0 || d.H % d.Hkv) return bad("bad head geometry");
    if (d.exc <= 0 || d.exc > d.n_local || d.block_size <= 0 || d.topk > d.max_cached || d.n_init < 0) return bad("bad knobs");
    if (infllm_resident_fits(desc) != 1) return bad("geometry without this path");
    if (d.ring_cap % kTile || d.ring_cap < (int64_t)d.n_local + 2 * d.exc + d.block_size) return bad("ring too small or unaligned");
    if (!d.d_ring_k_raw || !d.d_ring_k_rot || !d.d_ring_v || !d.d_ring_score || !d.d_init_kv || !d.d_ids || !d.d_pages || !d.d_log || !d.h_log ||
        !d.h_caches || !d.d_inv_freq)
        return bad("null buffer");
    if (d.log_slots < 2 || d.units_per_chunk < 1 || d.init_cap < 1 || d.max_pages < 1 || d.max_splits < 1 || d.num_cus < 1 || d.group_blocks < 1) return bad("bad capacities");
    Resident *R = new Resident();
    R->d = d;
    R->next_seq = d.first_seq;
    return R;
}

extern "C" int infllm_resident_destroy(void *handle) {
    Resident *R = (Resident *)handle;
    if (!R) return 0;
    for (auto &t : R->timer)
        for (hipEvent_t e : t.ev)
            if (e) (void)hipEventDestroy(e);
    delete R;
    return 0;
}

extern "C" int infllm_resident_set_state(void *handle, int64_t length, int64_t cursor, int32_t init_len, int32_t n_units) {
    INFLLM_REQUIRE(handle && length >= 0 && cursor >= 0 && cursor <= length && init_len >= 0 && n_units >= 0, "resident_set_state: bad state");
    Resident *R = (Resident *)handle;
    INFLLM_REQUIRE(init_len <= R->d.init_cap, "resident_set_state: %d init tokens", init_len);
    R->length = length;
    R->cursor = cursor;
    R->init_len = init_len;
    R->n_units = n_units;
    return 0;
}

extern "C" int infllm_resident_append(void *handle, const infllm_resident_call *a, void *stream) {
    INFLLM_REQUIRE(handle && a, "resident_append: null argument");
    Resident *R = (Resident *)handle;
    const infllm_resident_desc &d = R->d;
    INFLLM_REQUIRE(a->n >= 0 && a->call_tokens >= 0, "resident_append: negative length");
    if (a->n == 0) return 0;
    INFLLM_REQUIRE(a->d_q && a->d_k && a->d_v && a->d_out && a->d_q_loc && a->d_q_glb && a->d_qbar && a->d_o_part && a->d_lse_part, "resident_append: null pointer");
    INFLLM_REQUIRE(a->d_reps && a->h_chunks && a->d_chunks && a->d_unit_scores, "resident_append: null unit buffers");
    hipStream_t st = (hipStream_t)stream;
    R->last_stream = st;
    int rc = drain(R, false);
    if (rc) return rc;
    const int stretch = a->call_tokens > 0 ? a->call_tokens : d.exc;
    for (int64_t pos = 0; pos < a->n;) {
        const int n = (int)std::min<int64_t>(stretch, a->n - pos);
        INFLLM_REQUIRE(n <= a->max_tokens, "resident_append: %d tokens do not fit the buffers (%d)", n, a->max_tokens);
        if (n == 1) {
            INFLLM_REQUIRE(a->d_logits, "resident_append: null logits");
            rc = decode_step(R, a, pos, st);
        } else {
            INFLLM_REQUIRE(a->d_qpart && a->d_o_part2 && a->d_lse_part2 && a->d_lse && a->d_base && a->d_ticket, "resident_append: null pointer");
            rc = prompt_call(R, a, pos, n, st);
        }
        if (rc) return rc;
        pos += n;
    }
    return 0;
}

extern "C" int infllm_resident_state(void *handle, int32_t wait, int64_t *out) {
    INFLLM_REQUIRE(handle && out, "resident_state: null argument");
    Resident *R = (Resident *)handle;
    if (wait) {
        const int rc = drain(R, true);
        if (rc) return rc;
    }
    out[0] = R->length; out[1] = R->cursor; out[2] = R->init_len; out[3] = R->n_units;
    out[4] = R->blocks; out[5] = R->hits; out[6] = R->misses; out[7] = R->evictions; out[8] = R->ranked; out[9] = R->next_seq;
    return 0;
}

extern "C" int infllm_resident_timing(void *handle, int32_t capacity, int32_t stride) {
    INFLLM_REQUIRE(handle && capacity >= 0 && stride >= 1, "resident_timing: bad arguments");
    Resident *R = (Resident *)handle;
    for (auto &t : R->timer) {
        while ((int)t.ev.size() < 2 * capacity) {
            hipEvent_t e;
            HIP_OK(hipEventCreate(&e), "resident_timing");
            t.ev.push_back(e);
        }
        t.n_queries.resize(capacity);
        t.n_keys.resize(capacity);
        t.used = t.seen = 0;
    }
    R->timing_cap = capacity;
    R->timing_stride = stride;
    return 0;
}

extern "C" int infllm_resident_read_timing(void *handle, int32_t which, float *ms, int32_t *n_queries, int32_t *n_keys, int32_t capacity) {
    INFLLM_REQUIRE(handle && which >= 0 && which <= 2 && ms && capacity >= 0, "resident_read_timing: bad arguments");
    Resident *R = (Resident *)handle;
    Timer &t = R->timer[which];
    const int n = std::min(t.used, capacity);
    for (int i = 0; i < n; ++i) {
        HIP_OK(hipEventSynchronize(t.ev[2 * i + 1]), "resident_read_timing");
        HIP_OK(hipEventElapsedTime(&ms[i], t.ev[2 * i], t.ev[2 * i + 1]), "resident_read_timing");
        if (n_queries) n_queries[i] = t.n_queries[i];
        if (n_keys) n_keys[i] = t.n_keys[i];
    }
    return n;
}
