// A selection and what becomes of it on the device, for units resident in HBM (resident.hip; the launch that ends a block,
// score.hip, carries it along).
#pragma once
#include "common.h"

#include <type_traits>

constexpr int kRankEntries = 320;          // the k <= 64 best of the call's start + 256 units carved since
constexpr int kRankNew = 64;               // units carved by one block
constexpr int kRankChunks = 256;           // addresses of chunks of units that a ranking workgroup keeps

// The page table of a block: selected units, init tokens, overflow remainder of the ring (the order of the host-built
// tables of stream.hip).
struct PageList {
    infllm_page *out;                      // [B, n_pages]
    int32_t n_unit_pages, n_init_pages, n_pages, tiles_per_unit;
    int32_t Hkv, bs, init_len, dim;
    int64_t cursor, overflow_end, ring_cap, init_cap;
    const bf16_t *init_kv, *ring_k, *ring_v;
    const uint64_t *chunk;                 // device: chunks of units, [per_chunk, B, 2, Hkv, bs, dim] each
    int32_t per_chunk, B, n_chunks;
};

// Page p of batch row u.  ids: the selection, NULL: every unit in order; chunk: the table of addresses, where it has been read already.
__host__ __device__ __forceinline__ infllm_page page_of(const PageList &j, int u, int p, const int32_t *ids, const uint64_t *chunk) {
    const int64_t unit_elems = (int64_t)j.Hkv * j.bs * j.dim;
    infllm_page pg;
    pg.reserved = 0;
    if (p < j.n_unit_pages) {
        const int s = p / j.tiles_per_unit, t0 = (p - s * j.tiles_per_unit) * kTile;
        const int unit = ids ? ids[s] : s, ch = unit / j.per_chunk;
        const bf16_t *kb = (const bf16_t *)(uintptr_t)chunk[ch] + (((int64_t)(unit - ch * j.per_chunk) * j.B + u) * 2) * unit_elems + (int64_t)t0 * j.dim;
        pg.k = kb;
        pg.v = kb + unit_elems;
        pg.head_stride = (int64_t)j.bs * j.dim;
        pg.n_valid = j.bs - t0 < kTile ? j.bs - t0 : kTile;
    } else if (p < j.n_unit_pages + j.n_init_pages) {
        const int t0 = (p - j.n_unit_pages) * kTile;
        const bf16_t *ik = j.init_kv + (int64_t)u * 2 * j.Hkv * j.init_cap * j.dim + (int64_t)t0 * j.dim;
        pg.k = ik;
        pg.v = ik + (int64_t)j.Hkv * j.init_cap * j.dim;
        pg.head_stride = j.init_cap * j.dim;
        pg.n_valid = j.init_len - t0 < kTile ? j.init_len - t0 : kTile;
    } else {
        const int want = p - j.n_unit_pages - j.n_init_pages;
        int64_t pos = j.cursor, len = 0;
        for (int i = 0; i <= want; ++i) {          // runs of <= 64 rows that do not cross the end of the ring
            pos += len;
            const int64_t left = j.overflow_end - pos, lap = j.ring_cap - pos % j.ring_cap;
            len = left < kTile ? left : kTile;
            len = lap < len ? lap : len;
        }
        const int64_t row = pos % j.ring_cap;
        pg.k = j.ring_k + ((int64_t)u * j.Hkv * j.ring_cap + row) * j.dim;
        pg.v = j.ring_v + ((int64_t)u * j.Hkv * j.ring_cap + row) * j.dim;
        pg.head_stride = j.ring_cap * j.dim;
        pg.n_valid = (int)len;
    }
    return pg;
}

__device__ __forceinline__ void write_page(const PageList &j, int u, int p, const int32_t *ids, const uint64_t *chunk) {
    j.out[(int64_t)u * j.n_pages + p] = page_of(j, u, p, ids, chunk);
}

// After a block has carved units: every unit is scored under the mean queries of the call's later blocks, and block j_sel's list
// of the call's start is ranked against all units carved since; the selection becomes the block's page table.
struct RankJob {
    const bf16_t *reps;
    int64_t rep_sb, rep_su;
    const float *qbars;                    // [blocks][B][C]
    float *scores;                         // [blocks][B][cols]
    int64_t cols;
    const int32_t *base;                   // [blocks][B][k], n_list entries of a row are filled
    int32_t B, C, k, n_list, n_base, j0, j_sel;
    int32_t first_new, n_new;              // the units that have no scores under block j0 and later ones yet, from first_new on,
    int32_t n_before;                      // and how many of them were there before this launch
    int32_t *log;                          // pinned: [B][k] ids, then the sequence number
    int32_t seq;
    PageList pages;
};

template <int CPL>
struct RankLds {
    float q[CPL * 512];                    // the mean query
    float fresh[2 * kRankNew];
    uint64_t e_key[kRankEntries];
    int32_t sel[64];
    uint64_t chunk[kRankChunks];
};

// 256 threads: scores of n_new units from jb.first_new on under the mean query of block j0 + x, and the ranking if that is block
// j_sel (the sums are unit_scores_rows_kernel's, term by term: a unit's score does not depend on which kernel computed it).  All
// of it is a chain of trips to memory on the way to the next block, beside workgroups that keep the chip busy: everything whose
// address is known is requested at once, what depends on it next, and nothing is read behind the ranking.  all_pages: the pages
// behind the units' too (else another workgroup writes those, which depend on no selection).
template <int CPL>
__device__ __forceinline__ void rank_block(const RankJob &jb, int x, int n_new, bool all_pages, RankLds<CPL> &lds) {
    float *fresh = lds.fresh;
    uint64_t *e_key = lds.e_key;
    int32_t *sel = lds.sel;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, C = jb.C;
    const int j = jb.j0 + x;
    const bool is_sel = j == jb.j_sel;
    const int n = jb.n_list + jb.first_new + n_new - jb.n_base;
    const bool kept = is_sel && jb.pages.n_chunks <= kRankChunks;
    for (int u = 0; u < jb.B; ++u) {
        const float *qbar = jb.qbars + ((int64_t)j * jb.B + u) * C;
        float *scores = jb.scores + ((int64_t)j * jb.B + u) * jb.cols;
        // the ranking threads' entries, asked for ahead of the scoring
        int my_id[2] = {-1, -1};
        float my_score[2] = {0.f, 0.f};
        if (is_sel) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int e = tid + 256 * i;
                if (e < n) my_id[i] = e < jb.n_list ? jb.base[((int64_t)j * jb.B + u) * jb.k + e] : jb.n_base + (e - jb.n_list);
            }
        }
        u32x4 w[CPL];
        auto request = [&](int r) {
            const bf16_t *row = jb.reps + (int64_t)u * jb.rep_sb + (int64_t)(jb.first_new + r) * jb.rep_su + lane * 8;
#pragma unroll
            for (int c = 0; c < CPL; ++c) w[c] = c * 512 + lane * 8 < C ? *(const u32x4 *)(row + c * 512) : u32x4{0, 0, 0, 0};
        };
        if (wave < n_new) request(wave);
        constexpr int kQ = (CPL * 512 + 1023) / 1024;
        f32x4 q_in[kQ];
#pragma unroll
        for (int i = 0; i < kQ; ++i) q_in[i] = *(const f32x4 *)(qbar + min(i * 1024 + tid * 4, C - 4));
        uint64_t chunk_in = 0;
        if (kept && u == 0 && tid < jb.pages.n_chunks) chunk_in = jb.pages.chunk[tid];
#pragma unroll
        for (int i = 0; i < 2; ++i)
            if (is_sel && tid + 256 * i < n && my_id[i] < jb.first_new) my_score[i] = scores[my_id[i]];
#pragma unroll
        for (int i = 0; i < kQ; ++i) {
            const int e = i * 1024 + tid * 4;
            if (e < C) *(f32x4 *)(lds.q + e) = q_in[i];
        }
        if (kept && u == 0) lds.chunk[tid] = chunk_in;
        __syncthreads();
        for (int r = wave; r < n_new; r += 4) {
            float acc0 = 0.f, acc1 = 0.f;
#pragma unroll
            for (int c = 0; c < CPL; ++c) {
                if (c * 512 + lane * 8 >= C) continue;
                const f32x4 q[2] = {*(const f32x4 *)(lds.q + c * 512 + lane * 8), *(const f32x4 *)(lds.q + c * 512 + lane * 8 + 4)};
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    acc0 += bf16_bits_to_f32(w[c][i] & 0xffffu) * q[i >> 1][2 * (i & 1)];
                    acc1 += bf16_bits_to_f32(w[c][i] >> 16) * q[i >> 1][2 * (i & 1) + 1];
                }
            }
            if (r + 4 < n_new) request(r + 4);
            float acc = acc0 + acc1;
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
            if (lane == 0) {
                scores[jb.first_new + r] = acc;
                fresh[r] = acc;
            }
        }
        __syncthreads();
        if (!is_sel) continue;                                   // workgroup-uniform
#pragma unroll
        for (int i = 0; i < 2; ++i) {                            // descending score, equal scores in ascending id: all distinct
            const int e = tid + 256 * i;
            if (e >= n) continue;
            const float score = my_id[i] >= jb.first_new ? fresh[my_id[i] - jb.first_new] : my_score[i];
            e_key[e] = ((uint64_t)order_key(score) << 32) | (uint32_t)~my_id[i];
        }
        __syncthreads();
        auto count = [&](auto lanes) {                           // an entry's place is the number of entries in front of it: some lanes count
            constexpr int L = decltype(lanes)::value;
            for (int e0 = 0; e0 < n; e0 += 256 / L) {
                const int e = e0 + tid / L, p = tid % L;
                const uint64_t own = e_key[min(e, n - 1)];
                int rank = 0;
#pragma unroll 16
                for (int o = p; o < n; o += L) rank += e_key[o] > own ? 1 : 0;
#pragma unroll
                for (int o = 1; o < L; o <<= 1) rank += __shfl_xor(rank, o, 64);
                if (p == 0 && e < n && rank < jb.k) {
                    const int id = (int)~(uint32_t)own;
                    sel[rank] = id;
                    // (written through to the host's memory: a fence would write the whole L2 back)
                    __hip_atomic_store(jb.log + (int64_t)u * jb.k + rank, id, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                }
            }
        };
        if (n <= 64) count(std::integral_constant<int, 4>{});
        else count(std::integral_constant<int, 2>{});
        __syncthreads();
        const int n_write = all_pages ? jb.pages.n_pages : jb.pages.n_unit_pages;
        for (int p = tid; p < n_write; p += 256) write_page(jb.pages, u, p, sel, kept ? lds.chunk : jb.pages.chunk);
        __syncthreads();                                         // the lists are rewritten for the next row
    }
    if (is_sel) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");         // every wave's ids have arrived
        __syncthreads();
        if (tid == 0) __hip_atomic_store(jb.log + (int64_t)jb.B * jb.k, jb.seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}
