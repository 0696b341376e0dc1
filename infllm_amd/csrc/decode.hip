// Attention of ONE query per head over a list of key ranges: the decode step of every attention type
// (inf_llm/attention/dot_production_attention/torch_impl.py:39-96 for one query; stages joined by the merge).
//
// One query per head makes the step a read of K and V (2 FLOP per byte): bound by HBM, or for short ranges by the
// latency of two dependent round trips.  So nothing is staged: every wave streams blocks of 16 keys of one kv head
// straight from memory into registers, the next block's rows in flight while the current one is used, and the query
// heads that share the kv head (up to four) are handled together, so that K and V are read once for all of them.
//   S[key, head] = K . q^T by v_mfma_f32_16x16x32_bf16 (keys as rows, heads as columns): lane (head = lane & 15, row group
//   rg = lane >> 4) receives the logits of keys 4 * rg + 0..3 of its head;
//   the softmax runs per lane over those (its own running maximum and sum, no exchange between lanes);
//   O[head, d] += p[key] * v[key, d] on the vector units in fp32: a row group reads its own four keys' value rows
//   (16 lanes x 16 bytes), and a head's probability reaches the row's lanes by a DPP row broadcast.
// The states of all row groups and waves are joined through LDS at the end, the splits by the one that ends last, or by a merge
// or finishing kernel.
// A logit that is NaN or +infinity makes its query's row NaN, as the softmax has it: a lane that saw nothing but NaN still has
// its maximum at -infinity, so its sum is taken as it is, and a split whose sum is no number writes NaN rather than zeros.
// 32,768 keys x 8 kv heads (134 MB): 648 us with the tile kernel of attn.hip at one split, 33 us here.
#include "decode.h"
#include "rope.h"
#include "select.h"

#include <algorithm>
#include <numeric>
#include <type_traits>

namespace {

constexpr int kDecWaves = 8;                       // (see decode_attn_kernel)
constexpr float kLazyDec = 8.f;                    // the running maximum may lag the true one by 2^8

template <int N>
__device__ __forceinline__ float row_bcast(float x) {      // lane N of every row of 16 lanes, to the whole row
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0x150 + N, 0xf, 0xf, true));
}

template <int NG, int H0 = 0, typename F>
__device__ __forceinline__ void each_head(F &&f) {
    if constexpr (H0 < NG) {
        f(std::integral_constant<int, H0>{});
        each_head<NG, H0 + 1>(f);
    }
}

// D: head dimension (128 or 64); NG: query heads handled together (columns of the MFMA; heads beyond the group's last are
// zero queries whose results are not written)
//
// Front: the step's rows come as they are (StepQkv).  Rotating them in a launch in front cost 5 us on a chain of two, and its
// cache writes, copies included, were waited for by an attention that can read the old cache: here every workgroup rotates its
// heads' queries while its first rows are on their way, the last split attends the new key, and workgroups behind all splits
// write the cache (stream-llm, one token over 9,000: 25.4 -> 22.7 us; causal, over 8,192: 26.7 -> 24.0).  A step of the streaming memory
// that selects nothing has the rest of its prologue there (MemoryRows).
struct NoFront {};
struct MemoryRows : StepQkv {
    infllm_ingest_args in;
};
template <int D>
__device__ __forceinline__ void leave_rows(const StepRows &f, int b, int g, float2 *cs) {      // 256 threads
    constexpr int HALF = D / 2, C2 = D / 16;
    const int tid = threadIdx.x;
    const float freq = rope_freq<HALF>(f.inv_freq);
    u32x4 lo{}, hi{}, v{};
    if (tid < C2) {
        const bf16_t *src = f.k + (int64_t)b * f.k_sb + (int64_t)g * f.k_sh + tid * 8;
        lo = *(const u32x4 *)src, hi = *(const u32x4 *)(src + HALF);
    }
    if (tid < 2 * C2) v = *(const u32x4 *)(f.v + (int64_t)b * f.v_sb + (int64_t)g * f.v_sh + tid * 8);
    rope_angles<HALF>(f.pos, 1, f.glb_pos, f.distance_scale, freq, (float2(*)[HALF])cs, cs + HALF);
    __syncthreads();
    if (tid < C2) {
        const Rot8 r = rotate8(lo, hi, cs + tid * 8);
        bf16_t *dst = f.dk + (int64_t)b * f.dk_sb + (int64_t)g * f.dk_sh + tid * 8;
        *(u32x4 *)dst = r.lo, *(u32x4 *)(dst + HALF) = r.hi;
        if (f.raw) {
            dst = f.raw + (int64_t)b * f.raw_sb + (int64_t)g * f.raw_sh + tid * 8;
            *(u32x4 *)dst = lo, *(u32x4 *)(dst + HALF) = hi;
        }
    }
    if (tid < 2 * C2) *(u32x4 *)(f.dv + (int64_t)b * f.dv_sb + (int64_t)g * f.dv_sh + tid * 8) = v;
}

// SELECT: the units of the job are selected here (DecodeJob), by every workgroup that reads any of them, each for itself.  A launch that
// selects for all has to hand over inside: scores stored where every XCD sees them, a ticket, and one workgroup's trips to memory
// while the chip waits.  Here the others attend the window meanwhile, two thirds of the keys, which need no selection.  (Kernels of a
// step, 32 heads of 128: behind 64K tokens scores with selection 12.5 + attention 13.4 us, so 8.4 + 12.8; behind 512K 17.1 + 12.8,
// 11.8 + 14.6.  The window attended in the launch of the scores instead, beside the selection there: 18.5 + 9.8 and 25.7 + 9.6.)
//
// A split is a few microseconds of rows between a start and an end that are as long, so both are kept short.  What the host can divide it
// divides (DecodePlan), and a workgroup finds its block in two trips to the arguments (at_once).  At the end a wave adds up its four row
// groups by itself, and the waves' sums, each scaled to its wave's maximum, are read behind one barrier.
// Eight waves a workgroup, and a workgroup a CU: as many rows in flight as with two of four waves, for half the rotations and half the
// partial rows.  The split that ends last reads those of its heads, which is the work of one CU: 64 KB with 64 splits, and with two trips for
// them and a round of its L2's lines given up first (a fence; now what is read is asked for past that cache) 6 us of a step behind
// 9,000 tokens, of which 3 are left: 1.3 until the rows are asked for, 0.4 until they are there.  The step's own key is a block of the list
// like the others (as one more of the last wave it came behind a whole block's microsecond of every other wave).  One pass, 32 / 8 heads of
// 128, four waves and this: causal behind 9,000 tokens 17.8 and 13.8 us, behind 32,768 30.0 and 28.1, stream-llm with its window of 4,096
// 18.1 and 12.8, 4 batch rows and a window of 2,048 23.7 and 20.1; 36 heads of 64 behind 2,000 / 16,000 tokens 14.5 / 38.1, now 12.0 / 29.2, 4 batch
// rows of 8,000 68.5 and 52.9; the streaming memory behind 512K tokens 26.4 and 24.8 (behind less the host bounds it).
struct DecodePlan {
    int32_t G, chunks;                     // query heads of a kv head; workgroups that share them
    int32_t blocks;                        // of all ranges
    int32_t end[kDecodeSegs];              // blocks of the ranges up to this one's last; behind the last range: INT32_MAX
};
// The arguments that lead to a workgroup's first loads, in ONE trip to them: the compiler fetched each where it was first used, which were
// nine trips behind one another.  A word of every line that holds the ranges comes along, so that the range found is a trip to the cache.
__device__ __forceinline__ void at_once(const DecodeJob &j, int &G, int &chunks, int &B, int &n_split, int (&ends)[kDecodeSegs - 1], StepQkv &r) {
    static_assert(kDecodeSegs == 6 && sizeof(DecodeSeg) == 80);
    const int near[7] = {(int)j.seg[0].k_sb, j.seg[0].n_ids, j.seg[1].n_ids, j.seg[2].n_ids, j.seg[3].n_ids, j.seg[4].n_ids, j.seg[5].n_ids};
    asm volatile("" : "+s"(G), "+s"(chunks), "+s"(B), "+s"(n_split), "+s"(ends[0]), "+s"(ends[1]), "+s"(ends[2]), "+s"(ends[3]), "+s"(ends[4]),
                      "+s"(r.q), "+s"(r.k), "+s"(r.v), "+s"(r.q_sb)
                    : "s"(r.inv_freq), "s"(r.q_sh), "s"(r.k_sb), "s"(r.k_sh), "s"(r.v_sb), "s"(r.v_sh), "s"(near[0]), "s"(near[1]), "s"(near[2]), "s"(near[3]),
                      "s"(near[4]), "s"(near[5]), "s"(near[6]));
}
template <int D, int NG, bool LOGITS, bool JOIN, typename Front = NoFront, bool SELECT = false>
__global__ __launch_bounds__(kDecWaves * kWave, 2) void decode_attn_kernel(DecodeJob j, DecodePlan plan, Front f) {
    constexpr bool FRONT = !std::is_same_v<Front, NoFront>;
    constexpr bool UNITS = !std::is_same_v<Front, StepRows>;
    constexpr int NEW = FRONT;                     // the step's own key: a block behind the last
    constexpr int KK = D / 32;                     // k-steps of the first MFMA
    constexpr int LPR = D / 8;                     // lanes that hold a value row, 16 bytes each
    constexpr int VL = kDecodeBlock * LPR / 64;    // value loads per block: 4 (D = 128) or 2 (D = 64)
    constexpr int kRed = kDecWaves * NG * D, kSel = SELECT ? (int)sizeof(SelectLds<kDecWaves * kWave>) / 4 : 0;
    __shared__ __attribute__((aligned(16))) float red_room[kRed > kSel ? kRed : kSel];
    float(*red)[NG][D] = (float(*)[NG][D])red_room;
    __shared__ float sm[kDecWaves][NG], sl[kDecWaves][NG];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int col = lane & 15, rg = lane >> 4;
    const int split = blockIdx.x, b = blockIdx.z;
    int G = plan.G, chunks = plan.chunks, B = j.B, n_split = j.nsplit, ends[kDecodeSegs - 1];
#pragma unroll
    for (int i = 0; i < kDecodeSegs - 1; ++i) ends[i] = plan.end[i];
    StepQkv own_rows{};
    if constexpr (FRONT) own_rows = f;
    at_once(j, G, chunks, B, n_split, ends, own_rows);
    int g = blockIdx.y, c = 0;
    if (chunks > 1) g = (int)blockIdx.y / chunks, c = (int)blockIdx.y - g * chunks;
    // the ranges that this workgroup's split is one of, and which one of how many
    const bool lead = SELECT && split < j.lead_splits;
    const int seg_lo = SELECT && !lead ? j.lead_segs : 0, seg_hi = lead ? j.lead_segs : j.n_seg;
    const int part = SELECT && !lead ? split - j.lead_splits : split, n_part = !SELECT ? n_split : lead ? j.lead_splits : n_split - j.lead_splits;
    if constexpr (FRONT) {
        if (b >= B) {
            const int x = split + n_split * ((int)blockIdx.y + j.Hkv * chunks * (b - B)), n_rows = B * j.Hkv;
            if constexpr (std::is_same_v<Front, MemoryRows>) {
                if (threadIdx.x >= 256) return;
                if (x < n_rows) ingest_one<D>(f.in, x / j.Hkv, x % j.Hkv, (float2 *)red_room);
            } else {
                const int at = x - n_rows, bg = at / max(f.pieces, 1);
                if (at < 0) {
                    if (threadIdx.x < 256) leave_rows<D>(f, x / j.Hkv, x % j.Hkv, (float2 *)red_room);
                } else if (at < n_rows * f.pieces) copy_rows<D, kStepCopyRows, kDecWaves * kWave>(f.copy, at - bg * f.pieces, bg / j.Hkv, bg % j.Hkv);
            }
            return;
        }
    }
    const int h0 = g * G + c * NG, nh = min(NG, G - c * NG);
    const float scale = j.scale * 1.4426950408889634f;
    const float lazy = kLazyDec / scale;

    // ---- the list of blocks: every range rounded up to whole blocks (units: every unit by itself)
    const int seg_first = seg_lo > 0 ? plan.end[seg_lo - 1] : 0, n_blocks = (SELECT ? plan.end[seg_hi - 1] : plan.blocks) - seg_first + NEW;
    const int each = n_blocks / n_part, over = n_blocks - each * n_part;                   // (of n_blocks * part / n_part, below)
    const int b_lo = seg_first + each * part + over * part / n_part, b_hi = seg_first + each * (part + 1) + over * (part + 1) / n_part - (NEW && split == n_split - 1);
    __shared__ int32_t chosen[SELECT ? kSelectMost : 1];
    if constexpr (SELECT) {
        if (lead) {
            select_units<kDecWaves * kWave>(j.unit_scores + (int64_t)b * j.unit_scores_sb, j.n_scores, j.seg[0].n_ids, chosen, *(SelectLds<kDecWaves * kWave> *)red_room);
            if (split == 0 && blockIdx.y == 0)
                for (int i = threadIdx.x; i < j.seg[0].n_ids; i += kDecWaves * kWave) {
                    j.ids_out[(int64_t)b * j.seg[0].n_ids + i] = chosen[i];
                    if (j.log) __hip_atomic_store(j.log + (int64_t)b * j.seg[0].n_ids + i, chosen[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                }
        }
    }

    struct Block {
        const bf16_t *k, *v;
        int valid, q, row;                         // rows of the block, which query, where its logits go (-1: nowhere)
    };
    auto find = [&](int blk) {                     // wave-uniform
        int s = 0, first = 0;
#pragma unroll
        for (int i = 0; i < kDecodeSegs - 1; ++i)
            if (blk >= ends[i]) s = i + 1, first = ends[i];
        blk -= first;
        const DecodeSeg sg = j.seg[s];
        Block r{nullptr, nullptr, 0, sg.q, -1};
        if (UNITS && sg.n_ids > 0) {
            const int per = (sg.rows + kDecodeBlock - 1) / kDecodeBlock, i = blk / per, r0 = (blk - i * per) * kDecodeBlock;
            const int u = __builtin_amdgcn_readfirstlane(SELECT ? chosen[i] : sg.ids ? sg.ids[(int64_t)b * sg.n_ids + i] : i);
            const int ch = u / j.per_chunk;
            const bf16_t *base = (const bf16_t *)(uintptr_t)j.chunk[ch] + (int64_t)(u - ch * j.per_chunk) * j.unit_elems + (int64_t)b * j.row_elems +
                                 (int64_t)g * j.unit_sh + (int64_t)r0 * D;
            r.k = base;
            r.v = base + j.unit_v_off;
            r.valid = min(kDecodeBlock, sg.rows - r0);
        } else {
            const int r0 = blk * kDecodeBlock;
            r.k = sg.k + (int64_t)b * sg.k_sb + (int64_t)g * sg.k_sh + (int64_t)r0 * D;
            r.v = sg.v + (int64_t)b * sg.v_sb + (int64_t)g * sg.v_sh + (int64_t)r0 * D;
            r.valid = min(kDecodeBlock, sg.rows - r0);
            if (LOGITS && sg.logit0 >= 0) r.row = sg.logit0 + r0;
        }
        return r;
    };

    u32x4 kbuf[2][KK], vbuf[2][VL];
    auto load = [&](const Block &bl, int buf) {    // rows beyond the range: its last row again, masked below
        const bf16_t *kr = bl.k + min(col, bl.valid - 1) * D + rg * 8;
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) kbuf[buf][kk] = __builtin_nontemporal_load((const u32x4 *)(kr + kk * 32));
#pragma unroll
        for (int i = 0; i < VL; ++i) {
            const int key = D == 128 ? 4 * rg + i : 4 * rg + 2 * i + (col >> 3);
            vbuf[buf][i] = __builtin_nontemporal_load((const u32x4 *)(bl.v + min(key, bl.valid - 1) * D + (lane & (LPR - 1)) * 8));
        }
    };

    __shared__ __attribute__((aligned(16))) bf16_t new_rows[FRONT ? 2 * NG + 1 : 1][FRONT ? D : 8];      // the queries at both angles, the new key
    bf16x8 qreg[KK];
    auto load_q = [&](int which) {
        if constexpr (FRONT) {
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) {
                const u32x4 raw = *(const u32x4 *)&new_rows[which * NG + min(col, nh - 1)][rg * 8 + kk * 32];
                qreg[kk] = __builtin_bit_cast(bf16x8, col < nh ? raw : u32x4{0, 0, 0, 0});
            }
            return;
        }
        const bf16_t *q = j.q[which] + (int64_t)b * j.q_sb + (int64_t)(h0 + min(col, nh - 1)) * j.q_sh + rg * 8;
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
            const u32x4 raw = *(const u32x4 *)(q + kk * 32);
            qreg[kk] = __builtin_bit_cast(bf16x8, col < nh ? raw : u32x4{0, 0, 0, 0});
        }
    };

    float m = -INFINITY, l = 0.f, neg_ms = 0.f;
    float acc[NG][8];
#pragma unroll
    for (int h = 0; h < NG; ++h)
#pragma unroll
        for (int d = 0; d < 8; ++d) acc[h][d] = 0.f;

    auto step = [&](const Block &bl, int buf) {
        f32x4 s{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, kbuf[buf][kk]), qreg[kk], s, 0, 0, 0);
        if (LOGITS && bl.row >= 0 && col < nh) {
            float *dst = j.logits + ((int64_t)b * j.H + h0 + col) * j.logit_stride + bl.row + 4 * rg;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (4 * rg + r < bl.valid) dst[r] = s[r] * scale;
        }
        if (bl.valid < kDecodeBlock) {
#pragma unroll
            for (int r = 0; r < 4; ++r) s[r] = 4 * rg + r < bl.valid ? s[r] : -INFINITY;
        }
        const float t = fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]));
        const bool moved = t > m + lazy;
        if (__builtin_amdgcn_ballot_w64(moved) != 0) {
            const float mn = moved ? t : m;
            const float al = moved ? __builtin_amdgcn_exp2f((m - mn) * scale) : 1.f;
            l *= al;
            each_head<NG>([&](auto hc) {
                constexpr int h = decltype(hc)::value;
                const float a = row_bcast<h>(al);
#pragma unroll
                for (int d = 0; d < 8; ++d) acc[h][d] *= a;
            });
            m = mn;
            neg_ms = m == -INFINITY ? 0.f : -m * scale;
        }
        if (bl.valid < kDecodeBlock) {                     // the repeated rows: 0 x infinity would be NaN
#pragma unroll
            for (int i = 0; i < VL; ++i)
                if ((D == 128 ? 4 * rg + i : 4 * rg + 2 * i + (col >> 3)) >= bl.valid) vbuf[buf][i] = u32x4{0, 0, 0, 0};
        }
        float p[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) p[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], scale, neg_ms));
        l += (p[0] + p[1]) + (p[2] + p[3]);
#pragma unroll
        for (int i = 0; i < VL; ++i) {
            float v[8];
#pragma unroll
            for (int w = 0; w < 4; ++w) v[2 * w] = bf16_bits_to_f32(vbuf[buf][i][w] & 0xffffu), v[2 * w + 1] = __uint_as_float(vbuf[buf][i][w] & 0xffff0000u);
            each_head<NG>([&](auto hc) {
                constexpr int h = decltype(hc)::value;
                float pb;
                if constexpr (D == 128) pb = row_bcast<h>(p[i]);
                else {
                    const float lo = row_bcast<h>(p[2 * i]), hi = row_bcast<h>(p[2 * i + 1]);
                    pb = (col >> 3) ? hi : lo;
                }
#pragma unroll
                for (int d = 0; d < 8; ++d) acc[h][d] = __builtin_fmaf(pb, v[d], acc[h][d]);
            });
        }
    };

    // The step's own rows are asked for ahead of the cache's, which would otherwise be waited for with them before the angles' chain
    // begins; two microseconds of the first block's six (workgroups begin their products at 4.4 instead of 6.6 us of a step that slides;
    // causal, one token over 32,768, 8 key heads of 128: 32.9 -> 31.5 us a pass).
    const int own = threadIdx.x / (D / 16), own_at = threadIdx.x % (D / 16) * 8;
    const bool is_q = own < nh, is_k = own == NG, has_new = FRONT && split == n_split - 1 && wave == (b_hi - b_lo) % kDecWaves;
    u32x4 own_lo{}, own_hi{}, new_v{};
    float freq = 0.f;
    if constexpr (FRONT) {
        const StepQkv &r = own_rows;
        freq = rope_freq<D / 2>(r.inv_freq);
        const bf16_t *q_rows = r.q + (int64_t)b * r.q_sb + (int64_t)h0 * r.q_sh, *k_row = r.k + (int64_t)b * r.k_sb + (int64_t)g * r.k_sh;
        asm volatile("" : "+s"(q_rows), "+s"(k_row));            // (both addresses; not that of the one to be read)
        if (is_q || is_k) {
            const bf16_t *src = (is_q ? q_rows + (int64_t)own * r.q_sh : k_row) + own_at;
            own_lo = *(const u32x4 *)src, own_hi = *(const u32x4 *)(src + D / 2);
        }
        if (has_new) new_v = *(const u32x4 *)(r.v + (int64_t)b * r.v_sb + (int64_t)g * r.v_sh + (lane & (LPR - 1)) * 8);
        asm volatile("" ::: "memory");
    }
    int q_now = -1, blk = b_lo + wave;
    Block cur{};
    if (blk < b_hi) {
        cur = find(blk);
        load(cur, 0);
    }
    if constexpr (FRONT) {
        constexpr int HALF = D / 2;
        float2 *cs = (float2 *)red_room;
        rope_angles<HALF>(f.pos, 1, f.glb_pos, f.distance_scale, freq, (float2(*)[HALF])cs, cs + HALF);
        __syncthreads();
        if (is_q || is_k) {
            Rot8 x = rotate8(own_lo, own_hi, cs + own_at);
            bf16_t *dst = new_rows[is_q ? own : 2 * NG] + own_at;
            *(u32x4 *)dst = x.lo, *(u32x4 *)(dst + HALF) = x.hi;
            if (is_q) {
                x = rotate8(own_lo, own_hi, cs + HALF + own_at);
                dst = new_rows[NG + own] + own_at;
                *(u32x4 *)dst = x.lo, *(u32x4 *)(dst + HALF) = x.hi;
            }
        }
        __syncthreads();
    }
    if (blk < b_hi) {
        load_q(cur.q);
        q_now = cur.q;
        for (int buf = 0; blk < b_hi; blk += 2 * kDecWaves) {        // two blocks per turn, so that the buffers are fixed registers
            Block nxt{};
            const bool more = blk + kDecWaves < b_hi;
            if (more) {
                nxt = find(blk + kDecWaves);
                load(nxt, 1);
            }
            if (cur.q != q_now) load_q(q_now = cur.q);
            step(cur, 0);
            if (!more) break;
            if (blk + 2 * kDecWaves < b_hi) {
                cur = find(blk + 2 * kDecWaves);
                load(cur, 0);
            }
            if (nxt.q != q_now) load_q(q_now = nxt.q);
            step(nxt, 1);
        }
    }
    if constexpr (FRONT) {
        if (has_new) {                                                         // the new key: a block of one
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) kbuf[0][kk] = *(const u32x4 *)&new_rows[2 * NG][rg * 8 + kk * 32];
#pragma unroll
            for (int i = 0; i < VL; ++i) vbuf[0][i] = new_v;
            if (q_now != 0) load_q(0);
            step(Block{nullptr, nullptr, 1, 0, LOGITS ? j.new_logit : -1}, 0);
        }
    }

    // ---- join the row groups of the wave, then the waves (m == -infinity: nothing seen yet, or logits that are no numbers, whose
    //      sums have to stay NaN)
    const float mw = wave_max32(wave_max16(m));
    const float to_mw = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((m - mw) * scale);
    float lw = m == -INFINITY ? l : l * to_mw;
    lw = wave_sum32(wave_sum16(lw));
    if (lane < NG) {
        sm[wave][lane] = mw;
        sl[wave][lane] = lw;
    }
    // (The row groups' sums trade places as they are added: rows of 16 lanes keep a half of the numbers at each of two steps, so that a
    // quarter of them goes through LDS, and none more than once.)
    constexpr int N8 = NG * 8;
    float x[N8];
    each_head<NG>([&](auto hc) {
        constexpr int h = decltype(hc)::value;
        const float f = row_bcast<h>(to_mw);
#pragma unroll
        for (int d = 0; d < 8; ++d) x[h * 8 + d] = acc[h][d] * f;
    });
#pragma unroll
    for (int i = 0; i < N8 / 2; ++i) {
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x[i]), __float_as_uint(x[i + N8 / 2]), false, false);
        x[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
#pragma unroll
    for (int i = 0; i < N8 / 4; ++i) {
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x[i]), __float_as_uint(x[i + N8 / 4]), false, false);
        x[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
        if (D == 64) x[i] += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x[i]), 0x128, 0xf, 0xf, true));   // the row's other half
    }
    if (col < LPR) {
        const int first = rg * (N8 / 4);
        float *dst = &red[wave][first / 8][col * 8 + first % 8];
        if constexpr (NG == 1) *(float2 *)dst = float2{x[0], x[1]};
        else
#pragma unroll
            for (int i = 0; i < N8 / 4; i += 4) *(f32x4 *)(dst + i) = f32x4{x[i], x[i + 1], x[i + 2], x[i + 3]};
    }
    __syncthreads();
    const int64_t row0 = ((int64_t)split * j.B + b) * j.H + h0;
    for (int e = threadIdx.x * 2; e < nh * D; e += kDecWaves * kWave * 2) {
        const int h = e / D, d = e % D;
        float mx = -INFINITY, den = 0.f;
        float2 o{0.f, 0.f};
#pragma unroll
        for (int w = 0; w < kDecWaves; ++w) mx = fmaxf(mx, sm[w][h]);
#pragma unroll
        for (int w = 0; w < kDecWaves; ++w) {
            const float f = sm[w][h] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((sm[w][h] - mx) * scale);
            den += sm[w][h] == -INFINITY ? sl[w][h] : sl[w][h] * f;
            const float2 ow = *(const float2 *)&red[w][h][d];
            o.x += ow.x * f, o.y += ow.y * f;
        }
        const f16x2 part{(_Float16)(den == 0.f ? 0.f : o.x / den), (_Float16)(den == 0.f ? 0.f : o.y / den)};
        const float lse = den > 0.f ? mx * scale + log2f(den) : -INFINITY;
        uint32_t *dst = (uint32_t *)(j.o_part + (row0 + h) * D + d);
        if (!JOIN) {
            *dst = __builtin_bit_cast(uint32_t, part);
            if (d == 0) j.lse_part[row0 + h] = lse;
        } else {                                   // (performed where every XCD sees it: the split that ends last reads it)
            __hip_atomic_store(dst, __builtin_bit_cast(uint32_t, part), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (d == 0) __hip_atomic_store(j.lse_part + row0 + h, lse, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    if constexpr (JOIN) {
        // ---- The split that ends last joins them: a launch of its own is 4.8 us, of which next to nothing is work.  Every split's
        //      stores have been performed before its ticket is drawn, and nothing else crosses workgroups, so that none has to
        //      write its L2 back.  Wave w takes every eighth split, a lane one head's 8 elements (merge_piece's arithmetic).
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        __shared__ int last;
        uint32_t *ticket = j.ticket + (int64_t)b * (j.Hkv * chunks) + blockIdx.y;
        if (threadIdx.x == 0) last = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (uint32_t)n_split - 1;
        __syncthreads();
        if (!last) return;
        asm volatile("" ::: "memory");
        if (threadIdx.x == 0) __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const int h = lane / LPR, at = (lane & (LPR - 1)) * 8;                 // (heads of 64: four of them are 32 lanes)
        const bool on = h < nh;
        // (a scalar address for each split, one offset for the lane)
        const int64_t rows = (int64_t)j.B * j.H, lead_row = wave * rows + (int64_t)b * j.H + h0;
        const uint32_t lane_l = (on ? h : 0) * 4, lane_o = (on ? h : 0) * (D * 2) + at * 2;
        const char *from_l = (const char *)(j.lse_part + lead_row), *from_o = (const char *)(j.o_part + lead_row * D);
        float mx = -INFINITY, den = 0.f, o[8] = {};
        constexpr int kBatch = 8;                  // splits whose rows are requested together: all of a wave's, up to 64 splits
        for (int s0 = wave; s0 < n_split; s0 += kBatch * kDecWaves) {
            float l8[kBatch];
            uint64_t lo[kBatch], hi[kBatch];
#pragma unroll
            for (int i = 0; i < kBatch; ++i) {
                l8[i] = -INFINITY, lo[i] = hi[i] = 0;
                if (s0 + i * kDecWaves < n_split) {
                    l8[i] = __hip_atomic_load((const float *)(from_l + lane_l), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    lo[i] = __hip_atomic_load((const uint64_t *)(from_o + lane_o), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    hi[i] = __hip_atomic_load((const uint64_t *)(from_o + lane_o + 8), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    from_l += rows * (kDecWaves * 4), from_o += rows * (kDecWaves * D * 2);
                }
            }
            float mn = mx;
#pragma unroll
            for (int i = 0; i < kBatch; ++i) mn = fmaxf(mn, l8[i]);
            const float al = mx == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mx - mn), base = mn == -INFINITY ? 0.f : mn;
            if (mx != -INFINITY) {
                den *= al;
#pragma unroll
                for (int d = 0; d < 8; ++d) o[d] *= al;
            }
#pragma unroll
            for (int i = 0; i < kBatch; ++i) {     // exp2(-inf) = 0: empty splits hold zeros, those with a logit that was no number NaN
                if (s0 + i * kDecWaves >= n_split) break;
                const float w = __builtin_amdgcn_exp2f(l8[i] - base);
                const f16x4 x = __builtin_bit_cast(f16x4, lo[i]), y = __builtin_bit_cast(f16x4, hi[i]);
#pragma unroll
                for (int d = 0; d < 4; ++d) o[d] += (float)x[d] * w, o[4 + d] += (float)y[d] * w;
                den += w;
            }
            mx = mn;
        }
        if (on) {
            float *mine = &red[wave][h][at];
            *(f32x4 *)mine = f32x4{o[0], o[1], o[2], o[3]};
            *(f32x4 *)(mine + 4) = f32x4{o[4], o[5], o[6], o[7]};
            if (at == 0) sm[wave][h] = mx, sl[wave][h] = den;
        }
        __syncthreads();
        for (int e = threadIdx.x * 2; e < nh * D; e += kDecWaves * kWave * 2) {
            const int eh = e / D, d = e % D;
            float most = -INFINITY, all = 0.f;
            float2 x{0.f, 0.f};
#pragma unroll
            for (int w = 0; w < kDecWaves; ++w) most = fmaxf(most, sm[w][eh]);
            const float base = most == -INFINITY ? 0.f : most;
#pragma unroll
            for (int w = 0; w < kDecWaves; ++w) {
                // (a wave whose splits are all empty or no numbers: its sums are zeros or NaN, taken with weight 0)
                const float f = __builtin_amdgcn_exp2f(sm[w][eh] - base);
                const float2 xw = *(const float2 *)&red[w][eh][d];
                x.x += xw.x * f, x.y += xw.y * f;
                all += sl[w][eh] * f;
            }
            const float inv = all > 0.f ? 1.f / all : 0.f;
            *(uint32_t *)(j.out + (int64_t)b * j.out_sb + (int64_t)(h0 + eh) * j.out_sh + d) = pack_bf16x2(x.x * inv, x.y * inv);
        }
    }
}

DecodePlan plan_of(const DecodeJob *job, int NG) {
    DecodePlan p{};
    p.G = job->H / job->Hkv;
    p.chunks = (p.G + NG - 1) / NG;
    int32_t n = 0;
    for (int s = 0; s < kDecodeSegs; ++s) {
        if (s < job->n_seg) n += (job->seg[s].rows + kDecodeBlock - 1) / kDecodeBlock * (job->seg[s].n_ids > 0 ? job->seg[s].n_ids : 1);
        p.end[s] = s < job->n_seg ? n : INT32_MAX;
    }
    p.blocks = n;
    return p;
}

template <int D, bool LOGITS, bool JOIN, bool SELECT = false>
int launch(const DecodeJob *job, void *stream) {
    const int G = job->H / job->Hkv;
    const int NG = G >= 3 ? 4 : G;
    const dim3 grid(job->nsplit, job->Hkv * ((G + NG - 1) / NG), job->B);
    const auto kern = NG == 1 ? decode_attn_kernel<D, 1, LOGITS, JOIN, NoFront, SELECT> : NG == 2 ? decode_attn_kernel<D, 2, LOGITS, JOIN, NoFront, SELECT>
                                                                                                  : decode_attn_kernel<D, 4, LOGITS, JOIN, NoFront, SELECT>;
    hipLaunchKernelGGL(kern, grid, dim3(kDecWaves * kWave), 0, (hipStream_t)stream, *job, plan_of(job, NG), NoFront{});
    INFLLM_CHECK_LAUNCH("decode_attn");
    return 0;
}

template <int D>
int launch_step(const DecodeJob *job, const StepRows *rows, void *stream) {
    const int G = job->H / job->Hkv, NG = G >= 3 ? 4 : G;
    const int y = job->Hkv * ((G + NG - 1) / NG);
    // The workgroups that write the cache come behind all splits, in batch rows of their own.  In the grid's first dimension, behind the
    // splits of every head, they take places of splits and leave again, so that some CUs get two splits and some none, and a row of
    // them spreads the heads of a group, which read the same keys, over the XCDs.  (With workgroups of four waves: causal steps of 8 key heads
    // over 24,000 / 32,768 / 49,152 tokens 31.8 / 39.3 / 52.1 us so, 29.3 / 33.2 / 42.4 behind all, 32.5 / 36.5 / 45.7 as two launches; of 2 key
    // heads with 16 query heads each over 65,536 / 98,304 60.9 / 88.2, 38.1 / 54.1 and 47.2 / 63.1.)
    const int64_t extra = (int64_t)(1 + rows->pieces) * job->Hkv * job->B, planes = (extra + (int64_t)job->nsplit * y - 1) / ((int64_t)job->nsplit * y);
    if (job->B + planes > 65535 || extra >= (1ll << 30)) return 1;
    const dim3 grid(job->nsplit, y, (unsigned)(job->B + planes));
    const auto kern = NG == 1 ? decode_attn_kernel<D, 1, false, true, StepRows> : NG == 2 ? decode_attn_kernel<D, 2, false, true, StepRows>
                                                                                  : decode_attn_kernel<D, 4, false, true, StepRows>;
    hipLaunchKernelGGL(kern, grid, dim3(kDecWaves * kWave), 0, (hipStream_t)stream, *job, plan_of(job, NG), *rows);
    INFLLM_CHECK_LAUNCH("decode_step");
    return 0;
}

// A step of the streaming memory that selects nothing: all its ranges are known, so its prologue can ride along.
template <int D>
int launch_memory_step(const DecodeJob *job, const infllm_ingest_args *in, void *stream) {
    const int G = job->H / job->Hkv, NG = G >= 3 ? 4 : G;
    const int y = job->Hkv * ((G + NG - 1) / NG);
    const int64_t planes = ((int64_t)job->B * job->Hkv + (int64_t)job->nsplit * y - 1) / ((int64_t)job->nsplit * y);
    INFLLM_REQUIRE(job->B + planes <= 65535, "decode_memory_step: a batch of %d", job->B);
    MemoryRows rows{};
    (StepQkv &)rows = StepQkv{(const bf16_t *)in->d_q, (const bf16_t *)in->d_k, (const bf16_t *)in->d_v, in->q_sb, in->q_sh, in->k_sb, in->k_sh, in->v_sb,
                              in->v_sh, in->pos0, in->glb_pos, in->d_inv_freq, in->distance_scale};
    rows.in = *in;
    const auto kern = NG == 1 ? decode_attn_kernel<D, 1, true, false, MemoryRows> : NG == 2 ? decode_attn_kernel<D, 2, true, false, MemoryRows>
                                                                                            : decode_attn_kernel<D, 4, true, false, MemoryRows>;
    hipLaunchKernelGGL(kern, dim3(job->nsplit, y, (unsigned)(job->B + planes)), dim3(kDecWaves * kWave), 0, (hipStream_t)stream, *job, plan_of(job, NG), rows);
    INFLLM_CHECK_LAUNCH("decode_memory_step");
    return 0;
}

}  // namespace

// Key splits of a decode step over `blocks` blocks of 16 keys, at most max_splits.  Few heads: as many as have a block for each of their
// waves and a CU of their own (heads of 64: half of one), but for what the workgroups beside them take.
//
// More heads, or some workgroups for the heads of a group (chunks): the splits whose launch is estimated to take least.  A workgroup takes
// the time of 3 blocks to begin and end, and its blocks.  Workgroups of the chunks read the same keys, and where they go to other XCDs each
// of those fetches them: round-robin by id, so the chunks of a split are on min(chunks, 8 / gcd(8, splits)) of them, every one more
// taken for 0.3 of a block's time.  The launch takes its rounds of 256 workgroups (two on a CU share what it reads in a time), or, where that is longer,
// the work of all, those that copy 256 rows (2 blocks' time; heads of 64: 1) among it.  Those that write a row come last, in places that are
// free by then.  (They were taken off the places before, and nobody counted XCDs: 32 / 8 heads of 128, 16 batch rows behind 2,000 / 4,000 /
// 16,000 tokens 41.9 / 74.5 / 265 us a step, one split on half of the chip, now 28.9 / 49.6 / 171; 40 / 40 heads, 3 rows behind 8,000 131 and 84;
// 16 heads of one key head, 8 rows behind 16,000 51.6 with 7 splits, 36.1 with 8; 64 / 8 heads, 6 rows of a full window of 4,096 91.6 and 65.6.
// Against all counts of splits tried one by one, over 1,006 steps of 13 geometries, the rule takes 2 % longer than the best: 1 % for heads of 128.)
extern "C" int infllm_decode_splits(int32_t B, int32_t H, int32_t Hkv, int32_t dim, int64_t blocks, int32_t max_splits, int64_t rows, int64_t copies) {
    const int G = H / Hkv, NG = G >= 3 ? 4 : G, chunks = (G + NG - 1) / NG;
    const int64_t wgs = (int64_t)B * Hkv * chunks, places = (dim == 64 ? 512 : 256) - std::min<int64_t>(rows + copies, 128);
    const int64_t most = std::max<int64_t>(1, std::min<int64_t>((blocks + kDecWaves - 1) / kDecWaves, max_splits));
    if (chunks == 1 && wgs * (dim == 64 || copies ? 4 : 16) <= places) return (int)std::min(places / wgs, most);
    int best = 1;
    double best_time = INFINITY;
    for (int s = 1; s <= most; ++s) {
        const int xcds = std::min(chunks, 8 / std::gcd(8, s));
        const double one = 3 + (double)blocks / (kDecWaves * s) * (1 + 0.3 * (xcds - 1));
        const double time = std::max((double)((wgs * s + 255) / 256) * one, ((double)(wgs * s) * one + (double)copies * (dim == 64 ? 1 : 2)) / 256);
        if (time < best_time * (1 - 1e-9)) best = s, best_time = time;
    }
    return best;
}

static int check_job(const DecodeJob *job, int32_t dim) {
    INFLLM_REQUIRE(job && job->o_part && job->lse_part, "decode_attn: null pointer");
    INFLLM_REQUIRE(job->B > 0 && job->H > 0 && job->Hkv > 0 && job->H % job->Hkv == 0 && job->B <= 65535, "decode_attn: bad geometry B=%d H=%d Hkv=%d", job->B,
                   job->H, job->Hkv);
    INFLLM_REQUIRE(job->n_seg >= 0 && job->n_seg <= kDecodeSegs && job->nsplit >= 1 && job->nsplit <= 128, "decode_attn: %d ranges, %d splits", job->n_seg,
                   job->nsplit);
    for (int s = 0; s < job->n_seg; ++s) {
        const DecodeSeg &sg = job->seg[s];
        INFLLM_REQUIRE(sg.rows >= 0 && (sg.q == 0 || sg.q == 1), "decode_attn: bad range");
        if (sg.n_ids > 0) INFLLM_REQUIRE(job->chunk && job->per_chunk > 0, "decode_attn: units without an arena");
        else INFLLM_REQUIRE(sg.rows == 0 || (sg.k && sg.v), "decode_attn: null range");
    }
    INFLLM_REQUIRE(dim == 128 || dim == 64, "decode_attn: head_dim %d", dim);
    return 0;
}

// rows: the step's own (their strides multiples of 8 elements); job->out and job->ticket are set, the ranges are plain ones.  Returns
// 1, with nothing launched, where the grid does not hold the batch.
int infllm_decode_step(const DecodeJob *job, const StepRows *rows, int32_t dim, void *stream) {
    const int rc = check_job(job, dim);
    if (rc) return rc;
    INFLLM_REQUIRE(rows && rows->q && rows->k && rows->v && rows->inv_freq && rows->dk && rows->dv && rows->pieces >= 0, "decode_step: null pointer");
    INFLLM_REQUIRE(job->out && job->ticket && !job->logits && ((job->out_sb | job->out_sh) & 7) == 0, "decode_step: bad output");
    return dim == 128 ? launch_step<128>(job, rows, stream) : launch_step<64>(job, rows, stream);
}

// in: the prologue of the step, as infllm_ingest_dim takes it; the job's ranges leave out its key, job->new_logit is that key's place.
// (A batch of up to 32,767.)
int infllm_decode_memory_step(const DecodeJob *job, const infllm_ingest_args *in, int32_t dim, void *stream) {
    const int rc = check_job(job, dim);
    if (rc) return rc;
    INFLLM_REQUIRE(in && in->n == 1 && in->d_q && in->d_k && in->d_v && in->d_inv_freq && in->d_ring_k_raw && in->d_ring_k_rot && in->d_ring_v &&
                       in->d_ring_score && in->d_q_loc && in->d_q_glb && job->logits, "decode_memory_step: null pointer");
    INFLLM_REQUIRE(in->B == job->B && in->H == job->H && in->Hkv == job->Hkv && in->pos0 >= 0 && in->ring_cap > 0, "decode_memory_step: bad geometry");
    INFLLM_REQUIRE((in->q_sl % 8 | in->q_sh % 8 | in->q_sb % 8 | in->k_sl % 8 | in->k_sh % 8 | in->k_sb % 8 | in->v_sl % 8 | in->v_sh % 8 | in->v_sb % 8) == 0,
                   "decode_memory_step: strides must be multiples of 8 elements (16-byte rows)");
    return dim == 128 ? launch_memory_step<128>(job, in, stream) : launch_memory_step<64>(job, in, stream);
}

// How many of a launch's splits the ranges get that wait for a selection (lead_blocks of 16 keys) so that they end with the others: the
// selection is taken for as long as two blocks of a wave.  It reads all scores twice and lasts the longer the more there are, but with many
// splits the launch depends little on where between two and nine the line lies; few splits are cut differently.  (The kernel alone, us, taken for
// 1, 2, 3, 6 and 9 blocks.  32 / 8 heads of 128, 32 splits, 16 of 20 / 479 / 4,096 / 16,000 units: 13.8 11.1 11.2 11.3 11.1 / 13.3 11.6 11.4 11.9
// 11.8 / 14.0 11.8 12.0 11.8 12.0 / 17.1 14.8 14.8 14.8 14.6; 64 of 4,096: 20.6 20.5 21.0 20.6 20.6.  32 / 32 heads, 8 splits, 16 of 20 / 479:
// 21.6 21.7 24.8 24.8 30.5 / 22.4 22.5 22.7 25.0 30.3.  36 heads of 64, 14 splits, 16 of 512: 14.9 14.1 14.0 14.0 14.0.)
extern "C" int infllm_decode_lead_splits(int32_t nsplit, int64_t lead_blocks, int64_t blocks) {
    int best = 1;
    int64_t best_time = INT64_MAX;
    for (int s = 1; s < nsplit; ++s) {
        const int64_t lead = kDecWaves * s, rest = kDecWaves * (nsplit - s), time = std::max((lead_blocks + lead - 1) / lead + 2, (blocks + rest - 1) / rest);
        if (time < best_time) best = s, best_time = time;
    }
    return best;
}

int infllm_decode_attn(const DecodeJob *job, int32_t dim, void *stream) {
    const int rc = check_job(job, dim);
    if (rc) return rc;
    INFLLM_REQUIRE(job->q[0] && job->q[1] && job->n_seg >= 1, "decode_attn: no query or range");
    INFLLM_REQUIRE(!job->out || (!job->logits && job->ticket && ((job->out_sb | job->out_sh) & 7) == 0), "decode_attn: bad output");
    if (job->unit_scores) {
        INFLLM_REQUIRE(job->logits && job->ids_out && job->lead_segs >= 1 && job->lead_segs < job->n_seg && job->lead_splits >= 1 && job->lead_splits < job->nsplit,
                       "decode_attn: bad selection");
        for (int s = 0; s < job->n_seg; ++s)
            INFLLM_REQUIRE(s == 0 ? job->seg[s].n_ids >= 1 && job->seg[s].n_ids <= kSelectMost && job->seg[s].n_ids <= job->n_scores : job->seg[s].n_ids == 0,
                           "decode_attn: the first range, and no other, is that of the units");
        return dim == 128 ? launch<128, true, false, true>(job, stream) : launch<64, true, false, true>(job, stream);
    }
    if (job->logits) return dim == 128 ? launch<128, true, false>(job, stream) : launch<64, true, false>(job, stream);
    if (job->out) return dim == 128 ? launch<128, false, true>(job, stream) : launch<64, false, true>(job, stream);
    return dim == 128 ? launch<128, false, false>(job, stream) : launch<64, false, false>(job, stream);
}
