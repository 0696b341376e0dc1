// One call of an attention type with a plain cache - attention sinks + sliding window (inf_llm/attention/stream_llm.py:6-111,
// infinite_lm.py:6-100) or causal attention (origin.py:4-79) - in two or three launches: the new tokens' rows (rotary
// embedding, cache), the attention, and the merge of its key splits where several queries have any.  A step is one launch.
#include <algorithm>

#include "decode.h"
#include "rope.h"

int infllm_attn_window(const infllm_attn_args *local, const infllm_attn_args *sinks, const void *q_angles, const void *sink_angle, int32_t dim, void *d_out,
                       int64_t o_sb, int64_t o_sh, int64_t o_sl, void *stream);
bool infllm_attn_turns(int32_t H, int32_t Hkv, int32_t n_q, int64_t q_sl, int32_t dim);
namespace {

struct StageJob {
    const bf16_t *q, *k, *v;                   // new rows
    int64_t q_sb, q_sh, q_sl, k_sb, k_sh, k_sl, v_sb, v_sh, v_sl;
    int32_t B, H, Hkv, n;                      // n: rows of the q (or k / v) part
    int32_t do_q, do_kv;
    int64_t pos0, glb_pos;                     // position of row 0; the one angle of the sinks' queries
    const float *inv_freq;
    double distance_scale;
    bf16_t *q_loc, *q_glb;                     // [B, H, n, D]; q_glb NULL: not wanted
    float2 *pos_cs;                            // [n, D / 2] cosine and sine of every position and frequency (NULL: not wanted)
    float2 *glb_cs;                            // cosine and sine of every frequency at the sinks' angle (NULL: not wanted)
    bf16_t *dk, *dv;                           // where row 0 of head 0 goes, rotated / as it is
    int64_t dk_sb, dk_sh, dv_sb, dv_sh;
    // A second place for some of the rows (NULL: none): row p is row r = c_first + p of all that the call sees; those with
    // r < c_head go to row r, those with r >= c_tail to row c_head + r - c_tail.
    bf16_t *ck, *cv;
    int64_t ck_sb, ck_sh, cv_sb, cv_sh;
    int32_t c_first, c_head, c_tail;
    bf16_t *raw;                               // where un-rotated row 0 goes, rows [0, n_raw)
    int64_t raw_sb, raw_sh;
    int32_t n_raw;
    int32_t tiles;                             // workgroups along x that stage rows; the rest copy
    uint32_t *clear;                           // n_clear words to set to zero (tickets: of the decode kernel, or of steps to come)
    int32_t n_clear;
    RowCopy copy[kCopies];
};

// Bound by HBM for a prompt (a row read, one to three written), by the latency of the fp64 angles for a step.  grid =
// (position tiles of 16, then pieces of the row copies; batch rows; groups of KG kv heads): a workgroup rotates the query heads of its
// kv heads and their key heads at 16 positions.  (One wave per row with its own sincos, a launch for every tensor and
// angle, and torch.cat for the cache: 13 launches and 2.1 x the bytes per call.)
template <int D, int KG>
__global__ __launch_bounds__(256) void stage_rows_kernel(StageJob j) {
    constexpr int HALF = D / 2, C2 = D / 16;           // chunk pairs of a row
    __shared__ float2 cs_pos[kPosPerBlock][HALF];
    __shared__ float2 cs_glb[HALF];
    const int tid = threadIdx.x, b = blockIdx.y, g0 = blockIdx.z * KG, ng = KG == 1 ? 1 : min(KG, j.Hkv - g0);
    if ((int)blockIdx.x >= j.tiles) {
        for (int kg = 0; kg < ng; ++kg) copy_rows<D, kCopyRows>(j.copy, (int)blockIdx.x - j.tiles, b, g0 + kg);
        return;
    }
    if (blockIdx.x == 0 && b == 0 && g0 == 0)
        for (int i = tid; i < j.n_clear; i += 256) j.clear[i] = 0;
    const int h0 = g0 * (j.H / j.Hkv), n_heads = ng * (j.H / j.Hkv);
    const int p0 = blockIdx.x * kPosPerBlock, np = min(kPosPerBlock, j.n - p0);
    const float freq = rope_freq<HALF>(j.inv_freq);
    // ---- requests first: up to four query heads, the key heads, the value heads
    constexpr int kRound = 256 / (kPosPerBlock * C2), kItems = 4 / kRound;          // 2 (D = 128) or 1 (D = 64)
    constexpr int kKItems = (KG * kPosPerBlock * C2 + 255) / 256, kVItems = (KG * kPosPerBlock * 2 * C2 + 255) / 256;
    u32x4 q_lo[kItems], q_hi[kItems], k_lo[kKItems], k_hi[kKItems], v_row[kVItems];
    const bf16_t *q = j.q + (int64_t)b * j.q_sb + (int64_t)h0 * j.q_sh;
    const int qc = tid % C2, qp = tid / C2 % kPosPerBlock, qh = tid / (C2 * kPosPerBlock);
    if (j.do_q) {
#pragma unroll
        for (int i = 0; i < kItems; ++i)
            if (i * kRound + qh < n_heads && qp < np) {
                const bf16_t *src = q + (int64_t)(i * kRound + qh) * j.q_sh + (int64_t)(p0 + qp) * j.q_sl;
                q_lo[i] = *(const u32x4 *)(src + qc * 8);
                q_hi[i] = *(const u32x4 *)(src + HALF + qc * 8);
            }
    }
    if (j.do_kv) {
#pragma unroll
        for (int i = 0; i < kKItems; ++i) {
            const int e = tid + i * 256, c = e % C2, p = e / C2 % kPosPerBlock, kg = e / (C2 * kPosPerBlock);
            if (p < np && kg < ng) {
                const bf16_t *src = j.k + (int64_t)b * j.k_sb + (int64_t)(g0 + kg) * j.k_sh + (int64_t)(p0 + p) * j.k_sl;
                k_lo[i] = *(const u32x4 *)(src + c * 8);
                k_hi[i] = *(const u32x4 *)(src + HALF + c * 8);
            }
        }
#pragma unroll
        for (int i = 0; i < kVItems; ++i) {
            const int e = tid + i * 256, c = e % (2 * C2), p = e / (2 * C2) % kPosPerBlock, kg = e / (2 * C2 * kPosPerBlock);
            if (p < np && kg < ng) v_row[i] = *(const u32x4 *)(j.v + (int64_t)b * j.v_sb + (int64_t)(g0 + kg) * j.v_sh + (int64_t)(p0 + p) * j.v_sl + c * 8);
        }
    }
    rope_angles<HALF>(j.pos0 + p0, np, j.glb_pos, j.distance_scale, freq, cs_pos, cs_glb);
    __syncthreads();
    if (j.pos_cs && b == 0 && g0 == 0)
        for (int i = tid; i < np * HALF; i += 256) j.pos_cs[(int64_t)p0 * HALF + i] = cs_pos[0][i];
    if (j.glb_cs && blockIdx.x == 0 && b == 0 && g0 == 0 && tid < HALF) j.glb_cs[tid] = cs_glb[tid];
    if (j.do_q) {
        for (int hg0 = 0; hg0 < n_heads; hg0 += 4) {
#pragma unroll
            for (int i = 0; i < kItems; ++i) {
                const int hl = hg0 + i * kRound + qh;
                if (hl >= n_heads || qp >= np) continue;
                u32x4 lo = q_lo[i], hi = q_hi[i];
                if (hg0 > 0) {
                    const bf16_t *src = q + (int64_t)hl * j.q_sh + (int64_t)(p0 + qp) * j.q_sl;
                    lo = *(const u32x4 *)(src + qc * 8), hi = *(const u32x4 *)(src + HALF + qc * 8);
                }
                const int64_t o = (((int64_t)b * j.H + h0 + hl) * j.n + p0 + qp) * D;
                Rot8 r = rotate8(lo, hi, &cs_pos[qp][qc * 8]);
                *(u32x4 *)(j.q_loc + o + qc * 8) = r.lo;
                *(u32x4 *)(j.q_loc + o + HALF + qc * 8) = r.hi;
                if (j.q_glb) {
                    r = rotate8(lo, hi, &cs_glb[qc * 8]);
                    *(u32x4 *)(j.q_glb + o + qc * 8) = r.lo;
                    *(u32x4 *)(j.q_glb + o + HALF + qc * 8) = r.hi;
                }
            }
        }
    }
    if (j.do_kv) {
        auto second = [&](int p) {
            if (!j.ck) return -1;
            const int r = j.c_first + p;
            return r < j.c_head ? r : r >= j.c_tail ? j.c_head + r - j.c_tail : -1;
        };
#pragma unroll
        for (int i = 0; i < kKItems; ++i) {
            const int e = tid + i * 256, c = e % C2, p = e / C2 % kPosPerBlock, kg = e / (C2 * kPosPerBlock);
            if (p >= np || kg >= ng) continue;
            bf16_t *dst = j.dk + (int64_t)b * j.dk_sb + (int64_t)(g0 + kg) * j.dk_sh + (int64_t)(p0 + p) * D;
            const Rot8 r = rotate8(k_lo[i], k_hi[i], &cs_pos[p][c * 8]);
            *(u32x4 *)(dst + c * 8) = r.lo;
            *(u32x4 *)(dst + HALF + c * 8) = r.hi;
            const int at = second(p0 + p);
            if (at >= 0) {
                dst = j.ck + (int64_t)b * j.ck_sb + (int64_t)(g0 + kg) * j.ck_sh + (int64_t)at * D;
                *(u32x4 *)(dst + c * 8) = r.lo;
                *(u32x4 *)(dst + HALF + c * 8) = r.hi;
            }
            if (p0 + p < j.n_raw) {
                bf16_t *raw = j.raw + (int64_t)b * j.raw_sb + (int64_t)(g0 + kg) * j.raw_sh + (int64_t)(p0 + p) * D;
                *(u32x4 *)(raw + c * 8) = k_lo[i];
                *(u32x4 *)(raw + HALF + c * 8) = k_hi[i];
            }
        }
#pragma unroll
        for (int i = 0; i < kVItems; ++i) {
            const int e = tid + i * 256, c = e % (2 * C2), p = e / (2 * C2) % kPosPerBlock, kg = e / (2 * C2 * kPosPerBlock);
            if (p >= np || kg >= ng) continue;
            *(u32x4 *)(j.dv + (int64_t)b * j.dv_sb + (int64_t)(g0 + kg) * j.dv_sh + (int64_t)(p0 + p) * D + c * 8) = v_row[i];
            const int at = second(p0 + p);
            if (at >= 0) *(u32x4 *)(j.cv + (int64_t)b * j.cv_sb + (int64_t)(g0 + kg) * j.cv_sh + (int64_t)at * D + c * 8) = v_row[i];
        }
    }
}

int launch_stage_rows(StageJob &j, int dim, void *stream) {
    int pieces = 0;
    for (const RowCopy &c : j.copy) pieces += (c.n + kCopyRows - 1) / kCopyRows;
    j.tiles = j.do_q || j.do_kv ? (j.n + kPosPerBlock - 1) / kPosPerBlock : 0;
    if (j.tiles + pieces == 0) return 0;
    const int kg = heads_together(j.n, j.B, j.do_q ? j.H : j.Hkv, j.Hkv);
    const dim3 grid(j.tiles + pieces, j.B, (j.Hkv + kg - 1) / kg);
    const auto kern = dim == 128 ? (kg == 4 ? stage_rows_kernel<128, 4> : kg == 2 ? stage_rows_kernel<128, 2> : stage_rows_kernel<128, 1>)
                                 : (kg == 4 ? stage_rows_kernel<64, 4> : kg == 2 ? stage_rows_kernel<64, 2> : stage_rows_kernel<64, 1>);
    hipLaunchKernelGGL(kern, grid, dim3(256), 0, (hipStream_t)stream, j);
    INFLLM_CHECK_LAUNCH("stage_rows");
    return 0;
}

}  // namespace

// Key splits of a launch over `wgs` workgroups of up to `tiles` key tiles each, `mean_tiles` on average.  A workgroup costs
// about 6 us to start and drain plus 1.9 us per tile (a CU holds one), 256 of them run at a time, and splits cost a merge of
// 5 us; the smallest estimate wins.  Equal workgroups run in rounds; where the first queries see few keys (a prompt's first
// call) the short workgroups fill up behind the long ones, which start first, so that the launch lasts as long as its longest
// or as its sum, and a quarter of its longest more where the chip does not hold it at once (causal, one call of 32 heads:
// 1,500 tokens 60 -> 51 us and 2,048 tokens 77.7 -> 71.7 with two splits, where rounds said one).
// The constants are those of heads of 128.  Heads of 64 (a CU holds two of their workgroups) and the operator's stages take
// them too: against the best of 1, 2, 3, 4, 6 and 8 splits forced, whole passes - causal prompts of 1,500 / 2,500 / 4,001 tokens,
// 32 heads of 128: 71.3 / 110.3 / 179.2 us by the rule, 68.5 / 109.8 / 178.6 best; 36 heads of 64: 66.2 / 113.8 / 178.4, 64.2 /
// 113.7 / 177.2 best; the operator's two stages of 300 / 512 / 900 queries: 53.3 / 57.6 / 80.7, 52.5 / 57.8 / 82.8 best, 36 heads of
// 64 in rows of 128 120.5 / 124.9 / 178.8, 119.8 / 124.0 / 178.8 best; of 64 queries 58.9 by the rule (11 splits), 52.6 best (6).
// max_parts: splits that the partial rows have room for.
int infllm_attn_splits(int64_t wgs, int64_t tiles, int32_t max_parts, double mean_tiles) {
    const bool equal = mean_tiles > 0.9 * (double)tiles;
    int best = 1;
    double best_us = 0;
    for (int s = 1; s <= std::min(max_parts, 32) && (s == 1 || tiles / s >= 2); ++s) {
        const double longest = 6.0 + 1.9 * (double)((tiles + s - 1) / s);
        const double all = (double)(wgs * s) * (6.0 + 1.9 * mean_tiles / s) / 256.0;
        const double us = (equal ? (double)((wgs * s + 255) / 256) * longest : std::max(longest, all) + (wgs * s > 256 ? 0.25 * longest : 0.0)) +
                          (s > 1 ? 5.0 : 0.0);
        if (s == 1 || us < best_us) best = s, best_us = us;
    }
    return best;
}

extern "C" int infllm_window_forward(const infllm_window_args *a, void *stream) {
    INFLLM_REQUIRE(a != nullptr, "window_forward: null argument block");
    INFLLM_REQUIRE(a->dim == 128 || a->dim == 64, "window_forward: head_dim %d is not 64 or 128", a->dim);
    INFLLM_REQUIRE(a->B > 0 && a->H > 0 && a->Hkv > 0 && a->H % a->Hkv == 0 && a->B <= 65535 && a->Hkv <= 65535, "window_forward: bad geometry B=%d H=%d Hkv=%d",
                   a->B, a->H, a->Hkv);
    INFLLM_REQUIRE(a->n_q > 0 && a->n_new > 0 && a->kind >= 0 && a->kind <= 2 && a->n_init >= 0 && a->seen >= 0, "window_forward: bad sizes");
    INFLLM_REQUIRE(a->d_q && a->d_k && a->d_v && a->d_inv_freq && a->d_cache_k && a->d_cache_v && a->d_work && a->d_out, "window_forward: null pointer");
    INFLLM_REQUIRE(((a->q_sb | a->q_sh | a->q_sl | a->k_sb | a->k_sh | a->k_sl | a->v_sb | a->v_sh | a->v_sl | a->ok_sb | a->ok_sh | a->ov_sb | a->ov_sh |
                     a->ck_sb | a->ck_sh | a->cv_sb | a->cv_sh | a->o_sb | a->o_sh | a->o_sl) & 7) == 0,
                   "window_forward: strides must be multiples of 8 elements");
    const bool causal = a->kind == 0, inplace = a->d_old_k == a->d_cache_k && a->rows_old > 0;
    const int64_t rows_all = (int64_t)a->rows_old + a->n_new, len_k = a->seen + a->n_new;
    const bool cut = a->rows_new < rows_all;
    INFLLM_REQUIRE(a->rows_old >= 0 && a->rows_new > 0 && a->rows_new <= rows_all && (a->rows_old == 0 || (a->d_old_k && a->d_old_v)), "window_forward: bad cache rows");
    INFLLM_REQUIRE(a->rows_old <= a->seen && a->n_q <= rows_all, "window_forward: more cached rows or queries than tokens");
    INFLLM_REQUIRE(!cut || (!causal && a->rows_new >= a->n_init && a->rows_new - a->n_init >= std::min<int64_t>(a->n_local, rows_all)), "window_forward: cut cache too short");
    INFLLM_REQUIRE(!cut || a->d_all_k || (a->n_q == 1 && a->n_new == 1), "window_forward: a cut cache does not hold what several queries see");
    INFLLM_REQUIRE(!inplace || (!cut && a->ok_sb == a->ck_sb && a->ok_sh == a->ck_sh && a->d_old_v == a->d_cache_v && a->ov_sb == a->cv_sb && a->ov_sh == a->cv_sh),
                   "window_forward: in place needs the same strides and an uncut cache");
    INFLLM_REQUIRE((a->d_all_k != nullptr) == (a->d_all_v != nullptr), "window_forward: all_k without all_v");
    INFLLM_REQUIRE(a->softmax_scale > 0.f, "window_forward: softmax scale");
    const int D = a->dim;
    const int64_t q_elems = (int64_t)a->B * a->H * a->n_q * D;
    const bool sink_stage = !causal && len_k > a->n_local && a->n_init > 0;
    const int n_sink = sink_stage ? (int)std::min<int64_t>(a->n_init, rows_all) : 0;
    INFLLM_REQUIRE(!sink_stage || a->kind != 2 || (a->d_raw && a->raw_new >= n_sink), "window_forward: un-rotated sinks missing");
    const int64_t q_bytes = (causal ? 1 : 2) * q_elems * 2;
    const int64_t rows_q = (int64_t)a->B * a->H * a->n_q;
    // partial rows: what is left behind the queries (and a ticket per head, for a step)
    const int64_t part_rows = std::max<int64_t>(0, a->work_bytes - q_bytes - (a->n_q == 1 ? 4 * rows_q : 0)) / (2 * D + 4);
    const int max_parts = (int)std::min<int64_t>(part_rows / rows_q, 64);
    const bool step = a->n_q == 1 && max_parts >= 1;
    const bool fresh = a->d_ticket && a->ticket_fresh != 0;
    uint32_t *ticket = fresh ? (uint32_t *)a->d_ticket : (uint32_t *)((char *)a->d_work + q_bytes + part_rows * (2 * D + 4));
    INFLLM_REQUIRE(a->work_bytes >= q_bytes, "window_forward: scratch of %lld bytes for %lld", (long long)a->work_bytes, (long long)q_bytes);
    bf16_t *q_loc = (bf16_t *)a->d_work, *q_sink = causal ? nullptr : q_loc + q_elems;

    // ---- where the attention reads its keys: everything, or the new cache
    const bool all = a->d_all_k != nullptr;
    bf16_t *bk = (bf16_t *)(all ? a->d_all_k : a->d_cache_k), *bv = (bf16_t *)(all ? a->d_all_v : a->d_cache_v);
    const int64_t bk_sh = all ? rows_all * D : a->ck_sh, bk_sb = all ? bk_sh * a->Hkv : a->ck_sb;
    const int64_t bv_sh = all ? rows_all * D : a->cv_sh, bv_sb = all ? bv_sh * a->Hkv : a->cv_sb;
    const int64_t rows_base = all ? rows_all : a->rows_new;

    StageJob j{};
    j.B = a->B; j.H = a->H; j.Hkv = a->Hkv;
    j.q = (const bf16_t *)a->d_q; j.k = (const bf16_t *)a->d_k; j.v = (const bf16_t *)a->d_v;
    j.q_sb = a->q_sb; j.q_sh = a->q_sh; j.q_sl = a->q_sl;
    j.k_sb = a->k_sb; j.k_sh = a->k_sh; j.k_sl = a->k_sl;
    j.v_sb = a->v_sb; j.v_sh = a->v_sh; j.v_sl = a->v_sl;
    j.glb_pos = a->kind == 2 ? a->n_local - 1 : a->n_local + a->n_init - 1;
    j.inv_freq = a->d_inv_freq; j.distance_scale = a->distance_scale;
    j.q_loc = q_loc;
    // Queries are rotated to the sinks' angle where they are attended, by a table of it in their place, which two rows fill and one
    // row does not hold.
    const bool sink_turns = sink_stage && !step && rows_q >= 2;
    if (sink_turns) j.glb_cs = (float2 *)q_sink;
    else if (sink_stage) j.q_glb = q_sink;
    j.dk = bk + (rows_base - a->n_new) * D; j.dv = bv + (rows_base - a->n_new) * D;
    j.dk_sb = bk_sb; j.dk_sh = bk_sh; j.dv_sb = bv_sb; j.dv_sh = bv_sh;
    const int64_t raw_sh = (int64_t)a->raw_new * D;
    if (a->raw_new > a->raw_old) {
        INFLLM_REQUIRE(a->d_raw && a->raw_old == a->seen && a->raw_new - a->raw_old <= a->n_new && (a->raw_old == 0 || a->d_raw_old), "window_forward: bad sink rows");
        j.raw = (bf16_t *)a->d_raw + (int64_t)a->raw_old * D;
        j.raw_sh = raw_sh; j.raw_sb = raw_sh * a->Hkv;
        j.n_raw = a->raw_new - a->raw_old;
    }
    if (step || fresh) j.clear = ticket, j.n_clear = a->B * a->H;
    int nc = 0;
    auto copy = [&](const void *src, int64_t ss_b, int64_t ss_h, int64_t s_row, void *dst, int64_t ds_b, int64_t ds_h, int64_t d_row, int64_t n) {
        if (n > 0) j.copy[nc++] = RowCopy{(const bf16_t *)src + s_row * D, (bf16_t *)dst + d_row * D, ss_b, ss_h, ds_b, ds_h, (int32_t)n};
    };
    if (all || !cut) {
        if (!inplace) {
            copy(a->d_old_k, a->ok_sb, a->ok_sh, 0, bk, bk_sb, bk_sh, 0, a->rows_old);
            copy(a->d_old_v, a->ov_sb, a->ov_sh, 0, bv, bv_sb, bv_sh, 0, a->rows_old);
        }
    } else {                                    // one new row: the sinks, and the tail without its oldest rows
        const int64_t tail = a->rows_new - a->n_init - a->n_new, from = a->rows_old - tail;
        copy(a->d_old_k, a->ok_sb, a->ok_sh, 0, bk, bk_sb, bk_sh, 0, a->n_init);
        copy(a->d_old_v, a->ov_sb, a->ov_sh, 0, bv, bv_sb, bv_sh, 0, a->n_init);
        copy(a->d_old_k, a->ok_sb, a->ok_sh, from, bk, bk_sb, bk_sh, a->n_init, tail);
        copy(a->d_old_v, a->ov_sb, a->ov_sh, from, bv, bv_sb, bv_sh, a->n_init, tail);
    }
    if (all) {
        // The new cache - all rows, or the sinks and the tail - besides everything: old rows are copied to both places, new ones
        // written to both.  (Copied out of everything by a launch behind this
        // one: sinks + window over 16,001 tokens 1,077 us, so 1,063.)
        const int64_t head = cut ? a->n_init : a->rows_new, tail0 = rows_all - (a->rows_new - head), old_head = std::min<int64_t>(head, a->rows_old);
        copy(a->d_old_k, a->ok_sb, a->ok_sh, 0, a->d_cache_k, a->ck_sb, a->ck_sh, 0, old_head);
        copy(a->d_old_v, a->ov_sb, a->ov_sh, 0, a->d_cache_v, a->cv_sb, a->cv_sh, 0, old_head);
        copy(a->d_old_k, a->ok_sb, a->ok_sh, tail0, a->d_cache_k, a->ck_sb, a->ck_sh, head, a->rows_old - tail0);
        copy(a->d_old_v, a->ov_sb, a->ov_sh, tail0, a->d_cache_v, a->cv_sb, a->cv_sh, head, a->rows_old - tail0);
        j.ck = (bf16_t *)a->d_cache_k; j.cv = (bf16_t *)a->d_cache_v;
        j.ck_sb = a->ck_sb; j.ck_sh = a->ck_sh; j.cv_sb = a->cv_sb; j.cv_sh = a->cv_sh;
        j.c_first = a->rows_old; j.c_head = (int32_t)head; j.c_tail = (int32_t)tail0;
    }
    if (j.n_raw > 0 && a->raw_old > 0)
        copy(a->d_raw_old, (int64_t)a->raw_old * D * a->Hkv, (int64_t)a->raw_old * D, 0, a->d_raw, raw_sh * a->Hkv, raw_sh, 0, a->raw_old);
    // ---- A step whose old rows hold all it sees but its own key is one launch.
    int rc;
    const int64_t near_rows = causal ? rows_base : std::min<int64_t>(rows_base, a->n_local);       // of the new cache, the last of them the new one
    const int64_t far_rows = std::max<int64_t>(0, std::min<int64_t>(n_sink, len_k - a->n_local));  // sink j is seen from a distance of at least n_local
    const void *raw_from = a->raw_new > a->raw_old ? a->d_raw_old : a->d_raw;
    const int64_t raw_from_sh = (int64_t)(a->raw_new > a->raw_old ? a->raw_old : a->raw_new) * D;
    if (step && a->n_new == 1 && !all && a->d_ticket && !fresh && near_rows >= 1 && near_rows - 1 <= a->rows_old && far_rows <= a->rows_old &&
        (far_rows == 0 || a->kind != 2 || (raw_from && far_rows * D <= raw_from_sh))) {
        DecodeJob d{};
        d.B = a->B; d.H = a->H; d.Hkv = a->Hkv;
        d.scale = a->softmax_scale;
        const bf16_t *ok = (const bf16_t *)a->d_old_k, *ov = (const bf16_t *)a->d_old_v;
        const int64_t near_old = near_rows - 1, from = a->rows_old - near_old;
        if (near_old > 0) d.seg[d.n_seg++] = DecodeSeg{ok + from * D, ov + from * D, a->ok_sb, a->ok_sh, a->ov_sb, a->ov_sh, (int32_t)near_old, 0, 0, nullptr, -1};
        if (far_rows > 0)
            d.seg[d.n_seg++] = a->kind == 2 ? DecodeSeg{(const bf16_t *)raw_from, ov, raw_from_sh * a->Hkv, raw_from_sh, a->ov_sb, a->ov_sh, (int32_t)far_rows, 1, 0, nullptr, -1}
                                            : DecodeSeg{ok, ov, a->ok_sb, a->ok_sh, a->ov_sb, a->ov_sh, (int32_t)far_rows, 1, 0, nullptr, -1};
        StepRows f{};
        for (int i = 0; i < kCopies; ++i) {
            f.copy[i] = j.copy[i];
            f.pieces += (j.copy[i].n + kStepCopyRows - 1) / kStepCopyRows;
        }
        d.nsplit = infllm_decode_splits(a->B, a->H, a->Hkv, D, (near_old + kDecodeBlock - 1) / kDecodeBlock + (far_rows + kDecodeBlock - 1) / kDecodeBlock + 1, max_parts,
                                        (int64_t)a->Hkv * a->B, (int64_t)f.pieces * a->Hkv * a->B);
        d.o_part = (uint16_t *)((char *)a->d_work + q_bytes);
        d.lse_part = (float *)((char *)a->d_work + q_bytes + part_rows * 2 * D);
        d.out = (bf16_t *)a->d_out; d.out_sb = a->o_sb; d.out_sh = a->o_sh;
        d.ticket = (uint32_t *)a->d_ticket;
        f.q = j.q; f.k = j.k; f.v = j.v;
        f.q_sb = a->q_sb; f.q_sh = a->q_sh; f.k_sb = a->k_sb; f.k_sh = a->k_sh; f.v_sb = a->v_sb; f.v_sh = a->v_sh;
        f.pos = a->seen; f.glb_pos = j.glb_pos;
        f.inv_freq = a->d_inv_freq; f.distance_scale = a->distance_scale;
        f.dk = j.dk; f.dv = j.dv; f.dk_sb = j.dk_sb; f.dk_sh = j.dk_sh; f.dv_sb = j.dv_sb; f.dv_sh = j.dv_sh;
        if (j.n_raw > 0) f.raw = j.raw, f.raw_sb = j.raw_sb, f.raw_sh = j.raw_sh;
        rc = infllm_decode_step(&d, &f, D, stream);
        if (rc != 1) return rc;
    }
    // The attention rotates the queries itself, where it can, by a table of cosines and sines in their place (which hold it from two heads
    // on): the staging reads and writes 67 MB less of 4,096 tokens x 32 heads of 128.  Staged / so, 32 / 8 heads of 128, causal prompts of
    // 1,537 / 2,049 / 3,073 / 8,001 tokens 60.9 / 80.5 / 114.9 / 549.7 and 59.6 / 78.0 / 111.3 / 535.4 us; sinks + window of 1,024 over 1,537 /
    // 3,073 67.5 / 101.8 and 67.2 / 101.3; below, the host bounds them.
    // (Straight into LDS, 16 bytes a lane: rows that begin between two such pieces are staged, by loads into registers.)
    const bool turns = !step && a->n_q == a->n_new && (int64_t)a->B * a->H >= 2 && infllm_attn_turns(a->H, a->Hkv, a->n_q, a->q_sl, D) &&
                       ((uintptr_t)a->d_q & 15) == 0;
    if (a->n_q == a->n_new) {
        j.do_q = !turns;
        j.do_kv = 1;
        if (turns) j.pos_cs = (float2 *)q_loc;
        j.n = a->n_q;
        j.pos0 = a->seen;
        rc = launch_stage_rows(j, D, stream);
        if (rc) return rc;
    } else {                                    // queries and keys at different positions: a launch for each
        j.do_kv = 1;
        j.n = a->n_new;
        j.pos0 = a->seen;
        rc = launch_stage_rows(j, D, stream);
        if (rc) return rc;
        j.do_q = 1;
        j.do_kv = 0;
        j.n = a->n_q;
        j.pos0 = len_k - a->n_q;
        for (RowCopy &c : j.copy) c.n = 0;
        rc = launch_stage_rows(j, D, stream);
        if (rc) return rc;
    }
    // ---- attention
    const bf16_t *sk = a->kind == 2 ? (const bf16_t *)a->d_raw : bk;
    const int64_t sk_sh = a->kind == 2 ? raw_sh : bk_sh, sk_sb = a->kind == 2 ? raw_sh * a->Hkv : bk_sb;
    const float scale = a->softmax_scale;
    if (step) {
        DecodeJob d{};
        d.q[0] = q_loc; d.q[1] = sink_stage ? q_sink : q_loc;
        d.q_sb = (int64_t)a->H * D; d.q_sh = D;
        d.B = a->B; d.H = a->H; d.Hkv = a->Hkv;
        d.scale = scale;
        const int64_t near = near_rows;                                                              // the last rows
        d.seg[0] = DecodeSeg{bk + (rows_base - near) * D, bv + (rows_base - near) * D, bk_sb, bk_sh, bv_sb, bv_sh, (int32_t)near, 0, 0, nullptr, -1};
        d.n_seg = 1;
        const int64_t far = far_rows;
        if (far > 0) d.seg[d.n_seg++] = DecodeSeg{sk, bv, sk_sb, sk_sh, bv_sb, bv_sh, (int32_t)far, 1, 0, nullptr, -1};
        const int64_t blocks = (near + kDecodeBlock - 1) / kDecodeBlock + (far > 0 ? (far + kDecodeBlock - 1) / kDecodeBlock : 0);
        d.nsplit = infllm_decode_splits(a->B, a->H, a->Hkv, D, blocks, max_parts, 0, 0);
        d.o_part = (uint16_t *)((char *)a->d_work + q_bytes);
        d.lse_part = (float *)((char *)a->d_work + q_bytes + part_rows * 2 * D);
        d.out = (bf16_t *)a->d_out; d.out_sb = a->o_sb; d.out_sh = a->o_sh;
        d.ticket = ticket;
        return infllm_decode_attn(&d, D, stream);
    }
    infllm_attn_args l{}, s{};
    if (turns) {
        l.d_q = a->d_q;
        l.q_sl = a->q_sl; l.q_sh = a->q_sh; l.q_sb = a->q_sb;
    } else {
        l.d_q = q_loc;
        l.q_sl = D; l.q_sh = (int64_t)a->n_q * D; l.q_sb = (int64_t)a->H * a->n_q * D;
    }
    l.B = a->B; l.H = a->H; l.Hkv = a->Hkv; l.Lq = a->n_q;
    l.d_k = bk; l.d_v = bv;
    l.k_sl = l.v_sl = D;
    l.k_sh = bk_sh; l.k_sb = bk_sb; l.v_sh = bv_sh; l.v_sb = bv_sb;
    l.cap = 1ll << 40;
    l.mask = INFLLM_MASK_WINDOW;
    l.offset = rows_base - a->n_q;
    l.window = causal ? rows_base : a->n_local;
    l.j_lo = std::max<int64_t>(0, rows_base - a->n_q - l.window + 1);
    l.j_hi = rows_base;
    l.softmax_scale = scale;
    if (sink_stage) {
        s = l;
        if (sink_turns) {
            s.d_q = a->d_q;
            s.q_sl = a->q_sl; s.q_sh = a->q_sh; s.q_sb = a->q_sb;
        } else
            s.d_q = q_sink;
        s.d_k = sk; s.k_sh = sk_sh; s.k_sb = sk_sb;
        s.j_lo = 0; s.j_hi = n_sink;
        s.mask = INFLLM_MASK_COMPLEMENT;
        s.offset = len_k - a->n_q; s.window = a->n_local;
    }
    const int64_t wgs = ((int64_t)((a->n_q + 31) / 32) * (a->H / a->Hkv) + 7) / 8 * a->Hkv * a->B;
    const int64_t tiles = (std::min<int64_t>(l.window + 64, l.j_hi - l.j_lo) + kTile - 1) / kTile + (n_sink + kTile - 1) / kTile;
    // queries whose window is not full yet see half of what they could, on average
    const int64_t ramp = std::min<int64_t>(a->n_q, std::max<int64_t>(0, l.window - 1 - l.offset));
    const double near = ((double)ramp * ((double)l.offset + 0.5 * (double)(ramp + 1)) + (double)(a->n_q - ramp) * (double)l.window) / a->n_q;
    l.nsplit = infllm_attn_splits(wgs, tiles, max_parts, std::min((double)tiles, (near + n_sink) / kTile + 1.0));
    l.d_o_part = (uint16_t *)((char *)a->d_work + q_bytes);
    l.d_lse_part = (float *)((char *)a->d_work + q_bytes + part_rows * 2 * D);
    return infllm_attn_window(&l, sink_stage ? &s : nullptr, j.pos_cs, j.glb_cs, D, a->d_out, a->o_sb, a->o_sh, a->o_sl, stream);
}
