// Attention of ONE query per head (a decode step) over a list of key ranges; see decode.hip.
#pragma once
#include "common.h"

constexpr int kDecodeSegs = 6;
constexpr int kDecodeBlock = 16;           // keys a wave takes at a time

// `rows` consecutive rows of D elements, row stride D, of every (batch row, kv head).  With `n_ids` > 0 the rows are
// those of `n_ids` units of `rows` rows each, unit u of batch row b at chunk[u / per_chunk] + (u % per_chunk) * unit_elems + b *
// row_elems, where its keys are followed by its values (v_off elements on), heads k_sh apart.
struct DecodeSeg {
    const bf16_t *k, *v;
    int64_t k_sb, k_sh, v_sb, v_sh;
    int32_t rows, q;                       // q: which of the job's two rotations of the query this range is attended with
    int32_t n_ids;
    const int32_t *ids;                    // [B, n_ids] on the device, NULL: units 0, 1, .. (n_ids > 0) or a plain range
    int32_t logit0;                        // row r's scaled logit goes to logits[.., logit0 + r]; -1: not kept
};

struct DecodeJob {
    const bf16_t *q[2];                    // [B, H, D] (strides q_sb, q_sh), each
    int64_t q_sb, q_sh;
    int32_t B, H, Hkv, n_seg;
    float scale;                           // softmax scale (natural)
    int32_t nsplit;
    uint16_t *o_part;                      // [nsplit, B, H, D] fp16
    float *lse_part;                       // [nsplit, B, H]
    DecodeSeg seg[kDecodeSegs];
    // for ranges of units
    const uint64_t *chunk;                 // device: address of every chunk of units
    int32_t per_chunk;
    int64_t unit_elems, row_elems, unit_v_off, unit_sh;
    float *logits;                         // optional [B, H, logit_stride]: scaled logits in base 2 (see DecodeSeg)
    int64_t logit_stride;
    int32_t new_logit;                     // of a step with its rows: where the new key's logit goes (-1: not kept)
    // Optional: the launch selects the units itself (the one range of units, n_ids of them; `ids` is not read): the best of the
    // n_scores units with scores at unit_scores + b * unit_scores_sb, into ids_out [B, n_ids] too.  The first lead_segs ranges, with the
    // units among them, belong to the first lead_splits splits, the others to the rest.
    const float *unit_scores;
    int64_t unit_scores_sb;
    int32_t n_scores, lead_segs, lead_splits;
    int32_t *ids_out, *log;                // log (optional, the host's memory): [B, n_ids] too
    // Optional, without logits: the launch joins its splits itself, the finished row of head h goes to out + b * out_sb + h * out_sh.
    bf16_t *out;
    int64_t out_sb, out_sh;
    uint32_t *ticket;                      // [B * H] zeros, zeros again behind the launch
};

// rows [0, n) of a source to a destination, for every (batch row, kv head); rows are D elements apart on both sides
struct RowCopy {
    const bf16_t *src;
    bf16_t *dst;
    int64_t s_sb, s_sh, d_sb, d_sh;
    int32_t n;
};
constexpr int kCopies = 7;
// Rows that a copying workgroup moves: of a staging launch (256 threads), and beside the splits of a step (512), which waits for the last of
// them, where few and long ones find room.  (One token over a full window, 64 / 128 / 256 rows: 72 heads of 64, window of 2,048, 28.6 / 23.1 /
// 21.7 us; heads of 128 with workgroups of 256, window of 4,096: 64 rows 22.9, 256 rows 21.0.)
constexpr int kCopyRows = 64;
constexpr int kStepCopyRows = 256;

template <int D, int kRows, int THREADS = 256>
__device__ __forceinline__ void copy_rows(const RowCopy (&copies)[kCopies], int piece, int b, int g) {
    const int tid = threadIdx.x;
    int c = 0;
    for (; c < kCopies; ++c) {
        const int n = (copies[c].n + kRows - 1) / kRows;
        if (piece < n) break;
        piece -= n;
    }
    if (c == kCopies) return;
    const RowCopy &rc = copies[c];
    const int r0 = piece * kRows, m = min(kRows, rc.n - r0) * (D / 8);
    const u32x4 *src = (const u32x4 *)(rc.src + (int64_t)b * rc.s_sb + (int64_t)g * rc.s_sh + (int64_t)r0 * D);
    u32x4 *dst = (u32x4 *)(rc.dst + (int64_t)b * rc.d_sb + (int64_t)g * rc.d_sh + (int64_t)r0 * D);
    constexpr int U = kRows * (D / 8) / THREADS;
    u32x4 x[U];
#pragma unroll
    for (int i = 0; i < U; ++i) x[i] = src[min(tid + THREADS * i, m - 1)];              // (every one loaded: conditions here made the compiler spill)
#pragma unroll
    for (int i = 0; i < U; ++i)
        if (tid + THREADS * i < m) dst[tid + THREADS * i] = x[i];
}

// The rows of the step itself, as they come (DecodeJob's ranges are the rows that were there before, its q is not used): the
// launch rotates the query to its position and to the angle of the sinks or units, and attends the new key.
struct StepQkv {
    const bf16_t *q, *k, *v;               // [B, H, D], [B, Hkv, D]
    int64_t q_sb, q_sh, k_sb, k_sh, v_sb, v_sh;
    int64_t pos, glb_pos;
    const float *inv_freq;
    double distance_scale;
};
// ... of the sliding-window and causal types: it also leaves the key and the value where the cache has them, with the copies of
// old rows that the cache needs.
struct StepRows : StepQkv {
    bf16_t *dk, *dv, *raw;                 // rotated key, value, key as it is (NULL: nowhere)
    int64_t dk_sb, dk_sh, dv_sb, dv_sh, raw_sb, raw_sh;
    RowCopy copy[kCopies];
    int32_t pieces;                        // copying workgroups per (batch row, kv head)
};

int infllm_decode_step(const DecodeJob *job, const StepRows *rows, int32_t dim, void *stream);
// rows, copies: workgroups beside the splits that write a row each, and that copy rows
extern "C" int infllm_decode_splits(int32_t B, int32_t H, int32_t Hkv, int32_t dim, int64_t blocks, int32_t max_splits, int64_t rows, int64_t copies);
int infllm_decode_memory_step(const DecodeJob *job, const infllm_ingest_args *in, int32_t dim, void *stream);
int infllm_decode_attn(const DecodeJob *job, int32_t dim, void *stream);
extern "C" int infllm_decode_lead_splits(int32_t nsplit, int64_t lead_blocks, int64_t blocks);
