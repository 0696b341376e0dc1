// Attention of ONE query per head (a decode step) over a list of key ranges; see decode.hip.
#pragma once
#include "common.h"

constexpr int kDecodeSegs = 6;
constexpr int kDecodeBlock = 16;           // keys a wave takes at a time

// `rows` consecutive rows of D elements, row stride D, of every (batch row, kv head).  With `ids` the rows are those of
// `n_ids` units of `rows` rows each, unit u of batch row b at chunk[u / per_chunk] + (u % per_chunk) * unit_elems + b *
// row_elems, where its keys are followed by its values (v_off elements on), heads k_sh apart.
struct DecodeSeg {
    const bf16_t *k, *v;
    int64_t k_sb, k_sh, v_sb, v_sh;
    int32_t rows, q;                       // q: which of the job's two rotations of the query this range is attended with
    int32_t n_ids;
    const int32_t *ids;                    // [B, n_ids] on the device, NULL: a plain range
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
    // Optional, without logits: the launch joins its splits itself, the finished row of head h goes to out + b * out_sb + h * out_sh.
    bf16_t *out;
    int64_t out_sb, out_sh;
    uint32_t *ticket;                      // [B * H] zeros, zeros again behind the launch
};

int infllm_decode_splits(int32_t B, int32_t H, int32_t Hkv, int64_t blocks, int32_t max_splits);
int infllm_decode_attn(const DecodeJob *job, int32_t dim, void *stream);
