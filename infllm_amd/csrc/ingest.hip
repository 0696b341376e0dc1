// Prologue of the streaming path: RoPE of new tokens and their staging into the
// per-layer rings (inf_llm/attention/rope.py:89-112,
// inf_llm/attention/context_manager.py:719-747, 373-375).
#include "rope.h"

namespace {

// grid = (position tiles of 16, batch rows, groups of KG kv heads): a workgroup rotates the query heads of its kv heads plus
// their key heads, copies their value heads, and leaves the sum of its rotated-to-one-position queries over its positions in
// d_qpart (for the block's mean query; summed before the rounding to bf16, so the mean query carries no rounding of its own).
//
// Angles (rope_angles): the rows the workgroup will rotate are requested from memory BEFORE that arithmetic, so the
// two overlap.
//
// Bound by HBM, as long as the angles hide behind the rows (heads_together) and enough rows are on their way: the sums take their
// 16 KB of LDS for a round of heads at a time, so that six workgroups are on a CU (for all four heads at once 41 KB and three: 8,192
// tokens of 32 / 8 heads of 128 61.9 -> 53.3 us = 5.3 TB/s, 1,998 tokens 17.8 -> 14.6).
//
// D: head dimension (128 or 64).  qbar (optional): where the mean of the queries goes when the launch has a single
// position tile (a decode step), whose partial sum is the whole sum.
template <int D, int KG>
__global__ __launch_bounds__(256) void ingest_kernel(infllm_ingest_args a, float *qbar) {
    constexpr int kHalf = D / 2, C2 = D / 16;          // rotation pairs of a head; pairs of 16-byte chunks of a row
    constexpr int kRound = 256 / (kPosPerBlock * C2);  // query heads that 256 threads rotate at once: 2 (4)
    __shared__ float2 cs_pos[kPosPerBlock][kHalf];
    __shared__ float2 cs_glb[kHalf];
    __shared__ float red[kRound][kPosPerBlock][D];   // their q_glb, for the partial sums
    const int tid = threadIdx.x;
    const int b = blockIdx.y, g0 = blockIdx.z * KG, ng = KG == 1 ? 1 : min(KG, a.Hkv - g0);
    const int h0 = g0 * (a.H / a.Hkv), n_heads = ng * (a.H / a.Hkv);
    const int p0 = blockIdx.x * kPosPerBlock;
    const int np = min(kPosPerBlock, a.n - p0);

    const bf16_t *q = (const bf16_t *)a.d_q + (int64_t)b * a.q_sb + (int64_t)h0 * a.q_sh;
    const bf16_t *k = (const bf16_t *)a.d_k + (int64_t)b * a.k_sb + (int64_t)g0 * a.k_sh;
    const bf16_t *v = (const bf16_t *)a.d_v + (int64_t)b * a.v_sb + (int64_t)g0 * a.v_sh;
    bf16_t *q_loc = (bf16_t *)a.d_q_loc + ((int64_t)b * a.H + h0) * a.n * D;
    bf16_t *q_glb = (bf16_t *)a.d_q_glb + ((int64_t)b * a.H + h0) * a.n * D;
    const int64_t ring_g = ((int64_t)b * a.Hkv + g0) * a.ring_cap * D;
    const int n_tiles = (a.n + kPosPerBlock - 1) / kPosPerBlock;

    const float freq = rope_freq<kHalf>(a.d_inv_freq);
    // ---- requests first: the first (up to) 4 query heads, the key heads, the value heads
    constexpr int kQItems = 4 / kRound, kKItems = (KG * kPosPerBlock * C2 + 255) / 256, kVItems = (KG * kPosPerBlock * 2 * C2 + 255) / 256;
    u32x4 q_lo[kQItems], q_hi[kQItems], k_lo[kKItems], k_hi[kKItems], v_row[kVItems];
    const int qc = tid % C2, qp = tid / C2 % kPosPerBlock, qh = tid / (C2 * kPosPerBlock);      // of a round of heads
#pragma unroll
    for (int i = 0; i < kQItems; ++i) {
        if (qp < np && i * kRound + qh < n_heads) {
            const bf16_t *src = q + (int64_t)(i * kRound + qh) * a.q_sh + (int64_t)(p0 + qp) * a.q_sl;
            q_lo[i] = *(const u32x4 *)(src + qc * 8);
            q_hi[i] = *(const u32x4 *)(src + kHalf + qc * 8);
        }
    }
#pragma unroll
    for (int i = 0; i < kKItems; ++i) {
        const int e = tid + i * 256, c = e % C2, p = e / C2 % kPosPerBlock, kg = e / (C2 * kPosPerBlock);
        if (p < np && kg < ng) {
            const bf16_t *src = k + (int64_t)kg * a.k_sh + (int64_t)(p0 + p) * a.k_sl;
            k_lo[i] = *(const u32x4 *)(src + c * 8);
            k_hi[i] = *(const u32x4 *)(src + kHalf + c * 8);
        }
    }
#pragma unroll
    for (int i = 0; i < kVItems; ++i) {
        const int e = tid + i * 256, c = e % (2 * C2), p = e / (2 * C2) % kPosPerBlock, kg = e / (2 * C2 * kPosPerBlock);
        if (p < np && kg < ng) v_row[i] = *(const u32x4 *)(v + (int64_t)kg * a.v_sh + (int64_t)(p0 + p) * a.v_sl + c * 8);
    }

    // ---- angles
    rope_angles<kHalf>(a.pos0 + p0, np, a.glb_pos, a.distance_scale, freq, cs_pos, cs_glb);
    __syncthreads();

    // query heads, 4 at a time: C2 threads per (head, position) row
    for (int hg0 = 0; hg0 < n_heads; hg0 += 4) {
#pragma unroll
        for (int i = 0; i < kQItems; ++i) {
            const int h = hg0 + i * kRound + qh;
            if (qp < np && h < n_heads) {
                u32x4 lo = q_lo[i], hi = q_hi[i];
                if (hg0 > 0) {
                    const bf16_t *src = q + (int64_t)h * a.q_sh + (int64_t)(p0 + qp) * a.q_sl;
                    lo = *(const u32x4 *)(src + qc * 8), hi = *(const u32x4 *)(src + kHalf + qc * 8);
                }
                const int64_t o = ((int64_t)h * a.n + p0 + qp) * D;
                Rot8 r = rotate8(lo, hi, &cs_pos[qp][qc * 8]);
                *(u32x4 *)(q_loc + o + qc * 8) = r.lo;
                *(u32x4 *)(q_loc + o + kHalf + qc * 8) = r.hi;
                float raw[16];
                r = rotate8(lo, hi, &cs_glb[qc * 8], raw);
                *(u32x4 *)(q_glb + o + qc * 8) = r.lo;
                *(u32x4 *)(q_glb + o + kHalf + qc * 8) = r.hi;
                if (a.d_qpart || qbar) {
                    *(f32x4 *)&red[qh][qp][qc * 8] = f32x4{raw[0], raw[1], raw[2], raw[3]};
                    *(f32x4 *)&red[qh][qp][qc * 8 + 4] = f32x4{raw[4], raw[5], raw[6], raw[7]};
                    *(f32x4 *)&red[qh][qp][kHalf + qc * 8] = f32x4{raw[8], raw[9], raw[10], raw[11]};
                    *(f32x4 *)&red[qh][qp][kHalf + qc * 8 + 4] = f32x4{raw[12], raw[13], raw[14], raw[15]};
                }
            }
            if (a.d_qpart || qbar) {
                __syncthreads();
                const int d = tid % D, rh = tid / D, hs = hg0 + i * kRound + rh;
                static_assert(kRound * D == 256);
                if (hs < n_heads) {
                    float s = 0.f;
                    for (int p = 0; p < np; ++p) s += red[rh][p][d];          // fixed order
                    if (qbar) qbar[((int64_t)b * a.H + h0 + hs) * D + d] = s * (1.f / (float)a.n);
                    else a.d_qpart[(((int64_t)b * n_tiles + blockIdx.x) * a.H + h0 + hs) * D + d] = s;
                }
                __syncthreads();
            }
        }
    }
    // key heads: raw copy + rotated copy into the rings
#pragma unroll
    for (int i = 0; i < kKItems; ++i) {
        const int e = tid + i * 256, c = e % C2, p = e / C2 % kPosPerBlock, kg = e / (C2 * kPosPerBlock);
        if (p >= np || kg >= ng) continue;
        const int64_t o = ring_g + (kg * a.ring_cap + (a.pos0 + p0 + p) % a.ring_cap) * D;
        bf16_t *rk_raw = (bf16_t *)a.d_ring_k_raw + o, *rk_rot = (bf16_t *)a.d_ring_k_rot + o;
        *(u32x4 *)(rk_raw + c * 8) = k_lo[i];
        *(u32x4 *)(rk_raw + kHalf + c * 8) = k_hi[i];
        Rot8 r = rotate8(k_lo[i], k_hi[i], &cs_pos[p][c * 8]);
        *(u32x4 *)(rk_rot + c * 8) = r.lo;
        *(u32x4 *)(rk_rot + kHalf + c * 8) = r.hi;
    }
    // value heads: plain copy
#pragma unroll
    for (int i = 0; i < kVItems; ++i) {
        const int e = tid + i * 256, c = e % (2 * C2), p = e / (2 * C2) % kPosPerBlock, kg = e / (2 * C2 * kPosPerBlock);
        if (p < np && kg < ng) *(u32x4 *)((bf16_t *)a.d_ring_v + ring_g + (kg * a.ring_cap + (a.pos0 + p0 + p) % a.ring_cap) * D + c * 8) = v_row[i];
    }
    // the score track of a new token starts at zero (context_manager.py:733-741)
    for (int e = tid; e < n_heads * kPosPerBlock; e += 256) {
        const int p = e % kPosPerBlock, h = h0 + e / kPosPerBlock;
        if (p < np) a.d_ring_score[((int64_t)b * a.H + h) * a.ring_cap + (a.pos0 + p0 + p) % a.ring_cap] = 0.f;
    }
}

// out[b, c] = scale * sum_p parts[b, p, c], p ascending.  A workgroup owns 64 columns; its 4 waves fetch different
// partials, so that 32 of them are one round trip to memory (a chain of dependent loads is all latency, and that
// latency multiplies while a unit fetch keeps the memory fabric busy); the sum itself runs in the fixed order.
// With blockIdx.z > 0 the partials are those of several execution blocks ingested by one launch: block z owns
// blk_parts consecutive partials (the last block what is left of n_parts) and exc positions (the last what is left of
// n_rows), its mean goes to out[z, b, :] and its scale is 1 / (its positions).
__global__ __launch_bounds__(256) void reduce_partials_kernel(const float *parts, int n_parts, int C, float scale,
                                                              float *out, int blk_parts, int n_rows, int exc) {
    __shared__ float stage[32][64];
    const int lane = threadIdx.x & 63, grp = threadIdx.x >> 6;
    const int c = blockIdx.x * 64 + lane, b = blockIdx.y, z = blockIdx.z;
    const float *src = parts + ((int64_t)b * n_parts + (int64_t)z * blk_parts) * C + c;
    out += (int64_t)z * gridDim.y * C;
    if (blk_parts < n_parts) {
        n_parts = min(blk_parts, n_parts - z * blk_parts);
        scale = 1.f / (float)min(exc, n_rows - z * exc);
    }
    float s = 0.f;
    for (int p0 = 0; p0 < n_parts; p0 += 32) {
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int p = p0 + grp + 4 * i;
            v[i] = (c < C && p < n_parts) ? src[(int64_t)p * C] : 0.f;
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) stage[grp + 4 * i][lane] = v[i];
        __syncthreads();
        if (grp == 0) {
            const int m = min(32, n_parts - p0);
            for (int p = 0; p < m; ++p) s += stage[p][lane];
        }
        __syncthreads();
    }
    if (grp == 0 && c < C) out[(int64_t)b * C + c] = s * scale;
}

constexpr int kMeanThreads = 512;

// one workgroup per (block, head, batch row); fixed summation order => deterministic
__global__ __launch_bounds__(kMeanThreads) void block_mean_kernel(const bf16_t *q_glb, int H, int n, int exc,
                                                                 float *qbar, int n_blocks) {
    __shared__ float2 part[kMeanThreads / 64][64];
    const int blk = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
    const int lane = threadIdx.x & 63, grp = threadIdx.x >> 6;
    const int r0 = blk * exc, r1 = min(r0 + exc, n);
    const bf16_t *src = q_glb + ((int64_t)b * H + h) * (int64_t)n * kD;
    float s0 = 0.f, s1 = 0.f;
    for (int r = r0 + grp; r < r1; r += kMeanThreads / 64) {
        uint32_t w = *(const uint32_t *)(src + (int64_t)r * kD + lane * 2);
        s0 += bf16_bits_to_f32(w & 0xffffu);
        s1 += bf16_bits_to_f32(w >> 16);
    }
    part[grp][lane] = make_float2(s0, s1);
    __syncthreads();
    if (grp == 0) {
        float t0 = 0.f, t1 = 0.f;
        for (int g = 0; g < kMeanThreads / 64; ++g) {
            t0 += part[g][lane].x;
            t1 += part[g][lane].y;
        }
        float inv = 1.f / (float)(r1 - r0);
        float *dst = qbar + (((int64_t)b * n_blocks + blk) * H + h) * kD + lane * 2;
        dst[0] = t0 * inv;
        dst[1] = t1 * inv;
    }
}

// Mean global query of every execution block of a chunk, straight from the un-rotated input rows: the global
// query is rotated by ONE angle (rope.py:93-104), and a rotation is linear, so the mean is taken first (fp32)
// and rotated once.  One workgroup per (block, head, batch row).
__global__ __launch_bounds__(kMeanThreads) void chunk_qbar_kernel(const bf16_t *q, int64_t q_sb, int64_t q_sh, int64_t q_sl,
                                                                 int H, int n, int exc, const float *inv_freq,
                                                                 double distance_scale, int64_t glb_pos, float *qbar,
                                                                 int n_blocks) {
    __shared__ float2 part[kMeanThreads / 64][64];
    __shared__ float mean[kD];
    const int blk = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
    const int lane = threadIdx.x & 63, grp = threadIdx.x >> 6;
    const int r0 = blk * exc, r1 = min(r0 + exc, n);
    const bf16_t *src = q + (int64_t)b * q_sb + (int64_t)h * q_sh;
    float s0 = 0.f, s1 = 0.f;
    for (int r = r0 + grp; r < r1; r += kMeanThreads / 64) {
        uint32_t w = *(const uint32_t *)(src + (int64_t)r * q_sl + lane * 2);
        s0 += bf16_bits_to_f32(w & 0xffffu);
        s1 += bf16_bits_to_f32(w >> 16);
    }
    part[grp][lane] = make_float2(s0, s1);
    __syncthreads();
    if (grp == 0) {
        float t0 = 0.f, t1 = 0.f;
        for (int g = 0; g < kMeanThreads / 64; ++g) {
            t0 += part[g][lane].x;
            t1 += part[g][lane].y;
        }
        const float inv = 1.f / (float)(r1 - r0);
        mean[lane * 2] = t0 * inv;
        mean[lane * 2 + 1] = t1 * inv;
    }
    __syncthreads();
    if (threadIdx.x < kD / 2) {
        const int f = threadIdx.x;
        double sn, cs;
        sincos((double)glb_pos * distance_scale * (double)inv_freq[f], &sn, &cs);
        const float c = (float)cs, sgn = (float)sn, lo = mean[f], hi = mean[f + kD / 2];
        float *dst = qbar + (((int64_t)b * n_blocks + blk) * H + h) * kD;
        dst[f] = lo * c - hi * sgn;
        dst[f + kD / 2] = hi * c + lo * sgn;
    }
}

// RoPE of plain rows (rope.py:27-47, 93-104): out[b,h,r,:] = x[b,h,r,:] rotated by the angle of position
// pos0 + r * pos_step (pos_step 0: every row by the same angle).  One wave per row, a lane owns the pair
// (d, d + 64); the angle is formed in fp64 like in the stream prologue.
__global__ __launch_bounds__(256) void rope_rows_kernel(const bf16_t *x, int64_t sb, int64_t sh, int64_t sl, int H, int L,
                                                        int64_t pos0, int pos_step, const float *inv_freq,
                                                        double distance_scale, bf16_t *out) {
    const int lane = threadIdx.x & 63;
    const int r = blockIdx.x * 4 + (threadIdx.x >> 6), h = blockIdx.y, b = blockIdx.z;
    if (r >= L) return;
    const bf16_t *src = x + (int64_t)b * sb + (int64_t)h * sh + (int64_t)r * sl;
    bf16_t *dst = out + (((int64_t)b * H + h) * L + r) * kD;
    double sn, cs;
    sincos((double)(pos0 + (int64_t)r * pos_step) * distance_scale * (double)inv_freq[lane], &sn, &cs);
    const float c = (float)cs, s = (float)sn;
    const float lo = bf16_bits_to_f32(((const uint16_t *)src)[lane]), hi = bf16_bits_to_f32(((const uint16_t *)src)[lane + kD / 2]);
    ((uint16_t *)dst)[lane] = (uint16_t)(pack_bf16x2(lo * c - hi * s, 0.f) & 0xffffu);
    ((uint16_t *)dst)[lane + kD / 2] = (uint16_t)(pack_bf16x2(hi * c + lo * s, 0.f) & 0xffffu);
}

// grid.z = B, or 2*B to gather from a second ring (ring2 -> out2, same geometry) in the same launch
template <int D>
__global__ __launch_bounds__(256) void gather_rows_kernel(const bf16_t *ring, int64_t ring_cap, int Hkv, int64_t t0,
                                                          int n, int unit_rows, bf16_t *out, int64_t out_sb,
                                                          int64_t out_su, int64_t out_sh, int B, const bf16_t *ring2, bf16_t *out2) {
    const int b = blockIdx.z % B, h = blockIdx.y;
    if ((int)blockIdx.z >= B) {
        ring = ring2;
        out = out2;
    }
    const int e = blockIdx.x * 256 + threadIdx.x;      // (row, 16-byte chunk)
    if (e >= n * (D / 8)) return;
    int r = e / (D / 8), c = e % (D / 8);
    int64_t row = (t0 + r) % ring_cap;
    const bf16_t *src = ring + (((int64_t)b * Hkv + h) * ring_cap + row) * D + c * 8;
    *(u32x4 *)(out + (int64_t)b * out_sb + (int64_t)(r / unit_rows) * out_su + (int64_t)h * out_sh +
               (int64_t)(r % unit_rows) * D + c * 8) = *(const u32x4 *)src;
}

}  // namespace

extern "C" int infllm_ingest_dim(const infllm_ingest_args *a, int32_t dim, float *d_qbar, void *stream) {
    INFLLM_REQUIRE(a != nullptr, "ingest: null argument block");
    INFLLM_REQUIRE(a->d_q && a->d_k && a->d_v && a->d_inv_freq, "ingest: null input pointer");
    INFLLM_REQUIRE(a->d_ring_k_raw && a->d_ring_k_rot && a->d_ring_v && a->d_ring_score && a->d_q_loc && a->d_q_glb,
                   "ingest: null output pointer");
    INFLLM_REQUIRE(a->B > 0 && a->H > 0 && a->Hkv > 0 && a->H % a->Hkv == 0, "ingest: bad head geometry B=%d H=%d Hkv=%d",
                   a->B, a->H, a->Hkv);
    INFLLM_REQUIRE(a->n >= 0 && a->pos0 >= 0, "ingest: negative length or position");
    INFLLM_REQUIRE(a->ring_cap > 0 && a->n <= a->ring_cap, "ingest: %d new tokens do not fit a ring of %lld rows", a->n,
                   (long long)a->ring_cap);
    INFLLM_REQUIRE((a->q_sl % 8 | a->q_sh % 8 | a->q_sb % 8 | a->k_sl % 8 | a->k_sh % 8 | a->k_sb % 8 | a->v_sl % 8 |
                    a->v_sh % 8 | a->v_sb % 8) == 0,
                   "ingest: strides must be multiples of 8 elements (16-byte rows)");
    INFLLM_REQUIRE(dim == 128 || dim == 64, "ingest: head_dim %d", dim);
    INFLLM_REQUIRE(!d_qbar || a->n <= kPosPerBlock, "ingest: the mean of %d queries takes more than one tile", a->n);
    if (a->n == 0) return 0;
    const int kg = heads_together(a->n, a->B, a->H, a->Hkv);
    const dim3 grid((a->n + kPosPerBlock - 1) / kPosPerBlock, a->B, (a->Hkv + kg - 1) / kg);
    const auto kern = dim == 128 ? (kg == 4 ? ingest_kernel<128, 4> : kg == 2 ? ingest_kernel<128, 2> : ingest_kernel<128, 1>)
                                 : (kg == 4 ? ingest_kernel<64, 4> : kg == 2 ? ingest_kernel<64, 2> : ingest_kernel<64, 1>);
    hipLaunchKernelGGL(kern, grid, dim3(256), 0, (hipStream_t)stream, *a, d_qbar);
    INFLLM_CHECK_LAUNCH("ingest");
    return 0;
}

extern "C" int infllm_ingest(const infllm_ingest_args *a, void *stream) { return infllm_ingest_dim(a, kD, nullptr, stream); }

extern "C" int infllm_reduce_partials(const float *d_parts, int32_t B, int32_t n_parts, int32_t C, float scale, float *d_out,
                                      void *stream) {
    INFLLM_REQUIRE(d_parts && d_out, "reduce_partials: null pointer");
    INFLLM_REQUIRE(B > 0 && n_parts > 0 && C > 0, "reduce_partials: bad sizes B=%d n_parts=%d C=%d", B, n_parts, C);
    hipLaunchKernelGGL(reduce_partials_kernel, dim3((C + 63) / 64, B), dim3(256), 0, (hipStream_t)stream, d_parts, n_parts, C,
                       scale, d_out, n_parts, 0, 0);
    INFLLM_CHECK_LAUNCH("reduce_partials");
    return 0;
}

// library-internal: the mean rotated query of every execution block of one ingest launch over n positions (blocks of
// exc, a multiple of the ingest tile; the last may be shorter): d_parts [B, ceil(n / tile), C] -> d_out [blocks, B, C]
int infllm_reduce_partials_blocks(const float *d_parts, int32_t B, int32_t n, int32_t exc, int32_t C, float *d_out, void *stream) {
    INFLLM_REQUIRE(d_parts && d_out, "reduce_partials_blocks: null pointer");
    INFLLM_REQUIRE(B > 0 && n > 0 && C > 0 && exc > 0 && exc % kPosPerBlock == 0, "reduce_partials_blocks: bad sizes B=%d n=%d exc=%d C=%d", B, n, exc, C);
    const int n_parts = (n + kPosPerBlock - 1) / kPosPerBlock, n_blocks = (n + exc - 1) / exc;
    hipLaunchKernelGGL(reduce_partials_kernel, dim3((C + 63) / 64, B, n_blocks), dim3(256), 0, (hipStream_t)stream, d_parts, n_parts, C,
                       1.f / (float)n, d_out, n_blocks > 1 ? exc / kPosPerBlock : n_parts, n, exc);
    INFLLM_CHECK_LAUNCH("reduce_partials_blocks");
    return 0;
}

extern "C" int infllm_block_mean(const void *d_q_glb, int32_t B, int32_t H, int32_t n, int32_t exc, float *d_qbar,
                                 void *stream) {
    INFLLM_REQUIRE(d_q_glb && d_qbar, "block_mean: null pointer");
    INFLLM_REQUIRE(B > 0 && H > 0 && n > 0 && exc > 0, "block_mean: bad sizes B=%d H=%d n=%d exc=%d", B, H, n, exc);
    int n_blocks = (n + exc - 1) / exc;
    hipLaunchKernelGGL(block_mean_kernel, dim3(n_blocks, H, B), dim3(kMeanThreads), 0, (hipStream_t)stream,
                       (const bf16_t *)d_q_glb, H, n, exc, d_qbar, n_blocks);
    INFLLM_CHECK_LAUNCH("block_mean");
    return 0;
}

extern "C" int infllm_chunk_qbar(const void *d_q, int64_t q_sb, int64_t q_sh, int64_t q_sl, int32_t B, int32_t H, int32_t n,
                                 int32_t exc, const float *d_inv_freq, double distance_scale, int64_t glb_pos, float *d_qbar,
                                 void *stream) {
    INFLLM_REQUIRE(d_q && d_inv_freq && d_qbar, "chunk_qbar: null pointer");
    INFLLM_REQUIRE(B > 0 && H > 0 && n > 0 && exc > 0, "chunk_qbar: bad sizes B=%d H=%d n=%d exc=%d", B, H, n, exc);
    INFLLM_REQUIRE(q_sl % 2 == 0 && q_sh % 2 == 0 && q_sb % 2 == 0 && (uintptr_t)d_q % 4 == 0, "chunk_qbar: q rows must be 4-byte aligned");
    const int n_blocks = (n + exc - 1) / exc;
    hipLaunchKernelGGL(chunk_qbar_kernel, dim3(n_blocks, H, B), dim3(kMeanThreads), 0, (hipStream_t)stream, (const bf16_t *)d_q,
                       q_sb, q_sh, q_sl, H, n, exc, d_inv_freq, distance_scale, glb_pos, d_qbar, n_blocks);
    INFLLM_CHECK_LAUNCH("chunk_qbar");
    return 0;
}

extern "C" int infllm_rope_rows(const void *d_x, int64_t sb, int64_t sh, int64_t sl, int32_t B, int32_t H, int32_t L, int64_t pos0,
                                int32_t pos_step, const float *d_inv_freq, double distance_scale, void *d_out, void *stream) {
    INFLLM_REQUIRE(B >= 0 && H >= 0 && L >= 0 && pos0 >= 0 && (pos_step == 0 || pos_step == 1), "rope_rows: bad sizes B=%d H=%d L=%d", B, H, L);
    if (B == 0 || H == 0 || L == 0) return 0;
    INFLLM_REQUIRE(d_x && d_inv_freq && d_out, "rope_rows: null pointer");
    hipLaunchKernelGGL(rope_rows_kernel, dim3((L + 3) / 4, H, B), dim3(256), 0, (hipStream_t)stream, (const bf16_t *)d_x, sb, sh, sl,
                       H, L, pos0, pos_step, d_inv_freq, distance_scale, (bf16_t *)d_out);
    INFLLM_CHECK_LAUNCH("rope_rows");
    return 0;
}

extern "C" int infllm_gather_rows(const void *d_ring, int64_t ring_cap, int32_t B, int32_t Hkv, int64_t t0, int32_t n,
                                  int32_t unit_rows, void *d_out, int64_t out_sb, int64_t out_su, int64_t out_sh,
                                  void *stream) {
    INFLLM_REQUIRE(d_ring && d_out, "gather_rows: null pointer");
    INFLLM_REQUIRE(B > 0 && Hkv > 0 && ring_cap > 0 && t0 >= 0 && n >= 0 && n <= ring_cap,
                   "gather_rows: bad sizes B=%d Hkv=%d cap=%lld t0=%lld n=%d", B, Hkv, (long long)ring_cap, (long long)t0, n);
    INFLLM_REQUIRE(unit_rows > 0, "gather_rows: unit_rows must be positive");
    INFLLM_REQUIRE((out_sb % 8 | out_su % 8 | out_sh % 8) == 0, "gather_rows: output strides must be multiples of 8");
    if (n == 0) return 0;
    hipLaunchKernelGGL(gather_rows_kernel<kD>, dim3((n * 16 + 255) / 256, Hkv, B), dim3(256), 0, (hipStream_t)stream,
                       (const bf16_t *)d_ring, ring_cap, Hkv, t0, n, unit_rows, (bf16_t *)d_out, out_sb, out_su, out_sh, B,
                       (const bf16_t *)nullptr, (bf16_t *)nullptr);
    INFLLM_CHECK_LAUNCH("gather_rows");
    return 0;
}

// internal: the K and the V rows of the same stream positions in one launch (same arguments as infllm_gather_rows; rows of
// `dim` elements)
int infllm_gather_rows_pair(const void *d_ring_a, void *d_out_a, const void *d_ring_b, void *d_out_b, int64_t ring_cap, int32_t B,
                            int32_t Hkv, int64_t t0, int32_t n, int32_t unit_rows, int64_t out_sb, int64_t out_su, int64_t out_sh,
                            void *stream, int32_t dim) {
    INFLLM_REQUIRE(d_ring_a && d_out_a && d_ring_b && d_out_b, "gather_rows: null pointer");
    INFLLM_REQUIRE(B > 0 && Hkv > 0 && ring_cap > 0 && n >= 0 && n <= ring_cap && t0 >= 0 && unit_rows > 0, "gather_rows: bad sizes");
    INFLLM_REQUIRE((out_sb % 8 | out_su % 8 | out_sh % 8) == 0, "gather_rows: output strides must be multiples of 8");
    if (n == 0) return 0;
    INFLLM_REQUIRE(dim == 128 || dim == 64, "gather_rows: head_dim %d", dim);
    hipLaunchKernelGGL((dim == 64 ? gather_rows_kernel<64> : gather_rows_kernel<128>), dim3((n * (dim / 8) + 255) / 256, Hkv, 2 * B), dim3(256), 0,
                       (hipStream_t)stream, (const bf16_t *)d_ring_a, ring_cap, Hkv, t0, n, unit_rows, (bf16_t *)d_out_a, out_sb, out_su, out_sh, B,
                       (const bf16_t *)d_ring_b, (bf16_t *)d_out_b);
    INFLLM_CHECK_LAUNCH("gather_rows");
    return 0;
}
