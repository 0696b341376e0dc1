// Rotary embedding of rows, shared by the kernels that stage new tokens (inf_llm/attention/rope.py:89-112).
#pragma once
#include "common.h"

constexpr int kPosPerBlock = 16;   // stream positions handled by one workgroup

struct Rot8 {
    u32x4 lo, hi;
};

// rotate 8 pairs (lo[i], hi[i]) by (c[i], s[i]); fp32 math, one rounding to bf16.  `raw` (optional) receives the 16
// rotated values before that rounding: lo pairs first, then hi pairs.
__device__ __forceinline__ Rot8 rotate8(u32x4 xlo, u32x4 xhi, const float2 *cs, float *raw = nullptr) {
    Rot8 r;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        float a0 = bf16_bits_to_f32(xlo[w] & 0xffffu), a1 = bf16_bits_to_f32(xlo[w] >> 16);
        float b0 = bf16_bits_to_f32(xhi[w] & 0xffffu), b1 = bf16_bits_to_f32(xhi[w] >> 16);
        float2 c0 = cs[2 * w], c1 = cs[2 * w + 1];
        // x*cos + rotate_half(x)*sin, rotate_half = (-hi, lo)
        const float l0 = a0 * c0.x - b0 * c0.y, l1 = a1 * c1.x - b1 * c1.y;
        const float h0 = b0 * c0.x + a0 * c0.y, h1 = b1 * c1.x + a1 * c1.y;
        r.lo[w] = pack_bf16x2(l0, l1);
        r.hi[w] = pack_bf16x2(h0, h1);
        if (raw) {
            raw[2 * w] = l0, raw[2 * w + 1] = l1;
            raw[8 + 2 * w] = h0, raw[8 + 2 * w + 1] = h1;
        }
    }
    return r;
}

// This thread's frequency for rope_angles, to be asked for in front of the rows: what a wave requests comes back in that order, and the
// angles' chain is to run while the rows are on their way.  (A step's chain began when the last of the rows in front of it had come.)
template <int HALF>
__device__ __forceinline__ float rope_freq(const float *inv_freq) {
    const float f = inv_freq[threadIdx.x % HALF];
    asm volatile("" ::: "memory");                               // (no later load goes ahead of it)
    return f;
}

// cos / sin of (position x frequency) for the np <= 16 positions from pos0 on and for the one angle of position glb_pos,
// by a workgroup of at least HALF * 2 threads (HALF = head_dim / 2 frequencies).  Only the FIRST position and the step of
// one position are evaluated (fp64 sincos, one call per thread); the other positions follow by the angle-addition
// recurrence in fp64, whose error after 15 steps is a few 1e-16 - far below the fp32 value the rotation consumes.  The
// caller's barrier follows.
template <int HALF>
__device__ __forceinline__ void rope_angles(int64_t pos0, int np, int64_t glb_pos, double distance_scale, float freq,
                                            float2 (*cs_pos)[HALF], float2 *cs_glb) {
    const int tid = threadIdx.x;
    if (tid < HALF) {
        const double w = distance_scale * (double)freq;
        double s, c;
        sincos((double)pos0 * w, &s, &c);
        cs_pos[0][tid] = make_float2((float)c, (float)s);
        if (np > 1) {
            double2 cur = make_double2(c, s);
            sincos(w, &s, &c);
            const double2 step = make_double2(c, s);
            for (int p = 1; p < np; ++p) {                // (cos, sin)(x + w) from (cos, sin)(x)
                const double c2 = cur.x * step.x - cur.y * step.y, s2 = cur.y * step.x + cur.x * step.y;
                cur = make_double2(c2, s2);
                cs_pos[p][tid] = make_float2((float)c2, (float)s2);
            }
        }
    } else if (tid < 2 * HALF) {
        const int f = tid - HALF;
        double s, c;
        sincos((double)glb_pos * distance_scale * (double)freq, &s, &c);
        cs_glb[f] = make_float2((float)c, (float)s);
    }
}

// kv heads that a workgroup of a prompt's rows takes together: as many as make up to four query heads, where the workgroups of one
// kv head each are more than the chip holds at once.  The angles are the chain of one wave, and the first waves of a CU's workgroups
// share a SIMD: 36 key heads of 64 formed the angles of every 16 positions 36 times and waited for that SIMD and not for memory (ingest
// of 4,096 tokens 45.2 -> 33.9 us, of 1,500 17.2 -> 13.2; causal staging of 4,096 24.0 -> 20.9).  Below the line neither form is the
// faster one (300 - 450 tokens: 8 - 14 us either way), and copies of cached rows, in the same grid, want a workgroup for each head.
inline int heads_together(int64_t n, int32_t B, int32_t H, int32_t Hkv) {
    const int G = H / Hkv;
    return G >= 3 || (n + kPosPerBlock - 1) / kPosPerBlock * B * Hkv <= 1024 ? 1 : G == 2 ? 2 : 4;
}

// One new position (a decode step) of one kv head: its query heads rotated to their position and to the one angle of the units,
// its key and value into the rings, its scores at zero - what ingest_kernel does for a tile of one.  256 threads; cs: D float2.
template <int D>
__device__ __forceinline__ void ingest_one(const infllm_ingest_args &a, int b, int g, float2 *cs) {
    constexpr int HALF = D / 2, C2 = D / 16;
    const int tid = threadIdx.x, G = a.H / a.Hkv;
    const bf16_t *q = (const bf16_t *)a.d_q + (int64_t)b * a.q_sb + (int64_t)g * G * a.q_sh;
    const float freq = rope_freq<HALF>(a.d_inv_freq);
    u32x4 lo{}, hi{}, k_lo{}, k_hi{}, v_row{};
    if (tid < G * C2) {                                      // (more than 32 (64) heads: the rest below)
        lo = *(const u32x4 *)(q + (int64_t)(tid / C2) * a.q_sh + tid % C2 * 8);
        hi = *(const u32x4 *)(q + (int64_t)(tid / C2) * a.q_sh + HALF + tid % C2 * 8);
    }
    if (tid < C2) {
        const bf16_t *src = (const bf16_t *)a.d_k + (int64_t)b * a.k_sb + (int64_t)g * a.k_sh + tid * 8;
        k_lo = *(const u32x4 *)src, k_hi = *(const u32x4 *)(src + HALF);
    }
    if (tid < 2 * C2) v_row = *(const u32x4 *)((const bf16_t *)a.d_v + (int64_t)b * a.v_sb + (int64_t)g * a.v_sh + tid * 8);
    rope_angles<HALF>(a.pos0, 1, a.glb_pos, a.distance_scale, freq, (float2(*)[HALF])cs, cs + HALF);
    __syncthreads();
    for (int e = tid; e < G * C2; e += 256) {
        const int c = e % C2, h = e / C2;
        if (e >= 256) {
            lo = *(const u32x4 *)(q + (int64_t)h * a.q_sh + c * 8);
            hi = *(const u32x4 *)(q + (int64_t)h * a.q_sh + HALF + c * 8);
        }
        const int64_t o = ((int64_t)b * a.H + g * G + h) * D + c * 8;
        Rot8 r = rotate8(lo, hi, cs + c * 8);
        *(u32x4 *)((bf16_t *)a.d_q_loc + o) = r.lo;
        *(u32x4 *)((bf16_t *)a.d_q_loc + o + HALF) = r.hi;
        r = rotate8(lo, hi, cs + HALF + c * 8);
        *(u32x4 *)((bf16_t *)a.d_q_glb + o) = r.lo;
        *(u32x4 *)((bf16_t *)a.d_q_glb + o + HALF) = r.hi;
    }
    const int64_t slot = a.pos0 % a.ring_cap, at = (((int64_t)b * a.Hkv + g) * a.ring_cap + slot) * D;
    if (tid < C2) {
        *(u32x4 *)((bf16_t *)a.d_ring_k_raw + at + tid * 8) = k_lo;
        *(u32x4 *)((bf16_t *)a.d_ring_k_raw + at + HALF + tid * 8) = k_hi;
        const Rot8 r = rotate8(k_lo, k_hi, cs + tid * 8);
        *(u32x4 *)((bf16_t *)a.d_ring_k_rot + at + tid * 8) = r.lo;
        *(u32x4 *)((bf16_t *)a.d_ring_k_rot + at + HALF + tid * 8) = r.hi;
    }
    if (tid < 2 * C2) *(u32x4 *)((bf16_t *)a.d_ring_v + at + tid * 8) = v_row;
    for (int h = tid; h < G; h += 256) a.d_ring_score[((int64_t)b * a.H + g * G + h) * a.ring_cap + slot] = 0.f;
}
