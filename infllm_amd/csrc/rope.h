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

// cos / sin of (position x frequency) for the np <= 16 positions from pos0 on and for the one angle of position glb_pos,
// by a workgroup of at least HALF * 2 threads (HALF = head_dim / 2 frequencies).  Only the FIRST position and the step of
// one position are evaluated (fp64 sincos, one call per thread); the other positions follow by the angle-addition
// recurrence in fp64, whose error after 15 steps is a few 1e-16 - far below the fp32 value the rotation consumes.  The
// caller's barrier follows.
template <int HALF>
__device__ __forceinline__ void rope_angles(int64_t pos0, int np, int64_t glb_pos, double distance_scale, const float *inv_freq,
                                            float2 (*cs_pos)[HALF], float2 *cs_glb) {
    const int tid = threadIdx.x;
    if (tid < HALF) {
        const double w = distance_scale * (double)inv_freq[tid];
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
        sincos((double)glb_pos * distance_scale * (double)inv_freq[f], &s, &c);
        cs_glb[f] = make_float2((float)c, (float)s);
    }
}
