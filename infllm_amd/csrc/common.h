// Shared helpers for the gfx950 kernels of libinfllm_hip.so.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdarg.h>
#include <stdio.h>

#include "../../include/infllm_hip.h"

typedef __bf16 bf16_t;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

constexpr int kD = INFLLM_HEAD_DIM;       // head_dim
constexpr int kTile = INFLLM_KEY_TILE;    // keys per tile
constexpr int kInlinePages = 64;          // page table entries that a launch of the paged stage can carry
constexpr int kWave = 64;
constexpr float kLog2e = 1.4426950408889634f;

// thread-local error text, returned by infllm_last_error()
char *infllm_err_buf();
int infllm_fail(int code, const char *fmt, ...);

#define INFLLM_REQUIRE(cond, ...)                      \
    do {                                               \
        if (!(cond)) return infllm_fail(-1, __VA_ARGS__); \
    } while (0)

#define INFLLM_CHECK_LAUNCH(name)                                                     \
    do {                                                                              \
        hipError_t e_ = hipGetLastError();                                            \
        if (e_ != hipSuccess) return infllm_fail(-2, "%s: %s", name, hipGetErrorString(e_)); \
    } while (0)

__device__ __forceinline__ float bf16_bits_to_f32(uint32_t bits16) {
    return __uint_as_float(bits16 << 16);
}
// round-to-nearest-even fp32 -> bf16 bits (inputs are finite here; NaN kept quiet)
__device__ __forceinline__ uint32_t f32_to_bf16_bits(float f) {
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (u >> 16) | 0x40u;
    u += 0x7fffu + ((u >> 16) & 1u);
    return u >> 16;
}
// two fp32 -> packed bf16 pair, round-to-nearest-even (one v_cvt_pk_bf16_f32 on gfx950)
__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
    typedef float f32x2_t __attribute__((ext_vector_type(2)));
    typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
    f32x2_t v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
}
// ---- rows of D elements in LDS, their 16-byte chunk c at position c ^ swz(row): 16 consecutive rows, one chunk each, hit 16
//      different places, and so do the transposing reads of the attention kernel.
// Heads of 64: a row is 128 bytes (8 chunks), two rows share a 256-byte line.  16 consecutive rows, one chunk each, hit 16
// different places when the row pairs use 8 different positions; the four row pairs' bit that decides the upper or lower
// four chunks is the pair's lowest, so that the transposing read's 4 rows x 4 chunks x 2 halves are 32 different slots.
template <int D>
__device__ __forceinline__ int swz(int row) {
    return D == 128 ? ((row & 3) << 2) | ((row >> 2) & 3) : (((row >> 1) & 1) << 2) | ((row >> 2) & 3);
}

// Issued as inline assembly on purpose.  With the builtin, the compiler tracks the transfer as an LDS store that
// may alias every later LDS read and puts `s_waitcnt vmcnt(0)` in front of the first operand read of the tile being
// multiplied - which waits for the tiles just requested for LATER and serialises load and math completely.  The
// kernel orders the transfers itself: vmcnt(0) and a barrier before a buffer is read, a barrier before it is refilled.
// The row address is a scalar base and a 32-bit byte offset of the lane.  M0 is overwritten: nothing else in these kernels
// uses it (LDS instructions have not since gfx9).
__device__ __forceinline__ void load_to_lds4(const float *base, uint32_t lane_off, uint32_t lds) {      // 4 bytes a lane, at lds + 4 * lane
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" : : "s"(lds), "v"(lane_off), "s"(base) : "memory");
}
__device__ __forceinline__ void load_to_lds16(const bf16_t *base, uint32_t lane_off, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(lds), "v"(lane_off), "s"(base) : "memory");
}
__device__ __forceinline__ void load_to_lds16_at(const bf16_t *src, uint32_t lds) {                       // every lane from an address of its own
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(lds), "v"(src) : "memory");
}
__device__ __forceinline__ uint32_t lds_address(const char *p) { return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void *)p; }

__device__ __forceinline__ float wave_xor32(float x) {
    return __shfl_xor(x, 32, 64);
}

// A word of every line of the kernel's arguments (the first BYTES of them, a number of lines up to 16), in one trip: what is read of them
// where it is needed is then a trip to the scalar cache and not to memory.
template <int BYTES>
__device__ __forceinline__ void touch_arguments() {
    constexpr int kLines = (BYTES + 63) / 64;
    static_assert(kLines <= 16);
    auto *p = (const __attribute__((address_space(4))) uint32_t *)__builtin_amdgcn_kernarg_segment_ptr();
    uint32_t w[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) w[i] = i < kLines ? p[min(16 * i, BYTES / 4 - 1)] : 0;
    asm volatile("" : : "s"(w[0]), "s"(w[1]), "s"(w[2]), "s"(w[3]), "s"(w[4]), "s"(w[5]), "s"(w[6]), "s"(w[7]), "s"(w[8]), "s"(w[9]), "s"(w[10]), "s"(w[11]),
                 "s"(w[12]), "s"(w[13]), "s"(w[14]), "s"(w[15]));
}

// the larger of a lane's value and that of the lane 32 away, in both: vector instructions (a shuffle is a trip through LDS)
__device__ __forceinline__ float wave_max32(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// ... of the lane 16 away (the other row of 16 of its pair), and the sums
__device__ __forceinline__ float wave_max16(float x) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float wave_sum16(float x) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float wave_sum32(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

__device__ __forceinline__ uint32_t order_key(float f) {
    uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);       // larger float <=> larger key
}
__device__ __forceinline__ uint64_t shfl_xor_u64(uint64_t v, int o) {
    const uint32_t lo = __shfl_xor((uint32_t)v, o, 64), hi = __shfl_xor((uint32_t)(v >> 32), o, 64);
    return ((uint64_t)hi << 32) | lo;
}

// ---- the merge of partial attention outputs, shared by the merge kernels (attn.hip) and by the local-score launch
//      that carries the merge of its block along (score.hip)
// The partials of a merge may lie in two places: the first n_first of them behind the pointers the kernel is given,
// the rest wherever the second stage wrote them.  skip_l / skip_o are what has to be added to an index into the first
// buffers (log-sum-exps; fp16 elements beyond the row term) to land in the second.
struct PartSets {
    int32_t n_first;
    int64_t skip_l, skip_o;
    __device__ __forceinline__ int64_t l(int p, int64_t rows) const { return (int64_t)p * rows + (p >= n_first ? skip_l : 0); }
    __device__ __forceinline__ int64_t o(int p) const { return p >= n_first ? skip_o : 0; }
};

struct MergeJob {
    const _Float16 *o_part;            // [P, B, H, Lq, 128] normalised partial rows (see PartSets)
    const float *lse_part;             // [P, B, H, Lq] their base-2 log-sum-exps
    int32_t P, B, H, Lq;
    bf16_t *out;                       // rows [b, h, i] at b * o_sb + h * o_sh + i * o_sl
    int64_t o_sb, o_sh, o_sl;
    float *lse_out;                    // [B, H, Lq] with head rows lse_sh apart, or NULL
    PartSets ps;
    int32_t lse_sh;
};

// thread e of the merge: (row, 8 dims) = (e / 16, e % 16) for rows of 128 elements, (e / 8, e % 8) for rows of 64.  (inf_llm/attention/dot_production_attention/torch_impl.py:15-36)
template <int D = kD>
__device__ __forceinline__ void merge_piece(const MergeJob &mj, int64_t e) {
    const _Float16 *o_part = mj.o_part;
    const float *lse_part = mj.lse_part;
    const PartSets ps = mj.ps;
    const int P = mj.P, H = mj.H, Lq = mj.Lq;
    const int64_t rows = (int64_t)mj.B * H * Lq;                         // (fewer than 2^31)
    constexpr int kPieces = D / 8;
    if (e >= rows * kPieces) return;
    const uint32_t row = (uint32_t)(e / kPieces);
    const int c = (int)(e % kPieces);
    // partials in batches of 8 so that the loads of a batch are in flight together (decode-sized blocks merge
    // dozens of partials of very few rows: a chain of dependent loads would be all latency)
    float m = -INFINITY;
    for (int p0 = 0; p0 < P; p0 += 8) {
        float l8[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) l8[i] = p0 + i < P ? lse_part[ps.l(p0 + i, rows) + row] : -INFINITY;
#pragma unroll
        for (int i = 0; i < 8; ++i) m = fmaxf(m, l8[i]);
    }
    if (m == -INFINITY) m = 0.f;                                         // no partial with a finite sum: every weight is 0
    float acc[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] = 0.f;
    float den = 0.f;
    for (int p0 = 0; p0 < P; p0 += 8) {
        float l8[8];
        f16x8 o8[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const bool on = p0 + i < P;
            l8[i] = on ? lse_part[ps.l(p0 + i, rows) + row] : -INFINITY;
            o8[i] = on ? *(const f16x8 *)(o_part + (ps.l(p0 + i, rows) + row) * D + ps.o(p0 + i) + c * 8) : f16x8{0, 0, 0, 0, 0, 0, 0, 0};
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            // exp2(-inf) = 0: empty partials hold zeros, those with a logit that was no number NaN, which stays NaN
            const float w = __builtin_amdgcn_exp2f(l8[i] - m);
#pragma unroll
            for (int j = 0; j < 8; ++j) acc[j] += (float)o8[i][j] * w;
            den += w;
        }
    }
    const float inv = den > 0.f ? 1.f / den : 0.f;
    const uint32_t bh = row / (uint32_t)Lq, i = row - bh * (uint32_t)Lq, b = bh / (uint32_t)H, h = bh - b * (uint32_t)H;
    u32x4 packed{pack_bf16x2(acc[0] * inv, acc[1] * inv), pack_bf16x2(acc[2] * inv, acc[3] * inv),
                 pack_bf16x2(acc[4] * inv, acc[5] * inv), pack_bf16x2(acc[6] * inv, acc[7] * inv)};
    *(u32x4 *)(mj.out + (int64_t)b * mj.o_sb + (int64_t)h * mj.o_sh + (int64_t)i * mj.o_sl + c * 8) = packed;
    if (c == 0 && mj.lse_out) mj.lse_out[(int64_t)bh * mj.lse_sh + i] = den > 0.f ? m + log2f(den) : -INFINITY;
}


// ---- a call's selections from lists made once per call (retrieve.hip: call_rank_kernel; stream.hip drives it)
// For every later block of a prepared call the k best of the units that existed when the call began are known
// (`base`), and so are those units' scores under the block's mean query (`scores`).  After a block has carved
// n_new units, workgroup x of one launch scores them under the mean query of block j0 + x and, for the two blocks
// that need a list now, ranks the base list against all the units carved since the call began.
struct CallRankJob {
    const bf16_t *reps;                // [B][units][C] representatives
    int64_t rep_sb, rep_su;
    const float *qbars;                // [blocks][B][C] mean queries of the call's blocks
    float *scores;                     // [blocks][B][cols]
    int64_t cols;
    const int32_t *base;               // [blocks][B][k]
    int32_t B, k;
    int32_t n_base;                    // units that existed when the call began
    int32_t first_new, n_new;          // the units carved just now: [first_new, first_new + n_new)
    int32_t j0;                        // workgroup x works for block j0 + x
    int32_t j_sel, j_cand;             // blocks whose selection / candidate list leaves now (-1: none)
    int32_t *sel_out, *sel_flag;       // [B][k] ids, then the sequence number
    int32_t sel_seq;
    int32_t *cand_out, *cand_flag;
    int32_t cand_seq;
};
