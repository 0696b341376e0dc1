// What leaves the window: the units' rows out of the rings, and their representative keys
// (inf_llm/attention/context_manager.py:268-277, 652-675); shared by retrieve.hip and score.hip.
#pragma once
#include "common.h"

// The copy of the same units' K and V rows out of the rings into contiguous staging (what infllm_gather_rows does)
// can ride in the launch that picks their representatives: independent work, one launch less in the stream.
struct CarveCopy {
    const bf16_t *ring_a, *ring_b;
    bf16_t *out_a, *out_b;
    int64_t out_sb, out_su, out_sh;
    int32_t ring_cap, slot0;                       // n <= ring_cap rows from ring row slot0 on
    int32_t Hkv, B, n, unit_rows, x_extra;         // x_extra = extra workgroups along x (repr_keys_kernel; 0: no copy)
};

// element e = (ring, batch row, kv head, row, 16-byte chunk)
template <int D>
__device__ __forceinline__ void carve_copy(const CarveCopy &cc, int64_t e) {
    constexpr int kChunks = D / 8;
    if (e >= (int64_t)2 * cc.B * cc.Hkv * cc.n * kChunks) return;
    const int c = (int)(e % kChunks);
    uint32_t rest = (uint32_t)(e / kChunks);
    const int r = (int)(rest % (uint32_t)cc.n);
    rest /= (uint32_t)cc.n;
    const int hk = (int)(rest % (uint32_t)cc.Hkv);
    rest /= (uint32_t)cc.Hkv;
    const int bb = (int)(rest % (uint32_t)cc.B);
    const bool second = rest / (uint32_t)cc.B != 0;
    const int slot = cc.slot0 + r < cc.ring_cap ? cc.slot0 + r : cc.slot0 + r - cc.ring_cap;
    const bf16_t *src = (second ? cc.ring_b : cc.ring_a) + (((int64_t)bb * cc.Hkv + hk) * cc.ring_cap + slot) * D + c * 8;
    bf16_t *dst = (second ? cc.out_b : cc.out_a) + (int64_t)bb * cc.out_sb + (int64_t)((uint32_t)r / (uint32_t)cc.unit_rows) * cc.out_su +
                  (int64_t)hk * cc.out_sh + (int64_t)((uint32_t)r % (uint32_t)cc.unit_rows) * D + c * 8;
    *(u32x4 *)dst = *(const u32x4 *)src;
}

// the order of a unit's rows as representatives: larger is better, equal scores by lower row, NaN last; never 0
__device__ __forceinline__ uint64_t pick_key(float x, int r) { return ((uint64_t)(x == x ? order_key(x) : 1u) << 32) | (uint32_t)~r; }
