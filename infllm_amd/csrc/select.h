// The k best of N scores, by one workgroup that reads them from memory as often as it needs them.
#pragma once
#include "common.h"

constexpr int kSelectMost = 64;            // k at most

template <int THREADS>
struct SelectLds {
    static constexpr int kCap = 512;       // survivors
    uint64_t surv[kCap + 8];
    uint32_t gmax[THREADS / 64][64];
    int32_t hist[256];
    int32_t count, need, digit;
};

// The order is that of retrieve.hip's selections: composites order_key(score) << 32 | ~id, all distinct, larger = better score, equal
// scores by ascending id.  The scores are dealt to 16, 32 or 64 >= k groups of threads, those whose number is the same modulo that; the
// smallest of the groups' largest is a threshold that at least k units reach, and few more do.  Those are ranked against each other
// by counting.  Where more than fit reach it (equal scores, say) the k-th largest composite is found digit by digit instead.
// (select_topk_block of retrieve.hip is the same method for one workgroup behind a launch's last score, which fetches the scores once,
// from where other XCDs stored them, and keeps them in registers; here the kernel has neither the registers nor that need.)
// ids: the k, best first; a barrier has followed when the function returns.
template <int THREADS>
__device__ __forceinline__ void select_units(const float *scores, int N, int k, int32_t *ids, SelectLds<THREADS> &lds) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // Loads in flight.  (16: the kernel of a step that takes 16 of 100 / 479 / 2,048 units 0.3 / 0.5 / 0.1 us longer, 64 of them 1.0 / 1.2 /
    // 0.3; 16 of 4,096 / 8,192 / 16,384 0.2 / 0.9 / 1.4 shorter, 64 of them 0.6 / 1.4 / 1.9: a step seldom has more than 4,096.)
    constexpr int kBatch = 8;
    auto each = [&](auto &&f) {            // f(score's key, unit) of this thread's units
        for (int n0 = tid; n0 < N; n0 += kBatch * THREADS) {
            float sc[kBatch];
#pragma unroll
            for (int i = 0; i < kBatch; ++i) sc[i] = scores[min(n0 + i * THREADS, N - 1)];
#pragma unroll
            for (int i = 0; i < kBatch; ++i)
                if (n0 + i * THREADS < N) f(order_key(sc[i]), n0 + i * THREADS);
        }
    };
    auto composite = [](uint32_t key, int n) { return ((uint64_t)key << 32) | (uint32_t)~n; };
    uint32_t best = 0;
    each([&](uint32_t key, int) { best = max(best, key); });
    const int groups = k <= 16 ? 16 : k <= 32 ? 32 : 64;
    for (int o = 32; o >= groups; o >>= 1) best = max(best, (uint32_t)__shfl_xor(best, o, 64));
    lds.gmax[wave][lane] = best;
    if (tid == 0) lds.count = 0;
    __syncthreads();
    uint32_t tau = 0;
#pragma unroll
    for (int w = 0; w < THREADS / 64; ++w) tau = max(tau, lds.gmax[w][lane]);
    for (int o = 1; o < groups; o <<= 1) tau = min(tau, (uint32_t)__shfl_xor(tau, o, 64));
    auto collect = [&](uint64_t from) {    // composites >= from
        each([&](uint32_t key, int n) {
            const uint64_t c = composite(key, n);
            if (c < from) return;
            const int at = atomicAdd(&lds.count, 1);
            if (at < lds.kCap) lds.surv[at] = c;
        });
        __syncthreads();
    };
    collect((uint64_t)tau << 32);
    if (lds.count > lds.kCap) {
        uint64_t prefix = 0, known = 0;
        int need = k;                      // of the units whose composite agrees with prefix where it is known
        for (int shift = 56; shift >= 0; shift -= 8) {
            for (int i = tid; i < 256; i += THREADS) lds.hist[i] = 0;
            __syncthreads();
            each([&](uint32_t key, int n) {
                const uint64_t c = composite(key, n);
                if ((c & known) == prefix) atomicAdd(&lds.hist[(int)(c >> shift) & 255], 1);
            });
            __syncthreads();
            for (int d = tid; d < 256; d += THREADS) {         // the one digit that holds the need-th from the top
                int above = 0;
#pragma unroll 8
                for (int o = 255; o > 0; --o) above += o > d ? lds.hist[o] : 0;
                if (above < need && above + lds.hist[d] >= need) lds.digit = d, lds.need = need - above;
            }
            __syncthreads();
            prefix |= (uint64_t)lds.digit << shift, known |= (uint64_t)255 << shift, need = lds.need;
            __syncthreads();
        }
        if (tid == 0) lds.count = 0;
        __syncthreads();
        collect(prefix);                   // exactly k of them now
    }
    const int S = lds.count, S8 = (S + 7) & ~7;
    for (int i = S + tid; i < S8; i += THREADS) lds.surv[i] = 0;              // (below every real one)
    __syncthreads();
    for (int i = tid; i < S; i += THREADS) {
        const uint64_t mine = lds.surv[i];
        int rank = 0;
        for (int o = 0; o < S8; o += 8) {
            uint64_t other[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) other[e] = lds.surv[o + e];
#pragma unroll
            for (int e = 0; e < 8; ++e) rank += other[e] > mine ? 1 : 0;
        }
        if (rank < k) ids[rank] = (int32_t)~(uint32_t)mine;
    }
    __syncthreads();
}
