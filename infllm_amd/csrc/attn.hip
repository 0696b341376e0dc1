// Multi-stage attention for gfx950: one flash-style MFMA kernel per stage, and the
// merge that realises the joint softmax across stages
// (inf_llm/attention/dot_production_attention/torch_impl.py:15-96).
//
// Work split.  For one kv head the query heads that share it (GQA) are laid out as
// "wave tasks" (query tile of 32 rows, head-in-group); a workgroup of 8 waves takes 8
// consecutive tasks ordered tile-major/head-minor, so with 4 query heads per kv head
// the 8 waves hold two tiles of 32 queries of the 4 heads and walk the same keys.
// K and V tiles of 64 keys are staged through LDS once per workgroup.
//
// MFMA formulation (v_mfma_f32_32x32x16_bf16), all operands read as 16-byte vectors:
//   S^T[key, query] = K[key, :] . Q[query, :]       A = K rows (LDS), B = Q (registers)
//   O^T[d, query]  += V^T[d, key] . P^T[key, query]  A = V^T rows (LDS), B = P (registers)
// A lane owns ONE query column, so the running max / sum / rescale are per-lane scalars
// and P never leaves registers.  MFMA row r of a 32-key sub-tile is bound to key
// pi(r) = 16*(r>>4) + 8*((r>>2)&1) + 4*((r>>3)&1) + (r&3); with that binding the 16
// accumulator registers of a lane are two runs of 8 consecutive keys, which is exactly
// the k-slice the second MFMA wants from the lane.  V is transposed on its way out of LDS.
#include <cstdlib>

#include "common.h"
#include "decode.h"
#include "rope.h"

#include <algorithm>
#include <atomic>
#include <cstddef>
#include <cstring>
#include <type_traits>

namespace {

constexpr int kWaves = 8;                  // 2 per SIMD inside ONE workgroup: a K/V tile in LDS feeds 256 query rows
constexpr int kStages = 4;                 // K/V tiles resident in LDS
constexpr int kThreads = kWaves * kWave;
constexpr int kQTile = 32;                 // queries per wave
constexpr int kBig = 1 << 29;              // clamp for mask distances held in int32

// a wave-uniform distance clamped to int32, in scalar instructions (there is no scalar 64-bit comparison but for equality)
__device__ __forceinline__ int clamp_big(int64_t x) {
    return (uint64_t)(x + kBig) >> 30 == 0 ? (int)x : (int)(x >> 32) < 0 ? -kBig : kBig;
}

struct StageRange {
    int64_t lo, hi;   // key index range [lo, hi) visible to a span of queries
};

// keys visible to queries [i0, i1] under the stage mask, clipped to the source range
__device__ __forceinline__ StageRange visible_range(const infllm_attn_args &a, int64_t i0, int64_t i1) {
    StageRange r{a.j_lo, a.j_hi};
    if (a.mask == INFLLM_MASK_WINDOW) {
        r.lo = max(r.lo, i0 + a.offset - a.window + 1);
        r.hi = min(r.hi, i1 + a.offset + 1);
    } else if (a.mask == INFLLM_MASK_COMPLEMENT) {
        r.hi = min(r.hi, i1 + a.offset - a.window + 1);
    }
    return r;
}

__device__ __forceinline__ int floordiv64(int64_t x) { return (int)(x >> 6); }   // arithmetic shift = floor

// Division by a launch constant without the divide: q = (n * mul) >> shift is exact for every n < 2^31 when
// mul = floor(2^shift / d) + 1 and shift = 31 + ceil(log2 d) (the excess mul*d - 2^shift is at most d <= 2^ceil(log2 d),
// so the error term n * excess / (d * 2^shift) stays below 1/d).  The kernel's set-up is a chain of such divisions on
// the critical path of a workgroup that lives for only a handful of tiles; a hardware-less 64-bit divide costs
// some two hundred instructions.
struct FastDiv {
    uint32_t d, mul, shift;
};
inline FastDiv fast_div(uint32_t d) {
    uint32_t l = 0;
    while ((1ull << l) < d) ++l;
    return FastDiv{d, (uint32_t)((1ull << (31 + l)) / d + 1), 31 + l};
}
__device__ __forceinline__ uint32_t fdiv(uint32_t n, const FastDiv &f) { return (uint32_t)(((uint64_t)n * f.mul) >> f.shift); }

// launch constants the kernel would otherwise derive with divisions
struct StageGeom {
    // Cosines and sines by which the launch rotates queries that come as they are: of every query's position [Lq, 64] (kLinear and kSinks,
    // heads of 128; NULL: the linear stage's queries are rotated), of the sinks' one angle [D / 2] (kSinks).
    const float2 *q_angles, *sink_angle;
    FastDiv gx, gy, hkv, group, nsplit, cap_tiles;
    int32_t n_tasks;
    // Partial rows by execution block (out_exc > 0): the queries are those of several consecutive execution blocks of
    // out_exc rows (the last one may be shorter), and block k's partials form a [nsplit, B, H, n_k, 128] array of their
    // own at row k * out_block_rows of the partial buffers - where the merge of that block expects them.
    int32_t out_exc;
    int64_t out_block_rows;
    FastDiv out_exc_div;
    // A launch with one key split whose result nothing else joins (out != NULL) writes the finished bf16 rows itself:
    // row [b, h, i] at b * o_sb + h * o_sh + i * o_sl; no partial rows, no merge.
    bf16_t *out;
    int64_t o_sb, o_sh, o_sl;
    float scale;                            // what makes a logit of a product of rows, to base 2
};

// LDS layouts.  Tiles go from global memory straight into LDS (global_load_lds_dwordx4: lane l of a
// wave deposits its 16 bytes at base + 16*l, so one instruction fills 4 rows of 256 bytes), which leaves
// no staging registers; which 16-byte chunk of which row a lane FETCHES is free, and that is where the
// layout is decided:
//   Ks[buf][R][16 chunks]  LDS row R holds key k_lds_row(R) (bits 2 and 3 swapped inside each 32-key
//                          half, so the lane that owns MFMA row r reads LDS row r); chunk c of the row
//                          sits at position c ^ swz(R).  The LDS serves 256 bytes per cycle from 64 banks: a
//                          16-byte read is conflict free when the 16 lanes of a quarter wave hit 16 different
//                          chunk positions, an 8-byte transposing read when the 32 lanes of a half wave hit 32
//                          different 8-byte slots; swz() is a permutation of the 4 low row bits that gives both
//                          (K: 16 consecutive rows, one chunk each; V: 4 rows x 4 chunks x 2 halves).
//   Vs[buf][R][16 chunks]  natural rows, same swizzle; the V^T operand of the second MFMA is formed by
//                          the transposing read ds_read_b64_tr_b16: in a group of 16 lanes, lane 4*j + q
//                          supplies the address of 4 consecutive d of key j, and lane i receives element
//                          i of keys j = 0..3, i.e. 4 consecutive keys at one d.
__device__ __forceinline__ int k_lds_row(int key) { return (key & ~12) | ((key & 4) << 1) | ((key & 8) >> 1); }
typedef short s16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ s16x4 lds_read_tr(uint32_t at) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)(uintptr_t)at);
}
template <int D>
constexpr int kTileBytes = kTile * D * 2;         // one K (or V) tile in LDS
constexpr float kLazyLog2 = 8.f;                  // the running max may lag the true max by 2^8

template <int N>
struct IntC {
    static constexpr int value = N;
};

// MODE: what the launch walks.  kLinear: the linear source of `a`; kPaged: the page table of `a`; kBoth: the linear
// source of `a`, then the page table of `a2` with `a2`'s queries - both stages of the operator in one launch, as ONE
// list of tiles that the key splits divide between them (one set of partials, one fixed cost instead of two).  kSinks:
// the linear source of `a`, then the first j_hi rows of the linear source of `a2` (rows of D elements, no ring) under the
// complement mask with `a2`'s queries - the sliding window and the attention sinks of the sink + window types - which the launch
// rotates to the sinks' angle by the table of it that comes with them.  kSinksStaged: the same of queries that have been rotated, for
// the one call whose scratch does not hold the table (a mode of its own: asking at run time cost the others 0.5 to 1.3 %, sinks +
// window of 4,096 over 16,001 tokens 999 -> 1,013 us).
enum { kLinear = 0, kPaged = 1, kBoth = 2, kSinks = 3, kSinksStaged = 4 };

// The page table can ride in the launch itself (INLINE): the host passes up to kInlinePages entries by value, and the
// kernel reads them where they lie in its argument segment - scalar loads through the constant address space, like the
// table in device memory, but no kernel has to run beforehand to put it there.  The parameter is never touched as a
// C++ object (that would copy it to scratch memory for the dynamic index).
struct InlinePages {
    infllm_page p[kInlinePages];
};
struct NoInlinePages {};
struct KernargLayout {                     // the arguments as the launch lays them out: in order, naturally aligned
    infllm_attn_args a, a2;
    StageGeom geo;
    InlinePages pages;
};

// Heads of 64 leave room for two workgroups on a CU: half the accumulators and operands fit 128 registers (four waves per
// SIMD), the tiles 64 KB.  Their arithmetic per tile is bound by the exponentials (32 of 16 cycles a wave against 512 cycles
// of MFMA), and within one wave the two only add up; with four waves one's MFMAs run under another's exponentials (36 heads,
// prompt of 24,300 tokens, with the scores' smaller workgroups: 4474 -> 3550 us a pass).  The sinks' form, which took 129 registers when
// it was given more, fits as well: sinks + window of 2,048 over 16,001 tokens 773 -> 649 us, of 512 over 7,596 172 -> 147, 4 batch rows of
// 4,096 in a window of 4,000 667 -> 543.
template <int D>
constexpr int kWgsPerCu = D == 64 ? 2 : 1;

// The softmax scale is applied to products, in 32 bits.  In the queries, ahead of their rounding, it saves a score its multiply-add (causal,
// 8,001 tokens, 526 us, 518 so; sinks + window of 4,096 over 16,001 1,022 and 1,014) and costs exactness: pairs that are hardly turned lose
// little as they are rounded, and would as much as all others.  N(0, 1) rows, 1,500 tokens, base 1e6: outputs 2.69e-3 off 64 bits, 2.78e-3
// so; hardly any pair turned 2.16e-3 and 2.52e-3, and with logits up to 70 4.0e-3 and 6.4e-3.
template <int D, int MODE, bool INLINE = false>
__global__ __launch_bounds__(kThreads, 2 * kWgsPerCu<D>) void attn_stage_kernel(infllm_attn_args a, infllm_attn_args a2, StageGeom geo,
                                                                 std::conditional_t<INLINE, InlinePages, NoInlinePages>) {
    constexpr bool HAS_LIN = MODE != kPaged, HAS_PAG = MODE != kLinear, SINKS = MODE == kSinks || MODE == kSinksStaged, TWO = MODE == kBoth || SINKS;
    constexpr int kRow = D * 2, kTB = kTileBytes<D>;                     // bytes of a row, of a tile
    constexpr bool PING = D == 128, kTurns = D == 128 && (MODE == kLinear || MODE == kSinks);
    const infllm_attn_args &ap = TWO ? a2 : a;                 // the paged stage's arguments
    extern __shared__ __attribute__((aligned(1024))) char lds_dyn[];    // kStages K tiles, then kStages V tiles
    char *const Ks = lds_dyn, *const Vs = lds_dyn + kStages * kTB;
    __shared__ int wg_lo[kWaves], wg_hi[kWaves];
    __shared__ __attribute__((aligned(16))) float2 sink_cs[MODE == kSinks ? D / 2 : 2];

    // the wave index is the same in every lane: said so, what derives from it (the wave's queries, tile range, mask
    // distances) stays in scalar registers
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int col = lane & 31, grp = lane >> 5;
    const int G = (int)geo.group.d;
    // Workgroups go to the 8 XCDs round-robin by linear id, and each XCD has its own L2.  Renumber so that
    // one XCD runs a contiguous run of ids: the workgroups that share a (kv head, split) K/V range then sit
    // behind one L2 and that range leaves HBM once instead of once per XCD.  The splits of a head are next to each other, too: they read
    // the same queries (operator over 512 x (4,608 + 2,624) keys 96.5 -> 93.1 us, prompt of 24,300, 36 heads of 64, 2,861 -> 2,843).  Not so
    // over pages of heads of 128, where the heads of a split are (that stage of a block 30.3 us, so 31.4), and beside sinks (1,011 and 1,015).
    int bx = blockIdx.x, by = blockIdx.y, bz = blockIdx.z;
    {
        const int gx = gridDim.x, gy = gridDim.y, total = gx * gy * (int)gridDim.z;
        if ((total & 7) == 0) {
            const int lin = bx + gx * (by + gy * bz);
            const int id = (lin & 7) * (total >> 3) + (lin >> 3);
            const int rest = (int)fdiv(id, geo.gx);
            bx = id - rest * gx;
            if (D == 64 || !HAS_PAG) {                  // id = bx + gx * (bz + nsplit * by)
                by = (int)fdiv(rest, geo.nsplit);
                bz = rest - by * a.nsplit;
            } else {                                    // id = bx + gx * (by + gy * bz)
                bz = (int)fdiv(rest, geo.gy);
                by = rest - bz * gy;
            }
        }
        // a causal launch of more workgroups than the chip holds starts with the last queries, which see the most keys:
        // the short ones fill the end (7,904 causal keys, 512 workgroups: 281 -> 232 us)
        if (HAS_LIN && a.mask == INFLLM_MASK_WINDOW) bx = gx - 1 - bx;
    }
    const int b = (int)fdiv(by, geo.hkv), g = by - b * a.Hkv;
    const int split = bz;
    const int n_tasks = geo.n_tasks;

    // ---- this wave's task and the tiles it needs
    const int task = bx * kWaves + wave;
    const bool live = task < n_tasks;
    const int qt = live ? (int)fdiv(task, geo.group) : 0, hg = live ? task - qt * G : 0;
    const int h = g * G + hg;
    const int i0 = qt * kQTile, i1 = min(i0 + kQTile, a.Lq) - 1;

    if (MODE == kSinks && wave < D / 64)                         // 256 bytes a wave, there with the first tile
        load_to_lds4((const float *)geo.sink_angle, wave * 256 + lane * 4, lds_address((char *)sink_cs) + wave * 256);
    int w_t0 = 0, w_t1 = 0;              // this wave's range of LINEAR tiles (absolute tile numbers)
    if (HAS_LIN && live) {
        StageRange r = visible_range(a, i0, i1);
        if (r.hi > r.lo) {
            w_t0 = floordiv64(r.lo);
            w_t1 = floordiv64(r.hi - 1) + 1;
        }
    }
    // ---- workgroup range of linear tiles = union over its waves
    if (lane == 0) {
        wg_lo[wave] = w_t1 > w_t0 ? w_t0 : INT32_MAX;
        wg_hi[wave] = w_t1 > w_t0 ? w_t1 : INT32_MIN;
    }
    __syncthreads();
    int lin_t0 = INT32_MAX, lin_t1 = INT32_MIN;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
        lin_t0 = min(lin_t0, wg_lo[w]);
        lin_t1 = max(lin_t1, wg_hi[w]);
    }
    if (lin_t1 <= lin_t0) lin_t0 = lin_t1 = 0;
    // The unified tile list: u in [0, n_lin) is linear tile lin_t0 + u, u in [n_lin, n_lin + n_pag) is page u - n_lin.
    const int n_lin = lin_t1 - lin_t0, n_pag = SINKS ? ((int)ap.j_hi + kTile - 1) >> 6 : HAS_PAG ? ap.n_pages : 0;
    int g_t0, g_t1;                      // this split's share of the list
    {
        // n / nsplit tiles each; the n % nsplit left over go one each to a run of splits in the middle: the first and
        // the last split hold the tiles that need the mask (window start, causal diagonal) and take 1-2 us longer over
        // the same number of tiles, so with the extras at the ends the whole launch waited for them
        const uint32_t n = (uint32_t)(n_lin + n_pag), per = fdiv(n, geo.nsplit), rem = n - per * a.nsplit;
        const int first_extra = (int)((a.nsplit - rem) >> 1);
        const int before = min(max(split - first_extra, 0), (int)rem);            // extras given to lower splits
        const int mine = (split >= first_extra && split < first_extra + (int)rem) ? 1 : 0;
        g_t0 = (int)per * split + before;
        g_t1 = g_t0 + (int)per + mine;
    }
    const int wu0 = w_t0 - lin_t0, wu1 = w_t1 - lin_t0;     // this wave's linear tiles in list indices

    bf16x8 qreg[D / 16];                     // Q as the B operand: lane = (query col, k-group); loaded behind the first tiles

    // ---- per-lane LDS byte offsets of the MFMA operands (inside one tile buffer).  One address makes the others: the chunk
    //      bits of an address are the row's swizzle XOR the operand's number, so K operand kk of sub-tile 0 is at
    //      k_off ^ kk * 32 (sub-tile 1: + 32 rows), and the V^T operand of d-tile dt, key half e, of 16-key step gi at
    //      (v_off ^ (dt * 64 + e * 16)) + e * 4 rows + gi * 16 rows.  (Tile buffers begin at multiples of 256 bytes.)
    const uint32_t k_off = lds_address(Ks) + col * kRow + ((grp ^ swz<D>(col)) * 16);
    uint32_t v_off;
    {
        const int lam = lane & 15, g16 = lane >> 4;
        const int vr = 8 * (g16 >> 1) + (lam >> 2);              // lane 4*j + q addresses key j ...
        const int vc = 2 * (g16 & 1) + ((lam & 3) >> 1);         // ... at 4 consecutive d: 16-byte chunk
        const int vh = 8 * (lam & 1);                            //     and byte offset inside it
        v_off = lds_address(Vs) + vr * kRow + ((vc ^ swz<D>(vr)) * 16) + vh;
    }

    // ---- tile loads: an instruction fills 1024 bytes of LDS (4 rows of 128 elements or 8 of 64); wave w fills the 8 rows
    //      from 8*w on; lane -> (row, position).
    //      A wave issues an instruction every four to five cycles whatever its kind (a dependent scalar one every eight),
    //      so the some 300 scalar ones that a tile's addresses and checks used to take cost more than its MFMAs: the tile's
    //      base advances in scalar registers, and which tiles are whole, and which of them a wave sees without a mask, are
    //      ranges that are known before the loop.
    constexpr int kRowsPerLd = 1024 / kRow, kLd = kTile / (kRowsPerLd * kWaves);  // load instructions per wave and tile, for K and for V
    // byte offsets, from row `first` of a tile, of what this lane fetches for load i: rows of kd (vd) elements
    auto tile_row = [&](int i) { return kRowsPerLd * (kLd * wave + i) + lane / (D / 8); };      // row of the LDS tile
    auto k_offset = [&](int i, int64_t kd, int first) {                                          // (of a K tile: key k_lds_row of it)
        const int R = tile_row(i);
        return (uint32_t)((k_lds_row(R) - first) * kd + ((lane & (D / 8 - 1)) ^ swz<D>(R)) * 8) * 2;
    };
    auto v_offset = [&](int i, int64_t vd, int first) {
        const int R = tile_row(i);
        return (uint32_t)((R - first) * vd + ((lane & (D / 8 - 1)) ^ swz<D>(R)) * 8) * 2;
    };
    // Those of the linear source (of the pages, where there is nothing else).  Its rows may lie far apart: the base is that of the
    // first row the wave fetches, so that 32 bits have to reach over a wave's eight rows and not over the tile's 64.
    const int wave_rk = k_lds_row(kRowsPerLd * kLd * wave), wave_rv = kRowsPerLd * kLd * wave;
    uint32_t ld_k[kLd], ld_v[kLd];
#pragma unroll
    for (int i = 0; i < kLd; ++i) {
        ld_k[i] = k_offset(i, HAS_LIN ? a.k_sl : D, HAS_LIN ? wave_rk : 0);
        ld_v[i] = v_offset(i, HAS_LIN ? a.v_sl : D, HAS_LIN ? wave_rv : 0);
    }
    // the linear tile to load next (a tile never wraps: cap is a multiple of the tile), and tiles to the end of the ring
    const bf16_t *k_next = nullptr, *v_next = nullptr;
    const int64_t k_step = (int64_t)kTile * a.k_sl, v_step = (int64_t)kTile * a.v_sl;
    const int64_t ring_k = (int64_t)((uint64_t)a.cap * (uint64_t)a.k_sl), ring_v = (int64_t)((uint64_t)a.cap * (uint64_t)a.v_sl);
    int to_wrap = 0;
    if (HAS_LIN) {
        const int first = lin_t0 + min(g_t0, n_lin);
        const int slot = first - (int)(fdiv(first, geo.cap_tiles) * geo.cap_tiles.d);
        k_next = (const bf16_t *)a.d_k + (int64_t)b * a.k_sb + (int64_t)g * a.k_sh + ((int64_t)slot * kTile + wave_rk) * a.k_sl;
        v_next = (const bf16_t *)a.d_v + (int64_t)b * a.v_sb + (int64_t)g * a.v_sh + ((int64_t)slot * kTile + wave_rv) * a.v_sl;
        to_wrap = (int)min((uint32_t)INT32_MAX, geo.cap_tiles.d - (uint32_t)slot);
    }
    // linear tiles whose 64 rows are all in the source: list indices [whole_lo, whole_hi)
    const int whole_lo = HAS_LIN ? floordiv64(a.j_lo + kTile - 1) - lin_t0 : 0, whole_hi = HAS_LIN ? floordiv64(a.j_hi) - lin_t0 : 0;
    // The page table is read through the constant address space: the index is wave-uniform, so these become scalar
    // loads.  As vector loads they would share the vmcnt counter with the tile transfers, and waiting for a page
    // entry would wait for every tile in flight.  The table is written by an earlier kernel and is read-only here.
    const __attribute__((address_space(4))) infllm_page *page_table;
    if constexpr (INLINE)
        page_table = (const __attribute__((address_space(4))) infllm_page *)((const __attribute__((address_space(4))) char *)
                                                                             __builtin_amdgcn_kernarg_segment_ptr() +
                                                                             offsetof(KernargLayout, pages)) + (int64_t)b * n_pag;
    else
        page_table = (const __attribute__((address_space(4))) infllm_page *)(uintptr_t)ap.d_pages + (int64_t)b * n_pag;
    // the page to load next: its entry is read a tile ahead of its use
    const bf16_t *page_k = nullptr, *page_v = nullptr;
    int page_valid = 0;
    auto next_page = [&](int u) {
        const __attribute__((address_space(4))) infllm_page *entry = page_table + min(max(u - n_lin, 0), n_pag - 1);
        const int64_t hs = entry->head_stride;
        page_k = (const bf16_t *)entry->k + (int64_t)g * hs;
        page_v = (const bf16_t *)entry->v + (int64_t)g * hs;
        page_valid = entry->n_valid;
    };
    constexpr bool PAGES = MODE == kPaged || MODE == kBoth;
    if (PAGES && n_pag > 0) next_page(g_t0);
    const uint32_t lds_k = lds_address(Ks) + wave * (kLd * 1024), lds_v = lds_address(Vs) + wave * (kLd * 1024);
    // requests tile u into the tile buffer `at` bytes in; tiles are requested in ascending order.  Returns the rows of a page.
    bool whole = false;                      // the tile requested last was whole: 2 * kLd loads of this wave
    auto load_tile = [&](int u, uint32_t at) {
        const bf16_t *kbase, *vbase;
        const bool paged = MODE == kPaged || (TWO && u >= n_lin);
        int valid = kTile;
        if (SINKS && paged) {
            const int64_t j0 = (int64_t)(u - n_lin) * kTile;
            kbase = (const bf16_t *)ap.d_k + (int64_t)b * ap.k_sb + (int64_t)g * ap.k_sh + j0 * D;
            vbase = (const bf16_t *)ap.d_v + (int64_t)b * ap.v_sb + (int64_t)g * ap.v_sh + j0 * D;
            valid = (int)min((int64_t)kTile, ap.j_hi - j0);
            whole = valid == kTile;
        } else if (paged) {
            kbase = page_k, vbase = page_v, valid = page_valid;
            whole = valid == kTile;
            next_page(u + 1);
        } else {
            kbase = k_next, vbase = v_next;
            k_next += k_step, v_next += v_step;
            if (--to_wrap == 0) {
                asm volatile("" ::: "memory");         // (a branch, not selects on every tile)
                k_next -= ring_k, v_next -= ring_v;
                to_wrap = (int)geo.cap_tiles.d;
            }
            whole = u >= whole_lo && u < whole_hi;
        }
        const uint32_t kdst = lds_k + at, vdst = lds_v + at;
        uint32_t k_src[kLd], v_src[kLd];
#pragma unroll
        for (int i = 0; i < kLd; ++i) {
            k_src[i] = TWO && paged ? k_offset(i, D, 0) : ld_k[i];
            v_src[i] = TWO && paged ? v_offset(i, D, 0) : ld_v[i];
        }
        if (whole) {                                   // the common case: no per-lane predicate
#pragma unroll
            for (int i = 0; i < kLd; ++i) {
                load_to_lds16(kbase, k_src[i], kdst + i * 1024);
                load_to_lds16(vbase, v_src[i], vdst + i * 1024);
            }
        } else {
            int row_lo = 0, row_hi = valid;            // valid rows of this tile: [row_lo, row_hi)
            if (!paged) {
                const int64_t j0 = (int64_t)(lin_t0 + u) * kTile;
                row_lo = (int)max((int64_t)0, a.j_lo - j0);
                row_hi = (int)min((int64_t)kTile, a.j_hi - j0);
            }
            int ln = lane;
            uint32_t nil = 0;
            asm volatile("" : "+v"(ln), "+v"(nil));    // (places made here and not ahead of all tiles: registers are short)
            char *kz = Ks + at + wave * (kLd * 1024), *vz = Vs + at + wave * (kLd * 1024);
#pragma unroll
            for (int i = 0; i < kLd; ++i) {
                // rows outside the source are written as zeros: their keys are masked, but 0 * stale must stay 0
                const int rv = kRowsPerLd * (kLd * wave + i) + ln / (D / 8), rk = k_lds_row(rv);
                if (rk >= row_lo && rk < row_hi) load_to_lds16(kbase, k_src[i], kdst + i * 1024);
                else *(u32x4 *)(kz + i * 1024 + ln * 16) = u32x4{nil, nil, nil, nil};
                if (rv >= row_lo && rv < row_hi) load_to_lds16(vbase, v_src[i], vdst + i * 1024);
                else *(u32x4 *)(vz + i * 1024 + ln * 16) = u32x4{nil, nil, nil, nil};
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        }
        return valid;
    };

    // ---- running softmax state of this lane's query (max kept in raw logit units, allowed to lag)
    float m_run = -INFINITY, m_limit = -INFINITY, l_run = 0.f, neg_ms = 0.f;
    f32x16 oacc[D / 32];
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[dt][r] = 0.f;

    const float scale = geo.scale, lazy = kLazyLog2 / scale;
    typedef short s16x8 __attribute__((ext_vector_type(8)));
    // kb / vb: k_off / v_off in the tile's buffer
    auto k_operand = [&](uint32_t kb, int kk, int ks) {
        return *(const __attribute__((address_space(3))) u32x4 *)(uintptr_t)((kb ^ (kk * 32)) + ks * 32 * kRow);
    };
    auto v_operand = [&](uint32_t vb, int dt, int gi) {
        s16x8 v;
        v.lo = lds_read_tr((vb ^ (dt * 64)) + gi * 16 * kRow);
        v.hi = lds_read_tr((vb ^ (dt * 64 + 16)) + (gi * 16 + 4) * kRow);
        return __builtin_bit_cast(u32x4, v);
    };

    // Tiles that this wave sees whole, without a mask: of the linear ones [clear_lo, clear_hi), of the sinks' those in front
    // of clear_pag
    int clear_lo = whole_lo, clear_hi = whole_hi, clear_pag = 0;
    if (HAS_LIN) {
        const int64_t q0 = (int64_t)i0 + a.offset, q1 = (int64_t)i1 + a.offset;
        auto tile_of = [&](int64_t j) { return clamp_big(j >> 6); };
        if (a.mask == INFLLM_MASK_WINDOW) {            // every key at a distance of 0 or more from the first query, below the window from the last
            clear_lo = max(clear_lo, tile_of(q1 - a.window) + 1 - lin_t0);
            clear_hi = min(clear_hi, tile_of(q0 - (kTile - 1)) + 1 - lin_t0);
        } else if (a.mask == INFLLM_MASK_COMPLEMENT)
            clear_hi = min(clear_hi, tile_of(q0 - (kTile - 1) - a.window) + 1 - lin_t0);
        clear_hi = min(clear_hi, n_lin);
        if (SINKS) clear_pag = n_lin + min(floordiv64(ap.j_hi), tile_of((int64_t)i0 + ap.offset - (kTile - 1) - ap.window) + 1);
    }
    // the mask of a tile's scores (valid: rows of a page)
    auto mask = [&](f32x16 (&s)[2], int t, [[maybe_unused]] int valid) {
        const bool paged = MODE == kPaged || (TWO && t >= n_lin);
        if (!(PAGES && paged ? valid == kTile : TWO && paged ? t < clear_pag : t >= clear_lo && t < clear_hi)) {
            int ln = lane;
            asm volatile("" : "+v"(ln));
            const int col = ln & 31, grp = ln >> 5;
            int row_lo = 0, row_hi = kTile;
            int d0 = 0;                        // dist of (this lane's query, key 0 of the tile), clamped into int32
            if (SINKS && paged) {
                const int64_t j0 = (int64_t)(t - n_lin) * kTile, e0 = (int64_t)i0 + ap.offset - j0;
                row_hi = (int)min((int64_t)kTile, ap.j_hi - j0);
                d0 = clamp_big(e0) + col;
            } else if (paged) {
                row_hi = valid;
            } else {
                const int64_t j0 = (int64_t)(lin_t0 + t) * kTile, e0 = (int64_t)i0 + a.offset - j0;
                row_lo = (int)max((int64_t)0, a.j_lo - j0);
                row_hi = (int)min((int64_t)kTile, a.j_hi - j0);
                d0 = clamp_big(e0) + col;
            }
            // Whatever the mask, a lane's query sees ONE run of the tile's keys: its bounds are found once, and a key costs a
            // subtraction and a compare (a mask's conditions key by key: 150 branches in the sinks' form of the kernel).
            // dist = dl - kc; kc is the compile-time part of register r's key, which is kc + 8 * grp
            const int64_t win64 = SINKS && paged ? ap.window : a.window;
            const int win = (int)(win64 >> 32) >= 0 && (uint64_t)win64 >> 30 != 0 ? 2 * kBig : (int)win64, dl = d0 - 8 * grp;
            int lo_l = row_lo - 8 * grp, hi_l = row_hi - 8 * grp;
            if (SINKS && paged) {
                hi_l = min(hi_l, dl - win + 1);
            } else if (!paged) {
                if (a.mask == INFLLM_MASK_WINDOW) lo_l = max(lo_l, dl - win + 1), hi_l = min(hi_l, dl + 1);
                if (a.mask == INFLLM_MASK_COMPLEMENT) hi_l = min(hi_l, dl - win + 1);
            }
            const uint32_t n_l = (uint32_t)max(hi_l - lo_l, 0);
#pragma unroll
            for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int kc = ks * 32 + 16 * (r >> 3) + (r & 7);
                    const bool vis = MODE == kPaged ? kc < hi_l : (uint32_t)(kc - lo_l) < n_l;      // (a page begins with its rows)
                    s[ks][r] = vis ? s[ks][r] : -INFINITY;
                }
        }
    };
    // Row sums are taken over the probabilities AS ROUNDED to bf16, the values that P.V multiplies: the output is then an exact
    // convex combination of value rows (a row on which one key carries nearly all the weight comes out as that value row,
    // whatever the rounding of its weight).  In a product of 4 x 4 x 4 blocks every lane is a column of its own block, so
    // against ones it receives the sum of its own four values: 8 cycles of the matrix pipe for 4 keys.  (As one more 32 x
    // 32 x 16 product per step, 128 cycles a tile instead of 64, prompts of 131,072 tokens 26,020 -> 25,495 us, the operator over
    // 512 x (4,608 + 2,624) 102.7 -> 101.3; as 64 shifts and additions 220 cycles of the vector half.)
    uint32_t one_one;
    asm volatile("v_mov_b32 %0, 0x3f803f80" : "=v"(one_one));
    const s16x4 ones = __builtin_bit_cast(s16x4, u32x2{one_one, one_one});
    auto add_row_sums = [&](u32x4 p, f32x4 sums) {
        sums = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(ones, __builtin_bit_cast(s16x4, u32x2{p[0], p[1]}), sums, 0, 0, 0);
        return __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(ones, __builtin_bit_cast(s16x4, u32x2{p[2], p[3]}), sums, 0, 0, 0);
    };
    // the running max that a tile's scores move, and with it the accumulators
    auto max_and_rescale = [&](f32x16 (&s)[2]) {
        // (four chains: a dependent instruction waits twice as long as another)
        float tm[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
#pragma unroll
        for (int r = 0; r < 8; r += 2)
#pragma unroll
            for (int i = 0; i < 4; ++i) tm[i] = fmaxf(fmaxf(tm[i], s[i & 1][8 * (i >> 1) + r]), s[i & 1][8 * (i >> 1) + r + 1]);
        const float tmax = wave_max32(fmaxf(fmaxf(fmaxf(tm[0], tm[1]), tm[2]), tm[3]));
        // lazy running max: it only moves when a score would exceed it by more than 2^kLazyLog2 after scaling,
        // so the rescale of the output accumulators is rare; probabilities stay below 2^kLazyLog2
        const bool moved = tmax > m_limit;
        if (__builtin_amdgcn_ballot_w64(moved) != 0) {
            const float m_new = moved ? tmax : m_run;
            const float alpha = __builtin_amdgcn_exp2f((m_run - m_new) * scale);      // exp2(-inf) = 0 on the first move
            const float al = moved ? alpha : 1.f;
            l_run *= al;
#pragma unroll
            for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
                for (int r = 0; r < 16; ++r) oacc[dt][r] *= al;
            m_run = m_new;
            m_limit = m_new + lazy;
            neg_ms = (m_run == -INFINITY) ? 0.f : -m_run * scale;
        }
    };
    // heads of 64: a tile's arithmetic by itself; the SIMD's other three waves fill its waits.  Vector instructions go first, of whichever wave:
    // a wave that has nothing but MFMAs to issue keeps the matrix pipe busy with one every 32 cycles, and the others' exponentials are the
    // longer half (36 heads, prompt of 24,300 tokens: 2,902 -> 2,874 us a pass; MFMAs first 2,901, waves 4 - 7 first 2,901 against 2,889).
    auto tile_math = [&](int buf, int t) {
        uint32_t kb = k_off + buf * kTB, vb = v_off + buf * kTB;
        asm volatile("" : "+v"(kb), "+v"(vb));       // (an operand's address is made where it is read: registers are short)
        f32x16 s[2];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int r = 0; r < 16; ++r) s[ks][r] = 0.f;
        {
            // 8 K operands in groups of 2: a group is requested from LDS while the MFMAs of the previous one run;
            // scheduling fences keep the compiler from serialising read -> MFMA
            u32x4 ka[D / 16][2];
#pragma unroll
            for (int j = 0; j < 2; ++j) ka[0][j] = k_operand(kb, 0, j);
#pragma unroll
            for (int gi = 0; gi < D / 16; ++gi) {
                __builtin_amdgcn_sched_barrier(0);
                if (gi < D / 16 - 1) {
#pragma unroll
                    for (int j = 0; j < 2; ++j) ka[gi + 1][j] = k_operand(kb, gi + 1, j);
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int j = 0; j < 2; ++j) s[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, ka[gi][j]), qreg[gi], s[j], 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_s_setprio(1);
        mask(s, t, PAGES && (MODE == kPaged || t >= n_lin) ? page_table[t - n_lin].n_valid : kTile);
        max_and_rescale(s);
        f32x4 sums{0.f, 0.f, 0.f, 0.f};
        uint32_t pw[2][8];
        auto exps = [&](int ks, int r0, int r1) {
#pragma unroll
            for (int r = r0; r < r1; r += 2) {
                float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[ks][r], scale, neg_ms));
                float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[ks][r + 1], scale, neg_ms));
                pw[ks][r >> 1] = pack_bf16x2(p0, p1);
            }
        };
        exps(0, 0, 16);                        // the first 32 keys now; the other 32 beside the MFMAs that consume these
        {
            // 4 steps of 16 keys
#pragma unroll
            for (int gi = 0; gi < 4; ++gi) {
                u32x4 va[D / 32];
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int dt = 0; dt < D / 32; ++dt) va[dt] = v_operand(vb, dt, gi);
                const int ks = gi >> 1, mm = gi & 1;
                u32x4 praw{pw[ks][4 * mm], pw[ks][4 * mm + 1], pw[ks][4 * mm + 2], pw[ks][4 * mm + 3]};
                bf16x8 pb = __builtin_bit_cast(bf16x8, praw);
                // A wave's own vector-ALU work hides under its MFMAs when the two are interleaved instruction by
                // instruction (an MFMA holds the matrix pipe for 32 cycles and the issue port for a few): the
                // exponentials of the tile's second half go between the MFMAs of its first half.
                if (gi == 2) __builtin_amdgcn_s_setprio(0);
                if (gi < 2) exps(1, 8 * gi, 8 * gi + 8);
#pragma unroll
                for (int dt = 0; dt < D / 32; ++dt)
                    oacc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, va[dt]), pb, oacc[dt], 0, 0, 0);
                sums = add_row_sums(praw, sums);
                if (gi < 2) {
#pragma unroll
                    for (int dt = 0; dt < D / 32; ++dt) {
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);      // one MFMA
                        __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);      // multiply-adds, rounding, row sum
                        __builtin_amdgcn_sched_group_barrier(0x400, 2, 0);      // two exponentials
                        __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        l_run += sums[0];
    };

    // The sinks' queries are the step's own rows, rotated here to the one angle of the sinks: staged beside the others they were a third
    // of what the staging launch wrote (sinks + window of 4,096 over 16,001 tokens, 32 / 8 heads of 128: 1,063 -> 1,041 us; window of
    // 2,048 over two rows of 8,001: 633 -> 612; 36 heads of 64, whose sinks' queries are a seventh: 371 -> 370).
    auto load_q = [&](const infllm_attn_args &src, [[maybe_unused]] bool sinks) {
        const int qi = i0 + col;
        const bool ok = live && qi < src.Lq;
        const bf16_t *qrow = (const bf16_t *)src.d_q + (int64_t)b * src.q_sb + (int64_t)h * src.q_sh + (int64_t)qi * src.q_sl;
        if (MODE == kSinks && sinks) {                           // (a query behind the last: it again, never stored)
            qrow -= ok ? 0 : (int64_t)(qi - (src.Lq - 1)) * src.q_sl;
#pragma unroll
            for (int kk = 0; kk < D / 16; ++kk) qreg[kk] = __builtin_bit_cast(bf16x8, *(const u32x4 *)(qrow + kk * 16 + grp * 8));
#pragma unroll
            for (int kk = 0; kk < D / 32; ++kk) {                // in place, a pair at a time: registers are short
                __builtin_amdgcn_sched_barrier(0);
                const Rot8 r = rotate8(__builtin_bit_cast(u32x4, qreg[kk]), __builtin_bit_cast(u32x4, qreg[kk + D / 32]), sink_cs + kk * 16 + grp * 8);
                qreg[kk] = __builtin_bit_cast(bf16x8, r.lo);
                qreg[kk + D / 32] = __builtin_bit_cast(bf16x8, r.hi);
                asm volatile("" : "+v"(qreg[kk]), "+v"(qreg[kk + D / 32]));
            }
            return;
        }
#pragma unroll
        for (int kk = 0; kk < D / 16; ++kk) {
            u32x4 raw = ok ? *(const u32x4 *)(qrow + kk * 16 + grp * 8) : u32x4{0, 0, 0, 0};
            qreg[kk] = __builtin_bit_cast(bf16x8, raw);
        }
    };
    // does this wave see tile u at all?  (pages: every live wave; linear tiles: the wave's own visible range)
    auto mine = [&](int u) {
        if (SINKS && u >= n_lin) return live && (int64_t)i1 + ap.offset - ap.window >= (int64_t)(u - n_lin) * kTile;
        return (HAS_PAG && u >= n_lin) ? live : (u >= wu0 && u < wu1);
    };
    // the queries of the stage this split starts in; a split that crosses from the linear tiles into the pages swaps
    // them for the paged stage's queries at its first page (once per workgroup: that wait also covers the tiles in flight)
    bool q_paged = MODE == kPaged || (TWO && g_t0 >= n_lin);

    if constexpr (!PING) {
    // Tiles are handled in pairs: one barrier per two tiles.  While the pair (t, t+1) is multiplied, the next
    // pair is on its way into the other two buffers, which were last read before the previous barrier; the
    // loads of a pair are the only ones outstanding, so landing = vmcnt(0).
    static_assert(PING || kStages == 4, "two buffer pairs");
    for (int p = 0; p < 2; ++p)
        if (g_t0 + p < g_t1) load_tile(g_t0 + p, p * kTB);
    if (MODE == kSinks && q_paged) {                             // (a split that begins with the sinks: the angle first)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    }
    load_q(q_paged ? ap : a, q_paged);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    // The compiler does not know that the wait above also covered the query rows; passing them through an empty
    // asm makes it place its own wait for them HERE rather than in front of their first use inside the loop,
    // where a vmcnt(0) would wait for the tiles in flight.
#pragma unroll
    for (int kk = 0; kk < D / 16; ++kk) asm volatile("" : "+v"(qreg[kk]));
    __syncthreads();
    for (int t = g_t0; t < g_t1; t += 2) {
        const int buf = (t - g_t0) & 3;                          // 0 or 2
        if (t + 2 < g_t1) load_tile(t + 2, (buf ^ 2) * kTB);
        if (t + 3 < g_t1) load_tile(t + 3, ((buf ^ 2) + 1) * kTB);
#pragma unroll
        for (int e = 0; e < 2; ++e) {                            // wave-uniform conditions; barriers stay outside
            const int u = t + e;
            if (u >= g_t1) break;
            if (TWO && u >= n_lin && !q_paged) {
                load_q(ap, true);
                q_paged = true;
            }
            if (mine(u)) tile_math(buf + e, u);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    }
    } else {
    // Heads of 128.  A SIMD runs MFMAs of one wave beside vector instructions of another, but its two waves, at the same
    // place of the same code, want the same of the two at any time.  So waves w and w + 4, which share a SIMD, take turns:
    // while one multiplies - P.V of the tile before, then K.Q of this one, 36 MFMAs of 32 cycles -, the other forms its
    // probabilities.  The second four are half a tile behind, by one more barrier in front of their loop, and a barrier ends
    // each half.  A wave requests its rows of tile t + 2 while it multiplies with t and sees those of t + 1 through at the end
    // of that half, a tile's time after their request; the values of t - 2, whose buffer t + 2 takes, were last read a tile
    // earlier.  What the halves cost was found one instruction at a time (cycles of a tile and two waves; 4,200 with both
    // waves in step): the turns with the instructions of the old loop 4,600, row sums without dot instructions (they run on
    // the matrix pipe and wait until it is empty, also of the other wave's work) and MFMAs first (s_setprio) 4,450, addresses
    // and checks out of the loop 3,290, operand reads between the MFMAs instead of in runs of 8 and row sums as MFMAs 3,010,
    // the maximum in four chains and reads between the exponentials 2,800.  8,192 queries x 4,096 window keys, 32 heads:
    // 587 -> 500 us of N(0, 1) data, 510 -> 372 of zeros, on which the card does not lower its clock.
    f32x16 s[2];
    uint32_t pw[2][8];
    // A half's 32 operands, one per MFMA: 0-15 the V^T of the tile before (16-key step, then d-tile), 16-31 the K of this one.
    // Each is requested 8 MFMAs ahead, into the registers of the one that has just been used, and between the MFMAs: a run
    // of reads keeps the wave from issuing them.
    u32x4 op[8];
    uint32_t at = 0;                       // the buffer of the tile at hand
    auto request = [&](int i, uint32_t vb, uint32_t kb) {
        op[i & 7] = i < 16 ? v_operand(vb, (i & 3) % (D / 32), i >> 2) : k_operand(kb, ((i - 16) >> 1) % (D / 16), i & 1);
    };
    auto exps = [&](int ks, int r0, int r1) {
#pragma unroll
        for (int r = r0; r < r1; r += 2) {
            const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[ks][r], scale, neg_ms));
            const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[ks][r + 1], scale, neg_ms));
            pw[ks][r >> 1] = pack_bf16x2(p0, p1);
            asm volatile("" : "+v"(pw[ks][r >> 1]));                                // formed here, not where it is read
        }
    };
    // O += P.V of the tile before; the first 8 operands are on their way when it begins.
    auto pv_mul = [&](uint32_t vb, uint32_t kb, auto meanwhile) {
        f32x4 sums{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            __builtin_amdgcn_sched_barrier(0);
            meanwhile(g);
            const u32x4 praw{pw[g >> 1][4 * (g & 1)], pw[g >> 1][4 * (g & 1) + 1], pw[g >> 1][4 * (g & 1) + 2], pw[g >> 1][4 * (g & 1) + 3]};
            const bf16x8 pb = __builtin_bit_cast(bf16x8, praw);
#pragma unroll
            for (int dt = 0; dt < D / 32; ++dt) {
                oacc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, op[(4 * g + dt) & 7]), pb, oacc[dt], 0, 0, 0);
                request(4 * g + dt + 8, vb, kb);
            }
            sums = add_row_sums(praw, sums);
#pragma unroll
            for (int dt = 0; dt < D / 32; ++dt) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                  // one MFMA
                __builtin_amdgcn_sched_group_barrier(0x002, 1, 0);                  // an operand's address
                if (g < 2) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);       // its reads
                else __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        l_run += sums[0];
    };
    // S = K.Q of this tile; its first 8 operands are on their way
    auto qk_mul = [&](uint32_t kb) {
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int r = 0; r < 16; ++r) s[ks][r] = 0.f;
#pragma unroll
        for (int g = 4; g < 8; ++g) {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int i = 4 * g + j;
                s[i & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, op[i & 7]), qreg[((i - 16) >> 1) % (D / 16)], s[i & 1], 0, 0, 0);
                if (i + 8 < 32) request(i + 8, 0, kb);
            }
            if (g < 6) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // the vector half: max and rescale, the probabilities, the first 8 operands of P.V
    auto probabilities = [&]() {
        max_and_rescale(s);
        __builtin_amdgcn_sched_barrier(0);
        exps(0, 0, 16);
        exps(1, 0, 16);
#pragma unroll
        for (int i = 0; i < 8; ++i) request(i, v_off + at, 0);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);                      // two keys' multiply-adds
            __builtin_amdgcn_sched_group_barrier(0x400, 2, 0);                      // their exponentials
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);                      // a read
            __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);                      // rounding, an address
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto half_end = [&]() { asm volatile("s_barrier" ::: "memory"); };
    auto all_but_last = [&]() { asm volatile("s_waitcnt vmcnt(%0)" ::"i"(2 * kLd) : "memory"); };      // but the rows of one whole tile
    auto landed = [&]() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); };
    const bool second = wave >= 4;
    int t = g_t0;                          // the tile at hand, and rows of the pages t, t + 1, t + 2
    int valid0 = kTile, valid1 = kTile, valid2 = kTile;
    // The wave's queries, the first tile and the second are requested at once, and only the second may still be on its way when
    // the loop begins.  The queries come by way of LDS - the two buffers that the third and fourth tile take -, because a load
    // into registers is waited for by the compiler, which knows of no other: with everything in flight.  (With the second tile
    // behind the first one's arrival and queries into registers: operator over 512 x (4,608 + 2,624) keys 101.0 -> 102.2 us,
    // causal prompt of 8,001 tokens 536 -> 540.  Pages, whose second tile's address is an entry of its own to wait for, gain
    // nothing by it: prompt of 131,072 25,690 us with, 25,350 without.)
    const infllm_attn_args &first = q_paged ? ap : a;
    // Rows to be rotated come that way too, and their angles (512 bytes a query) into the second tile's buffer, which is requested when
    // they have been read.  (By lanes that each fetch their own query's pieces, 32 lines an instruction: sinks + window of 4,096 over 16,001
    // tokens 1,060 -> 1,041 us, of 512 over 7,596 174.7 -> 167.2, causal prompt of 8,001 542 -> 535.)
    // (Two tiles of queries a workgroup at most: infllm_attn_turns.)
    const bool turn_lds = kTurns && geo.q_angles && !q_paged;
    if (turn_lds) {
        const int qt0 = (int)fdiv(bx * kWaves, geo.group), half = wave >> 2;
        const uint32_t at_q = (wave < 4 ? lds_address(Ks) : lds_address(Vs)) + 2 * kTB + (wave & 3) * (kQTile * kRow);
        const bf16_t *rows = (const bf16_t *)a.d_q + (int64_t)b * a.q_sb + (int64_t)h * a.q_sh + (int64_t)i0 * a.q_sl;
#pragma unroll
        for (int i = 0; i < kQTile * kRow / 1024; ++i) {
            const int r = kRowsPerLd * i + lane / (D / 8);                              // (rows behind the last: it again, never stored)
            load_to_lds16(rows, (uint32_t)(min(r, a.Lq - 1 - i0) * (int)a.q_sl + ((lane & (D / 8 - 1)) ^ swz<D>(r)) * 8) * 2, at_q + i * 1024);
        }
        const uint32_t angles = lds_address(half == 0 ? Ks : Vs) + kTB;                 // waves 0 - 3: of the first query tile, 4 - 7: of the second
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = ((wave & 3) * 4 + i) * 2 + (lane >> 5), q = min((qt0 + half) * kQTile + r, a.Lq - 1);
            load_to_lds16((const bf16_t *)geo.q_angles, (uint32_t)q * (D * 4) + ((lane & 31) ^ r) * 16, angles + ((wave & 3) * 4 + i) * 1024);
        }
        if (t < g_t1) valid0 = load_tile(t, 0);
        landed();
        half_end();
        const uint32_t own = at_q + col * kRow + ((grp ^ swz<D>(col)) * 16);
        const uint32_t own_angles = lds_address(qt == qt0 ? Ks : Vs) + kTB + col * (D * 4);
#pragma unroll
        for (int kk = 0; kk < D / 32; ++kk) {
            const u32x4 lo = *(const __attribute__((address_space(3))) u32x4 *)(uintptr_t)(own ^ (kk * 32));
            const u32x4 hi = *(const __attribute__((address_space(3))) u32x4 *)(uintptr_t)(own ^ ((kk + D / 32) * 32));
            f32x4 cs[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) cs[i] = *(const __attribute__((address_space(3))) f32x4 *)(uintptr_t)(own_angles + (((kk * 8 + grp * 4 + i) ^ col) * 16));
            const Rot8 r = rotate8(lo, hi, (const float2 *)cs);
            qreg[kk] = __builtin_bit_cast(bf16x8, r.lo);
            qreg[kk + D / 32] = __builtin_bit_cast(bf16x8, r.hi);
            asm volatile("" : "+v"(qreg[kk]), "+v"(qreg[kk + D / 32]));                 // (read before the barrier)
        }
    } else if (MODE != kPaged && !(SINKS && q_paged) && (uint64_t)first.q_sl < (uint64_t)1 << 26) {
        const uint32_t at_q = (wave < 4 ? lds_address(Ks) : lds_address(Vs)) + 2 * kTB + (wave & 3) * (kQTile * kRow);
        const bf16_t *rows = (const bf16_t *)first.d_q + (int64_t)b * first.q_sb + (int64_t)h * first.q_sh + (int64_t)i0 * first.q_sl;
#pragma unroll
        for (int i = 0; i < kQTile * kRow / 1024; ++i) {
            const int r = kRowsPerLd * i + lane / (D / 8);                              // (rows behind the last: it again, never stored)
            load_to_lds16(rows, (uint32_t)(min(r, first.Lq - 1 - i0) * (int)first.q_sl + ((lane & (D / 8 - 1)) ^ swz<D>(r)) * 8) * 2, at_q + i * 1024);
        }
        if (t < g_t1) valid0 = load_tile(t, 0);
        whole = false;
        if (t + 1 < g_t1) valid1 = load_tile(t + 1, kTB);
        if (whole) all_but_last();
        else landed();
        const uint32_t own = at_q + col * kRow + ((grp ^ swz<D>(col)) * 16);
#pragma unroll
        for (int kk = 0; kk < D / 16; ++kk) {
            qreg[kk] = __builtin_bit_cast(bf16x8, *(const __attribute__((address_space(3))) u32x4 *)(uintptr_t)(own ^ (kk * 32)));
            asm volatile("" : "+v"(qreg[kk]));                                          // (read before the barrier)
        }
    } else {                               // pages, and rows that a 32-bit offset does not reach: far apart, or backwards
        if (t < g_t1) valid0 = load_tile(t, 0);
        if (MODE == kSinks && q_paged) {                         // (a split that begins with the sinks: the angle first)
            landed();
            half_end();
        }
        load_q(first, q_paged);
        landed();
#pragma unroll
        for (int kk = 0; kk < D / 16; ++kk) asm volatile("" : "+v"(qreg[kk]));
        if (t + 1 < g_t1) valid1 = load_tile(t + 1, kTB);
    }
    half_end();
    if (turn_lds) {
        whole = false;
        if (t + 1 < g_t1) valid1 = load_tile(t + 1, kTB);
    }
    if (second) half_end();
    bool have_p = false;                   // the tile before has probabilities that wait for their values
    // A tile with nothing special about it - whole, seen without a mask, the tile before seen too and the one to request
    // whole - takes the form without branches.  Of the pages that is known one at a time.
    const int hot_lo = max(max(wu0 + 1, g_t0 + 1), clear_lo), hot_hi = min(min(min(wu1, clear_hi), min(whole_hi, g_t1) - 2), n_lin - 2);
    auto is_hot = [&]() {
        if (MODE == kPaged) return t + 2 < g_t1 && valid0 == kTile && page_valid == kTile;
        return t < hot_hi;
    };
    const int64_t k_back = k_step - ring_k, v_back = v_step - ring_v;
    auto hot = [&]() {
        const uint32_t kb = k_off + at, vb = v_off + ((at - kTB) & (4 * kTB - 1));
        const uint32_t to = (at + 2 * kTB) & (4 * kTB - 1), kdst = lds_k + to, vdst = lds_v + to;
        const bf16_t *kbase = k_next, *vbase = v_next;
        if (MODE == kPaged)
            kbase = page_k, vbase = page_v;
        else {
            --to_wrap;
            k_next += to_wrap == 0 ? k_back : k_step;
            v_next += to_wrap == 0 ? v_back : v_step;
            to_wrap = to_wrap == 0 ? (int)geo.cap_tiles.d : to_wrap;
        }
        __builtin_amdgcn_s_setprio(1);       // the MFMAs go first
        pv_mul(vb, kb, [&](int g) {          // the tile after next: a request beside each of the four steps
            static_assert(D != 128 || kLd == 2, "two loads of K and of V a wave");
            if (g < kLd) load_to_lds16(kbase, ld_k[g % kLd], kdst + g * 1024);
            else load_to_lds16(vbase, ld_v[g % kLd], vdst + (g - kLd) * 1024);
        });
        qk_mul(kb);
        if (MODE == kPaged) next_page(t + 3);
        all_but_last();
        half_end();
        __builtin_amdgcn_s_setprio(0);
        probabilities();
        half_end();
        at = (at + kTB) & (4 * kTB - 1);
        if (PAGES) valid0 = valid1, valid1 = kTile;
        ++t;
    };
    auto special = [&]() {
        whole = false;
        if (t + 2 < g_t1) valid2 = load_tile(t + 2, (at + 2 * kTB) & (4 * kTB - 1));
        if (TWO && t >= n_lin && !q_paged) {
            load_q(ap, true);
            q_paged = true;
        }
        const bool see = mine(t);
        const uint32_t kb = k_off + at;
        __builtin_amdgcn_s_setprio(1);
        if (have_p) pv_mul(v_off + ((at - kTB) & (4 * kTB - 1)), kb, [](int) {});
        else {
#pragma unroll
            for (int i = 16; i < 24; ++i) request(i, 0, kb);
        }
        if (see) qk_mul(kb);
        if (whole) all_but_last();
        else landed();
        half_end();
        __builtin_amdgcn_s_setprio(0);
        if (see) {
            mask(s, t, valid0);
            probabilities();
        }
        have_p = see;
        half_end();
        at = (at + kTB) & (4 * kTB - 1);
        if (PAGES) valid0 = valid1, valid1 = valid2;
        ++t;
    };
    while (t < g_t1) {
        if (have_p && (MODE == kPaged || t >= hot_lo) && is_hot())
            do hot();
            while (is_hot());
        special();
    }
    if (have_p) pv_mul(v_off + ((at - kTB) & (4 * kTB - 1)), k_off, [](int) {});
    if (!second) half_end();
    half_end();                            // every tile has been read: the epilogue stages rows in the buffers
    }

    // ---- epilogue: normalised partial + base-2 log-sum-exp.  The accumulators hold O^T (a lane owns a query and
    //      scattered 4-float pieces of its row); they go through this wave's 16 KB of the now idle tile buffers so
    //      that every store instruction writes two whole 512-byte rows.
    if (!live) return;
    const float l_tot = l_run + wave_xor32(l_run);
    const int qi = i0 + col;
    const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
    int64_t row0 = (((int64_t)split * a.B + b) * a.H + h) * a.Lq + i0;            // row of this wave's first query
    int rows_left = a.Lq - i0;                                                     // valid queries of this tile
    if (geo.out_exc > 0) {                    // a query tile lies inside one execution block (out_exc is a multiple of the tile)
        const int blk = (int)fdiv(i0, geo.out_exc_div), in_blk = i0 - blk * geo.out_exc;
        const int n_blk = min(geo.out_exc, a.Lq - blk * geo.out_exc);
        row0 = (int64_t)blk * geo.out_block_rows + (((int64_t)split * a.B + b) * a.H + h) * n_blk + in_blk;
        rows_left = n_blk - in_blk;
    }
    const int64_t row = row0 + col;
    char *stage = lds_dyn + wave * (kQTile * kRow);
    constexpr int kChunks = D / 8;                                                 // 16-byte chunks of a row
    constexpr int kRowsPerSt = 64 / kChunks;                                       // rows a wave stores per instruction
    if (geo.out) {                                                                 // the finished rows, rounded to bf16 once
#pragma unroll
        for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4) {
                const u32x2 o4{pack_bf16x2(oacc[dt][4 * q4] * inv, oacc[dt][4 * q4 + 1] * inv),
                               pack_bf16x2(oacc[dt][4 * q4 + 2] * inv, oacc[dt][4 * q4 + 3] * inv)};
                const int chunk = dt * 4 + q4;
                *(u32x2 *)(stage + col * kRow + ((chunk ^ col) & (kChunks - 1)) * 16 + grp * 8) = o4;
            }
        const int piece = lane & (kChunks - 1);
        bf16_t *dst = geo.out + (int64_t)b * geo.o_sb + (int64_t)h * geo.o_sh + (int64_t)i0 * geo.o_sl + piece * 8;
#pragma unroll
        for (int k4 = 0; k4 < kQTile / kRowsPerSt; ++k4) {
            const int qr = kRowsPerSt * k4 + lane / kChunks;
            const u32x4 o8 = *(const u32x4 *)(stage + qr * kRow + ((piece ^ qr) & (kChunks - 1)) * 16);
            if (qr < rows_left) *(u32x4 *)(dst + (int64_t)qr * geo.o_sl) = o8;
        }
        return;
    }
    {
        // fp16 keeps 11 bits of a value that ends up rounded to bf16's 8, and halves what the partials cost in HBM
        // (with few tiles per workgroup their write is a tenth of the kernel); staged rows are 256 bytes, a lane's
        // 4-value piece is 8 bytes, and 16-byte chunks are swizzled by the row
#pragma unroll
        for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4) {
                const f16x4 o4{(_Float16)(oacc[dt][4 * q4] * inv), (_Float16)(oacc[dt][4 * q4 + 1] * inv),
                               (_Float16)(oacc[dt][4 * q4 + 2] * inv), (_Float16)(oacc[dt][4 * q4 + 3] * inv)};
                const int chunk = dt * 4 + q4;                                     // 16-byte chunk of the row; grp picks its half
                *(f16x4 *)(stage + col * kRow + ((chunk ^ col) & (kChunks - 1)) * 16 + grp * 8) = o4;
            }
        const int piece = lane & (kChunks - 1);
        _Float16 *o_part = (_Float16 *)a.d_o_part;
#pragma unroll
        for (int k4 = 0; k4 < kQTile / kRowsPerSt; ++k4) {
            const int qr = kRowsPerSt * k4 + lane / kChunks;
            const u32x4 o8 = *(const u32x4 *)(stage + qr * kRow + ((piece ^ qr) & (kChunks - 1)) * 16);
            if (qr < rows_left) *(u32x4 *)(o_part + (row0 + qr) * D + piece * 8) = o8;
        }
    }
    if (qi >= a.Lq) return;
    if (grp == 0) a.d_lse_part[row] = l_tot > 0.f ? m_run * scale + log2f(l_tot) : -INFINITY;
}

// one thread per (row, 8 dims): P fp16 partials -> bf16 output row + final lse (merge_piece, common.h)
template <int D>
__global__ __launch_bounds__(256) void attn_merge_kernel(MergeJob job) { merge_piece<D>(job, (int64_t)blockIdx.x * 256 + threadIdx.x); }

// ... of several execution blocks' partials (infllm_attn_stage_blocked), blockIdx.y one of them
template <int D>
__global__ __launch_bounds__(256) void attn_merge_blocked_kernel(MergeJob job, int64_t block_rows, int32_t exc, int32_t n) {
    const int32_t q0 = (int32_t)blockIdx.y * exc;
    job.Lq = min(exc, n - q0);
    job.o_part += blockIdx.y * block_rows * D;
    job.lse_part += blockIdx.y * block_rows;
    job.out += q0 * job.o_sl;
    job.lse_out += q0;
    merge_piece<D>(job, (int64_t)blockIdx.x * 256 + threadIdx.x);
}

// the log-sum-exp half of the merge alone: one thread per row
__global__ __launch_bounds__(256) void attn_merge_lse_kernel(const float *lse_part, int P, int64_t rows, float *lse_out, PartSets ps) {
    const int64_t row = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (row >= rows) return;
    float m = -INFINITY, den = 0.f;
    for (int p0 = 0; p0 < P; p0 += 8) {                 // online over batches of 8 independent loads
        float l8[8], m8 = -INFINITY;
#pragma unroll
        for (int i = 0; i < 8; ++i) l8[i] = p0 + i < P ? lse_part[ps.l(p0 + i, rows) + row] : -INFINITY;
#pragma unroll
        for (int i = 0; i < 8; ++i) m8 = fmaxf(m8, l8[i]);
        if (m8 == -INFINITY) continue;
        const float m_new = fmaxf(m, m8);
        den *= __builtin_amdgcn_exp2f(m - m_new);
#pragma unroll
        for (int i = 0; i < 8; ++i) den += __builtin_amdgcn_exp2f(l8[i] - m_new);
        m = m_new;
    }
    lse_out[row] = den > 0.f ? m + log2f(den) : -INFINITY;
}

// The same two merges for few rows and many partials (decode-sized blocks: a handful of query rows, dozens of key
// splits).  16 adjacent lanes share a row piece and take every 16th partial each, so all partials are one or two
// round trips to memory instead of a chain; the lanes' sums are then joined by a fixed butterfly.
__device__ __forceinline__ float group16_max(float v) {
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    return v;
}
__device__ __forceinline__ float group16_sum(float v) {
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

template <int D>
__global__ __launch_bounds__(256) void attn_merge_wide_kernel(const _Float16 *o_part, const float *lse_part, int P, int B, int H,
                                                              int Lq, bf16_t *out, int64_t o_sb, int64_t o_sh, int64_t o_sl,
                                                              float *lse_out, PartSets ps) {
    const int64_t rows = (int64_t)B * H * Lq;
    const int64_t e = ((int64_t)blockIdx.x * 256 + threadIdx.x) >> 4;       // (row, 8 dims)
    const int pl = threadIdx.x & 15;
    constexpr int kPieces = D / 8;
    const int64_t row = e / kPieces;
    const int c = (int)(e % kPieces);
    if (row >= rows) return;                                                 // whole 16-lane groups leave together
    constexpr int kMine = 8;                                                 // partials per lane: P <= 128
    float l[kMine];
    f16x8 o[kMine];
    float m = -INFINITY;
#pragma unroll
    for (int i = 0; i < kMine; ++i) {
        const int p = pl + 16 * i;
        const bool on = p < P;
        l[i] = on ? lse_part[ps.l(p, rows) + row] : -INFINITY;
        o[i] = on ? *(const f16x8 *)(o_part + (ps.l(p, rows) + row) * D + ps.o(p) + c * 8) : f16x8{0, 0, 0, 0, 0, 0, 0, 0};
        m = fmaxf(m, l[i]);
    }
    m = group16_max(m);
    if (m == -INFINITY) m = 0.f;                                             // as in merge_piece
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, den = 0.f;
#pragma unroll
    for (int i = 0; i < kMine; ++i) {
        const float w = __builtin_amdgcn_exp2f(l[i] - m);
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[j] += (float)o[i][j] * w;
        den += w;
    }
    den = group16_sum(den);
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] = group16_sum(acc[j]);
    if (pl != 0) return;
    const float inv = den > 0.f ? 1.f / den : 0.f;
    const int i = (int)(row % Lq), h = (int)((row / Lq) % H), b = (int)(row / ((int64_t)Lq * H));
    u32x4 packed{pack_bf16x2(acc[0] * inv, acc[1] * inv), pack_bf16x2(acc[2] * inv, acc[3] * inv),
                 pack_bf16x2(acc[4] * inv, acc[5] * inv), pack_bf16x2(acc[6] * inv, acc[7] * inv)};
    *(u32x4 *)(out + (int64_t)b * o_sb + (int64_t)h * o_sh + (int64_t)i * o_sl + c * 8) = packed;
    if (c == 0 && lse_out) lse_out[row] = den > 0.f ? m + log2f(den) : -INFINITY;
}

__global__ __launch_bounds__(256) void attn_merge_lse_wide_kernel(const float *lse_part, int P, int64_t rows, float *lse_out, PartSets ps) {
    const int64_t row = ((int64_t)blockIdx.x * 256 + threadIdx.x) >> 4;
    const int pl = threadIdx.x & 15;
    if (row >= rows) return;
    constexpr int kMine = 8;
    float l[kMine], m = -INFINITY;
#pragma unroll
    for (int i = 0; i < kMine; ++i) {
        const int p = pl + 16 * i;
        l[i] = p < P ? lse_part[ps.l(p, rows) + row] : -INFINITY;
        m = fmaxf(m, l[i]);
    }
    m = group16_max(m);
    float den = 0.f;
    if (m > -INFINITY) {
#pragma unroll
        for (int i = 0; i < kMine; ++i) den += __builtin_amdgcn_exp2f(l[i] - m);
    }
    den = group16_sum(den);
    if (pl == 0) lse_out[row] = den > 0.f ? m + log2f(den) : -INFINITY;
}

}  // namespace

#define HIP_OK_ATTN(call, what)                                                         \
    do {                                                                                \
        hipError_t e_ = (call);                                                         \
        if (e_ != hipSuccess) return infllm_fail(-2, "%s: %s", what, hipGetErrorString(e_)); \
    } while (0)

namespace {

int check_linear_stage(const infllm_attn_args *a) {
    INFLLM_REQUIRE(a->j_hi <= a->j_lo || (a->d_k && a->d_v), "attn_stage: null k / v pointer");
    INFLLM_REQUIRE(a->cap > 0 && a->cap % kTile == 0, "attn_stage: cap %lld is not a positive multiple of %d",
                   (long long)a->cap, kTile);
    INFLLM_REQUIRE(a->j_lo >= 0 && a->j_hi - a->j_lo <= a->cap, "attn_stage: key range [%lld,%lld) exceeds cap %lld",
                   (long long)a->j_lo, (long long)a->j_hi, (long long)a->cap);
    INFLLM_REQUIRE(a->mask >= 0 && a->mask <= 2, "attn_stage: unknown mask %d", a->mask);
    INFLLM_REQUIRE(a->j_hi < (1ll << 36), "attn_stage: key range beyond 2^36 rows");
    INFLLM_REQUIRE((a->k_sl % 8 | a->k_sh % 8 | a->k_sb % 8 | a->v_sl % 8 | a->v_sh % 8 | a->v_sb % 8) == 0,
                   "attn_stage: k/v strides must be multiples of 8");
    // A lane's offset is 32 bits of bytes, from the first row that its wave fetches of a tile: up to 11 keys (k_lds_row), as many as there are.
    const int64_t rows = a->j_hi - a->j_lo, far = rows <= 0 ? 0 : std::min<int64_t>(11, a->j_lo % kTile + rows - 1);
    const int64_t most = far == 0 ? INT64_MAX : ((1ll << 31) - 128) / far;
    INFLLM_REQUIRE(far == 0 || (a->k_sl >= 0 && a->v_sl >= 0 && a->k_sl <= most && a->v_sl <= most), "attn_stage: k/v rows of %lld / %lld elements apart",
                   (long long)a->k_sl, (long long)a->v_sl);
    return 0;
}

int check_common(const infllm_attn_args *a) {
    INFLLM_REQUIRE(a->d_q, "attn_stage: null q pointer");
    INFLLM_REQUIRE(a->B > 0 && a->H > 0 && a->Hkv > 0 && a->H % a->Hkv == 0 && a->Lq > 0,
                   "attn_stage: bad geometry B=%d H=%d Hkv=%d Lq=%d", a->B, a->H, a->Hkv, a->Lq);
    INFLLM_REQUIRE(a->nsplit >= 1 && a->nsplit <= 64, "attn_stage: nsplit %d out of range", a->nsplit);
    INFLLM_REQUIRE((a->q_sl % 8 | a->q_sh % 8 | a->q_sb % 8) == 0, "attn_stage: q strides must be multiples of 8");
    return 0;
}

// Where a launch's rows go besides the argument block's partial buffers, and what it rotates its queries by: see StageGeom
struct StageOut {
    int out_exc = 0;
    int64_t out_block_rows = 0;
    bf16_t *out = nullptr;
    int64_t o_sb = 0, o_sh = 0, o_sl = 0;
    const float2 *q_angles = nullptr, *sink_angle = nullptr;
};

template <int D, int MODE, bool INLINE, typename Pages>
int launch_mode(dim3 grid, const infllm_attn_args &a, const infllm_attn_args &a2, const StageGeom &geo, const Pages &pages, void *stream) {
    constexpr size_t lds_bytes = 2 * kStages * kTileBytes<D>;
    static std::atomic<bool> lds_set{false};                  // dynamic LDS above 64 KiB must be enabled once per kernel
    if (!lds_set.load(std::memory_order_acquire)) {
        const hipError_t e = hipFuncSetAttribute((const void *)attn_stage_kernel<D, MODE, INLINE>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
        if (e != hipSuccess) return infllm_fail(-2, "attn_stage: %s", hipGetErrorString(e));
        lds_set.store(true, std::memory_order_release);
    }
    hipLaunchKernelGGL((attn_stage_kernel<D, MODE, INLINE>), grid, dim3(kThreads), lds_bytes, (hipStream_t)stream, a, a2, geo, pages);
    INFLLM_CHECK_LAUNCH("attn_stage");
    return 0;
}

// mode: kLinear (a), kPaged (a), kBoth / kSinks / kSinksStaged (a = linear stage, a2 = the other stage); h_pages: NULL, or the paged
// stage's table [B, n_pages] in HOST memory, B * n_pages <= kInlinePages, which then travels in the launch (d_pages is
// not read)
template <int D = kD>
int launch_stage(int mode, const infllm_attn_args *a, const infllm_attn_args *a2, void *stream, const infllm_page *h_pages = nullptr,
                 const StageOut &so = StageOut()) {
    const int G = a->H / a->Hkv;
    const int n_tasks = ((a->Lq + kQTile - 1) / kQTile) * G;
    dim3 grid((n_tasks + kWaves - 1) / kWaves, a->B * a->Hkv, a->nsplit);
    INFLLM_REQUIRE((int64_t)grid.x * grid.y * grid.z < (1ll << 31), "attn_stage: grid too large");
    StageGeom geo{so.q_angles, so.sink_angle, fast_div(grid.x), fast_div(grid.y), fast_div((uint32_t)a->Hkv), fast_div((uint32_t)G),
                  fast_div((uint32_t)a->nsplit), fast_div(1), n_tasks, so.out_exc, so.out_block_rows,
                  fast_div((uint32_t)(so.out_exc > 0 ? so.out_exc : 1)), so.out, so.o_sb, so.o_sh, so.o_sl, a->softmax_scale * kLog2e};
    // tile indices stay below 2^30, so any ring of 2^31 tiles or more never wraps: one divisor stands for all of them
    if (mode != kPaged) geo.cap_tiles = fast_div((uint32_t)std::min<int64_t>(a->cap / kTile, 1ll << 31));
    const infllm_attn_args &second = a2 ? *a2 : *a;
    if (h_pages) {
        const infllm_attn_args &pg = mode == kBoth ? second : *a;
        INFLLM_REQUIRE((mode == kPaged || mode == kBoth) && pg.n_pages >= 0 && (int64_t)pg.B * pg.n_pages <= kInlinePages,
                       "attn_stage: %d x %d pages do not fit a launch", pg.B, pg.n_pages);
        InlinePages table;
        memcpy(table.p, h_pages, sizeof(infllm_page) * pg.B * pg.n_pages);
        return mode == kPaged ? launch_mode<D, kPaged, true>(grid, *a, second, geo, table, stream)
                              : launch_mode<D, kBoth, true>(grid, *a, second, geo, table, stream);
    }
    constexpr NoInlinePages none{};
    switch (mode) {
        case kLinear: return launch_mode<D, kLinear, false>(grid, *a, second, geo, none, stream);
        case kPaged: return launch_mode<D, kPaged, false>(grid, *a, second, geo, none, stream);
        case kBoth: return launch_mode<D, kBoth, false>(grid, *a, second, geo, none, stream);
        case kSinks: return launch_mode<D, kSinks, false>(grid, *a, second, geo, none, stream);
        default: return launch_mode<D, kSinksStaged, false>(grid, *a, second, geo, none, stream);
    }
}

}  // namespace

extern "C" int infllm_attn_stage(const infllm_attn_args *a, void *stream) {
    INFLLM_REQUIRE(a != nullptr, "attn_stage: null argument block");
    INFLLM_REQUIRE(a->d_o_part && a->d_lse_part, "attn_stage: null output pointer");
    int rc = check_common(a);
    if (rc) return rc;
    if (a->d_pages) {
        INFLLM_REQUIRE(a->n_pages >= 0, "attn_stage: negative page count");
        return launch_stage(kPaged, a, nullptr, stream);
    }
    rc = check_linear_stage(a);
    if (rc) return rc;
    if (a->Lq == 1 && a->k_sl == kD && a->v_sl == kD) {
        // One query: what it sees is a range of keys, at most two runs of ring rows - the streaming kernel, which reads a
        // kv head's rows once for its query heads (4097 ring rows, 32 splits: 9.6 -> 5 us).
        int64_t lo = a->j_lo, hi = a->j_hi;
        if (a->mask == INFLLM_MASK_WINDOW) lo = std::max(lo, a->offset - a->window + 1), hi = std::min(hi, a->offset + 1);
        else if (a->mask == INFLLM_MASK_COMPLEMENT) hi = std::min(hi, a->offset - a->window + 1);
        DecodeJob d{};
        d.q[0] = d.q[1] = (const bf16_t *)a->d_q;
        d.q_sb = a->q_sb; d.q_sh = a->q_sh;
        d.B = a->B; d.H = a->H; d.Hkv = a->Hkv;
        d.scale = a->softmax_scale;
        d.nsplit = a->nsplit;
        d.o_part = a->d_o_part; d.lse_part = a->d_lse_part;
        for (int64_t pos = lo; pos < hi;) {
            const int64_t row = pos % a->cap, n = std::min(hi - pos, a->cap - row);
            INFLLM_REQUIRE(n < (1ll << 31), "attn_stage: key range too long");
            d.seg[d.n_seg++] = DecodeSeg{(const bf16_t *)a->d_k + row * kD, (const bf16_t *)a->d_v + row * kD, a->k_sb, a->k_sh, a->v_sb, a->v_sh, (int32_t)n,
                                         0, 0, nullptr, -1};
            pos += n;
        }
        if (d.n_seg == 0) d.n_seg = 1;                 // nothing visible: empty partials
        return infllm_decode_attn(&d, kD, stream);
    }
    return launch_stage(kLinear, a, nullptr, stream);
}

int infllm_attn_splits(int64_t wgs, int64_t tiles, int32_t max_parts, double mean_tiles);
extern "C" int infllm_attn_stage_splits(const infllm_attn_args *a, int32_t max_splits) {
    INFLLM_REQUIRE(a && a->B > 0 && a->H > 0 && a->Hkv > 0 && a->H % a->Hkv == 0 && a->Lq > 0 && max_splits >= 1, "attn_stage_splits: bad arguments");
    int64_t keys = a->d_pages ? (int64_t)a->n_pages * kTile : a->j_hi - a->j_lo;
    if (!a->d_pages && a->mask == INFLLM_MASK_WINDOW) keys = std::min<int64_t>(keys, a->window + kTile);
    keys = std::max<int64_t>(keys, 1);
    if (a->Lq == 1 && !a->d_pages) return infllm_decode_splits(a->B, a->H, a->Hkv, kD, (keys + kDecodeBlock - 1) / kDecodeBlock, std::min(max_splits, 64), 0, 0);
    const int64_t wgs = ((int64_t)((a->Lq + kQTile - 1) / kQTile) * (a->H / a->Hkv) + kWaves - 1) / kWaves * a->Hkv * a->B;
    const int64_t tiles = (keys + kTile - 1) / kTile;
    return infllm_attn_splits(wgs, tiles, std::min(max_splits, 64), (double)tiles);
}

// library-internal: a linear stage over the queries of several consecutive execution blocks of `exc` rows (the last
// may be shorter); block k's partial rows and log-sum-exps start at row k * block_rows of d_o_part / d_lse_part and
// are laid out [nsplit, B, H, n_k, 128] / [nsplit, B, H, n_k], as infllm_attn_merge takes them for that block.
int infllm_attn_stage_blocked(const infllm_attn_args *a, int32_t exc, int64_t block_rows, void *stream, int32_t dim) {
    INFLLM_REQUIRE(a && a->d_o_part && a->d_lse_part && !a->d_pages, "attn_stage_blocked: null argument or paged source");
    INFLLM_REQUIRE(exc > 0 && exc % kQTile == 0, "attn_stage_blocked: blocks of %d rows are not whole query tiles", exc);
    INFLLM_REQUIRE(block_rows >= (int64_t)a->nsplit * a->B * a->H * (a->Lq < exc ? a->Lq : exc), "attn_stage_blocked: block stride too small");
    int rc = check_common(a);
    if (rc) return rc;
    rc = check_linear_stage(a);
    if (rc) return rc;
    StageOut so;
    so.out_exc = exc;
    so.out_block_rows = block_rows;
    INFLLM_REQUIRE(dim == 128 || dim == 64, "attn_stage_blocked: head_dim %d", dim);
    return dim == 128 ? launch_stage<128>(kLinear, a, nullptr, stream, nullptr, so) : launch_stage<64>(kLinear, a, nullptr, stream, nullptr, so);
}

// library-internal: the paged stage over a table in device memory, or (h_pages != NULL, B * n_pages <=
// infllm_inline_page_limit()) one in host memory that the launch carries, for heads of 128 or 64
int infllm_attn_paged(const infllm_attn_args *a, const infllm_page *h_pages, void *stream, int32_t dim) {
    INFLLM_REQUIRE(a && a->d_o_part && a->d_lse_part && (h_pages || a->d_pages) && a->n_pages >= 0, "attn_paged: null argument");
    INFLLM_REQUIRE(dim == 128 || dim == 64, "attn_paged: head_dim %d", dim);
    const int rc = check_common(a);
    if (rc) return rc;
    return dim == 128 ? launch_stage<128>(kPaged, a, nullptr, stream, h_pages) : launch_stage<64>(kPaged, a, nullptr, stream, h_pages);
}

// library-internal: the paged stage (local == NULL) or both stages in one launch, with the page table [B, n_pages]
// given in HOST memory and carried by the launch; global->d_pages is not read.  B * n_pages <= infllm_inline_page_limit().
int infllm_inline_page_limit() { return kInlinePages; }
int infllm_attn_paged_inline(const infllm_attn_args *local, const infllm_attn_args *global, const infllm_page *h_pages, void *stream) {
    INFLLM_REQUIRE(global && h_pages && global->d_o_part && global->d_lse_part, "attn_paged_inline: null argument");
    int rc = check_common(global);
    if (rc) return rc;
    if (!local) return launch_stage(kPaged, global, nullptr, stream, h_pages);
    INFLLM_REQUIRE(local->d_o_part && local->d_lse_part && !local->d_pages, "attn_paged_inline: bad local stage");
    INFLLM_REQUIRE(local->B == global->B && local->H == global->H && local->Hkv == global->Hkv && local->Lq == global->Lq &&
                       local->softmax_scale == global->softmax_scale,
                   "attn_paged_inline: the two stages disagree");
    rc = check_common(local);
    if (rc) return rc;
    rc = check_linear_stage(local);
    return rc ? rc : launch_stage(kBoth, local, global, stream, h_pages);
}

extern "C" int infllm_attn_stages_fused(const infllm_attn_args *local, const infllm_attn_args *global, void *stream) {
    INFLLM_REQUIRE(local && global, "attn_stages_fused: null argument block");
    INFLLM_REQUIRE(local->d_o_part && local->d_lse_part, "attn_stages_fused: null output pointer");
    INFLLM_REQUIRE(!local->d_pages && global->d_pages && global->n_pages >= 0,
                   "attn_stages_fused: the first stage must be linear, the second paged");
    INFLLM_REQUIRE(local->B == global->B && local->H == global->H && local->Hkv == global->Hkv && local->Lq == global->Lq,
                   "attn_stages_fused: the two stages disagree on B / H / Hkv / Lq");
    INFLLM_REQUIRE(local->softmax_scale == global->softmax_scale, "attn_stages_fused: the two stages disagree on the softmax scale");
    int rc = check_common(local);
    if (rc) return rc;
    rc = check_common(global);
    if (rc) return rc;
    rc = check_linear_stage(local);
    return rc ? rc : launch_stage(kBoth, local, global, stream);
}

extern "C" int infllm_attn_merge(const uint16_t *d_o_part, const float *d_lse_part, int32_t P, int32_t B, int32_t H,
                                 int32_t Lq, void *d_out, int64_t o_sb, int64_t o_sh, int64_t o_sl, float *d_lse,
                                 void *stream);

extern "C" int infllm_attn_fwd(const infllm_attn_args *local, const infllm_attn_args *global, void *d_out, int64_t o_sb,
                               int64_t o_sh, int64_t o_sl, float *d_lse, void *stream) {
    INFLLM_REQUIRE(local || global, "attn_fwd: no stage given");
    INFLLM_REQUIRE(d_out || d_lse, "attn_fwd: neither output nor lse requested");
    const infllm_attn_args *first = local ? local : global;
    int parts = first->nsplit;
    if (local && global) {
        INFLLM_REQUIRE(local->B == global->B && local->H == global->H && local->Lq == global->Lq,
                       "attn_fwd: the two stages disagree on B / H / Lq");
        const int64_t rows = (int64_t)local->B * local->H * local->Lq;
        INFLLM_REQUIRE(global->d_o_part == local->d_o_part + (int64_t)local->nsplit * rows * kD &&
                           global->d_lse_part == local->d_lse_part + (int64_t)local->nsplit * rows,
                       "attn_fwd: the global stage's partials must follow the local stage's in one buffer");
        parts += global->nsplit;
    }
    int rc = local ? infllm_attn_stage(local, stream) : 0;
    if (rc) return rc;
    rc = global ? infllm_attn_stage(global, stream) : 0;
    if (rc) return rc;
    return infllm_attn_merge(first->d_o_part, first->d_lse_part, parts, first->B, first->H, first->Lq, d_out, o_sb, o_sh, o_sl,
                             d_lse, stream);
}

// ---- the forward for callers that cannot allocate
// The stages' partial rows are scratch memory: infllm_attn_fwd takes them from the caller.  A caller under HIP graph
// capture, in a tight serving loop or in a harness that forbids hipMalloc has nowhere to get them from, so this
// variant keeps them in an array of the library's own image.  Every GPU the library runs on holds its own copy of the
// array (at its own address) until the process ends; every call on a GPU uses that GPU's copy, so calls that overlap on
// one GPU race.  Nothing has to be cleared between calls: each split writes all of its rows and log-sum-exps before
// the merge reads them.
constexpr int64_t kStaticPartRows = INFLLM_NOALLOC_MAX_PART_ROWS;            // (split, batch row, head, query) rows
static __device__ __align__(256) unsigned char attn_static_scratch[kStaticPartRows * (kD * 2 + 4)];
constexpr int kMaxDevices = 64;
// per device: where ITS copy of the array lives.  Atomic: two threads making their first call on a device both look the
// address up and store the same value
static std::atomic<unsigned char *> static_scratch_ptr[kMaxDevices];

extern "C" int infllm_attn_fwd_noalloc(const infllm_attn_args *local, const infllm_attn_args *global, void *d_out, int64_t o_sb,
                                       int64_t o_sh, int64_t o_sl, float *d_lse, void *stream) {
    INFLLM_REQUIRE(local || global, "attn_fwd_noalloc: no stage given");
    const infllm_attn_args *first = local ? local : global;
    INFLLM_REQUIRE(first->B > 0 && first->H > 0 && first->Lq > 0, "attn_fwd_noalloc: bad geometry");
    if (local && global)
        INFLLM_REQUIRE(local->B == global->B && local->H == global->H && local->Lq == global->Lq,
                       "attn_fwd_noalloc: the two stages disagree on B / H / Lq");
    const int parts = (local ? local->nsplit : 0) + (global ? global->nsplit : 0);
    const int64_t rows = (int64_t)first->B * first->H * first->Lq;
    INFLLM_REQUIRE(parts >= 1 && parts <= 128, "attn_fwd_noalloc: %d key splits", parts);
    INFLLM_REQUIRE(parts * rows <= kStaticPartRows,
                   "attn_fwd_noalloc: %d splits x %lld rows exceed the built-in scratch of %lld partial rows (use infllm_attn_fwd "
                   "with a workspace of your own)", parts, (long long)rows, (long long)kStaticPartRows);
    int dev = -1;
    HIP_OK_ATTN(hipGetDevice(&dev), "attn_fwd_noalloc");
    INFLLM_REQUIRE(dev >= 0 && dev < kMaxDevices, "attn_fwd_noalloc: device %d", dev);
    unsigned char *scratch = static_scratch_ptr[dev].load(std::memory_order_acquire);
    if (!scratch) {                            // once per device, with that device current: the symbol's address THERE
        void *p = nullptr;
        HIP_OK_ATTN(hipGetSymbolAddress(&p, HIP_SYMBOL(attn_static_scratch)), "attn_fwd_noalloc: hipGetSymbolAddress");
        INFLLM_REQUIRE(p != nullptr, "attn_fwd_noalloc: no address for the scratch array");
        scratch = (unsigned char *)p;
        static_scratch_ptr[dev].store(scratch, std::memory_order_release);
    }
    // o partials first (fp16 rows), the log-sum-exps behind all of them; the global stage's follow the local stage's
    uint16_t *o_part = (uint16_t *)scratch;
    float *lse_part = (float *)(scratch + kStaticPartRows * kD * 2);
    infllm_attn_args l{}, g{};
    if (local) {
        l = *local;
        l.d_o_part = o_part;
        l.d_lse_part = lse_part;
    }
    if (global) {
        g = *global;
        const int64_t skip = local ? (int64_t)local->nsplit * rows : 0;
        g.d_o_part = o_part + skip * kD;
        g.d_lse_part = lse_part + skip;
    }
    return infllm_attn_fwd(local ? &l : nullptr, global ? &g : nullptr, d_out, o_sb, o_sh, o_sl, d_lse, stream);
}

// library-internal: the description of a merge over two sets of partials, P1 behind (d_o_part, d_lse_part) and P2
// behind (d_o_part2, d_lse_part2), in that order; P2 == 0 is the plain merge.  dim: elements of a row, 128 or 64.
int infllm_merge_job(const uint16_t *d_o_part, const float *d_lse_part, int32_t P1, const uint16_t *d_o_part2, const float *d_lse_part2,
                     int32_t P2, int32_t B, int32_t H, int32_t Lq, void *d_out, int64_t o_sb, int64_t o_sh, int64_t o_sl, float *d_lse,
                     MergeJob *job, int32_t dim) {
    INFLLM_REQUIRE(d_o_part && d_lse_part && job, "attn_merge: null pointer");
    INFLLM_REQUIRE(P1 >= 1 && P2 >= 0 && (P2 == 0 || (d_o_part2 && d_lse_part2)), "attn_merge: bad partial sets %d + %d", P1, P2);
    INFLLM_REQUIRE(B > 0 && H > 0 && Lq > 0, "attn_merge: bad sizes B=%d H=%d Lq=%d", B, H, Lq);
    INFLLM_REQUIRE((int64_t)B * H * Lq < (1ll << 31), "attn_merge: %lld rows", (long long)B * H * Lq);
    INFLLM_REQUIRE(dim == 128 || dim == 64, "attn_merge: rows of %d elements", dim);
    INFLLM_REQUIRE((o_sl % 8 | o_sh % 8 | o_sb % 8) == 0, "attn_merge: output strides must be multiples of 8");
    PartSets ps{P1 + P2, 0, 0};
    if (P2 > 0) {
        const int64_t rows_ = (int64_t)B * H * Lq;
        ps.n_first = P1;
        // index (p * rows + row) of the first buffers -> index ((p - P1) * rows + row) of the second
        ps.skip_l = (int64_t)(((intptr_t)d_lse_part2 - (intptr_t)d_lse_part) / (intptr_t)sizeof(float)) - (int64_t)P1 * rows_;
        ps.skip_o = (int64_t)(((intptr_t)d_o_part2 - (intptr_t)d_o_part) / 2) - (int64_t)P1 * rows_ * dim - ps.skip_l * dim;
    }
    *job = MergeJob{(const _Float16 *)d_o_part, d_lse_part, P1 + P2, B, H, Lq, (bf16_t *)d_out, o_sb, o_sh, o_sl, d_lse, ps, Lq};
    return 0;
}

// library-internal: the merge of the partials that infllm_attn_stage_blocked left for n queries in blocks of exc (P of them a
// block, blocks block_rows apart), in one launch: rows of all blocks to d_out, their joint log-sum-exps [B, H, n] to d_lse
int infllm_attn_merge_blocked(const uint16_t *d_o_part, const float *d_lse_part, int32_t P, int32_t B, int32_t H, int32_t n, int32_t exc, int64_t block_rows,
                              void *d_out, int64_t o_sb, int64_t o_sh, int64_t o_sl, float *d_lse, void *stream, int32_t dim) {
    INFLLM_REQUIRE(n > 0 && exc > 0 && d_out && d_lse && (n + exc - 1) / exc <= 65535, "attn_merge_blocked: bad arguments");
    MergeJob job;
    const int rc = infllm_merge_job(d_o_part, d_lse_part, P, nullptr, nullptr, 0, B, H, std::min(n, exc), d_out, o_sb, o_sh, o_sl, d_lse, &job, dim);
    if (rc) return rc;
    job.lse_sh = n;
    const int64_t threads = (int64_t)B * H * std::min(n, exc) * (dim / 8);
    hipLaunchKernelGGL((dim == 64 ? attn_merge_blocked_kernel<64> : attn_merge_blocked_kernel<128>), dim3((unsigned)((threads + 255) / 256), (n + exc - 1) / exc),
                       dim3(256), 0, (hipStream_t)stream, job, block_rows, exc, n);
    INFLLM_CHECK_LAUNCH("attn_merge_blocked");
    return 0;
}

// library-internal: the merge over two sets of partials
int infllm_attn_merge2(const uint16_t *d_o_part, const float *d_lse_part, int32_t P1, const uint16_t *d_o_part2,
                       const float *d_lse_part2, int32_t P2, int32_t B, int32_t H, int32_t Lq, void *d_out, int64_t o_sb,
                       int64_t o_sh, int64_t o_sl, float *d_lse, void *stream, int32_t dim) {
    MergeJob job;
    const int jrc = infllm_merge_job(d_o_part, d_lse_part, P1, d_o_part2, d_lse_part2, P2, B, H, Lq, d_out, o_sb, o_sh, o_sl, d_lse, &job, dim);
    if (jrc) return jrc;
    const int32_t P = P1 + P2;
    const PartSets ps = job.ps;
    // few rows, many partials (decode-sized blocks): 16 lanes per row piece, each taking every 16th partial
    const bool wide = P > 8 && P <= 128 && (int64_t)B * H * Lq <= 2048;
    if (!d_out) {                                     // log-sum-exp only
        INFLLM_REQUIRE(d_lse, "attn_merge: neither output nor lse requested");
        const int64_t rows = (int64_t)B * H * Lq;
        if (wide)
            hipLaunchKernelGGL(attn_merge_lse_wide_kernel, dim3((unsigned)((rows * 16 + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                               d_lse_part, P, rows, d_lse, ps);
        else
            hipLaunchKernelGGL(attn_merge_lse_kernel, dim3((unsigned)((rows + 255) / 256)), dim3(256), 0, (hipStream_t)stream, d_lse_part,
                               P, rows, d_lse, ps);
        INFLLM_CHECK_LAUNCH("attn_merge (lse)");
        return 0;
    }
    const int64_t threads = (int64_t)B * H * Lq * (dim / 8);
    if (wide)
        hipLaunchKernelGGL((dim == 64 ? attn_merge_wide_kernel<64> : attn_merge_wide_kernel<128>), dim3((unsigned)((threads * 16 + 255) / 256)),
                           dim3(256), 0, (hipStream_t)stream, (const _Float16 *)d_o_part, d_lse_part, P, B, H, Lq, (bf16_t *)d_out, o_sb, o_sh, o_sl, d_lse, ps);
    else
        hipLaunchKernelGGL((dim == 64 ? attn_merge_kernel<64> : attn_merge_kernel<128>), dim3((unsigned)((threads + 255) / 256)), dim3(256), 0,
                           (hipStream_t)stream, job);
    INFLLM_CHECK_LAUNCH("attn_merge");
    return 0;
}

extern "C" int infllm_attn_merge(const uint16_t *d_o_part, const float *d_lse_part, int32_t P, int32_t B, int32_t H,
                                 int32_t Lq, void *d_out, int64_t o_sb, int64_t o_sh, int64_t o_sl, float *d_lse,
                                 void *stream) {
    return infllm_attn_merge2(d_o_part, d_lse_part, P, nullptr, nullptr, 0, B, H, Lq, d_out, o_sb, o_sh, o_sl, d_lse, stream, kD);
}

extern "C" int infllm_attn_merge_pair(const uint16_t *d_o_part, const float *d_lse_part, int32_t P1, const uint16_t *d_o_part2, const float *d_lse_part2,
                                      int32_t P2, int32_t B, int32_t H, int32_t Lq, void *d_out, int64_t o_sb, int64_t o_sh, int64_t o_sl, float *d_lse,
                                      void *stream) {
    return infllm_attn_merge2(d_o_part, d_lse_part, P1, d_o_part2, d_lse_part2, P2, B, H, Lq, d_out, o_sb, o_sh, o_sl, d_lse, stream, kD);
}

// library-internal: whether a launch rotates its linear queries itself.  A workgroup has room for the angles of two tiles of queries:
// its eight waves take eight consecutive (tile, query head of the group) pairs from a multiple of eight on, and those lie in two tiles
// at most of groups of four heads and of six and more.  Six and seven are still staged; rotated here they would be the faster too (48 / 8
// and 28 / 4 heads, causal prompts of 1,537 / 3,073 / 8,001 tokens 67.3 / 157.8 / 745.5 us and 63.2 / 126.6 / 459.3 staged, 63.7 / 150.4 /
// 719.5 and 61.7 / 123.1 / 446.1 so).  Heads of 64 take their queries another way.  32-bit offsets have to reach rows and angles.
bool infllm_attn_turns(int32_t H, int32_t Hkv, int32_t n_q, int64_t q_sl, int32_t dim) {
    const int G = H / Hkv;
    return dim == 128 && (G == 4 || G >= 8) && q_sl >= 0 && q_sl < 1 << 26 && n_q < 1 << 22;
}

// library-internal: a linear stage and (sinks != NULL) the rows of a second source under the complement mask, under one
// softmax, as rows of `dim` elements (128 or 64) in the caller's layout; local->nsplit key splits of the joint tile list,
// with partial rows at local->d_o_part / d_lse_part when there is more than one
// q_angles: NULL, or cosine and sine of every query's angles [Lq, 64], by which the launch rotates local's rows (infllm_attn_turns);
// sink_angle: NULL, or of the one angle of the sinks' queries [dim / 2], by which it rotates theirs
int infllm_attn_window(const infllm_attn_args *local, const infllm_attn_args *sinks, const void *q_angles, const void *sink_angle, int32_t dim, void *d_out,
                       int64_t o_sb, int64_t o_sh, int64_t o_sl, void *stream) {
    INFLLM_REQUIRE(local && d_out && (dim == 128 || dim == 64), "attn_window: bad arguments");
    int rc = check_common(local);
    if (rc) return rc;
    rc = check_linear_stage(local);
    if (rc) return rc;
    if (sinks) {
        INFLLM_REQUIRE(sinks->d_q && sinks->d_k && sinks->d_v && sinks->j_lo == 0 && sinks->j_hi >= 0 && sinks->k_sl == dim && sinks->v_sl == dim,
                       "attn_window: bad sink rows");
        INFLLM_REQUIRE(sinks->Lq == local->Lq && sinks->B == local->B && sinks->H == local->H && ((sinks->q_sl | sinks->q_sh | sinks->q_sb) & 7) == 0,
                       "attn_window: the two stages disagree");
    }
    INFLLM_REQUIRE(!q_angles || infllm_attn_turns(local->H, local->Hkv, local->Lq, local->q_sl, dim), "attn_window: queries that are not rotated");
    StageOut so;
    so.q_angles = (const float2 *)q_angles;
    so.sink_angle = (const float2 *)sink_angle;
    if (local->nsplit == 1) {
        so.out = (bf16_t *)d_out;
        so.o_sb = o_sb; so.o_sh = o_sh; so.o_sl = o_sl;
    } else
        INFLLM_REQUIRE(local->d_o_part && local->d_lse_part, "attn_window: splits without partial rows");
    const int mode = !sinks ? kLinear : sink_angle ? kSinks : kSinksStaged;
    rc = dim == 128 ? launch_stage<128>(mode, local, sinks, stream, nullptr, so) : launch_stage<64>(mode, local, sinks, stream, nullptr, so);
    if (rc || local->nsplit == 1) return rc;
    return infllm_attn_merge2(local->d_o_part, local->d_lse_part, local->nsplit, nullptr, nullptr, 0, local->B, local->H, local->Lq, d_out, o_sb, o_sh, o_sl,
                              nullptr, stream, dim);
}
