// Top-k over the logits of the tied LM head: rlx_cpu::lm_head::gguf_tied_lm_topk (rlx-cpu/src/lm_head.rs:172-198) and
// topk_from_scores (:130-141) keep the `cap` largest (token, logit) pairs, largest first. The reference visits the
// rows one after another against a rising floor; here the decode kernel writes all logits and a selection over
// (value, row) keys follows. Keys order as in the argmax: larger value first, among equal values the smaller row; a NaN
// logit is no candidate; every key is unique, so "the cap-th largest" is one key.
//
// Few winners are taken one by one, many through a threshold found by bisection over the bits of the key, a count per step,
// after which every survivor counts the keys above its own:
//   rlx_topk_serial  one wave per 1024 candidates, sixteen per lane, sorted once per lane; cap rounds of a wave-wide maximum of the
//                    lanes' heads, the lane that held the winner moves its list up. Writes its cap winners as keys or, as
//                    the only wave, the answer. No LDS, no barrier.
//   rlx_topk_select  one wave per 1024 candidates, sixteen per lane, leaves their `cap` best in any order.
//   rlx_topk_finish  one workgroup, up to 8192 candidates, eight per thread: writes rows and values, largest first.
// All are bound by latency (launch, one load, the chain of rounds or counts), not by bandwidth: 128256 logits are 0.5 MB. The whole
// LM-head call at [128256, 4096] Q4_K, cap 40: 63 us, about 53 of it the matmul. Where the lines between them lie: host/ops.cpp.
#include "common.h"

namespace rlx {

constexpr int TOPK_PER_LANE = 16, TOPK_GROUP = 64 * TOPK_PER_LANE;       // candidates per wave of rlx_topk_serial / rlx_topk_select
constexpr int TOPK_PER_THREAD = 8, TOPK_FINISH = 1024 * TOPK_PER_THREAD;  // candidates rlx_topk_finish takes
constexpr int TOPK_SURVIVORS = 128;                                       // keys it puts in order (cap <= 64)
constexpr int TOPK_FEW = 256;                                             // keys rlx_topk_select counts four per lane

__device__ __forceinline__ unsigned long long topk_key_of(float v, uint32_t row) {
    const uint32_t b = __builtin_bit_cast(uint32_t, v + 0.0f);  // -0 and +0 compare equal
    const uint32_t ordered = (b & 0x80000000u) ? ~b : (b | 0x80000000u);
    return ((unsigned long long)ordered << 32) | (uint32_t)~row;
}

// Reduction over the 64 lanes, returned in a scalar register: four DPP steps leave every row of 16 lanes with its result,
// four lane reads and three scalar operations finish it.
template <typename Op>
__device__ __forceinline__ uint32_t wave_reduce_u32(uint32_t v, Op op) {
    v = op(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, true));   // quad_perm [1,0,3,2]
    v = op(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xF, 0xF, true));   // quad_perm [2,3,0,1]
    v = op(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xF, 0xF, true));  // row_half_mirror
    v = op(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x140, 0xF, 0xF, true));  // row_mirror
    const uint32_t r0 = (uint32_t)__builtin_amdgcn_readlane((int)v, 0), r1 = (uint32_t)__builtin_amdgcn_readlane((int)v, 16);
    const uint32_t r2 = (uint32_t)__builtin_amdgcn_readlane((int)v, 32), r3 = (uint32_t)__builtin_amdgcn_readlane((int)v, 48);
    return op(op(r0, r1), op(r2, r3));
}
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
    return wave_reduce_u32(v, [](uint32_t x, uint32_t y) { return max(x, y); });
}
__device__ __forceinline__ uint32_t wave_min_u32(uint32_t v) {
    return wave_reduce_u32(v, [](uint32_t x, uint32_t y) { return min(x, y); });
}

struct TopkArgs {
    const float *vals;                  // first pass: [n] logits; null afterwards
    const unsigned long long *keys_in;  // later passes: [n] keys, zero = no candidate
    int n;                              // candidates in all; wave g of rlx_topk_serial / _select takes [g * TOPK_GROUP, (g + 1) * TOPK_GROUP)
    int cap;
    unsigned long long *keys_out;       // rlx_topk_select and all but a last rlx_topk_serial: [waves][cap] keys
    uint32_t *out_idx;                  // last launch: [cap] rows and values; (0, -inf) where no candidate is left
    float *out_val;
};

// N candidates per lane, `stride` apart from `first` on. All loads are issued before the first one is used: behind a branch each they
// were N latencies one after the other, and logits that other XCDs have just written are 0.5 us away (6 of the 12 us of a
// rlx_topk_select).
template <int N>
__device__ __forceinline__ void topk_load(const TopkArgs &a, long long first, int stride, unsigned long long (&key)[N]) {
    const long long last = a.n - 1;
    if (a.vals) {
        float v[N];
#pragma unroll
        for (int e = 0; e < N; e++) v[e] = a.vals[min(first + (long long)e * stride, last)];
#pragma unroll
        for (int e = 0; e < N; e++) {
            const long long i = first + (long long)e * stride;
            key[e] = i <= last && v[e] == v[e] ? topk_key_of(v[e], (uint32_t)i) : 0;
        }
    } else {
#pragma unroll
        for (int e = 0; e < N; e++) key[e] = a.keys_in[min(first + (long long)e * stride, last)];
#pragma unroll
        for (int e = 0; e < N; e++) key[e] = first + (long long)e * stride <= last ? key[e] : 0;
    }
}

}  // namespace rlx

extern "C" __global__ __launch_bounds__(64) void rlx_topk_serial(rlx::TopkArgs a) {
    using namespace rlx;
    const int lane = threadIdx.x;
    const long long base = (long long)blockIdx.x * TOPK_GROUP;
    unsigned long long mine[TOPK_PER_LANE];
    topk_load(a, base + lane, 64, mine);
    // this lane's candidates in descending order (bitonic network over registers: every index is a constant)
#pragma unroll
    for (int k = 2; k <= TOPK_PER_LANE; k <<= 1)
#pragma unroll
        for (int j = k >> 1; j > 0; j >>= 1)
#pragma unroll
            for (int i = 0; i < TOPK_PER_LANE; i++) {
                const int l = i ^ j;
                if (l > i) {
                    const unsigned long long x = mine[i], y = mine[l];
                    const bool desc = (i & k) == 0;  // descending runs first, so the last merge leaves the whole list descending
                    const bool swap = desc ? (x < y) : (x > y);
                    mine[i] = swap ? y : x;
                    mine[l] = swap ? x : y;
                }
            }
    for (int r = 0; r < a.cap; r++) {
        const uint32_t hi = (uint32_t)(mine[0] >> 32), lo = (uint32_t)mine[0];
        const uint32_t whi = wave_max_u32(hi);
        const uint32_t wlo = wave_max_u32(hi == whi ? lo : 0u);  // keys are unique (they carry the row): one lane matches both
        const unsigned long long win = ((unsigned long long)whi << 32) | wlo;
        if (win != 0 && mine[0] == win) {  // the lane that held the winner moves its list up
#pragma unroll
            for (int e = 0; e + 1 < TOPK_PER_LANE; e++) mine[e] = mine[e + 1];
            mine[TOPK_PER_LANE - 1] = 0;
        }
        if (lane == 0) {
            if (a.keys_out) {
                a.keys_out[(long long)blockIdx.x * a.cap + r] = win;
            } else {
                const uint32_t ordered = (uint32_t)(win >> 32);
                const uint32_t b = (ordered & 0x80000000u) ? (ordered & 0x7FFFFFFFu) : ~ordered;
                a.out_idx[r] = win ? ~(uint32_t)win : 0u;
                a.out_val[r] = win ? __builtin_bit_cast(float, b) : -__builtin_inff();
            }
        }
    }
}

// The bound comes first: the cap-th largest of the 64 lanes' own maxima, one ballot a step. At least cap keys reach it, and few more do
// (about 62 of 1024 at cap 40 where the values lie in no particular order, exactly 40 where they rise or fall), so the search for the
// cap-th largest key counts four keys per lane instead of sixteen: the whole LM-head call at [128256, 4096] Q4_K, cap 40, 67.1 -> 63.2 us
// with loads that do not wait for each other. Where more than 256 survive (many equal values, or the best ones in fewer lanes than
// cap: every 64th value belongs to a lane) it counts all sixteen.
extern "C" __global__ __launch_bounds__(64) void rlx_topk_select(rlx::TopkArgs a) {
    using namespace rlx;
    __shared__ unsigned long long few[TOPK_FEW];
    const int lane = threadIdx.x;
    const long long base = (long long)blockIdx.x * TOPK_GROUP;
    unsigned long long mine[TOPK_PER_LANE];
    topk_load(a, base + lane, 64, mine);
    uint32_t best = 0;
#pragma unroll
    for (int e = 0; e < TOPK_PER_LANE; e++) best = max(best, (uint32_t)(mine[e] >> 32));
    const uint32_t top = wave_max_u32(best), low = wave_min_u32(best);
    uint32_t bound = low;  // all 64 >= cap maxima reach it
    if (top != low) {
        const int open = 32 - __builtin_clz(top ^ low);  // undecided low bits
        bound = open < 32 ? top >> open << open : 0u;
        for (int bit = open - 1; bit >= 0; bit--) {
            const uint32_t trial = bound | (1u << bit);
            if (__builtin_popcountll(__ballot(best >= trial)) >= a.cap) bound = trial;
        }
    }
    if (bound == 0) bound = 1;  // fewer than cap lanes have a candidate, an absent one is key 0
    unsigned long long t = (unsigned long long)bound << 32;  // keys >= t are taken in the end
    int count = 0;
#pragma unroll
    for (int e = 0; e < TOPK_PER_LANE; e++) count += __builtin_popcountll(__ballot(mine[e] >= t));
    auto write = [&](auto &keys) {
        int at = 0;
#pragma unroll
        for (unsigned e = 0; e < sizeof(keys) / 8; e++) {
            const bool take = keys[e] >= t;
            const unsigned long long who = __ballot(take);
            const int pos = at + __builtin_popcountll(who & ((1ull << lane) - 1ull));
            if (take) a.keys_out[(long long)blockIdx.x * a.cap + pos] = keys[e];
            at += __builtin_popcountll(who);
        }
        if (at + lane < a.cap) a.keys_out[(long long)blockIdx.x * a.cap + at + lane] = 0;
    };
    // t: the largest value with at least cap keys >= t, a bit a step
    auto search = [&](auto &keys) {
        const int bits = top == bound ? 32 : 64 - __builtin_clz(top ^ bound);  // undecided low bits of t
        t = bits < 64 ? (unsigned long long)top << 32 >> bits << bits : 0;
        for (int bit = bits - 1; bit >= 0; bit--) {
            const unsigned long long trial = t | (1ull << bit);
            int c = 0;
#pragma unroll
            for (unsigned e = 0; e < sizeof(keys) / 8; e++) c += __builtin_popcountll(__ballot(keys[e] >= trial));
            if (c >= a.cap) t = trial;
            if (c == a.cap) break;
        }
    };
    if (count <= a.cap) {
        write(mine);
    } else if (count <= TOPK_FEW) {
        int at = 0;
#pragma unroll
        for (int e = 0; e < TOPK_PER_LANE; e++) {
            const bool take = mine[e] >= t;
            const unsigned long long who = __ballot(take);
            if (take) few[at + __builtin_popcountll(who & ((1ull << lane) - 1ull))] = mine[e];
            at += __builtin_popcountll(who);
        }
        __syncthreads();
        unsigned long long kept[TOPK_FEW / 64];
#pragma unroll
        for (int e = 0; e < TOPK_FEW / 64; e++) kept[e] = lane + 64 * e < count ? few[lane + 64 * e] : 0;
        search(kept);
        write(kept);
    } else {
        search(mine);
        write(mine);
    }
}

extern "C" __global__ __launch_bounds__(1024) void rlx_topk_finish(rlx::TopkArgs a) {
    using namespace rlx;
    __shared__ uint32_t wave_hi[16], wave_lo[16];
    __shared__ uint32_t counts[2][3][16];                      // [step parity][trial][wave]
    __shared__ unsigned long long survivors[TOPK_SURVIVORS];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    unsigned long long mine[TOPK_PER_THREAD];
    topk_load(a, tid, 1024, mine);
    uint32_t best = 0;
#pragma unroll
    for (int e = 0; e < TOPK_PER_THREAD; e++) best = max(best, (uint32_t)(mine[e] >> 32));
    if (tid < TOPK_SURVIVORS) survivors[tid] = 0;
    // As above, with the maxima of the 64 rows of 16 lanes: every one of them is a key, so 64 >= cap keys reach the smallest.
    uint32_t rowbest = best;
    rowbest = max(rowbest, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)rowbest, 0xB1, 0xF, 0xF, true));
    rowbest = max(rowbest, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)rowbest, 0x4E, 0xF, 0xF, true));
    rowbest = max(rowbest, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)rowbest, 0x141, 0xF, 0xF, true));
    rowbest = max(rowbest, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)rowbest, 0x140, 0xF, 0xF, true));
    const uint32_t wtop = wave_max_u32(best), wlow = wave_min_u32(rowbest);
    if (lane == 0) {
        wave_hi[wave] = wtop;
        wave_lo[wave] = wlow;
    }
    __syncthreads();
    const uint32_t top = wave_max_u32(wave_hi[lane & 15]), low = wave_min_u32(wave_lo[lane & 15]);
    // t: at least cap keys are >= t; two bits a step, until no more than TOPK_SURVIVORS keys are left. Keys are unique,
    // so the end of the bits is the end of the search at the latest.
    int bits = top == low ? 32 : 64 - __builtin_clz(top ^ low);  // undecided low bits of t
    bits = (bits + 1) & ~1;
    unsigned long long t = bits >= 64 ? 0 : (unsigned long long)top << 32 >> bits << bits;
    bool done = false;
    for (int step = 0; bits > 0 && !done; step++) {
        bits -= 2;
#pragma unroll
        for (int q = 1; q <= 3; q++) {
            const unsigned long long trial = t | ((unsigned long long)q << bits);
            int c = 0;
#pragma unroll
            for (int e = 0; e < TOPK_PER_THREAD; e++) c += __builtin_popcountll(__ballot(mine[e] >= trial));
            if (lane == 0) counts[step & 1][q - 1][wave] = (uint32_t)c;
        }
        __syncthreads();  // the other parity is written next: a wave still reading this one is not overtaken
        const unsigned long long t0 = t;
#pragma unroll
        for (int q = 1; q <= 3; q++) {  // counts fall with q
            const uint32_t c = wave_reduce_u32(lane < 16 ? counts[step & 1][q - 1][lane] : 0u, [](uint32_t x, uint32_t y) { return x + y; });
            if (c >= (uint32_t)a.cap) {
                t = t0 | ((unsigned long long)q << bits);
                done = c <= (uint32_t)TOPK_SURVIVORS;
            }
        }
    }
    if (t == 0) t = 1;
    // survivors, in any order: every wave counts its own, takes its place among the waves, writes
    int c = 0;
#pragma unroll
    for (int e = 0; e < TOPK_PER_THREAD; e++) c += __builtin_popcountll(__ballot(mine[e] >= t));
    __syncthreads();
    if (lane == 0) wave_hi[wave] = (uint32_t)c;
    __syncthreads();
    int at = (int)wave_reduce_u32(lane < wave ? wave_hi[lane & 15] : 0u, [](uint32_t x, uint32_t y) { return x + y; });
#pragma unroll
    for (int e = 0; e < TOPK_PER_THREAD; e++) {
        const bool take = mine[e] >= t;
        const unsigned long long who = __ballot(take);
        const int pos = at + __builtin_popcountll(who & ((1ull << lane) - 1ull));
        if (take && pos < TOPK_SURVIVORS) survivors[pos] = mine[e];
        at += __builtin_popcountll(who);
    }
    __syncthreads();
    // rank = keys above; eight neighbouring threads share a survivor, sixteen comparisons each
    const unsigned long long key = survivors[tid >> 3];
    uint32_t above = 0;
#pragma unroll
    for (int i = 0; i < TOPK_SURVIVORS / 8; i++) above += survivors[i * 8 + (tid & 7)] > key ? 1u : 0u;
    above += (uint32_t)__shfl_xor((int)above, 1);
    above += (uint32_t)__shfl_xor((int)above, 2);
    above += (uint32_t)__shfl_xor((int)above, 4);
    if ((tid & 7) == 0 && key != 0 && above < (uint32_t)a.cap) {
        const uint32_t ordered = (uint32_t)(key >> 32);
        const uint32_t b = (ordered & 0x80000000u) ? (ordered & 0x7FFFFFFFu) : ~ordered;
        a.out_idx[above] = ~(uint32_t)key;
        a.out_val[above] = __builtin_bit_cast(float, b);
    }
    // fewer candidates than cap: the rest of the list
    const int total = (int)wave_reduce_u32(lane < 16 ? wave_hi[lane] : 0u, [](uint32_t x, uint32_t y) { return x + y; });
    if (tid >= total && tid < a.cap) {
        a.out_idx[tid] = 0u;
        a.out_val[tid] = -__builtin_inff();
    }
}
