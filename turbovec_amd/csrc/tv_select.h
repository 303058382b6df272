// Selection by counting, shared by the kernels that pick the best of a few thousand keys in a workgroup.
#pragma once
#include "tv_device.h"

namespace tv {

constexpr uint32_t kSelectBins = 1024;
constexpr uint32_t kSelectKept = 1024;     // keys left to rank by comparison

struct SelectShared {
    uint32_t bins[kSelectBins];            // all zero between uses
    uint32_t w_sum[16], w_max[16], w_min[16];
    uint32_t bin, at, above;
};

// A threshold that at least `need` and at most kSelectKept of the keys reach: counting passes into 1024
// bins between the smallest (its score word given inverted) and the largest score word, from the top; a
// bin that still holds too many is divided again.  `each(f)` calls f with every key of the calling
// thread; keys are distinct, and at least `need` of them exist.  Met by all T threads.
template <uint32_t T, typename Each>
__device__ __forceinline__ uint64_t select_threshold(const Each &each, uint32_t mx, uint32_t mn_inv, uint32_t need, SelectShared &sh) {
    constexpr uint32_t W = T / 64, kPerBin = kSelectBins / T;
    const uint32_t t = threadIdx.x, lane = t & 63u, wv = t >> 6;
    // keys lie in [low, low + 2^width): 1024 bins of 2^shift; `above` of them were counted beyond that range
    // before, and `rest` are still wanted from it
    uint64_t low = uint64_t(~mn_inv) << 32;
    uint32_t width = 32u + (mx == ~mn_inv ? 0u : 32u - uint32_t(__clz(int(mx - ~mn_inv))));
    uint32_t above = 0u, rest = need;
    for (;;) {
        const uint32_t shift = width > 10u ? width - 10u : 0u;
        each([&](uint64_t k) {
            const uint64_t d = k - low;
            if (k >= low && (width >= 64u || (d >> width) == 0ull)) atomicAdd(&sh.bins[uint32_t(d >> shift)], 1u);
        });
        __syncthreads();
        // from the top: the bin in which the count passes `rest`
        uint32_t own[kPerBin], sum = 0u;
#pragma unroll
        for (uint32_t i = 0; i < kPerBin; ++i) { own[i] = sh.bins[kSelectBins - 1u - (t * kPerBin + i)]; sum += own[i]; }
        uint32_t run = sum;
        for (int off = 1; off < 64; off <<= 1) {
            const uint32_t v = __shfl_up(run, off);
            if (lane >= uint32_t(off)) run += v;
        }
        if (lane == 63u) sh.w_sum[wv] = run;
        __syncthreads();
        uint32_t before = run - sum;
        for (uint32_t w = 0; w < W; ++w) if (w < wv) before += sh.w_sum[w];
#pragma unroll
        for (uint32_t i = 0; i < kPerBin; ++i) {
            if (before < rest && before + own[i] >= rest) {
                sh.bin = kSelectBins - 1u - (t * kPerBin + i);
                sh.above = before;
                sh.at = before + own[i];
            }
            before += own[i];
            sh.bins[kSelectBins - 1u - (t * kPerBin + i)] = 0u;
        }
        __syncthreads();
        low += uint64_t(sh.bin) << shift;
        if (above + sh.at <= kSelectKept) break;               // (a bin of width one holds one key: this ends)
        above += sh.above;
        rest -= sh.above;
        width = shift;
        __syncthreads();                                       // sh.* are read by all before they are written again
    }
    return low;
}

// A score word that at least `need` of the threads' words reach, or 1 where the threads hold fewer: the need-th largest of the
// best words of groups of threads, 64 of them or, from 17 on, 256.  For words dealt out at random few more than `need` reach it
// (k = 10 of 64 groups: 10.8; 100 of 256: 126): one pass over them and one barrier (two), where counting them into bins takes a range and two
// passes of four barriers.  Words that lie with few threads (rows laid out by score) give a low one
// or none; up to kSelectKept keys are ranked all the same, which is still the faster way (100K x 128 by rising score, 64 queries, k = 100
// 56 us a search, with more than 256 counted out 60; 2M x 128 by falling score, k = 10 83 and 94).
// `most`: the largest of the calling thread's words, 0 for none.  Met by all T threads.
constexpr uint32_t kSelectTopFew = 16;         // (of 64 groups)
struct TopShared {
    __attribute__((aligned(16))) uint32_t groups[256 + 16];      // (four words of padding after every 64: lanes that read 64 apart spread over the banks)
    uint32_t w_top[16];
};
template <uint32_t T>
__device__ __forceinline__ uint32_t select_top(uint32_t most, uint32_t need, TopShared &sh) {
    constexpr uint32_t W = T / 64;
    const uint32_t t = threadIdx.x, lane = t & 63u, wv = t >> 6;
    auto other = [](uint32_t v, auto ctrl) { return uint32_t(__builtin_amdgcn_update_dpp(0, int(v), decltype(ctrl)::value, 0xf, 0xf, false)); };
    auto reached = [&](uint32_t from, uint32_t count, uint32_t v) -> uint32_t {      // words of groups[from .. from + count) not below v
        uint32_t n = 0u;
        for (uint32_t g = from; g < from + count; g += 4u) {
            const uint4 x = *reinterpret_cast<const uint4 *>(&sh.groups[g + (g >> 6) * 4u]);
            n += (x.x >= v ? 1u : 0u) + (x.y >= v ? 1u : 0u) + (x.z >= v ? 1u : 0u) + (x.w >= v ? 1u : 0u);
        }
        return n;
    };
    const bool few = need <= kSelectTopFew;
    // (groups of T / 64 lanes, or of T / 256)
    if (few || T >= 512) most = max(most, other(most, IntC<0xB1>{}));       // quad_perm [1,0,3,2]
    if (few || T >= 1024) most = max(most, other(most, IntC<0x4E>{}));      // quad_perm [2,3,0,1]
    if (few && T >= 512) most = max(most, other(most, IntC<0x141>{}));      // row_half_mirror
    if (few && T >= 1024) most = max(most, other(most, IntC<0x140>{}));     // row_mirror
    const uint32_t per = few ? T / 64u : T / 256u, g = t / per;
    if (t % per == 0u) sh.groups[g + (g >> 6) * 4u] = most;
    __syncthreads();
    if (few) {      // every wave for itself
        const uint32_t v = sh.groups[lane], top = wave_umax(v != 0u && reached(0u, 64u, v) >= need ? v : 0u);
        return max(top, 1u);
    }
    constexpr uint32_t kWords = 256u / W, kLanes = 64u / kWords;              // words of a wave, lanes to a word
    const uint32_t mine = wv * kWords + lane / kLanes, v = sh.groups[mine + (mine >> 6) * 4u];
    uint32_t n = reached(lane % kLanes * (256u / kLanes), 256u / kLanes, v);
    if (kLanes >= 2u) n += other(n, IntC<0xB1>{});
    if (kLanes >= 4u) n += other(n, IntC<0x4E>{});
    const uint32_t top = wave_umax(v != 0u && n >= need ? v : 0u);
    if (lane == 0u) sh.w_top[wv] = top;
    __syncthreads();
    uint32_t all = 1u;
    for (uint32_t w = 0; w < W; ++w) all = max(all, sh.w_top[w]);
    return all;
}

// Largest score word and largest inverted score word over all T threads' keys.  Met by all T threads.
template <uint32_t T>
__device__ __forceinline__ void select_range(uint32_t hi_max, uint32_t hi_min_inv, SelectShared &sh, uint32_t &mx, uint32_t &mn_inv) {
    constexpr uint32_t W = T / 64;
    hi_max = wave_umax(hi_max);
    hi_min_inv = wave_umax(hi_min_inv);
    if ((threadIdx.x & 63u) == 63u) { sh.w_max[threadIdx.x >> 6] = hi_max; sh.w_min[threadIdx.x >> 6] = hi_min_inv; }
    __syncthreads();
    mx = 0u;
    mn_inv = 0u;
    for (uint32_t w = 0; w < W; ++w) { mx = max(mx, sh.w_max[w]); mn_inv = max(mn_inv, sh.w_min[w]); }
}

// Keys greater than k among kept[0 .. n), which is followed by two zero keys (read in pairs).
__device__ __forceinline__ uint32_t rank_in(const uint64_t *kept, uint32_t n, uint64_t k) {
    uint32_t rank = 0u;
    for (uint32_t j = 0; j < n; j += 2u) {
        const ulonglong2 o = *reinterpret_cast<const ulonglong2 *>(&kept[j]);
        rank += (o.x > k ? 1u : 0u) + (o.y > k ? 1u : 0u);
    }
    return rank;
}

// The keys whose score words reach `least`, which at least `need` of all keys do or which no key is below, into kept, two zeros behind
// them: how many.  Where they are too many for it, a threshold is counted out.  n_kept is 0, and its writing has been seen or is seen
// behind a barrier that comes between; met by all T threads.  count: there are too many for it.
template <uint32_t T, typename Each>
__device__ __forceinline__ uint32_t keep_best(const Each &each, uint32_t least, uint32_t need, uint64_t *kept, uint32_t &n_kept, SelectShared &sh,
                                              bool count = false) {
    const uint32_t t = threadIdx.x;
    uint32_t n = kSelectKept + 1u;
    if (!count) {
        each([&](uint64_t k) {
            if (uint32_t(k >> 32) < least) return;
            const uint32_t at = atomicAdd(&n_kept, 1u);
            if (at < kSelectKept) kept[at] = k;
        });
        __syncthreads();
        n = n_kept;
    }
    if (n > kSelectKept) {
        for (uint32_t i = t; i < kSelectBins; i += T) sh.bins[i] = 0u;
        uint32_t hi_max = 0u, hi_min_inv = 0u, mx, mn_inv;
        each([&](uint64_t k) {
            hi_max = max(hi_max, uint32_t(k >> 32));
            hi_min_inv = max(hi_min_inv, ~uint32_t(k >> 32));
        });
        select_range<T>(hi_max, hi_min_inv, sh, mx, mn_inv);       // (everyone has read n_kept)
        const uint64_t threshold = select_threshold<T>(each, mx, mn_inv, need, sh);
        if (t == 0) n_kept = 0u;
        __syncthreads();
        each([&](uint64_t k) {
            if (k >= threshold) kept[atomicAdd(&n_kept, 1u)] = k;
        });
        __syncthreads();
        n = n_kept;
    }
    if (t < 2u) kept[n + t] = 0ull;
    __syncthreads();
    return n;
}

}  // namespace tv
