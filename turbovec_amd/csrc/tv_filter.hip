// Filtered searches on the allowed rows alone: the rows a mask allows are gathered, in their order, into dense blocks
// of the native layout, and the search runs over those as over any index.  A mask of rows picked at random leaves hardly any
// block of 32 without one (1 %: 28 % of the blocks; 10 %: 97 %), and a scan pays for whole blocks: matrix tiles for
// rows it may not return.  Results are the same bits: a row's score depends on its own codes alone, and the
// order of rows, which decides ties, is kept.
#include <algorithm>

#include "tv_device.h"
#include "tv_internal.h"

namespace tv {

constexpr int kMaskThreads = 256;
constexpr uint32_t kMaskWords = 512;       // mask words (of 64 rows) one workgroup counts: two to a thread

__device__ __forceinline__ uint64_t mask_word(const uint64_t *mask, uint32_t w, uint32_t n_words, uint32_t n) {
    if (w >= n_words) return 0ull;
    const uint64_t x = mask[w];
    const uint32_t left = n - w * 64u;      // (bits at or past n do not count)
    return left < 64u ? x & ((1ull << left) - 1ull) : x;
}
__device__ __forceinline__ uint32_t wave_sum(uint32_t v) {
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) v += __shfl_xor(v, d);
    return v;
}

// Per workgroup: allowed rows, blocks with one.  1.25 MB for 10M rows: as long as a launch.
__global__ __launch_bounds__(kMaskThreads) void k_mask_count(const uint64_t *mask, uint32_t n, uint32_t n_words, uint2 *counts) {
    __shared__ uint2 part[kMaskThreads / 64];
    uint32_t rows = 0, live = 0;
#pragma unroll
    for (uint32_t u = 0; u < kMaskWords / kMaskThreads; ++u) {
        const uint64_t x = mask_word(mask, blockIdx.x * kMaskWords + u * kMaskThreads + threadIdx.x, n_words, n);
        rows += uint32_t(__popcll(x));
        live += (uint32_t(x) != 0u) + (uint32_t(x >> 32) != 0u);
    }
    rows = wave_sum(rows);
    live = wave_sum(live);
    if ((threadIdx.x & 63u) == 0u) part[threadIdx.x >> 6] = make_uint2(rows, live);
    __syncthreads();
    if (threadIdx.x != 0u) return;
    uint2 s = part[0];
    for (int w = 1; w < kMaskThreads / 64; ++w) { s.x += part[w].x; s.y += part[w].y; }
    counts[blockIdx.x] = s;
}

// The allowed rows in order, at most `room` of them; the last workgroup leaves both totals in `totals`.  A wave writes a word's rows
// at once, a lane to a bit (a thread writing its own words' rows one after the other: 40 us more where whole words are allowed).
__global__ __launch_bounds__(kMaskThreads) void k_mask_slots(const uint64_t *mask, uint32_t n, uint32_t n_words, const uint2 *counts,
                                                             uint32_t *slots, uint32_t room, uint32_t *totals) {
    __shared__ uint2 part[kMaskThreads / 64];
    const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
    uint2 before = make_uint2(0u, 0u);
    for (uint32_t i = t; i < blockIdx.x; i += kMaskThreads) { before.x += counts[i].x; before.y += counts[i].y; }
    before.x = wave_sum(before.x);
    before.y = wave_sum(before.y);
    if (lane == 0u) part[wave] = before;
    __syncthreads();
    uint32_t at = 0, live = 0;
    for (int w = 0; w < kMaskThreads / 64; ++w) { at += part[w].x; live += part[w].y; }
    __syncthreads();
    if (blockIdx.x == gridDim.x - 1u && t == 0u) {
        totals[0] = at + counts[blockIdx.x].x;
        totals[1] = live + counts[blockIdx.x].y;
        __threadfence_system();      // (the host looks for the third word)
        *static_cast<volatile uint32_t *>(totals + 2) = 1u;
    }
    // a thread's words are neighbours: one running position over them
    constexpr uint32_t kPer = kMaskWords / kMaskThreads;
    uint64_t x[kPer];
    uint32_t mine = 0;
#pragma unroll
    for (uint32_t u = 0; u < kPer; ++u) {
        x[u] = mask_word(mask, blockIdx.x * kMaskWords + t * kPer + u, n_words, n);
        mine += uint32_t(__popcll(x[u]));
    }
    uint32_t upto = mine;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t o = __shfl_up(upto, d);
        if (int(lane) >= d) upto += o;
    }
    if (lane == 63u) part[wave].x = upto;
    __syncthreads();
    at += upto - mine;
    for (uint32_t w = 0; w < wave; ++w) at += part[w].x;
    for (uint32_t l = 0; l < 64u; ++l) {
        uint32_t from = __builtin_amdgcn_readlane(at, l);
#pragma unroll
        for (uint32_t u = 0; u < kPer; ++u) {
            const uint32_t lo = __builtin_amdgcn_readlane(uint32_t(x[u]), l), hi = __builtin_amdgcn_readlane(uint32_t(x[u] >> 32), l);
            const uint64_t word = uint64_t(hi) << 32 | lo;
            const uint32_t to = from + __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, 0u));
            if ((word >> lane & 1ull) && to < room) slots[to] = (blockIdx.x * kMaskWords + (t - lane + l) * kPer + u) * 64u + lane;
            from += uint32_t(__popcll(word));
        }
    }
}

// One wave per gathered block and run of up to eight chunks, all of them on their way at once: a lane brings the 16
// bytes a chunk holds of one row's half, so a line of 128 bytes is read whole for the one to eight rows of it that are
// allowed.  Bound by HBM: the lines with an allowed row once, the gathered rows written.
constexpr int kGatherRun = 8;
__global__ __launch_bounds__(256) void k_gather_rows(const uint4 *codes, const float *scales, uint32_t nch, uint32_t runs, uint32_t run, const uint32_t *slots,
                                                     uint32_t n, uint32_t n_blocks, uint4 *out, float *out_scales) {
    const uint32_t lane = threadIdx.x & 63u, unit = blockIdx.x * 4u + (threadIdx.x >> 6);
    const uint32_t b = unit / runs, c0 = unit % runs * run;
    if (b >= n_blocks) return;
    const uint32_t row = b * 32u + (lane & 31u), m = min(run, nch - c0);
    const bool real = row < n;
    const uint32_t slot = real ? slots[row] : 0u;
    const uint4 *from = codes + (size_t(slot >> 5) * nch + c0) * 64 + (lane >> 5) * 32 + (slot & 31u);
    uint4 *to = out + (size_t(b) * nch + c0) * 64 + lane;
    uint4 v[kGatherRun];
#pragma unroll
    for (int u = 0; u < kGatherRun; ++u) v[u] = real && uint32_t(u) < m ? from[u * 64] : make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
    for (int u = 0; u < kGatherRun; ++u)
        if (uint32_t(u) < m) to[u * 64] = v[u];
    if (c0 == 0u && lane < 32u) out_scales[row] = real ? scales[slot] : 0.0f;
}

// A scan of rows in place addresses a block's rows with 32 bits from the first one's block.
__global__ __launch_bounds__(256) void k_rows_apart(const uint32_t *slots, uint32_t n, uint32_t block_bytes, uint32_t *far) {
    const uint32_t i = (blockIdx.x * 256u + threadIdx.x) * 32u;
    if (i >= n) return;
    const uint32_t a = slots[i] >> 5, b = slots[min(i + 31u, n - 1u)] >> 5;
    if (uint64_t(b - a + 1u) * block_bytes > 0xffffffffull) *far = 1u;
}

// Results of the exact path name gathered rows: back to the index's own.  (What is no row, a place beyond the last one with a score, stays.)
__global__ __launch_bounds__(256) void k_map_slots(int64_t *idx, size_t count, const uint32_t *slots, uint32_t n) {
    const size_t i = size_t(blockIdx.x) * 256 + threadIdx.x;
    if (i >= count) return;
    const int64_t v = idx[i];
    if (v >= 0 && v < int64_t(n)) idx[i] = int64_t(slots[v]);
}

size_t mask_counts(size_t n) { return ((n + 63) / 64 + kMaskWords - 1) / kMaskWords; }

hipError_t launch_mask_slots(const uint64_t *mask, size_t n, uint32_t *counts, uint32_t *slots, size_t room, uint32_t *totals, hipStream_t s) {
    if (n == 0 || n >= (size_t(1) << 31) || room > n) return hipErrorInvalidValue;
    const unsigned grid = unsigned(mask_counts(n));
    const uint32_t n_words = uint32_t((n + 63) / 64);
    hipLaunchKernelGGL(k_mask_count, dim3(grid), dim3(kMaskThreads), 0, s, mask, uint32_t(n), n_words, reinterpret_cast<uint2 *>(counts));
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_mask_slots, dim3(grid), dim3(kMaskThreads), 0, s, mask, uint32_t(n), n_words, reinterpret_cast<const uint2 *>(counts), slots,
                       uint32_t(room), totals);
    return hipGetLastError();
}

hipError_t launch_gather_rows(const uint8_t *codes, const float *scales, int nch, const uint32_t *slots, size_t n, uint8_t *out, float *out_scales, hipStream_t s) {
    const size_t n_blocks = (n + kVecBlock - 1) / kVecBlock, runs = size_t(nch + kGatherRun - 1) / kGatherRun, run = (size_t(nch) + runs - 1) / runs;
    if (n == 0 || nch <= 0 || (n_blocks * runs + 3) / 4 > 0x7fffffffull) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_gather_rows, dim3(unsigned((n_blocks * runs + 3) / 4)), dim3(256), 0, s, reinterpret_cast<const uint4 *>(codes), scales, uint32_t(nch),
                       uint32_t(runs), uint32_t(run), slots, uint32_t(n), uint32_t(n_blocks), reinterpret_cast<uint4 *>(out), out_scales);
    return hipGetLastError();
}

hipError_t launch_rows_apart(const uint32_t *slots, size_t n, size_t block_bytes, uint32_t *far, hipStream_t s) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_rows_apart, dim3(unsigned((n + 8191) / 8192)), dim3(256), 0, s, slots, uint32_t(n), uint32_t(block_bytes), far);
    return hipGetLastError();
}

hipError_t launch_map_slots(int64_t *idx, size_t count, const uint32_t *slots, size_t n, hipStream_t s) {
    if (count == 0) return hipSuccess;
    hipLaunchKernelGGL(k_map_slots, dim3(unsigned((count + 255) / 256)), dim3(256), 0, s, idx, count, slots, uint32_t(n));
    return hipGetLastError();
}

}  // namespace tv
