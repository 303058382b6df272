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
constexpr uint32_t kMaskWaves = kMaskThreads / 64;
constexpr uint32_t kMaskWords = 128;       // mask words (of 64 rows) in a piece: counted by a wave, its rows listed by a workgroup

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

// Per piece: allowed rows, blocks with one.  1.25 MB for 10M rows: as long as a launch.  A host that waits for the sums finds each
// workgroup's in a word of its own in host memory.
__global__ __launch_bounds__(kMaskThreads) void k_mask_count(const uint64_t *mask, uint32_t n, uint32_t n_words, uint32_t pieces, uint2 *counts, uint64_t *totals) {
    __shared__ uint64_t part[kMaskWaves];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    uint64_t all = 0;
    for (uint32_t piece = blockIdx.x * kMaskWaves + wave; piece < pieces; piece += gridDim.x * kMaskWaves) {
        uint32_t rows = 0, live = 0;
#pragma unroll
        for (uint32_t u = 0; u < kMaskWords / 64u; ++u) {
            const uint64_t x = mask_word(mask, piece * kMaskWords + u * 64u + lane, n_words, n);
            rows += uint32_t(__popcll(x));
            live += (uint32_t(x) != 0u) + (uint32_t(x >> 32) != 0u);
        }
        rows = wave_sum(rows);
        live = wave_sum(live);
        if (lane == 0u) counts[piece] = make_uint2(rows, live);
        all += mask_total(rows, live);
    }
    if (totals == nullptr) return;
    if (lane == 0u) part[wave] = all;
    __syncthreads();
    if (threadIdx.x != 0u) return;
    for (uint32_t w = 1; w < kMaskWaves; ++w) all += part[w];
    __hip_atomic_store(totals + blockIdx.x, all | kMaskCounted, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The allowed rows in order, at most `room` of them, a workgroup to a piece.  A wave writes a word's rows at once, a lane to a bit (a
// thread writing its own words' rows one after the other: 40 us more where whole words are allowed), and takes every
// fourth word: with both kernels on pieces of 512 words, 64 steps of two words to a wave, and the sums by the second one,
// a search of 1 % of 1M x 768, 300 queries, took 73 us, now 69; one that counts and then reads the mask (100K x 1536, 300 queries, a
// range of 20 %) 101, now 96.
__global__ __launch_bounds__(kMaskThreads) void k_mask_slots(const uint64_t *mask, uint32_t n, uint32_t n_words, const uint2 *counts,
                                                             uint32_t *slots, uint32_t room) {
    __shared__ uint32_t part[kMaskWaves], ends[kMaskWords / 64u], place[kMaskWords];
    __shared__ uint64_t word[kMaskWords];
    const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
    uint32_t before = 0;
    for (uint32_t i = t; i < blockIdx.x; i += kMaskThreads) before += counts[i].x;
    before = wave_sum(before);
    if (lane == 0u) part[wave] = before;
    if (t < kMaskWords) {      // (whole waves)
        const uint64_t x = mask_word(mask, blockIdx.x * kMaskWords + t, n_words, n);
        const uint32_t mine = uint32_t(__popcll(x));
        uint32_t upto = mine;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t o = __shfl_up(upto, d);
            if (int(lane) >= d) upto += o;
        }
        word[t] = x;
        place[t] = upto - mine;
        if (lane == 63u) ends[wave] = upto;
    }
    __syncthreads();
    uint32_t at = 0;
    for (uint32_t w = 0; w < kMaskWaves; ++w) at += part[w];
#pragma unroll 4
    for (uint32_t i = wave; i < kMaskWords; i += kMaskWaves) {
        const uint64_t x = word[i];
        uint32_t to = at + place[i] + __builtin_amdgcn_mbcnt_hi(uint32_t(x >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(x), 0u));
        for (uint32_t w = 0; w < i / 64u; ++w) to += ends[w];
        if ((x >> lane & 1ull) && to < room) slots[to] = (blockIdx.x * kMaskWords + i) * 64u + lane;
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
size_t mask_totals(size_t n) { return std::min((mask_counts(n) + kMaskWaves - 1) / kMaskWaves, kMaxMaskTotals); }

hipError_t launch_mask_count(const uint64_t *mask, size_t n, uint32_t *counts, uint64_t *totals, hipStream_t s) {
    if (n == 0 || n >= (size_t(1) << 31)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_mask_count, dim3(unsigned(mask_totals(n))), dim3(kMaskThreads), 0, s, mask, uint32_t(n), uint32_t((n + 63) / 64),
                       uint32_t(mask_counts(n)), reinterpret_cast<uint2 *>(counts), totals);
    return hipGetLastError();
}

hipError_t launch_mask_slots(const uint64_t *mask, size_t n, const uint32_t *counts, uint32_t *slots, size_t room, hipStream_t s) {
    if (n == 0 || n >= (size_t(1) << 31) || room > n) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_mask_slots, dim3(unsigned(mask_counts(n))), dim3(kMaskThreads), 0, s, mask, uint32_t(n), uint32_t((n + 63) / 64),
                       reinterpret_cast<const uint2 *>(counts), slots, uint32_t(room));
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
