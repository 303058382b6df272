// Search of a small index without sampling: one pass that keeps, per query and block of 32 rows, only the
// best allowed row's score, then one launch that finds the k best blocks of each query, scores their rows
// once more and ranks them.
//
// The k best rows lie in the k blocks whose best rows rank first: a row outside them has k rows, one per
// such block, ranked before it (score, then lower slot; blocks follow the slots, so equal best scores
// order blocks as they order rows).  So there is no floor to estimate, no candidate segment to overflow
// and nothing to repeat: three dependent launches instead of five, and a (block, query) pair costs one
// 4-byte store instead of the appends of an open first level.
#include <algorithm>

#include "tv_device.h"
#include "tv_internal.h"
#include "tv_select.h"

namespace tv {

// ===========================================================================
// Score mode P: best row per (block, query) over NT query tiles per workgroup, their weights in LDS.
// grid = (block groups, tile groups); a wave decodes a block's chunk on the vector ALU (about 60
// instructions, 240 cycles) and feeds NT tiles' MFMAs from it (64 NT cycles), so four tiles balance the
// two units.  The tiles are split over workgroups because a small index has few blocks: 100K rows are
// 3125 of them, which fill 65 of the 256 workgroups of a kernel that takes all queries through one.
// 100K x 128, 1000 queries: 31 us, the vector ALU busy in 55 % of the clocks and the matrix unit in 15 %.  Rows that
// short have two chunks, so of the 456 vector instructions per block and four tiles the decode is 120, the rest epilogue.
// Weights in plane order, or (kBestSplit) in the order of k_scan_p4, whose operands then take four byte permutes a chunk.  kBestRows: plane order,
// and every row's score instead of the block's best (ScanArgs::best_rows; an instance of its own, as two of the others would spill).
// a.b_step: every so many blocks only (the sample a floor is taken from), recorded by their place in the sample.
// ===========================================================================
enum { kBestPlane, kBestSplit, kBestRows };
constexpr int kBestThreads = 512;
constexpr int kBestWaves = kBestThreads / 64;

// ONE: rows of U chunks.  (Their first product takes the constant zero as its addend, which saves 16 moves a tile: 100K x 128, 1000 queries
// 65 us a search and 60.7, x 64 56 and 54.  A first turn of its own for longer rows spills, and so do four chunks at once or two with two tiles.)
template <int NT, int U, int FORM, bool ONE>
__global__ __launch_bounds__(kBestThreads, NT <= 2 ? 4 : 2) void k_scan_p4_best(ScanArgs a) {
    extern __shared__ __align__(16) uint8_t smem[];
    const int nch = a.nch, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, qn = lane & 31, h = lane >> 5;
    const int tile0 = int(blockIdx.y) * NT;
    const int nt = min(NT, (a.nq_tile + kQTile - 1) / kQTile - tile0);
    const uint32_t stride = gridDim.x * kBestWaves, step = a.b_step, nj = (a.n_blocks + step - 1) / step;
    const uint4 *codes = reinterpret_cast<const uint4 *>(a.codes) + lane;
    const float nan = __int_as_float(0x7fc00000);
    auto store = [&](int t, uint32_t j, uint32_t word) {
        const int q = (tile0 + t) * kQTile + qn;
        if (h == 0 && t < nt && q < a.nq_tile) a.best_out[size_t(q) * a.best_stride + j] = word;
    };
    // (a.best_rows) the scores of the lane's sixteen rows of block j, four side by side
    auto store_rows = [&](int t, uint32_t j, auto &&score) {
        const int q = (tile0 + t) * kQTile + qn;
        if (t >= nt || q >= a.nq_tile) return;
        float4 *to = reinterpret_cast<float4 *>(reinterpret_cast<float *>(a.best_out) + size_t(q) * a.best_stride + j * 32u + 4u * uint32_t(h));
#pragma unroll
        for (int r = 0; r < 16; r += 4) to[r >> 1] = float4{score(r), score(r + 1), score(r + 2), score(r + 3)};
    };
    // the next block from j on with an allowed row; the ones without are recorded on the way
    auto live_from = [&](uint32_t j) -> uint32_t {
        if (a.mask == nullptr) return j;
        for (; j < nj; j += stride) {
            const uint32_t b = j * step;
            if (uint32_t(a.mask[b >> 1] >> ((b & 1) * 32)) != 0u) break;
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                if constexpr (FORM == kBestRows) store_rows(t, j, [&](int) { return nan; });
                else store(t, j, 0u);
            }
        }
        return j;
    };
    // the wave's first codes are on their way while the workgroup sets up its LDS
    uint32_t j = live_from(blockIdx.x * kBestWaves + wave);
    uint4 buf[U];
    if (j < nj) {
#pragma unroll
        for (int u = 0; u < U; ++u) buf[u] = codes[(size_t(j) * step * nch + u) * 64];
    }
    {
        const uint4 *src = reinterpret_cast<const uint4 *>(a.tables) + size_t(tile0) * nch * 128;
        uint4 *dst = reinterpret_cast<uint4 *>(smem);
        const int n16 = nt * nch * 128;
        constexpr int kBatch = 8;
        for (int i0 = tid; i0 < n16; i0 += kBestThreads * kBatch) {
            uint4 tmp[kBatch];
#pragma unroll
            for (int u = 0; u < kBatch; ++u) tmp[u] = i0 + u * kBestThreads < n16 ? src[i0 + u * kBestThreads] : make_uint4(0, 0, 0, 0);
#pragma unroll
            for (int u = 0; u < kBatch; ++u)
                if (i0 + u * kBestThreads < n16) dst[i0 + u * kBestThreads] = tmp[u];
        }
    }
    float qs[NT], qb[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int q = (tile0 + t) * kQTile + qn;
        qs[t] = q < a.nq_tile ? a.qscale[q] : 0.0f;
        qb[t] = q < a.nq_tile ? a.qbias[q] : 0.0f;
    }
    __syncthreads();
    const uint32_t t0 = a.lv[0], t1 = a.lv[1], t2 = a.lv[2], t3 = a.lv[3];
    const v4i *w = reinterpret_cast<const v4i *>(smem) + lane;

    while (j < nj) {
        const uint32_t jn = live_from(j + stride), b = j * step;
        // row scales, NaN where a row may not be returned
        const uint32_t slot0 = b * 32u;
        uint32_t mw = a.mask != nullptr ? uint32_t(a.mask[b >> 1] >> ((b & 1) * 32)) : 0xffffffffu;
        if (slot0 + 32u > a.n) mw &= (1u << (a.n - slot0)) - 1u;
        float vs[16];
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
            const float4 f = *reinterpret_cast<const float4 *>(a.scales + slot0 + 8 * q4 + 4 * h);
            vs[q4 * 4 + 0] = f.x; vs[q4 * 4 + 1] = f.y; vs[q4 * 4 + 2] = f.z; vs[q4 * 4 + 3] = f.w;
        }
        v16i acc[NT];
        auto chunks = [&](int c0, auto first) {
            uint4 cur[U];
#pragma unroll
            for (int u = 0; u < U; ++u) cur[u] = buf[u];
            const bool more = !ONE && c0 + U < nch;
            if (more || jn < nj) {
                const uint4 *from = codes + (more ? size_t(b) * nch + c0 + U : size_t(jn) * step * nch) * 64;
#pragma unroll
                for (int u = 0; u < U; ++u) buf[u] = from[u * 64];
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const uint32_t x[4] = {cur[u].x, cur[u].y, cur[u].z, cur[u].w};
                v4i lo, hi;
#pragma unroll
                for (int d = 0; d < 4; ++d) {
                    lo[d] = int(levels_of(x[d] & 0x0f0f0f0fu, t0, t1, t2, t3));
                    hi[d] = int(levels_of((x[d] >> 4) & 0x0f0f0f0fu, t0, t1, t2, t3));
                }
                if constexpr (FORM == kBestSplit) {
                    const v4i l = lo, g = hi;
                    lo = v4i{l[0], g[0], l[1], g[1]};
                    hi = v4i{int(__builtin_amdgcn_perm(uint32_t(g[2]), uint32_t(l[2]), 0x05010400u)), int(__builtin_amdgcn_perm(uint32_t(g[2]), uint32_t(l[2]), 0x07030602u)),
                             int(__builtin_amdgcn_perm(uint32_t(g[3]), uint32_t(l[3]), 0x05010400u)), int(__builtin_amdgcn_perm(uint32_t(g[3]), uint32_t(l[3]), 0x07030602u))};
                }
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const v4i *wt = w + ((t * nch + c0 + u) * 2) * 64;
                    const v16i zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
                    acc[t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(lo, wt[0], decltype(first)::value != 0 && u == 0 ? zero : acc[t], 0, 0, 0);
                    acc[t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(hi, wt[64], acc[t], 0, 0, 0);
                }
            }
        };
        if constexpr (ONE) {
            chunks(0, IntC<1>{});
        } else {
#pragma unroll
            for (int t = 0; t < NT; ++t) acc[t] = v16i{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
            for (int c0 = 0; c0 < nch; c0 += U) chunks(c0, IntC<0>{});
        }
        // lane: query qn of each tile, rows 8 (r / 4) + 4 h + r % 4 (search.rs:1519-1524)
        if (mw != 0xffffffffu) {
#pragma unroll
            for (int r = 0; r < 16; ++r) vs[r] = ((mw >> (8 * (r >> 2) + 4 * h + (r & 3))) & 1u) ? vs[r] : nan;
        }
        if constexpr (FORM == kBestRows) {
#pragma unroll
            for (int t = 0; t < NT; ++t) store_rows(t, j, [&](int r) { return fmaf(float(acc[t][r]), qs[t], qb[t]) * vs[r]; });
            j = jn;
            continue;
        }
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            float m = -__int_as_float(0x7f800000);
#pragma unroll
            for (int r = 0; r < 16; ++r) m = fmaxf(m, fmaf(float(acc[t][r]), qs[t], qb[t]) * vs[r]);   // (NaN never wins)
            store(t, j, best_word(fmaxf(m, __shfl_xor(m, 32))));
        }
        j = jn;
    }
}

// Query tiles per workgroup: as many as the LDS holds beside another workgroup's -- four at most -- but no
// more than leave the chip with a workgroup per CU.  Three where that makes no more groups (us a search with four and three: 3 tiles
// 310K x 384 53.5 and 51.3; 5 tiles 537K x 352 110 and 94, 35K x 640 43.2 and 41.4; 9 tiles 269K x 640 133 and 116, 152K x 384 68 and 63).
static int best_tiles(int nch, size_t n_blocks, int tiles, int cus) {
    int nt = tiles == 3 || tiles == 5 || tiles == 6 || tiles == 9 ? 3 : std::min(tiles, 4);
    while (nt > 1 && size_t(nt) * nch * 2048 > 80 * 1024) nt = nt == 3 ? 2 : nt / 2;
    const size_t groups = (n_blocks + kBestWaves - 1) / kBestWaves;
    while (nt > 1 && groups * size_t((tiles + nt - 1) / nt) < size_t(cus)) nt = nt == 3 ? 2 : nt / 2;
    return nt;
}
bool best_serves(int nch) { return size_t(nch) * 2048 <= 160 * 1024; }

template <int NT, int U, int FORM, bool ONE>
static hipError_t launch_best_one(const ScanArgs &a, uint32_t nj, int device, hipStream_t s) {
    const int tiles = (a.nq_tile + kQTile - 1) / kQTile, groups_y = (tiles + NT - 1) / NT;
    const size_t lds = size_t(NT) * a.nch * 2048;
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(k_scan_p4_best<NT, U, FORM, ONE>), hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
    if (e != hipSuccess) return e;
    // A workgroup keeps its weights for all its blocks: as many workgroups as are resident, and none more, which would
    // start when the others end (us a search with 258 or 260 for 256 places and so: 194K x 560, 696 queries 241 and 173, 350K x 512, 300
    // 184 and 134, 1M x 256, 600 464 and 314; 513 for 512: 333K x 2424, 67 280 and 249, 50K x 3072, 96 106 and 91).
    const unsigned per_cu = unsigned(std::min<size_t>(NT <= 2 ? 2 : 1, 160 * 1024 / lds));
    const unsigned resident = unsigned(device_cus(device)) * std::max(1u, per_cu);
    const unsigned x = std::max(1u, std::min((nj + kBestWaves - 1) / kBestWaves, resident / unsigned(groups_y)));
    hipLaunchKernelGGL((k_scan_p4_best<NT, U, FORM, ONE>), dim3(x, groups_y), dim3(kBestThreads), lds, s, a);
    return hipGetLastError();
}
template <int NT, int U, int FORM>
static hipError_t launch_best_n(const ScanArgs &a, uint32_t nj, int device, hipStream_t s) {
    if constexpr (U <= 2 && !(U == 2 && NT == 2))
        if (a.nch == U) return launch_best_one<NT, U, FORM, true>(a, nj, device, s);
    return launch_best_one<NT, U, FORM, false>(a, nj, device, s);
}
template <int NT, int FORM>
static hipError_t launch_best_u(const ScanArgs &a, uint32_t nj, int device, hipStream_t s) {
    // (two tiles' accumulators and bursts of four chunks do not fit the 128 registers of four waves per SIMD)
    if constexpr (NT != 2) {
        if (a.nch % 4 == 0) return launch_best_n<NT, 4, FORM>(a, nj, device, s);
    }
    return a.nch % 2 == 0 ? launch_best_n<NT, 2, FORM>(a, nj, device, s) : launch_best_n<NT, 1, FORM>(a, nj, device, s);
}
// a.nq_tile = all queries of the launch, a.tables = their weight tiles, a.best_out / a.best_stride = the result.
hipError_t launch_scan_p4_best(const ScanArgs &a, bool split, int device, hipStream_t s) {
    const uint32_t nj = a.b_step ? (a.n_blocks + a.b_step - 1) / a.b_step : 0u;
    if (a.nq_tile <= 0 || nj == 0 || !best_serves(a.nch) || a.best_out == nullptr || a.best_stride / (a.best_rows ? 32u : 1u) < nj || (a.best_rows && (a.b_step != 1 || split))) return hipErrorInvalidValue;
    const int nt = best_tiles(a.nch, nj, (a.nq_tile + kQTile - 1) / kQTile, device_cus(device));
    if (nt == 1)
        if (const int parts = p4_parts(a.nch, nj, (a.nq_tile + kQTile - 1) / kQTile, device_cus(device)); parts > 1) return launch_scan_p4_parts(a, split, parts, device, s);
    auto form = [&](auto f) -> hipError_t {
        constexpr int F = decltype(f)::value;
        return nt == 1 ? launch_best_u<1, F>(a, nj, device, s) : nt == 2 ? launch_best_u<2, F>(a, nj, device, s) : nt == 3 ? launch_best_u<3, F>(a, nj, device, s) : launch_best_u<4, F>(a, nj, device, s);
    };
    return a.best_rows ? form(IntC<kBestRows>{}) : split ? form(IntC<kBestSplit>{}) : form(IntC<kBestPlane>{});
}

// ===========================================================================
// The floor a sample's best rows give: a workgroup per query takes the k_floor-th best of the sampled blocks' best
// scores, which k_floor scanned rows reach.
// ===========================================================================
constexpr uint32_t kFloorThreads = 512, kFloorHeld = kMaxFloorBlocks / kFloorThreads;
__global__ __launch_bounds__(kFloorThreads) void k_floor_of_best(const uint32_t *__restrict__ words, uint32_t stride, uint32_t n, uint32_t k_floor,
                                                        int *tau_out, int tau_stride_q, uint64_t *stamp) {
    constexpr uint32_t T = kFloorThreads;
    __shared__ __align__(16) uint64_t kept[kSelectKept + 2];
    __shared__ SelectShared sh;
    __shared__ TopShared top;
    __shared__ uint32_t n_kept;
    const uint32_t qi = blockIdx.x, t = threadIdx.x;
    const uint32_t *best = words + size_t(qi) * stride;
    uint32_t v[kFloorHeld];
#pragma unroll
    for (uint32_t e = 0; e < kFloorHeld; ++e) v[e] = e * T + t < n ? best[e * T + t] : 0u;
    if (t == 0) n_kept = 0u;
    uint32_t most = 0u;
#pragma unroll
    for (uint32_t e = 0; e < kFloorHeld; ++e) most = max(most, v[e]);
    auto each = [&](auto &&f) {
#pragma unroll
        for (uint32_t e = 0; e < kFloorHeld; ++e)
            if (v[e] != 0u) f((uint64_t(v[e]) << 32) | ~(e * T + t));
    };
    // (256 words are ranked as they are)
    if (n <= 256u) __syncthreads();
    const uint32_t n_of = keep_best<T>(each, n <= 256u ? 1u : select_top<T>(most, k_floor, top), k_floor, kept, n_kept, sh);
    int *out = tau_out + (qi / uint32_t(tau_stride_q)) * kQTile + qi % uint32_t(tau_stride_q);
    if (n_of < k_floor) {      // (a mask that leaves the sample too few rows)
        if (t == 0) *out = kTauInit;
    } else {
        for (uint32_t i = t; i < n_of; i += T)
            if (rank_in(kept, n_of, kept[i]) + 1u == k_floor) *out = int(uint32_t(kept[i] >> 32) ^ 0x80000000u);
    }
    if (t == 0 && stamp != nullptr && qi + 1u == gridDim.x) *stamp = wall_clock64();      // (among the last to end)
}
hipError_t launch_floor(const uint32_t *words, uint32_t stride, uint32_t n, int k_floor, int nq, int *tau_out, int tau_stride_q, uint64_t *stamp,
                        hipStream_t s) {
    if (nq <= 0) return hipSuccess;
    if (n > kMaxFloorBlocks || n > stride || k_floor <= 0 || k_floor > int(kSelectKept)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_floor_of_best, dim3(unsigned(nq)), dim3(kFloorThreads), 0, s, words, stride, n, uint32_t(k_floor), tau_out, tau_stride_q, stamp);
    return hipGetLastError();
}

// ===========================================================================
// A workgroup per query, or several that share its work: the k_eff best blocks (select_top, and counting where many tie), their rows scored as the
// scans score them, ranked.  All latency (k = 10, a thousand queries: 16 us over 100K x 128; at 3072 dimensions, twenty-four
// times the row, 133 over 200K, where it takes workgroups of 1024).  With the threshold from groups' best words
// instead of counted out, us a search: 100K x 128, 1 query 30.2 -> 27.9, 64 queries, k = 100 41.8 -> 40.4; and of the floors' kernel 500K x
// 768, 45 queries, k = 64 109 -> 92, 1M x 1536, 64 queries 198 -> 194.
// ===========================================================================
// A query's part of the memory that its workgroups share: how many rows each found, and each one's rows.
constexpr uint32_t kMaxShares = 8;
__host__ __device__ constexpr uint32_t pick_shared_words(uint32_t k_eff) { return kMaxShares + (k_eff + kMaxShares) * 32u; }
struct PickArgs {
    const uint32_t *best;
    uint32_t best_stride, n_blocks, n;
    const uint8_t *codes;
    const float *scales;
    const uint64_t *mask;
    const uint8_t *tables;
    const float *qscale, *qbias;
    uint32_t lv[4];
    int nch, k_eff, split;
    float *out_scores;
    int64_t *out_idx;
    const uint32_t *slots;      // when given: the slot of each row, for out_idx
    uint32_t *overflow;
    uint32_t nq, shares, parts;
    uint64_t *counts, *lists;   // shares > 1: per query the number of workgroups that are through with it, and what they found (pick_shared_words)
    uint64_t *stamp;
};
// Chunks of a query to score again (of tables: thirds), from where sharing them pays (less: 100K x 768, 64 queries, k = 10 43.3 us and, shared,
// 44.2; 100K x 512 2-bit, one query 35.1 and 36.4; 20K x 384, one query, k = 20 31.9 and 31.1).
constexpr size_t kSharedWork = 200;
// What a part of a block costs beside its chunks, and parts at all -- two barriers, the sums' way through LDS -- in chunks' time.
constexpr size_t kPartCost = 1, kPartsCost = 3;
// H: blocks a thread keeps in registers -- all of them, T * H at most.
// LUT: score mode L with the u32 epilogue.
// Scoring a block again is 70 (LUT: 200) vector instructions a chunk, on one CU for all of a query's blocks.  Where queries are too few for
// all CUs, several workgroups choose the same blocks, score their share of them and write its rows to memory;
// the one that finds itself last ranks it.  Nobody waits for another.  us a search with one workgroup each and so: 100K x 768, one query, k = 50
// 60.6 -> 43.5; 100K x 1536, 8 queries, k = 25 66.5 -> 54.5, one query, k = 10 55.4 -> 52.6; 778K x 1000 3-bit, 37 queries, k = 33 218 -> 216 (this
// kernel 37 -> 25).
// PARTS: a block's chunks in parts to several waves (launch_pick; an instance of its own, as the others lost 2 to 5 % to it).
template <uint32_t T, uint32_t H, bool LUT, bool SHARED, bool PARTS>
__global__ __launch_bounds__(T) void k_pick(PickArgs a) {
    constexpr uint32_t W = T / 64;
    extern __shared__ __align__(16) uint8_t dyn[];
    __shared__ __align__(16) uint64_t kept[kSelectKept + 2];
    __shared__ SelectShared sh;
    __shared__ TopShared top;
    __shared__ uint32_t blocks[kMaxPickK];
    __shared__ uint32_t n_kept, n_list, s_floor, s_last;
    uint64_t *list = reinterpret_cast<uint64_t *>(dyn);                     // rows of the chosen blocks that can still matter
    uint8_t *wts = dyn + size_t(a.k_eff) * 32 * 8;                          // this query's weights
    int *s_acc = reinterpret_cast<int *>(wts + size_t(a.nch) * (LUT ? 1024 : 64));     // parts > 1: sums of rows scored in parts
    const uint32_t qi = SHARED ? blockIdx.x % a.nq : blockIdx.x, share = SHARED ? blockIdx.x / a.nq : 0u, shares = SHARED ? a.shares : 1u;
    const uint32_t t = threadIdx.x, lane = t & 63u, wv = t >> 6;
    const uint32_t k_eff = uint32_t(a.k_eff);
    const uint32_t *best = a.best + size_t(qi) * a.best_stride;
    if (a.stamp != nullptr && blockIdx.x + t == 0) *a.stamp = wall_clock64();
    uint32_t v[H];
#pragma unroll
    for (uint32_t e = 0; e < H; ++e) v[e] = e * T + t < a.n_blocks ? best[e * T + t] : 0u;
    // the tile's weights lie [chunk][fragment][half * 32 + query] in 16-byte pieces; here [chunk][half][fragment]
    if constexpr (LUT) {
        // (two tables of 16 entries per byte-group, as they are)
        const uint4 *src = reinterpret_cast<const uint4 *>(a.tables) + size_t(qi) * a.nch * 64;
        for (int i = int(t); i < a.nch * 64; i += int(T)) reinterpret_cast<uint4 *>(wts)[i] = src[i];
    } else {
        const uint4 *src = reinterpret_cast<const uint4 *>(a.tables) + size_t(qi / kQTile) * a.nch * 128 + qi % kQTile;
        for (int i = int(t); i < a.nch * 4; i += int(T))
            reinterpret_cast<uint4 *>(wts)[i] = src[(i >> 2) * 128 + (i & 1) * 64 + ((i >> 1) & 1) * 32];
    }
    if (t == 0) { n_kept = 0u; n_list = 0u; s_floor = 0u; }
    uint32_t most = 0u;
#pragma unroll
    for (uint32_t e = 0; e < H; ++e) most = max(most, v[e]);
    auto each = [&](auto &&f) {
#pragma unroll
        for (uint32_t e = 0; e < H; ++e)
            if (v[e] != 0u) f((uint64_t(v[e]) << 32) | ~(e * T + t));
    };
    // (256 blocks are ranked as they are)
    if (a.n_blocks <= 256u) __syncthreads();
    uint32_t n = keep_best<T>(each, a.n_blocks <= 256u ? 1u : select_top<T>(most, k_eff, top), k_eff, kept, n_kept, sh);
    const uint32_t need = min(k_eff, n);
    for (uint32_t i = t; i < n; i += T) {
        const uint64_t k = kept[i];
        const uint32_t rank = rank_in(kept, n, k);
        if (rank < need) blocks[rank] = ~uint32_t(k);
        // k_eff blocks have a row that reaches the last one's best: nothing below it is wanted
        if (rank + 1u == k_eff) s_floor = uint32_t(k >> 32);
    }
    __syncthreads();
    // the chosen blocks' rows, a block per wave: lane = row lane % 32, sixteen code bytes of each chunk
    const uint32_t floor_word = s_floor, h = lane >> 5;
    const float qs = a.qscale[qi], qb = a.qbias[qi];
    const uint32_t t0 = a.lv[0], t1 = a.lv[1], t2 = a.lv[2], t3 = a.lv[3];
    // blocks of this workgroup's share: numbers share, share + shares, ...; parts (a power of two) of a block's chunks to as many waves
    const uint32_t mine = need > share ? (need - share + shares - 1u) / shares : 0u, log_parts = PARTS ? uint32_t(__builtin_ctz(a.parts)) : 0u;
    const uint32_t lds_w = uint32_t(reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) uint8_t *)wts));
    auto take = [&](uint32_t b, uint32_t row, int acc, float vs) {
        const uint32_t slot = b * 32u + row;
        const float s = LUT ? ((float(acc) * qs) + qb) * vs : fmaf(float(acc), qs, qb) * vs;      // search.rs:1174-1177, 1519-1524
        // (A score of -infinity does not count here either, as it does not in a block's best word: rows that tie there
        // with rows of blocks that were not chosen are for the exact path to order.)
        bool ok = slot < a.n && s > -__int_as_float(0x7f800000);
        if (ok && a.mask != nullptr) ok = (uint32_t(a.mask[b >> 1] >> ((b & 1) * 32)) >> row) & 1u;
        const uint64_t key = sort_key(s, slot);
        if (ok && uint32_t(key >> 32) >= floor_word) list[atomicAdd(&n_list, 1u)] = key;
    };
    if constexpr (PARTS) {
        for (uint32_t i = t; i < mine * 32u; i += T) s_acc[i] = 0;
        __syncthreads();
    }
    for (uint32_t it = wv; it < mine << log_parts; it += W) {
        const uint32_t at = it >> log_parts, part = PARTS ? it & (a.parts - 1u) : 0u, b = blocks[at * shares + share];
        const int first = PARTS ? int(uint32_t(a.nch) * part >> log_parts) : 0, end = PARTS ? int(uint32_t(a.nch) * (part + 1u) >> log_parts) : a.nch;
        const float vs = a.scales[b * 32u + (lane & 31u)];      // (requested ahead of the codes)
        const uint4 *src = reinterpret_cast<const uint4 *>(a.codes) + size_t(b) * a.nch * 64 + lane;
        int acc = 0;
        constexpr int kBurst = 8;
        for (int c0 = first; c0 < end; c0 += kBurst) {
            uint4 x[kBurst];
#pragma unroll
            for (int u = 0; u < kBurst; ++u) x[u] = c0 + u < end ? src[(c0 + u) * 64] : make_uint4(0, 0, 0, 0);
#pragma unroll
            for (int u = 0; u < kBurst; ++u) {
                if (c0 + u >= end) break;
                const uint32_t d[4] = {x[u].x, x[u].y, x[u].z, x[u].w};
                if constexpr (LUT) {
                    const uint32_t row = lds_w + uint32_t(((c0 + u) * 32 + int(h) * 16) * 32);
                    static_for<16>([&](auto ee) {
                        constexpr int e = decltype(ee)::value;
                        const uint32_t high = (d[e >> 2] >> 4) & 0x0f0f0f0fu, low = d[e >> 2] & 0x0f0f0f0fu;
                        acc += int(reinterpret_cast<LdsByte *>(uintptr_t(plus_byte<(e & 3)>(row, high)))[e * 32]) +
                               int(reinterpret_cast<LdsByte *>(uintptr_t(plus_byte<(e & 3)>(row, low)))[e * 32 + 16]);
                    });
                    continue;
                }
                const uint4 *wq = reinterpret_cast<const uint4 *>(wts) + ((c0 + u) * 2 + h) * 2;
                const uint4 f0 = wq[0], f1 = wq[1];
                uint32_t lo[4], hi[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    lo[e] = levels_of(d[e] & 0x0f0f0f0fu, t0, t1, t2, t3);
                    hi[e] = levels_of((d[e] >> 4) & 0x0f0f0f0fu, t0, t1, t2, t3);
                }
                const uint32_t g0[4] = {f0.x, f0.y, f0.z, f0.w}, g1[4] = {f1.x, f1.y, f1.z, f1.w};
                if (a.split) {
                    // bytes 0..7 as (low, high) dwords of four, bytes 8..15 as (low, high) byte pairs (k_scan_p4)
                    acc = __builtin_amdgcn_sdot4(int(lo[0]), int(g0[0]), acc, false);
                    acc = __builtin_amdgcn_sdot4(int(hi[0]), int(g0[1]), acc, false);
                    acc = __builtin_amdgcn_sdot4(int(lo[1]), int(g0[2]), acc, false);
                    acc = __builtin_amdgcn_sdot4(int(hi[1]), int(g0[3]), acc, false);
#pragma unroll
                    for (int e = 2; e < 4; ++e) {
                        acc = __builtin_amdgcn_sdot4(int(__builtin_amdgcn_perm(hi[e], lo[e], 0x05010400u)), int(g1[2 * e - 4]), acc, false);
                        acc = __builtin_amdgcn_sdot4(int(__builtin_amdgcn_perm(hi[e], lo[e], 0x07030602u)), int(g1[2 * e - 3]), acc, false);
                    }
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        acc = __builtin_amdgcn_sdot4(int(lo[e]), int(g0[e]), acc, false);
                        acc = __builtin_amdgcn_sdot4(int(hi[e]), int(g1[e]), acc, false);
                    }
                }
            }
        }
        acc += __shfl_xor(acc, 32);
        if (lane < 32u) {
            if constexpr (PARTS) atomicAdd(&s_acc[at * 32u + lane], acc);
            else take(b, lane, acc, vs);
        }
    }
    if constexpr (PARTS) {
        __syncthreads();
        for (uint32_t i = t; i < mine * 32u; i += T) {
            const uint32_t b = blocks[(i >> 5) * shares + share];
            take(b, i & 31u, s_acc[i], a.scales[b * 32u + (i & 31u)]);
        }
    }
    if constexpr (SHARED) {
        __syncthreads();
        const uint32_t cap = (k_eff + shares - 1u) / shares * 32u, own = n_list;
        uint64_t *area = a.lists + size_t(qi) * pick_shared_words(k_eff);
        // What is handed over goes through put and get alone: the order below rests on every word of it passing the caches on both
        // sides, which the language's memory model does not promise.  A plain store or load among them may come late or find old bytes.
        auto put = [](uint64_t *to, uint64_t v) { __hip_atomic_store(to, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
        auto get = [](uint64_t *from) { return __hip_atomic_load(from, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
        for (uint32_t i = t; i < own; i += T) put(&area[kMaxShares + share * cap + i], list[i]);
        if (t == 0) put(&area[share], own);
        // This thread's words are there before its workgroup is counted: they go past the caches, like the count and
        // like the loads below, so the stores' completion is enough (a fence writes the whole cache of the die back, and
        // with 200 workgroups of 16 waves takes 80 us).
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (t == 0) s_last = atomicAdd(reinterpret_cast<unsigned long long *>(&a.counts[qi]), 1ull) + 1ull == shares ? 1u : 0u;
        __syncthreads();
        if (s_last == 0u) return;
        uint32_t all = 0u;
        for (uint32_t o = 0; o < shares; ++o) {
            const uint32_t theirs = uint32_t(get(&area[o]));
            for (uint32_t i = t; i < theirs; i += T) list[all + i] = get(&area[kMaxShares + o * cap + i]);
            all += theirs;
        }
        if (t == 0) n_list = all;
    }
    __syncthreads();
    const uint32_t m = n_list;
    // (fewer rows with a score than wanted -- an overstated count of allowed rows, scores of NaN or -infinity: the exact
    // path takes the query)
    if (t == 0) a.overflow[qi] = m < k_eff ? 2u : 0u;
    if (m < k_eff) return;
    auto each_row = [&](auto &&f) {
        for (uint32_t i = t; i < m; i += T) f(list[i]);
    };
    if (t == 0) n_kept = 0u;
    __syncthreads();
    n = keep_best<T>(each_row, 1u, k_eff, kept, n_kept, sh);       // (all of them, but for many ties)
    for (uint32_t i = t; i < n; i += T) {
        const uint64_t k = kept[i];
        const uint32_t rank = rank_in(kept, n, k);
        if (rank >= k_eff) continue;
        float s; uint32_t idx;
        sort_unkey(k, s, idx);
        a.out_scores[size_t(qi) * k_eff + rank] = s;
        a.out_idx[size_t(qi) * k_eff + rank] = int64_t(a.slots != nullptr ? a.slots[idx] : idx);
    }
}

// ===========================================================================
// Few rows (a filter's, as a rule): the scan has kept every row's score, and nothing is scored again.  Writing and reading
// a score per row and query takes less than k_pick's second scoring of whole blocks (2000 rows x 3072, 1024 queries, k = 10: this kernel 6 to 11 us,
// k_pick 80; all latency at that size).
// ===========================================================================
template <uint32_t T, uint32_t H>
__global__ __launch_bounds__(T) void k_pick_rows(const float *__restrict__ scores, uint32_t stride, uint32_t n, uint32_t k_eff, float *out_scores,
                                                 int64_t *out_idx, const uint32_t *slots, uint32_t *overflow, uint64_t *stamp) {
    __shared__ __align__(16) uint64_t kept[kSelectKept + 2];
    __shared__ SelectShared sh;
    __shared__ TopShared top;
    __shared__ uint32_t n_kept;
    const uint32_t qi = blockIdx.x, t = threadIdx.x;
    if (stamp != nullptr && qi + t == 0) *stamp = wall_clock64();
    const float *mine = scores + size_t(qi) * stride;
    float v[H];
#pragma unroll
    for (uint32_t e = 0; e < H; ++e) v[e] = e * T + t < n ? mine[e * T + t] : __int_as_float(0x7fc00000);
    if (t == 0) n_kept = 0u;
    // (a score of -infinity does not count, as in k_pick)
    auto word = [&](uint32_t e) { return v[e] == v[e] ? best_word(v[e]) : 0u; };
    uint32_t most = 0u;
#pragma unroll
    for (uint32_t e = 0; e < H; ++e) most = max(most, word(e));
    auto each = [&](auto &&f) {
#pragma unroll
        for (uint32_t e = 0; e < H; ++e)
            if (word(e) != 0u) f(sort_key(v[e], e * T + t));
    };
    const uint32_t m = keep_best<T>(each, select_top<T>(most, k_eff, top), k_eff, kept, n_kept, sh);
    if (t == 0) overflow[qi] = m < k_eff ? 2u : 0u;
    if (m < k_eff) return;
    for (uint32_t i = t; i < m; i += T) {
        const uint64_t k = kept[i];
        const uint32_t rank = rank_in(kept, m, k);
        if (rank >= k_eff) continue;
        float s; uint32_t idx;
        sort_unkey(k, s, idx);
        out_scores[size_t(qi) * k_eff + rank] = s;
        out_idx[size_t(qi) * k_eff + rank] = int64_t(slots != nullptr ? slots[idx] : idx);
    }
}
hipError_t launch_pick_rows(const float *scores, uint32_t stride, uint32_t n, int k_eff, int nq, float *out_scores, int64_t *out_idx, const uint32_t *slots,
                            uint32_t *overflow, uint64_t *stamp, hipStream_t s) {
    if (nq <= 0) return hipSuccess;
    if (n > kMaxPickRows || n > stride || k_eff <= 0 || k_eff > kMaxPickK) return hipErrorInvalidValue;
    if (nq > 256) hipLaunchKernelGGL((k_pick_rows<256, 16>), dim3(unsigned(nq)), dim3(256), 0, s, scores, stride, n, uint32_t(k_eff), out_scores, out_idx, slots, overflow, stamp);
    else hipLaunchKernelGGL((k_pick_rows<1024, 4>), dim3(unsigned(nq)), dim3(1024), 0, s, scores, stride, n, uint32_t(k_eff), out_scores, out_idx, slots, overflow, stamp);
    return hipGetLastError();
}

static size_t pick_sum_bytes(size_t k_eff) { return k_eff * 32 * 4; }      // (where a block's chunks go to several waves)
size_t pick_lds_bytes(int nch, size_t k_eff, bool lut) { return k_eff * 32 * 8 + size_t(nch) * (lut ? 1024 : 64) + pick_sum_bytes(k_eff); }
int pick_shares(int device, int nch, size_t k_eff, size_t nq, bool lut) {
    // (a SIMD's worth of blocks at least for each workgroup)
    if (nq == 0 || k_eff * size_t(nch) * (lut ? 3 : 1) < kSharedWork) return 1;
    return int(std::max<size_t>(1, std::min<size_t>({kMaxShares, k_eff / 4, size_t(device_cus(device)) / nq})));
}
size_t pick_shared_bytes(size_t k_eff, size_t nq) { return nq * (1 + pick_shared_words(uint32_t(k_eff))) * sizeof(uint64_t); }

// The scan's arguments say what was scanned; a.tables: its weight tiles, or (lut) the queries' tables as k_prep_lut leaves them.
hipError_t launch_pick(const ScanArgs &a, bool lut, bool split, int k_eff, float *out_scores, int64_t *out_idx, const uint32_t *slots, uint32_t *overflow,
                       int shares, uint64_t *shared, uint64_t *stamp, hipStream_t s) {
    if (a.nq_tile <= 0) return hipSuccess;
    if (shares < 1 || (shares > 1 && shared == nullptr)) return hipErrorInvalidValue;
    const size_t most_lds = pick_lds_bytes(a.nch, size_t(k_eff), lut);
    if (k_eff <= 0 || k_eff > kMaxPickK || most_lds > kPickLds || a.b_step != 1 || a.n_blocks > kMaxPickBlocks) return hipErrorInvalidValue;
    PickArgs p;
    p.best = a.best_out; p.best_stride = a.best_stride; p.n_blocks = a.n_blocks; p.n = a.n;
    p.codes = a.codes; p.scales = a.scales; p.mask = a.mask; p.tables = a.tables;
    p.qscale = a.qscale; p.qbias = a.qbias;
    for (int i = 0; i < 4; ++i) p.lv[i] = a.lv[i];
    p.nch = a.nch; p.k_eff = k_eff; p.split = split ? 1 : 0;
    p.out_scores = out_scores; p.out_idx = out_idx; p.slots = slots; p.overflow = overflow; p.stamp = stamp;
    p.nq = uint32_t(a.nq_tile); p.shares = uint32_t(shares); p.counts = shared; p.lists = shared + a.nq_tile;
    // few queries leave the chip empty: as many waves as there are blocks to score again
    const bool small = a.nq_tile > 256 && a.n_blocks <= 256 * 16;
    // A block to a wave leaves most of sixteen waves without one where results are few, and the others with a row's chunks one after the
    // other: so many parts of a block's chunks go to as many waves as make the longest wave's time least, by turns of a wave, chunks of a part and what comes on
    // top, where a workgroup has a CU to itself and there are no more blocks than waves (more of them fill the waves whole: 23 blocks of 20 chunks in 1, 2, 4, 8 and 16
    // parts 49.1, 52.0, 52.4, 57.6 and 64.1 us a search).  11 500 shapes, every number of parts: 2.5 % less time than with whole blocks on the mean, 0.6 % more than with
    // the best number each, and 1 in 2000 shapes more than 3 % slower than with whole blocks.  us a search with whole blocks and so: 60K x 3072, one query, k = 1 60.1 and 51.2; 40K x 3032 3-bit, k = 4 88.8 and 82.4; 24K
    // x 2760 2-bit, k = 2 62.4 and 58.1; 50K x 768, 8 queries, k = 1 33.1 and 31.7.  Seven blocks of 20 chunks in 1, 2, 4, 8 and 16 parts 33.2, 33.1, 31.7, 33.7 and 37.4; two
    // workgroups a CU, 352 queries, k = 1, 7 chunks 3-bit, 41.5, 47.8, 47.1, 47.0 and 47.1.
    const size_t waves = 16, share_blocks = (size_t(k_eff) + size_t(shares) - 1) / size_t(shares);
    p.parts = 1;
    if (size_t(a.nq_tile) * size_t(shares) <= 256 && share_blocks <= waves) {
        auto longest = [&](size_t parts) {
            return (share_blocks * parts + waves - 1) / waves * (kPartCost + (size_t(a.nch) + parts - 1) / parts) + (parts > 1 ? kPartsCost : 0);
        };
        for (uint32_t parts = 2; parts <= 16 && int(parts) <= a.nch; parts *= 2)
            if (longest(parts) < longest(p.parts)) p.parts = parts;
    }
    // (LDS decides how many queries' workgroups a CU runs at once: with room for sums that are not used 5K x 320 3-bit, 750 queries, k = 92
    // 128.7 us a search and 106, 10.9K x 64 4-bit, 910, k = 82 68.4 and 57.0, 27K x 768 2-bit, 610, k = 98 217 and 177)
    const size_t lds = most_lds - (p.parts > 1 ? 0 : pick_sum_bytes(size_t(k_eff)));
    auto launch = [&](auto kernel, unsigned threads) -> hipError_t {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(kernel, dim3(unsigned(a.nq_tile) * unsigned(shares)), dim3(threads), lds, s, p);
        return hipGetLastError();
    };
    auto form = [&](auto lut_, auto shared_) -> hipError_t {
        constexpr bool L = decltype(lut_)::value != 0, S = decltype(shared_)::value != 0;
        if constexpr (!S) {
            if (small) return launch(k_pick<256, 16, L, S, false>, 256);
        }
        if (p.parts > 1) return a.n_blocks > 1024 * 16 ? launch(k_pick<1024, 32, L, S, true>, 1024) : launch(k_pick<1024, 16, L, S, true>, 1024);
        return a.n_blocks > 1024 * 16 ? launch(k_pick<1024, 32, L, S, false>, 1024) : launch(k_pick<1024, 16, L, S, false>, 1024);
    };
    if (shares > 1) return lut ? form(IntC<1>{}, IntC<1>{}) : form(IntC<0>{}, IntC<1>{});
    return lut ? form(IntC<1>{}, IntC<0>{}) : form(IntC<0>{}, IntC<0>{});
}

}  // namespace tv
