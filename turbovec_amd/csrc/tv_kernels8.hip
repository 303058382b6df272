// The best row of every block where blocks are few and rows long: a block's chunks over several waves.
//
// k_scan_p4_best, k_scan_lut and k_scan_lut_bt carry a block through the row on one wave, a burst of loads after another, each a microsecond
// of latency: where the blocks are fewer than the chip's waves the launch takes the serial walk of one block, however few there are.  Here 2
// to 16 waves of a workgroup take as many parts of the block's chunks, and their integer sums, which add up in any order, meet in LDS.  Every
// float operation is the one of those kernels, on the same sum.
//
// us a search with one wave a block and with parts: 4-bit 4K x 3072, 5 queries 42.7 and 30.8; 6K x 2048, 1 query 44.8 and 37.2; 20K x 1192, 32
// queries 38.3 and 36.5; 2-bit 1 query 11K x 3048 58.3 and 45.6, 52K x 2656 58.1 and 40.9, 94K x 1024 41.6 and 37.3; 3-bit 1 query 20K x 3072
// 74.8 and 60.6, 7K x 768 39.8 and 31.9; 2 queries 24K x 2048 78 and 64; 8 queries 22K x 2048 61.7 and 55.9.
#include <algorithm>

#include "tv_device.h"
#include "tv_internal.h"

namespace tv {

// Parts of a block, up to `most`: as many as leave every wave a place among `waves` and `least` chunks to work on.
static int parts_of(size_t items, int nch, size_t waves, int least, int most) {
    int p = 1;
    while (p < most && items * size_t(p) * 2 <= waves && nch >= least * p * 2) p *= 2;
    return p;
}
// Blocks of a workgroup of so many waves: no more than spread them over the chip.
static uint32_t blocks_of(size_t items, int cus, int waves, int parts) {
    return uint32_t(std::min<size_t>(size_t(waves / parts), std::max<size_t>(1, (items + cus - 1) / cus)));
}
// The chunks of one part.
struct Part { int from, to; };
static __device__ __forceinline__ Part part_of(int nch, int parts, int part) { return {nch * part / parts, nch * (part + 1) / parts}; }

// ===========================================================================
// Score mode P (k_scan_p4_best, whose forms these are): one tile of queries a workgroup, grid = (block groups, tiles).  A weight is
// used by the few waves that share a part, so it is read from the L2 where it is used; a wave has the codes and weights of kBurst chunks on
// their way while it works on as many.
// ===========================================================================
enum { kPartsPlane, kPartsSplit, kPartsRows };
constexpr int kPartsThreads = 512, kPartsWaves = kPartsThreads / 64;

template <int FORM>
__global__ __launch_bounds__(kPartsThreads, 4) void k_scan_p4_parts(ScanArgs a, int parts, uint32_t per) {
    __shared__ v4i s_acc[kPartsWaves][4][64];
    const int nch = a.nch, lane = threadIdx.x & 63, qn = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)), part = wave & (parts - 1), tile = int(blockIdx.y);
    const uint32_t step = a.b_step, nj = (a.n_blocks + step - 1) / step, j = blockIdx.x * per + uint32_t(wave / parts);
    const uint32_t b = j * step, slot0 = b * 32u;
    const bool there = j < nj;
    uint32_t mw = there && a.mask != nullptr ? uint32_t(a.mask[b >> 1] >> ((b & 1) * 32)) : 0xffffffffu;
    const bool live = there && mw != 0u;
    v16i acc = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    float vs[16];
    if (live) {
        const Part mine = part_of(nch, parts, part);
        const uint4 *codes = reinterpret_cast<const uint4 *>(a.codes) + size_t(b) * nch * 64 + lane;
        const v4i *w = reinterpret_cast<const v4i *>(a.tables) + size_t(tile) * nch * 128 + lane;
        const uint32_t t0 = a.lv[0], t1 = a.lv[1], t2 = a.lv[2], t3 = a.lv[3];
        constexpr int kBurst = 2;
        uint4 x[kBurst];
        v4i wl[kBurst], wh[kBurst];
        auto request = [&](int c0) {
#pragma unroll
            for (int u = 0; u < kBurst; ++u) {
                const int c = min(c0 + u, mine.to - 1);      // (what lies past the part is loaded again, not used)
                x[u] = codes[c * 64];
                wl[u] = w[c * 128];
                wh[u] = w[c * 128 + 64];
            }
        };
        request(mine.from);
        if (part == 0) {
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4) {
                const float4 f = *reinterpret_cast<const float4 *>(a.scales + slot0 + 8 * q4 + 4 * h);
                vs[q4 * 4 + 0] = f.x; vs[q4 * 4 + 1] = f.y; vs[q4 * 4 + 2] = f.z; vs[q4 * 4 + 3] = f.w;
            }
        }
        for (int c0 = mine.from; c0 < mine.to; c0 += kBurst) {
            uint4 cx[kBurst];
            v4i cl[kBurst], ch[kBurst];
#pragma unroll
            for (int u = 0; u < kBurst; ++u) cx[u] = x[u], cl[u] = wl[u], ch[u] = wh[u];
            if (c0 + kBurst < mine.to) request(c0 + kBurst);
#pragma unroll
            for (int u = 0; u < kBurst; ++u) {
                if (c0 + u >= mine.to) break;
                const uint32_t y[4] = {cx[u].x, cx[u].y, cx[u].z, cx[u].w};
                v4i lo, hi;
#pragma unroll
                for (int d = 0; d < 4; ++d) {
                    lo[d] = int(levels_of(y[d] & 0x0f0f0f0fu, t0, t1, t2, t3));
                    hi[d] = int(levels_of((y[d] >> 4) & 0x0f0f0f0fu, t0, t1, t2, t3));
                }
                if constexpr (FORM == kPartsSplit) {
                    const v4i l = lo, g = hi;
                    lo = v4i{l[0], g[0], l[1], g[1]};
                    hi = v4i{int(__builtin_amdgcn_perm(uint32_t(g[2]), uint32_t(l[2]), 0x05010400u)), int(__builtin_amdgcn_perm(uint32_t(g[2]), uint32_t(l[2]), 0x07030602u)),
                             int(__builtin_amdgcn_perm(uint32_t(g[3]), uint32_t(l[3]), 0x05010400u)), int(__builtin_amdgcn_perm(uint32_t(g[3]), uint32_t(l[3]), 0x07030602u))};
                }
                acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(lo, cl[u], acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(hi, ch[u], acc, 0, 0, 0);
            }
        }
        if (part != 0) {
#pragma unroll
            for (int r = 0; r < 4; ++r) s_acc[wave][r][lane] = v4i{acc[4 * r], acc[4 * r + 1], acc[4 * r + 2], acc[4 * r + 3]};
        }
    }
    __syncthreads();
    if (part != 0 || !there) return;
    const int q = tile * kQTile + qn;
    const float nan = __int_as_float(0x7fc00000);
    float4 *rows = reinterpret_cast<float4 *>(reinterpret_cast<float *>(a.best_out) + size_t(q) * a.best_stride + j * 32u + 4u * uint32_t(h));
    if (!live) {      // (no row of the block is allowed)
        if (q >= a.nq_tile) return;
        if constexpr (FORM == kPartsRows) {
#pragma unroll
            for (int r = 0; r < 4; ++r) rows[2 * r] = float4{nan, nan, nan, nan};
        } else if (h == 0) a.best_out[size_t(q) * a.best_stride + j] = 0u;
        return;
    }
    for (int p = 1; p < parts; ++p) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const v4i s = s_acc[wave + p][r][lane];
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[4 * r + e] += s[e];
        }
    }
    const float qs = q < a.nq_tile ? a.qscale[q] : 0.0f, qb = q < a.nq_tile ? a.qbias[q] : 0.0f;
    // rows 8 (r / 4) + 4 h + r % 4 (turbovec/src/search.rs:1519-1524); NaN for those that may not be returned
    if (slot0 + 32u > a.n) mw &= (1u << (a.n - slot0)) - 1u;
    float s[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const float v = ((mw >> (8 * (r >> 2) + 4 * h + (r & 3))) & 1u) ? vs[r] : nan;
        s[r] = fmaf(float(acc[r]), qs, qb) * v;
    }
    if constexpr (FORM == kPartsRows) {
        if (q >= a.nq_tile) return;
#pragma unroll
        for (int r = 0; r < 4; ++r) rows[2 * r] = float4{s[4 * r], s[4 * r + 1], s[4 * r + 2], s[4 * r + 3]};
    } else {
        float m = -__int_as_float(0x7f800000);
#pragma unroll
        for (int r = 0; r < 16; ++r) m = fmaxf(m, s[r]);      // (NaN never wins)
        m = fmaxf(m, __shfl_xor(m, 32));
        if (h == 0 && q < a.nq_tile) a.best_out[size_t(q) * a.best_stride + j] = best_word(m);
    }
}

// Two waves to a SIMD -- beyond, one wave a block is level or better (us one wave and two, 12 to 24 chunks: 843 blocks 36.1 and 34.4, 856 45.4 and 43.0,
// 918 43.0 and 39.5, 1116 32.9 and 33.3, 1338 48.0 and 48.6, 1854 42.1 and 43.1) -- and four chunks each: with parts of two chunks 7K x 488, 100 queries are 33.9 us against 32.2, 20K x 768, 32
// queries 31.0 against 30.4 (and 372 x 392 23.6 against 25.4); longer rows do not care.
int p4_parts(int nch, size_t n_blocks, int tiles, int cus) { return parts_of(n_blocks * size_t(tiles), nch, size_t(cus) * 8, 4, kPartsWaves); }

hipError_t launch_scan_p4_parts(const ScanArgs &a, bool split, int parts, int device, hipStream_t s) {
    const uint32_t nj = a.b_step ? (a.n_blocks + a.b_step - 1) / a.b_step : 0u;
    if (a.nq_tile <= 0 || nj == 0 || a.best_out == nullptr || a.best_stride / (a.best_rows ? 32u : 1u) < nj || (a.best_rows && (a.b_step != 1 || split)) ||
        (parts != 2 && parts != 4 && parts != 8))
        return hipErrorInvalidValue;
    const uint32_t tiles = uint32_t(a.nq_tile + kQTile - 1) / kQTile, per = blocks_of(size_t(nj) * tiles, device_cus(device), kPartsWaves, parts);
    const dim3 grid((nj + per - 1) / per, tiles), threads(64 * per * uint32_t(parts));
    if (a.best_rows) hipLaunchKernelGGL((k_scan_p4_parts<kPartsRows>), grid, threads, 0, s, a, parts, per);
    else if (split) hipLaunchKernelGGL((k_scan_p4_parts<kPartsSplit>), grid, threads, 0, s, a, parts, per);
    else hipLaunchKernelGGL((k_scan_p4_parts<kPartsPlane>), grid, threads, 0, s, a, parts, per);
    return hipGetLastError();
}

// ===========================================================================
// Score modes L, u32 epilogue: QL queries, their tables in LDS with the queries' entries side by side (k_scan_lut), one block a group of
// waves, one block a workgroup where the CUs are as many.  Nibble tables also for one query: byte tables (k_scan_lut_bt) halve the reads,
// but setting out 32 times as many entries as a block has look-ups takes longer than the reads they save.
// ===========================================================================
constexpr int kMaxLutGroups = 8;
constexpr int kLutPartsThreads = 1024, kLutPartsWaves = kLutPartsThreads / 64;

// Four words, each four entries of one query, as four words, each an entry of the four.
static __device__ __forceinline__ void transpose4(uint32_t (&w)[4]) {
    const uint32_t a = __builtin_amdgcn_perm(w[1], w[0], 0x05010400u), b = __builtin_amdgcn_perm(w[3], w[2], 0x05010400u);
    const uint32_t c = __builtin_amdgcn_perm(w[1], w[0], 0x07030602u), d = __builtin_amdgcn_perm(w[3], w[2], 0x07030602u);
    w[0] = __builtin_amdgcn_perm(b, a, 0x05040100u);
    w[1] = __builtin_amdgcn_perm(b, a, 0x07060302u);
    w[2] = __builtin_amdgcn_perm(d, c, 0x05040100u);
    w[3] = __builtin_amdgcn_perm(d, c, 0x07060302u);
}
template <int QL> struct PartsWord;
template <> struct PartsWord<1> { typedef uint8_t type; };
template <> struct PartsWord<2> { typedef uint16_t type; };
template <> struct PartsWord<4> { typedef uint32_t type; };
template <> struct PartsWord<8> { typedef uint32_t type __attribute__((ext_vector_type(2))); };

template <int QL>
__global__ __launch_bounds__(kLutPartsThreads) void k_scan_lut_parts(ScanArgs a, int parts, uint32_t per) {
    typedef typename PartsWord<QL>::type word_t;
    typedef const __attribute__((address_space(3))) word_t lds_word_t;
    extern __shared__ __align__(16) uint8_t smem[];
    const int nch = a.nch, tid = threadIdx.x, lane = tid & 63, vi = lane & 31, h = lane >> 5, q0 = int(blockIdx.y) * QL, nq = min(QL, a.nq_tile - q0);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), part = wave & (parts - 1), block = wave / parts;
    uint32_t *s_sum = reinterpret_cast<uint32_t *>(smem + size_t(nch) * 1024 * QL);      // [block][query][row]
    const uint32_t step = a.b_step, nj = (a.n_blocks + step - 1) / step, j = blockIdx.x * per + uint32_t(block);
    const uint32_t b = j * step, slot0 = b * 32u;
    const bool there = uint32_t(block) < per && j < nj;      // (waves without a block help to set out the tables)
    uint32_t mw = there && a.mask != nullptr ? uint32_t(a.mask[b >> 1] >> ((b & 1) * 32)) : 0xffffffffu;
    const bool live = there && mw != 0u;
    const Part mine = part_of(nch, parts, part);
    const uint4 *codes = reinterpret_cast<const uint4 *>(a.codes) + size_t(live ? b : 0u) * nch * 64 + lane;
    constexpr int kBurst = 2;
    uint4 x[kBurst];
    auto request = [&](int c0) {
#pragma unroll
        for (int u = 0; u < kBurst; ++u) x[u] = codes[min(c0 + u, mine.to - 1) * 64];
    };
    request(mine.from);      // (on their way while the tables are set out)
    const float vs = live ? a.scales[slot0 + vi] : 0.0f;
    for (int w = tid; w < nch * 256; w += kLutPartsThreads) {
        uint32_t v[QL < 4 ? 4 : QL] = {};
#pragma unroll
        for (int qq = 0; qq < QL; ++qq)
            v[qq] = reinterpret_cast<const uint32_t *>(a.tables + size_t(q0 + min(qq, nq - 1)) * nch * 1024)[w];      // (sums of queries past the last are not read)
        if constexpr (QL == 1) reinterpret_cast<uint32_t *>(smem)[w] = v[0];
        if constexpr (QL == 2) {
            reinterpret_cast<uint2 *>(smem)[w] = make_uint2(__builtin_amdgcn_perm(v[1], v[0], 0x05010400u), __builtin_amdgcn_perm(v[1], v[0], 0x07030602u));
        }
        if constexpr (QL == 4) {
            transpose4(v);
            reinterpret_cast<uint4 *>(smem)[w] = make_uint4(v[0], v[1], v[2], v[3]);
        }
        if constexpr (QL == 8) {
            uint32_t lo[4] = {v[0], v[1], v[2], v[3]}, hi[4] = {v[4], v[5], v[6], v[7]};
            transpose4(lo);
            transpose4(hi);
            reinterpret_cast<uint4 *>(smem)[2 * w] = make_uint4(lo[0], hi[0], lo[1], hi[1]);
            reinterpret_cast<uint4 *>(smem)[2 * w + 1] = make_uint4(lo[2], hi[2], lo[3], hi[3]);
        }
    }
    for (int i = tid; i < int(per) * QL * 32; i += kLutPartsThreads) s_sum[i] = 0u;
    __syncthreads();
    if (live) {
        const uint32_t base = uint32_t(reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) uint8_t *)smem));
        constexpr int kSh = QL == 1 ? 0 : QL == 2 ? 1 : QL == 4 ? 2 : 3;      // (a nibble times the entries' size still fits a byte)
        uint32_t acc[QL] = {};
        for (int c0 = mine.from; c0 < mine.to; c0 += kBurst) {
            uint4 cx[kBurst];
#pragma unroll
            for (int u = 0; u < kBurst; ++u) cx[u] = x[u];
            if (c0 + kBurst < mine.to) request(c0 + kBurst);
#pragma unroll
            for (int u = 0; u < kBurst; ++u) {
                if (c0 + u >= mine.to) break;
                const uint32_t y[4] = {cx[u].x, cx[u].y, cx[u].z, cx[u].w};
                const uint32_t at = base + uint32_t((c0 + u) * 32 + 16 * h) * 32 * QL;
#pragma unroll
                for (int d = 0; d < 4; ++d) {
                    const uint32_t plo = (y[d] << kSh) & (0x0f0f0f0fu << kSh), phi = (y[d] >> (4 - kSh)) & (0x0f0f0f0fu << kSh);
                    auto add = [&](auto ec) {
                        constexpr int e = decltype(ec)::value;
                        const int g = d * 4 + e;
                        const word_t vh = *reinterpret_cast<lds_word_t *>(plus_byte<e>(at, phi) + g * 32 * QL);
                        const word_t vl = *reinterpret_cast<lds_word_t *>(plus_byte<e>(at, plo) + (g * 32 + 16) * QL);
                        // (entries are at most 127, so the two add bytewise without a carry)
                        if constexpr (QL == 1) acc[0] += uint32_t(vh) + uint32_t(vl);
                        if constexpr (QL == 2 || QL == 4) {
                            const uint32_t s = uint32_t(vh) + uint32_t(vl);
#pragma unroll
                            for (int qq = 0; qq < QL; ++qq) acc[qq] = __builtin_amdgcn_udot4(s, 1u << (8 * qq), acc[qq], false);
                        }
                        if constexpr (QL == 8) {
                            const word_t s = vh + vl;
#pragma unroll
                            for (int qq = 0; qq < 4; ++qq) {
                                acc[qq] = __builtin_amdgcn_udot4(s.x, 1u << (8 * qq), acc[qq], false);
                                acc[4 + qq] = __builtin_amdgcn_udot4(s.y, 1u << (8 * qq), acc[4 + qq], false);
                            }
                        }
                    };
                    add(IntC<0>{}); add(IntC<1>{}); add(IntC<2>{}); add(IntC<3>{});
                }
            }
        }
#pragma unroll
        for (int qq = 0; qq < QL; ++qq) atomicAdd(&s_sum[(block * QL + qq) * 32 + vi], acc[qq]);      // (both halves of the wave, all parts)
    }
    __syncthreads();
    if (!there) return;
    if (slot0 + 32u > a.n) mw &= (1u << (a.n - slot0)) - 1u;
    for (int qq = part; qq < nq; qq += parts) {
        // ((f32(sum) * scale) + bias) * vec_scale (turbovec/src/search.rs:1174-1177); NaN never wins
        const float score = ((float(int(s_sum[(block * QL + qq) * 32 + vi])) * a.qscale[q0 + qq]) + a.qbias[q0 + qq]) * vs;
        float m = -__int_as_float(0x7f800000);
        if ((mw >> vi) & 1u) m = fmaxf(m, score);
#pragma unroll
        for (int d = 1; d < 32; d <<= 1) m = fmaxf(m, __shfl_xor(m, d));
        if (lane == 0) a.best_out[size_t(q0 + qq) * a.best_stride + j] = live ? best_word(m) : 0u;
    }
}

static size_t lut_parts_lds(int nch, int ql) { return size_t(nch) * 1024 * size_t(ql) + size_t(kLutPartsWaves / 2) * size_t(ql) * 32 * 4; }
// Queries of a workgroup: all of up to eight, as far as their tables fit.
static int lut_parts_queries(int nch, int nq) {
    int ql = nq <= 1 ? 1 : nq <= 2 ? 2 : nq <= 4 ? 4 : 8;
    while (ql > 1 && lut_parts_lds(nch, ql) > 160 * 1024) ql /= 2;
    return ql;
}

// As many waves as are resident -- up to two queries, whose look-ups the LDS bounds: more queries add up on the vector ALU what k_scan_lut adds on the
// matrix unit, and pay only where the chip is rather empty (us one wave a block and parts on four times as many waves: 8 queries 99K x 960 2-bit 42 and
// 51, 56K x 728 3-bit 49 and 52; 4 queries 67K x 1024 3-bit, filtered, 44 and 52).  Queries beyond a workgroup's go to more of them, side by
// side, where there is room by the same count; k_scan_lut16 takes sixteen at a time, but wants its tables in another order, 5 to 7 us a launch
// more (us so and with parts: 500 x 2880 2-bit, 16 queries 49 and 36; 5K x 1024 2-bit, 16 43 and 34; 1.5K x 448 3-bit, 47 38 and 31; 5K x 3072 2-bit, 5 68 and 51;
// 25K x 3072 3-bit, 3 80 and 64; on twice the waves 22K x 1024 3-bit, 22 57 and 74, but 24K x 384 2-bit, 15 44 and 39: rows up to three chunks have twice).
int lut_parts(int nch, int nq, size_t n_blocks, int cus) {
    const int ql = lut_parts_queries(nch, nq), groups = (nq + ql - 1) / ql;
    const size_t lds = lut_parts_lds(nch, ql);
    if (groups > kMaxLutGroups || lds > 160 * 1024) return 1;
    const size_t waves = ql > 4 ? kLutPartsWaves / (nch <= 3 ? 1 : 2) : ql > 2 || lds > 80 * 1024 ? kLutPartsWaves : 2 * kLutPartsWaves;
    return parts_of(n_blocks * size_t(groups), nch, size_t(cus) * waves, 1, kLutPartsWaves);
}

hipError_t launch_scan_lut_parts(const ScanArgs &a, int parts, int device, hipStream_t s) {
    const uint32_t nj = a.b_step ? (a.n_blocks + a.b_step - 1) / a.b_step : 0u;
    const int ql = lut_parts_queries(a.nch, a.nq_tile), groups = (a.nq_tile + ql - 1) / ql;
    const size_t lds = lut_parts_lds(a.nch, ql);
    if (a.nq_tile <= 0 || groups > kMaxLutGroups || nj == 0 || a.best_out == nullptr || a.best_stride < nj || a.classic != 0 || lds > 160 * 1024 ||
        (parts != 2 && parts != 4 && parts != 8 && parts != 16))
        return hipErrorInvalidValue;
    const uint32_t per = blocks_of(size_t(nj) * groups, device_cus(device), kLutPartsWaves, parts);
    auto launch = [&](auto q) -> hipError_t {
        constexpr int Q = decltype(q)::value;
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(k_scan_lut_parts<Q>), hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL((k_scan_lut_parts<Q>), dim3((nj + per - 1) / per, groups), dim3(kLutPartsThreads), lds, s, a, parts, per);
        return hipGetLastError();
    };
    return ql == 1 ? launch(IntC<1>{}) : ql == 2 ? launch(IntC<2>{}) : ql == 4 ? launch(IntC<4>{}) : launch(IntC<8>{});
}

}  // namespace tv
