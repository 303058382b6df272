// Second step of the two-step table scan: rows that the int8 scan in front (k_scan_p4_wide's instances for 2- and 3-bit codes)
// left in are scored from the u8 tables, term for term as k_scan_lut does (turbovec/src/search.rs:2856-2994, 1174-1177), and
// those that reach the floor go to the query's candidate segments.
//
// A workgroup holds the tables of QW neighbouring queries in LDS and takes a share of the stage's blocks; the words of
// its queries for eight blocks are neighbours in memory.  A wave collects set bits in a queue of its own and scores 64 rows
// at a time, one per lane: at every step all lanes look up the same byte-group, of QW tables laid out a bank group
// apart, so that two lanes meet in a bank only on the same dword.  Rows lie one after the other (the scan wrote them so): a lane reads
// its row's lines whole -- where they lie in the index's blocks a row of 384 bytes is spread over 24 lines.
//
// What bounds it: one LDS instruction per look-up, six clocks each with 32 waves per CU (no bank conflicts by the counters; one or
// two vector instructions beside it), and the latency of a row's first line.  10M rows x 1536 2-bit, 1024 queries, k = 100: 14 000 rows
// a query, 2.9 ms of the search's 15.2 to 16.4.  With eight queries and sixteen waves per CU, where the tables of four would let 32
// run, 20 to 40 % longer over short stages (890K x 920, 640 queries: 66 us a launch and 45), level over long ones.
#include "tv_device.h"
#include "tv_internal.h"

namespace tv {

constexpr int kNearThreads = 1024, kNearWaves = kNearThreads / 64;
constexpr uint32_t kNearQueue = 128;      // entries of a wave's queue: fewer than 64 left over, and 64 more at a time
// A workgroup that meets more than one in so many of its (row, query) pairs gives up: the floors of its queries are far too low,
// and the caller repeats them.
constexpr uint32_t kNearGiveUp = 8;
constexpr uint32_t kNearSubs = 8;         // most segments a workgroup keeps per query: neighbouring rows, often neighbours of one query, go to different ones
constexpr uint32_t kNearGaveUp = 0xffffffffu;

__host__ __device__ constexpr uint32_t near_table_stride(int nch) { return uint32_t(nch) * 1024u + 16u; }
constexpr size_t near_lds_bytes(int nch, int qw) {
    return size_t(qw) * near_table_stride(nch) + size_t(kNearWaves) * kNearQueue * 8 + size_t(qw) * (12 + 4 * kNearSubs) + 64;
}

template <int QW>
__global__ __launch_bounds__(kNearThreads, QW <= 4 ? 8 : 4) void k_near_rescore(NearRescore a) {
    static_assert(QW >= 1 && QW <= 8 && 8 % QW == 0, "a wave's 64 words are whole groups of eight blocks");
    constexpr uint32_t kSub = 8 / QW;                     // groups of eight blocks a wave takes at a time
    extern __shared__ __align__(16) uint8_t smem[];
    const uint32_t stride = near_table_stride(a.nch);
    uint2 *queue = reinterpret_cast<uint2 *>(smem + QW * stride);
    float *s_q = reinterpret_cast<float *>(queue + kNearWaves * kNearQueue);     // [QW]: qscale, qbias, floor
    uint32_t *s_cnt = reinterpret_cast<uint32_t *>(s_q + QW * 3);                // [QW][kNearSubs] candidates appended
    uint32_t *s_met = s_cnt + QW * kNearSubs;                                    // pairs met so far
    const uint32_t n_groups_q = (uint32_t(a.nq) + QW - 1) / QW;
    const uint32_t part = blockIdx.x / n_groups_q, q0 = blockIdx.x % n_groups_q * QW;
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = uint32_t(__builtin_amdgcn_readfirstlane(int(tid >> 6)));
    const uint32_t active = min(uint32_t(QW), uint32_t(a.nq) - q0);
    const uint32_t lo = uint32_t(uint64_t(a.stage.groups) * part / a.splits), hi = uint32_t(uint64_t(a.stage.groups) * (part + 1) / a.splits);
    const uint32_t seg = a.seg0 + part * a.sub;
    // (given up in the stage before: in all that follow)
    const bool given_up = a.seg0 != 0u && a.cand_cnt[size_t(q0) * a.seg_stride + seg - a.splits * a.sub] == kNearGaveUp;
    const uint32_t limit = max((hi - lo) * (kNearBlocks * kVecBlock / kNearGiveUp) * active, 4096u);

    for (uint32_t q = 0; q < active; ++q) {
        const uint4 *src = reinterpret_cast<const uint4 *>(a.tables + size_t(q0 + q) * a.nch * 1024);
        uint4 *dst = reinterpret_cast<uint4 *>(smem + q * stride);
        for (uint32_t i = tid; i < uint32_t(a.nch) * 64u; i += kNearThreads) dst[i] = src[i];
    }
    if (tid < QW) {
        const bool act = tid < active;
        s_q[tid * 3 + 0] = act ? a.qscale[q0 + tid] : 0.0f;
        s_q[tid * 3 + 1] = act ? a.qbias[q0 + tid] : 0.0f;
        s_q[tid * 3 + 2] = act ? order_unkey(a.gtau[q0 + tid]) : __int_as_float(0x7fc00000);
    }
    if (tid < QW * kNearSubs) s_cnt[tid] = 0u;
    if (tid == 0) *s_met = 0u;
    __syncthreads();

    uint2 *mine = queue + wave * kNearQueue;
    const uint32_t lds_b = uint32_t(reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) uint8_t *)smem));
    // `count` queued rows from place `at` on, one per lane.
    auto score = [&](uint32_t at, uint32_t count) {
        const uint2 e = mine[at + (lane < count ? lane : 0u)];
        const bool on = lane < count && e.y < a.n;      // (places behind the last row have no bound, and may be in)
        const uint32_t ql = e.x >> 29, slot = e.y;
        const u32x4 *row = reinterpret_cast<const u32x4 *>(a.stage.rows + size_t(e.x & 0x1fffffffu) * (uint32_t(a.nch) * 32u));
        const float scale = a.scales[min(slot, a.n - 1u)];
        uint32_t tab = lds_b + ql * stride;
        uint32_t sum = 0u;
        auto look_up = [&](const u32x4 &x, uint32_t at) {
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                const uint32_t high = (x[d] >> 4) & 0x0f0f0f0fu, low = x[d] & 0x0f0f0f0fu;
                static_for<4>([&](auto bb) {
                    constexpr int b = decltype(bb)::value;
                    sum += uint32_t(reinterpret_cast<LdsByte *>(uintptr_t(plus_byte<b>(at, high)))[(d * 4 + b) * 32]) +
                           uint32_t(reinterpret_cast<LdsByte *>(uintptr_t(plus_byte<b>(at, low)))[(d * 4 + b) * 32 + 16]);
                });
                if (d & 1) asm volatile("" : "+v"(sum));      // (sixteen at a time: added up late, they would take every register)
            }
        };
        u32x4 c0 = row[0], c1 = row[1];
#pragma unroll 1
        for (int c = 0; c < a.nch; ++c) {
            const int from = 2 * min(c + 1, a.nch - 1);
            const u32x4 n0 = row[from], n1 = row[from + 1];
            __builtin_amdgcn_sched_barrier(0);
            look_up(c0, tab);
            look_up(c1, tab + 512u);
            tab += 1024u;
            c0 = n0;
            c1 = n1;
        }
        const float s = ((float(sum) * s_q[ql * 3]) + s_q[ql * 3 + 1]) * scale;
        if (on && s >= s_q[ql * 3 + 2]) {
            const uint32_t my_sub = slot & (a.sub - 1u), pos = atomicAdd(&s_cnt[ql * kNearSubs + my_sub], 1u);
            if (pos < kSegCap) a.cand[(size_t(q0 + ql) * a.seg_stride + seg + my_sub) * kSegCap + pos] = sort_key(s, slot);
        }
    };

    // lane: query ql, group x of the stage, block w of it
    const uint32_t ql = lane / 8u % QW, w = lane & 7u, sub = lane / (8u * QW);
    const uint32_t *words = reinterpret_cast<const uint32_t *>(a.stage.masks) +
                            size_t(q0 / kQTile) * a.stage.groups * (kQTile * kNearBlocks) + (q0 % kQTile + ql) * kNearBlocks + w;
    constexpr uint32_t kStep = kNearWaves * kSub;
    const uint32_t gstep = uint32_t(uint64_t(kStep) * a.stage.mul % a.stage.total);
    uint32_t x = lo + wave * kSub + sub;                              // of the word in `left`; the next ones are on their way
    uint32_t group = near_group(a.stage, a.stage.first + x);
    auto word_at = [&](uint32_t xu) { return xu < hi && ql < active ? words[size_t(xu) * (kQTile * kNearBlocks)] : 0u; };
    uint32_t left = word_at(x), w1 = word_at(x + kStep), w2 = word_at(x + 2 * kStep), w3 = word_at(x + 3 * kStep);
    uint32_t queued = 0u, met = 0u, x0 = lo + wave * kSub;            // (x0: uniform over the wave)
    if (given_up) x0 = hi;
    for (;;) {
        while (queued < 64u && x0 < hi) {
            const uint64_t any = __ballot(left != 0u);
            if (any == 0ull) {
                left = w1;
                w1 = w2;
                w2 = w3;
                x += kStep;
                x0 += kStep;
                w3 = word_at(x + 3 * kStep);
                group += gstep;
                if (group >= a.stage.total) group -= a.stage.total;
                continue;
            }
            if (left != 0u) {
                const uint32_t bit = uint32_t(__builtin_ctz(left)), r = 15u - (bit & 15u), i = 8u * (r >> 2) + 4u * (bit >> 4) + (r & 3u);
                left &= left - 1u;
                const uint32_t pos = queued + uint32_t(__popcll(any & ((1ull << lane) - 1ull)));
                mine[pos] = make_uint2(ql << 29 | ((x * uint32_t(kNearBlocks) + w) * uint32_t(kVecBlock) + i), near_block(a.stage, group, w) * uint32_t(kVecBlock) + i);
            }
            queued += uint32_t(__popcll(any));
        }
        if (queued == 0u) break;
        const uint32_t n = min(queued, 64u);
        queued -= n;
        met += n;
        score(queued, n);
        if (met >= 1024u) {
            if (lane == 0) atomicAdd(s_met, met);
            met = 0u;
            if (*reinterpret_cast<volatile uint32_t *>(s_met) > limit) break;
        }
    }
    if (lane == 0 && met != 0u) atomicAdd(s_met, met);
    __syncthreads();
    const bool over = *s_met > limit || given_up;
    for (uint32_t i = 0; i < active * a.sub; ++i) {
        const uint32_t q = i / a.sub, sb = i % a.sub, n = s_cnt[q * kNearSubs + sb];
        const size_t at = size_t(q0 + q) * a.seg_stride + seg + sb;
        // (a segment given up reads as full: places not written hold candidates that rank behind all others -- each of another
        // slot, as the selection counts on keys that differ; nothing of such a query is returned)
        if (over)
            for (uint32_t e = n + tid; e < uint32_t(kSegCap); e += kNearThreads)
                a.cand[at * kSegCap + e] = sort_key(-__int_as_float(0x7f800000), (seg + sb) * uint32_t(kSegCap) + e);
        if (tid == 0) a.cand_cnt[at] = over ? kNearGaveUp : n;
    }
}

int near_rescore_queries(int nch) {
    for (int qw = 8; qw >= 1; qw /= 2)
        if (near_lds_bytes(nch, qw) <= 80 * 1024) return qw;
    for (int qw = 8; qw >= 1; qw /= 2)
        if (near_lds_bytes(nch, qw) <= 160 * 1024) return qw;
    return 0;
}

template <int QW>
static hipError_t launch_rescore(const NearRescore &a, hipStream_t s) {
    const size_t lds = near_lds_bytes(a.nch, QW);
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(k_near_rescore<QW>), hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
    if (e != hipSuccess) return e;
    const unsigned grid = (unsigned(a.nq) + QW - 1) / QW * a.splits;
    hipLaunchKernelGGL((k_near_rescore<QW>), dim3(grid), dim3(kNearThreads), lds, s, a);
    return hipGetLastError();
}
hipError_t launch_near_rescore(const NearRescore &a, hipStream_t s) {
    if (a.nq <= 0 || a.stage.groups == 0 || a.splits == 0 || a.sub == 0 || a.sub > kNearSubs || (a.sub & (a.sub - 1)) != 0 || size_t(a.seg0) + size_t(a.splits) * a.sub > a.seg_stride) return hipErrorInvalidValue;
    if (size_t(a.stage.groups) * kNearBlocks * kVecBlock > (size_t(1) << 29)) return hipErrorInvalidValue;
    switch (near_rescore_queries(a.nch)) {
        case 8: return launch_rescore<8>(a, s);
        case 4: return launch_rescore<4>(a, s);
        case 2: return launch_rescore<2>(a, s);
        case 1: return launch_rescore<1>(a, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace tv
