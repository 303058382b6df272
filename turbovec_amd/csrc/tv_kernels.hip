// HIP kernels of the turbovec search path for gfx950 (MI355X).
//
// Compiled with -ffp-contract=off: every float expression keeps the separate
// multiplies and adds the reference performs, and fmaf appears only where the
// reference fuses.
#include "tv_device.h"
#include "tv_internal.h"
#include "tv_select.h"

#include <cfloat>
#include <climits>
#include <cstdlib>

namespace tv {



// ===========================================================================
// Layout transforms between the persisted sequential-blocked layout
// (turbovec/src/pack.rs:336-361) and the native chunked layout.
// ===========================================================================

// One workgroup per (block, chunk): a 1 KiB tile of 32 groups x 32 lanes is
// transposed through LDS so both sides move as dwords.
__global__ __launch_bounds__(256) void k_seq_to_native(const uint8_t *__restrict__ seq, uint8_t *__restrict__ nat,
                                                       int G, int nch, size_t first_block) {
    __shared__ uint8_t tile[32 * 36];  // [group][lane], rows padded to 36 bytes
    const size_t b = first_block + blockIdx.x / nch;
    const int c = blockIdx.x % nch;
    const int t = threadIdx.x;
    {   // read: dword t covers group gl = t/8, lanes 4*(t%8)..+3
        const int gl = t >> 3, l4 = (t & 7) * 4;
        const int g = c * 32 + gl;
        uint32_t v = 0;
        if (g < G) v = *reinterpret_cast<const uint32_t *>(seq + ((b - first_block) * size_t(G) + g) * 32 + l4);
        *reinterpret_cast<uint32_t *>(tile + gl * 36 + l4) = v;
    }
    __syncthreads();
    {   // write: dword t of the chunk = lane l = t/4 (h = l/32, i = l%32), bytes j0..j0+3
        const int l = t >> 2, j0 = (t & 3) * 4;
        const int h = l >> 5, i = l & 31;
        uint32_t v = 0;
        for (int j = 0; j < 4; ++j) v |= uint32_t(tile[(16 * h + j0 + j) * 36 + i]) << (8 * j);
        *reinterpret_cast<uint32_t *>(nat + (b * size_t(nch) + c) * 1024 + size_t(t) * 4) = v;
    }
}

__global__ __launch_bounds__(256) void k_native_to_seq(const uint8_t *__restrict__ nat, uint8_t *__restrict__ seq,
                                                       int G, int nch, size_t first_block, size_t block_bytes,
                                                       const float *__restrict__ scales) {
    __shared__ uint8_t tile[32 * 36];
    const size_t b = first_block + blockIdx.x / nch;
    const int c = blockIdx.x % nch;
    const int t = threadIdx.x;
    {
        const int l = t >> 2, j0 = (t & 3) * 4;
        const int h = l >> 5, i = l & 31;
        const uint32_t v = *reinterpret_cast<const uint32_t *>(nat + (b * size_t(nch) + c) * 1024 + size_t(t) * 4);
        for (int j = 0; j < 4; ++j) tile[(16 * h + j0 + j) * 36 + i] = uint8_t(v >> (8 * j));
    }
    __syncthreads();
    {
        const int gl = t >> 3, l4 = (t & 7) * 4;
        const int g = c * 32 + gl;
        if (g < G)
            *reinterpret_cast<uint32_t *>(seq + (b - first_block) * block_bytes + size_t(g) * 32 + l4) =
                *reinterpret_cast<const uint32_t *>(tile + gl * 36 + l4);
    }
    // (a snapshot's unit: the block's row scales behind its codes)
    if (scales != nullptr && c == 0 && t < 32)
        *reinterpret_cast<float *>(seq + (b - first_block) * block_bytes + size_t(G) * 32 + t * 4) = scales[b * 32 + t];
}

__device__ __forceinline__ size_t native_byte_index(size_t v, int g, int nch) {
    const size_t b = v >> 5;
    const int i = int(v & 31);
    return ((b * size_t(nch) + size_t(g >> 5)) * 64 + size_t(((g & 31) >> 4) * 32 + i)) * 16 + size_t(g & 15);
}

// rows[r*G + g] -> lane of vector old_n + r (turbovec/src/pack.rs:211-233 append_lanes).
__global__ void k_append_rows(const uint8_t *__restrict__ rows, uint8_t *__restrict__ nat, int G, int nch,
                              size_t old_n, size_t n_new) {
    const size_t idx = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (idx >= n_new * size_t(G)) return;
    const size_t r = idx / G;
    const int g = int(idx % G);
    nat[native_byte_index(old_n + r, g, nch)] = rows[idx];
}

// turbovec/src/lib.rs:2964-3003: move_lane(last -> idx), zero_lane(last), scale move.
__global__ void k_move_lane(uint8_t *__restrict__ nat, float *__restrict__ scales, int G, int nch, size_t src,
                            size_t dst) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g < G) {
        const size_t s = native_byte_index(src, g, nch);
        if (src != dst) nat[native_byte_index(dst, g, nch)] = nat[s];
        nat[s] = 0;
    }
    if (g == 0) {
        if (src != dst) scales[dst] = scales[src];
        scales[src] = 0.0f;
    }
}

// Queries whose candidates overflowed, packed for one more full scan: row r of the packed batch
// is query rows[r] of the chunk, its floor the raised one k_final left for it, placed where the
// scan kernels read the floors of tile r / tile_q.
__global__ __launch_bounds__(256) void k_gather_redo(const float *__restrict__ q, const uint32_t *__restrict__ rows,
                                                     const int *__restrict__ raised, int dim, int tile_q,
                                                     float *__restrict__ q_out, int *__restrict__ tau_out) {
    const uint32_t r = blockIdx.x, o = rows[r];
    for (int i = threadIdx.x; i < dim; i += 256) q_out[size_t(r) * dim + i] = q[size_t(o) * dim + i];
    if (threadIdx.x == 0) tau_out[(r / tile_q) * kQTile + r % tile_q] = raised[o];
}

__global__ void k_fill_i32(int *p, int v, size_t n) {
    const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// A new index's tables, read from pinned host memory, and its open floors in one launch, which the call that makes the index waits for
// (a copy and a fill one after the other: 1500 rows of 1536 dimensions into a new index 133 us a pass, and so 121).
__global__ void k_lay_tables(const uint32_t *__restrict__ from, uint32_t *__restrict__ to, uint32_t n, int *__restrict__ floors, int v, uint32_t n_floors) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) to[i] = from[i];
    else if (i - n < n_floors) floors[i - n] = v;
}

// ===========================================================================
// Scan, score mode P: 4-bit codes -> int8 codebook levels -> i8 MFMA against
// int8 query weights (turbovec/src/search.rs:1392-1567 computes the same
// integers with vpdpbusd).  acc = sum_d w[d] * level[code[d]], exact in i32;
// score = fma(f32(acc), scale, bias) * vec_scale (search.rs:1519-1524).
//
// k_scan_p4 decodes half of a chunk through LDS: a 256-entry table maps a code
// byte to the two levels of its nibbles (low nibble's in the low byte); two
// entries make one dword of an A operand -- one shift (the byte's table
// offset), one LDS read and half a merge per code byte, against 3.75
// vector-ALU instructions per byte for the in-register lookup, which alone held
// this kernel below the HBM stream (as does one LDS instruction per byte alone).
// The table sits at the start of the kernel's LDS (there is no static
// allocation before it), so a byte's offset is its address.
// ===========================================================================
// 16 bytes of LDS per lane, requested like the table entries (lds_u16): behind the compiler's
// wait-count bookkeeping, lds_settle being the matching wait.
template <int OFF>
__device__ __forceinline__ void lds_b128(v4i &dst, uint32_t addr) {
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=&v"(dst) : "v"(addr), "n"(OFF));
}
// Hold until at most N LDS requests younger than those feeding e, o, w0 and w1 are outstanding.
template <int N>
__device__ __forceinline__ void lds_settle(uint32_t (&e)[4], uint32_t (&o)[4], v4i &w0, v4i &w1) {
    asm volatile("s_waitcnt lgkmcnt(%10)" : "+v"(e[0]), "+v"(e[1]), "+v"(e[2]), "+v"(e[3]), "+v"(o[0]), "+v"(o[1]), "+v"(o[2]), "+v"(o[3]), "+v"(w0), "+v"(w1) : "n"(N));
}

// The same with a run-time address, and a full wait tied to the registers a step is about to use.
__device__ __forceinline__ void lds_b128_at(v4i &dst, uint32_t addr) {
    asm volatile("ds_read_b128 %0, %1" : "=&v"(dst) : "v"(addr));
}
// (the same for two table dwords)
template <int NT>
__device__ __forceinline__ void lds_settle_all(uint32_t (&e)[2], uint32_t (&o)[2], v4i (&w)[NT]) {
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(e[0]), "+v"(e[1]), "+v"(o[0]), "+v"(o[1]));
#pragma unroll
    for (int t = 0; t < NT; ++t) asm volatile("" : "+v"(w[t]));
}
template <int NT>
__device__ __forceinline__ void lds_settle_all(uint32_t (&e)[4], uint32_t (&o)[4], v4i (&w)[NT]) {
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(e[0]), "+v"(e[1]), "+v"(e[2]), "+v"(e[3]), "+v"(o[0]), "+v"(o[1]), "+v"(o[2]), "+v"(o[3]));
#pragma unroll
    for (int t = 0; t < NT; ++t) asm volatile("" : "+v"(w[t]));
}

// n16 16-byte words from global memory into LDS by a workgroup of THREADS, twelve loads per thread
// in flight at a time: a scan launch that reads a block or two per wave (a sampling level, a
// small index) is as long as its set-up, and word after word the copy is a chain of trips to L2.
template <int THREADS>
__device__ __forceinline__ void stage_to_lds(uint4 *dst, const uint4 *src, int n16, int tid) {
    constexpr int kBatch = 12;
    for (int i0 = tid; i0 < n16; i0 += THREADS * kBatch) {
        uint4 tmp[kBatch];
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
            const int i = i0 + u * THREADS;
            tmp[u] = i < n16 ? src[i] : make_uint4(0, 0, 0, 0);
        }
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
            const int i = i0 + u * THREADS;
            if (i < n16) dst[i] = tmp[u];
        }
    }
}

template <int U, int MODE, bool W_LDS, int THREADS = kScanThreads>
__global__ __launch_bounds__(THREADS) void k_scan_p4(ScanArgs a) {
    extern __shared__ __align__(16) uint8_t smem[];
    constexpr bool LISTS = MODE == kModeLists, DUMP = MODE == kModeDump, BEST = MODE == kModeBest;
    constexpr bool APPEND = MODE == kModeAppend || BEST;     // both fill the candidate segments
    if (APPEND && launch_switched_off(a.run_if)) return;
    const int nch = a.nch, k = a.k;
    uint8_t *sW = smem + kDecodeBytes;
    const size_t w_bytes = kDecodeBytes + (W_LDS ? size_t(nch) * 2048 : 0);
    float *ls = reinterpret_cast<float *>(smem + w_bytes);
    uint32_t *li = reinterpret_cast<uint32_t *>(ls + (LISTS ? k * THREADS : 0));
    int *stau = reinterpret_cast<int *>(li + (LISTS ? k * THREADS : 0));
    uint32_t *scnt = reinterpret_cast<uint32_t *>(stau);  // append mode: candidates per query of this workgroup

    // A workgroup of more than four waves is GROUPS four-wave groups that share the weights in LDS
    // and are, in every other respect, workgroups vb of a launch of a.vgrid four-wave workgroups:
    // the same blocks per wave, a candidate segment per group.
    constexpr int GROUPS = THREADS / kScanThreads;
    static_assert(THREADS % kScanThreads == 0 && (GROUPS == 1 || APPEND), "wave groups are an append-mode form");
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = (tid >> 6) % (kScanThreads / 64);
    const int qn = lane & 31, h = lane >> 5;
    const uint32_t vgrid = GROUPS > 1 ? a.vgrid : gridDim.x;
    const uint32_t vb = GROUPS > 1 ? blockIdx.x * GROUPS + uint32_t(tid) / kScanThreads : blockIdx.x;
    if (GROUPS > 1) scnt += (tid / kScanThreads) * kQTile;

    // Logical blocks j = 0..nj-1 stand for physical blocks j*step (step > 1 samples the index).
    const uint32_t step = a.b_step;
    const uint32_t nj = (a.n_blocks + step - 1) / step;
    const uint32_t total_waves = vgrid * (kScanThreads / 64);
    const uint32_t gw = wave * vgrid + vb;  // consecutive blocks go to different workgroups
    // Blocks are dealt round-robin to the waves of the grid: wave gw takes logical blocks gw,
    // gw + total_waves, ...  Neighbouring rows (clustered data, contiguous allowlists) then spread
    // over all workgroups instead of piling into one.
    const uint32_t j_begin = gw, j_end = (GROUPS > 1 && vb >= vgrid) ? 0u : nj;   // (a group beyond the launch's last has no blocks)
    const uint4 *codes = reinterpret_cast<const uint4 *>(a.codes) + lane;

    // first block with at least one allowed slot (search.rs:3015-3029)
    auto live_from = [&](uint32_t j) -> uint32_t {
        if (a.mask == nullptr) return j;
        while (j < j_end) {
            const uint32_t b = j * step;
            const uint64_t w = a.mask[b >> 1];
            if (uint32_t(w >> ((b & 1) * 32)) != 0u) break;
            j += total_waves;
        }
        return j;
    };

    // the wave's first codes are on their way from HBM while the workgroup sets up its LDS
    uint32_t j = live_from(j_begin);
    uint4 buf[U];
    if (j < j_end) {
#pragma unroll
        for (int u = 0; u < U; ++u) buf[u] = load_stream16(&codes[(size_t(j) * step * nch + u) * 64]);
    }

    if (W_LDS) stage_to_lds<THREADS>(reinterpret_cast<uint4 *>(sW), reinterpret_cast<const uint4 *>(a.tables), nch * 128, tid);
    for (int b = tid; b < 256; b += THREADS) {
        const uint32_t lo = (a.lv[(b & 15) >> 2] >> (8 * (b & 3))) & 0xffu;
        const uint32_t hi = (a.lv[b >> 6] >> (8 * ((b >> 4) & 3))) & 0xffu;
        reinterpret_cast<uint16_t *>(smem)[b] = uint16_t(lo | (hi << 8));
    }
    if (LISTS && tid < kQTile) stau[tid] = a.gtau[tid];
    if (APPEND && (tid % kScanThreads) < kQTile) scnt[tid % kScanThreads] = 0u;
    __syncthreads();

    const bool active = qn < a.nq_tile;
    const float qs = active ? a.qscale[qn] : 0.0f;
    const float qb = active ? a.qbias[qn] : 0.0f;
    const uint32_t t0 = a.lv[0], t1 = a.lv[1], t2 = a.lv[2], t3 = a.lv[3];
    // append mode: a fixed per-query floor; NaN for idle lanes so no compare passes
    const float tau_fixed = (APPEND && !BEST) ? (active ? order_unkey(a.gtau[qn]) : __int_as_float(0x7fc00000)) : 0.0f;

    LaneList L{0, 0.0f, 0u, 0};
    const uint4 *wglob = reinterpret_cast<const uint4 *>(a.tables) + lane;

    while (j < j_end) {
        const uint32_t nj_live = live_from(j + total_waves);
        const uint32_t b = j * step;
        v16i acc = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
        for (int c0 = 0; c0 < nch; c0 += U) {
            // the next U chunks (of this block, or the head of the next one) are requested as one
            // contiguous burst before the current U are consumed
            uint4 cur[U];
#pragma unroll
            for (int u = 0; u < U; ++u) cur[u] = buf[u];
            if (c0 + U < nch) {
#pragma unroll
                for (int u = 0; u < U; ++u) buf[u] = load_stream16(&codes[(size_t(b) * nch + c0 + U + u) * 64]);
            } else if (nj_live < j_end) {
#pragma unroll
                for (int u = 0; u < U; ++u) buf[u] = load_stream16(&codes[(size_t(nj_live) * step * nch + u) * 64]);
            }
            // A chunk gives two A operands.  The first, from code bytes 0..7 of the lane, is decoded
            // on the vector ALU: dwords (low-nibble levels of bytes 0..3, high-nibble levels of bytes
            // 0..3, the same for bytes 4..7).  The second, from bytes 8..15, through the byte table:
            // dword r from bytes 8+2r (low half) and 9+2r (high half), each as its (low nibble, high
            // nibble) pair of levels.  Either unit alone is slower than the HBM stream (3.75 ALU
            // instructions per byte; one LDS instruction per byte); half each fits under it.  The
            // LDS requests of chunk u+1 are issued before chunk u is waited for.
            uint32_t e[2][4], o[2][4];
            v4i bw0[2], bw1[2];
            const uint32_t w_addr = uint32_t(kDecodeBytes + c0 * 2048 + lane * 16);
            auto request = [&](auto uc) {
                constexpr int u = decltype(uc)::value, p = u & 1;
                if (W_LDS) {
                    lds_b128<u * 2048>(bw0[p], w_addr);
                } else {
                    const uint4 w = wglob[(size_t(c0 + u) * 2) * 64];
                    bw0[p] = v4i{int(w.x), int(w.y), int(w.z), int(w.w)};
                }
                const uint32_t xa = cur[u].z, xb = cur[u].w;
                lds_u16(e[p][0], byte_x2<0>(xa)); lds_u16(o[p][0], byte_x2<1>(xa));
                lds_u16(e[p][1], byte_x2<2>(xa)); lds_u16(o[p][1], byte_x2<3>(xa));
                lds_u16(e[p][2], byte_x2<0>(xb)); lds_u16(o[p][2], byte_x2<1>(xb));
                lds_u16(e[p][3], byte_x2<2>(xb)); lds_u16(o[p][3], byte_x2<3>(xb));
                if (W_LDS) {
                    lds_b128<u * 2048 + 1024>(bw1[p], w_addr);
                } else {
                    const uint4 w = wglob[(size_t(c0 + u) * 2 + 1) * 64];
                    bw1[p] = v4i{int(w.x), int(w.y), int(w.z), int(w.w)};
                }
            };
            request(IntC<0>{});
            static_for<U>([&](auto uc) {
                constexpr int u = decltype(uc)::value, p = u & 1;
                if constexpr (u + 1 < U) request(IntC<u + 1>{});
                const v4i a0 = {int(levels_of(cur[u].x & 0x0f0f0f0fu, t0, t1, t2, t3)),
                                int(levels_of((cur[u].x >> 4) & 0x0f0f0f0fu, t0, t1, t2, t3)),
                                int(levels_of(cur[u].y & 0x0f0f0f0fu, t0, t1, t2, t3)),
                                int(levels_of((cur[u].y >> 4) & 0x0f0f0f0fu, t0, t1, t2, t3))};
                if constexpr (u + 1 < U) lds_settle<W_LDS ? 10 : 8>(e[p], o[p], bw0[p], bw1[p]);
                else lds_settle<0>(e[p], o[p], bw0[p], bw1[p]);
                acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(a0, bw0[p], acc, 0, 0, 0);
                const v4i a1 = {int(e[p][0] | (o[p][0] << 16)), int(e[p][1] | (o[p][1] << 16)),
                                int(e[p][2] | (o[p][2] << 16)), int(e[p][3] | (o[p][3] << 16))};
                acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(a1, bw1[p], acc, 0, 0, 0);
            });
        }

        // ---- epilogue: lane owns query qn and rows 8*(r/4) + 4*h + r%4 ----
        const uint32_t slot0 = b * 32u;
        uint32_t mw = 0xffffffffu;
        if (a.mask != nullptr) mw = uint32_t(a.mask[b >> 1] >> ((b & 1) * 32));
        float vs[16];
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
            const float4 f = *reinterpret_cast<const float4 *>(a.scales + slot0 + 8 * q4 + 4 * h);
            vs[q4 * 4 + 0] = f.x; vs[q4 * 4 + 1] = f.y; vs[q4 * 4 + 2] = f.z; vs[q4 * 4 + 3] = f.w;
        }
        if (DUMP) {
            if (active) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int i = 8 * (r >> 2) + 4 * h + (r & 3);
                    const uint32_t slot = slot0 + i;
                    if (slot < a.n) {
                        const float s = fmaf(float(acc[r]), qs, qb) * vs[r];
                        const size_t o = size_t(qn) * a.n + slot;
                        if (a.acc_out) a.acc_out[o] = acc[r];
                        if (a.score_out) a.score_out[o] = ((mw >> i) & 1u) ? s : __int_as_float(0x7fc00000);
                    }
                }
            }
        } else if (BEST) {
            // A first sampling level without a floor: one candidate per block and query, the best
            // allowed row of the block (a real score of a real row, so the k-th best of these is a
            // floor at least k scanned rows reach, and with rows in no particular order it is the
            // k-th best row of the sample but for the odd pair that shares a block).
            float bs = 0.0f;
            uint32_t bslot = 0xffffffffu;      // none yet
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int i = 8 * (r >> 2) + 4 * h + (r & 3);
                const uint32_t slot = slot0 + i;
                const float s = fmaf(float(acc[r]), qs, qb) * vs[r];
                const bool ok = active && slot < a.n && ((mw >> i) & 1u) && s == s;
                if (ok && (bslot == 0xffffffffu || ranks_before(s, slot, bs, bslot))) { bs = s; bslot = slot; }
            }
            const float os_ = __shfl_xor(bs, 32);
            const uint32_t oslot = __shfl_xor(bslot, 32);
            if (oslot != 0xffffffffu && (bslot == 0xffffffffu || ranks_before(os_, oslot, bs, bslot))) { bs = os_; bslot = oslot; }
            if (h == 0 && bslot != 0xffffffffu) {
                const uint32_t pos = atomicAdd(&scnt[qn], 1u);
                if (pos < kSegCap) a.cand[(size_t(qn) * a.seg_stride + vb) * kSegCap + pos] = sort_key(bs, bslot);
            }
        } else if (APPEND) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float s = fmaf(float(acc[r]), qs, qb) * vs[r];
                if (s >= tau_fixed) {
                    const int i = 8 * (r >> 2) + 4 * h + (r & 3);
                    const uint32_t slot = slot0 + i;
                    if (slot < a.n && ((mw >> i) & 1u)) {
                        const uint32_t pos = atomicAdd(&scnt[qn], 1u);
                        if (pos < kSegCap)
                            a.cand[(size_t(qn) * a.seg_stride + vb) * kSegCap + pos] = sort_key(s, slot);
                    }
                }
            }
        } else {
            if (a.share_tau && (j & 3u) == 0u && lane < kQTile) atomicMax(&stau[lane], a.gtau[lane]);
            const float tau = order_unkey(stau[qn]);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int i = 8 * (r >> 2) + 4 * h + (r & 3);
                const uint32_t slot = slot0 + i;
                const float s = fmaf(float(acc[r]), qs, qb) * vs[r];
                if (active && s >= tau && (L.cnt < k || ranks_before(s, slot, L.worst_s, L.worst_i))) {
                    if (slot < a.n && ((mw >> i) & 1u)) {
                        if (list_offer(L, ls, li, THREADS, tid, k, s, slot) && a.share_tau) {
                            const int key = order_key(L.worst_s);
                            if (atomicMax(&stau[qn], key) < key) atomicMax(&a.gtau[qn], key);
                        }
                    }
                }
            }
        }
        j = nj_live;
    }

    if (LISTS) {
        const size_t total_threads = size_t(gridDim.x) * THREADS;
        const size_t gt = size_t(blockIdx.x) * THREADS + tid;
        a.part_cnt[gt] = L.cnt;
        for (int e = 0; e < L.cnt; ++e) {
            a.part_scores[size_t(e) * total_threads + gt] = ls[e * THREADS + tid];
            a.part_idx[size_t(e) * total_threads + gt] = li[e * THREADS + tid];
        }
    }
    if (APPEND) {
        __syncthreads();
        const int t = tid % kScanThreads;
        if (t < a.nq_tile && vb < vgrid) a.cand_cnt[size_t(t) * a.seg_stride + vb] = scnt[t];
    }
}

// ===========================================================================
// Multi-tile scan, score mode P, append mode only: the weights of NT query
// tiles stay resident in LDS for the whole launch (NT * dim bytes), every wave
// decodes a chunk once and feeds NT tiles' MFMAs from it.  No barrier in the
// main loop.  Used when NT * dim fits the 160 KiB of LDS.
// ===========================================================================

// LB = code bytes of a lane's sixteen that are decoded through the LDS byte table (8: bytes 8..15;
// 4: bytes 12..15, bytes 8..11 then go through the vector ALU like bytes 0..7 and are interleaved
// into the table's (low, high) order by two byte permutes: fewer LDS reads in flight and fewer
// registers, which lets the three-tile instance run four waves per SIMD).
template <int NT, int U, int THREADS, int LB>
__global__ __launch_bounds__(THREADS) void k_scan_p4_multi(ScanArgs a) {
    static_assert(LB == 8 || LB == 4, "table bytes per lane and chunk");
    extern __shared__ __align__(16) uint8_t smem[];
    if (launch_switched_off(a.run_if)) return;
    const int nch = a.nch;
    uint8_t *sW = smem + kDecodeBytes;                             // [NT][nch][2][64 lanes][16], after the byte table
    uint32_t *scnt = reinterpret_cast<uint32_t *>(sW + size_t(NT) * nch * 2048);
    const int tid = threadIdx.x, lane = tid & 63;
    const int qn = lane & 31, h = lane >> 5;
    const int nt_active = (a.nq_tile + kQTile - 1) / kQTile;
    {
        const int live16 = nt_active * nch * 128;
        stage_to_lds<THREADS>(reinterpret_cast<uint4 *>(sW), reinterpret_cast<const uint4 *>(a.tables), live16, tid);
        for (int i = live16 + tid; i < NT * nch * 128; i += THREADS) reinterpret_cast<uint4 *>(sW)[i] = make_uint4(0, 0, 0, 0);
    }
    for (int b = tid; b < 256; b += THREADS) {   // code byte -> (level of its low nibble, level of its high nibble)
        const uint32_t lo = (a.lv[(b & 15) >> 2] >> (8 * (b & 3))) & 0xffu;
        const uint32_t hi = (a.lv[b >> 6] >> (8 * ((b >> 4) & 3))) & 0xffu;
        reinterpret_cast<uint16_t *>(smem)[b] = uint16_t(lo | (hi << 8));
    }
    uint32_t *snext = scnt + NT * kQTile;   // next unclaimed block of this workgroup
    // Per query, in LDS (a block's epilogue reads them; registers are for the stream): scale, bias
    // and floor, and the accumulator bound of k_scan_p4_wide -- a row reaches its query's floor only
    // if its integer sum reaches  floor / (qscale * largest row scale of the block) - qbias / qscale,
    // taken conservatively (1e-5 relative, 2 + 1 absolute), so a tile of a block is scored in
    // floats only when some lane's largest sum is at the bound.  Floors, query scales and biases
    // outside 1e-30 .. 1e30 switch the bound off for that query (every tile scored).
    float4 *s_q = reinterpret_cast<float4 *>(snext + 4);      // [NT * 32] (scale, bias, floor, -)
    float2 *s_b = reinterpret_cast<float2 *>(s_q + NT * kQTile);   // [NT * 32] (ta, tb) of the bound
    float *s_vs = reinterpret_cast<float *>(s_b + NT * kQTile) + (tid >> 6) * 32;   // this wave's: the row scales of the block it finishes, NaN where not allowed
    for (int q = tid; q < NT * kQTile; q += THREADS) {
        scnt[q] = 0u;
        const bool act = q < a.nq_tile;
        const float qs = act ? a.qscale[q] : 0.0f, qb = act ? a.qbias[q] : 0.0f;
        const float tau = act ? order_unkey(a.gtau[q]) : __int_as_float(0x7fc00000);  // NaN: nothing passes
        s_q[q] = make_float4(qs, qb, tau, 0.0f);
        const float inf = __int_as_float(0x7f800000);
        const bool bounded = tau >= 1e-30f && tau <= 1e30f && qs >= 1e-30f && qs <= 1e30f && fabsf(qb) <= 1e30f &&
                             tau / qs < inf;
        const float rb = qb / qs;
        s_b[q] = make_float2(!act ? inf : bounded ? (tau / qs) * (1.0f - 1e-5f) : -inf,
                             act && bounded ? rb + 1e-5f * fabsf(rb) + 2.0f : 0.0f);
    }
    if (tid == 0) *snext = 0u;
    __syncthreads();

    const uint32_t t0 = a.lv[0], t1 = a.lv[1], t2 = a.lv[2], t3 = a.lv[3];
    const uint32_t step = a.b_step;
    const uint32_t nj = (a.n_blocks + step - 1) / step;
    const uint4 *codes = reinterpret_cast<const uint4 *>(a.codes) + lane;
    const uint32_t w_base = uint32_t(kDecodeBytes + lane * 16), w_tile = uint32_t(nch) * 2048u;

    // Blocks are dealt round-robin to workgroups (logical block m * gridDim.x + blockIdx.x belongs
    // to this one), so neighbouring rows -- clustered data, contiguous allowlists -- spread over
    // all of them; inside a workgroup the waves claim blocks from a shared counter as they go,
    // so all of them finish within one block of each other whatever the SIMD arbitration did.
    // Returns the next block with at least one allowed slot (search.rs:3015-3029), or >= nj.
    auto claim = [&]() -> uint32_t {
        for (;;) {
            uint32_t m = 0;
            if (lane == 0) m = atomicAdd(snext, 1u);
            m = uint32_t(__builtin_amdgcn_readfirstlane(int(m)));
            const uint32_t j = m * gridDim.x + blockIdx.x;
            if (j >= nj || a.mask == nullptr) return j;
            const uint32_t b = j * step;
            if (uint32_t(a.mask[b >> 1] >> ((b & 1) * 32)) != 0u) return j;
        }
    };

    // The wave's work is one stream of U-chunk groups running through its blocks.  Two register
    // sets take turns: while one group is decoded and multiplied, the next group's codes (of this
    // block, or the head of the next live one) are in flight into the other set, requested as one
    // contiguous burst.  Every group issues the same loads in the same order -- the row scale of
    // its block, then the burst -- so the number of younger loads behind any register is fixed:
    // before chunk u of the current set, 2U - u of them may still be outstanding.
    v16i acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = v16i{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    uint32_t j = claim();
    int c0 = 0;
    const uint8_t *code_bytes = reinterpret_cast<const uint8_t *>(codes);   // lane offset included

    auto issue = [&](u32x4 (&dst)[U], float &sc, uint32_t jb_phys, int c) {
        load4_async(sc, a.scales + jb_phys * 32u + qn);
        const uint8_t *p = code_bytes + (size_t(jb_phys) * nch + c) * 1024;
        load16_async<0>(dst[0], p);
        if (U > 1) load16_async<1024>(dst[U > 1 ? 1 : 0], p);
        if (U > 2) load16_async<2048>(dst[U > 2 ? 2 : 0], p);
        if (U > 3) load16_async<3072>(dst[U > 3 ? 3 : 0], p);
        static_assert(U <= 4, "immediate offsets cover four chunks");
    };

    auto finish_block = [&](uint32_t b, float my_scale) {
        const uint32_t slot0 = b * 32u;
        uint32_t mw = 0xffffffffu;
        if (a.mask != nullptr) mw = uint32_t(a.mask[b >> 1] >> ((b & 1) * 32));
        // Rows past the end of the index or outside the allowlist get a NaN scale: their scores
        // then fail the floor compare by themselves, and the per-score path has no other test.
        if (slot0 + 32u > a.n) mw &= (a.n > slot0) ? (0xffffffffu >> (slot0 + 32u - a.n)) : 0u;
        // the block's largest allowed row scale; a negative, huge or non-finite scale (no encoder
        // writes such) or a largest one below 1e-30 switches the bound off for the block
        // (the lane's query number through a move the compiler cannot see through: the addresses of
        // its records are then formed here, per block, instead of living in registers through the stream)
        int qrec = qn;
        asm volatile("v_mov_b32 %0, %0" : "+v"(qrec));
        const bool ok = (mw >> qn) & 1u;
        const bool odd = ok && !(my_scale >= 0.0f && my_scale <= 1e30f);
        // (non-negative floats order like their bit patterns: the maximum on the data-parallel path, no LDS)
        const float vmax = __uint_as_float(wave_umax(ok && !odd ? __float_as_uint(my_scale) : 0u));
        const float inv = 1.0f / vmax;       // all scales zero: +inf, no sum reaches the bound, and every score is zero
        if (lane < 32) s_vs[lane] = ok ? my_scale : __int_as_float(0x7fc00000);   // for the tiles scored below (read by this wave only)
        const bool odd_block = __any(odd) || (vmax > 0.0f && vmax < 1e-30f);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const float2 tq = s_b[t * kQTile + qrec];
            const float bf = fmaf(tq.x, inv, -tq.y) - 1.0f;
            int bound;
            asm("v_cvt_i32_f32 %0, %1" : "=v"(bound) : "v"(bf));   // saturates; NaN gives 0
            if (odd_block) bound = int(0x80000000);
            const v16i &c = acc[t];
            int m = max(max(c[0], c[1]), c[2]);       // (one running maximum: the kernel has no register to spare)
            m = max(max(m, c[3]), c[4]);
            m = max(max(m, c[5]), c[6]);
            m = max(max(m, c[7]), c[8]);
            m = max(max(m, c[9]), c[10]);
            m = max(max(m, c[11]), c[12]);
            m = max(max(m, c[13]), c[14]);
            m = max(m, c[15]);
            if (m >= bound) {
                const float4 qp = s_q[t * kQTile + qrec];
                const float *vs = s_vs + 4 * h;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int i = 8 * (r >> 2) + 4 * h + (r & 3);
                    const float s = fmaf(float(acc[t][r]), qp.x, qp.y) * vs[8 * (r >> 2) + (r & 3)];
                    if (s >= qp.z) {
                        const int q = t * kQTile + qn;
                        const uint32_t pos = atomicAdd(&scnt[q], 1u);
                        if (pos < kSegCap)
                            a.cand[(size_t(q) * a.seg_stride + blockIdx.x) * kSegCap + pos] = sort_key(s, slot0 + i);
                    }
                }
            }
        }
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t] = v16i{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    };

    // One group: request the following group into `nxt`, consume `cur`.  Returns false after the
    // wave's last group (whose request re-reads the current group: a valid address, never used).
    auto phase = [&](u32x4 (&cur)[U], float &cur_sc, u32x4 (&nxt)[U], float &nxt_sc) -> bool {
        const uint32_t b = j * step;
        const bool block_ends = c0 + U >= nch;
        uint32_t pj = j;
        int pc = c0 + U;
        if (block_ends) { pj = claim(); pc = 0; }
        const bool more = pj < nj;
        issue(nxt, nxt_sc, (more ? pj : j) * step, more ? pc : c0);
        // the group's weights: one address per tile, the chunk and the operand as immediate offsets
        uint32_t w_at[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) w_at[t] = w_base + (uint32_t(c0) * 2048u + uint32_t(t) * w_tile);
        static_for<U>([&](auto uc) {
            constexpr int u = decltype(uc)::value;
            wait_vm<2 * U - u>(cur[u]);
            // Split decode as in k_scan_p4: code bytes 8..15 of the lane through the byte table
            // (requested first), bytes 0..7 on the vector ALU while those reads and the first
            // operand's weights are on their way; the second operand's weights travel during the
            // first operand's MFMAs.  All LDS traffic of the loop is requested and waited for by
            // hand, so the counts below are exact.
            constexpr int kTab = LB / 2;      // dwords of the second operand that come from the table (two code bytes each)
            uint32_t e[kTab], o[kTab];
            if constexpr (LB == 8) {
                lds_u16(e[0], byte_x2<0>(cur[u].z)); lds_u16(o[0], byte_x2<1>(cur[u].z));
                lds_u16(e[1], byte_x2<2>(cur[u].z)); lds_u16(o[1], byte_x2<3>(cur[u].z));
            }
            lds_u16(e[kTab - 2], byte_x2<0>(cur[u].w)); lds_u16(o[kTab - 2], byte_x2<1>(cur[u].w));
            lds_u16(e[kTab - 1], byte_x2<2>(cur[u].w)); lds_u16(o[kTab - 1], byte_x2<3>(cur[u].w));
            v4i b0[NT], b1[NT];
            static_for<NT>([&](auto tc) {
                constexpr int t = decltype(tc)::value;
                lds_b128<u * 2048>(b0[t], w_at[t]);
            });
            const v4i a0 = {int(levels_of(cur[u].x & 0x0f0f0f0fu, t0, t1, t2, t3)),
                            int(levels_of((cur[u].x >> 4) & 0x0f0f0f0fu, t0, t1, t2, t3)),
                            int(levels_of(cur[u].y & 0x0f0f0f0fu, t0, t1, t2, t3)),
                            int(levels_of((cur[u].y >> 4) & 0x0f0f0f0fu, t0, t1, t2, t3))};
            uint32_t z01[2] = {0u, 0u};       // LB = 4: the second operand's first two dwords, from bytes 8..11
            if constexpr (LB == 4) {
                const uint32_t lo = levels_of(cur[u].z & 0x0f0f0f0fu, t0, t1, t2, t3);
                const uint32_t hi = levels_of((cur[u].z >> 4) & 0x0f0f0f0fu, t0, t1, t2, t3);
                z01[0] = __builtin_amdgcn_perm(hi, lo, 0x05010400u);      // (low, high) of byte 8, of byte 9
                z01[1] = __builtin_amdgcn_perm(hi, lo, 0x07030602u);      // of bytes 10 and 11
            }
            lds_settle_all(e, o, b0);
            static_for<NT>([&](auto tc) {
                constexpr int t = decltype(tc)::value;
                lds_b128<u * 2048 + 1024>(b1[t], w_at[t]);
            });
#pragma unroll
            for (int t = 0; t < NT; ++t) acc[t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a0, b0[t], acc[t], 0, 0, 0);
            v4i a1;
            if constexpr (LB == 8) {
                a1 = v4i{int(e[0] | (o[0] << 16)), int(e[1] | (o[1] << 16)), int(e[2] | (o[2] << 16)), int(e[3] | (o[3] << 16))};
            } else {
                a1 = v4i{int(z01[0]), int(z01[1]), int(e[0] | (o[0] << 16)), int(e[1] | (o[1] << 16))};
            }
            lds_settle_all(e, o, b1);
#pragma unroll
            for (int t = 0; t < NT; ++t) acc[t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a1, b1[t], acc[t], 0, 0, 0);
        });
        if (block_ends) {
            wait_vm<U + 1>(cur_sc);   // this group's own scale: only the request issued above is younger
            finish_block(b, cur_sc);
        }
        j = pj;
        c0 = pc;
        return more;
    };

    if (j < nj) {
        u32x4 bufA[U], bufB[U];
        float scA, scB;
        issue(bufA, scA, j * step, 0);
        while (phase(bufA, scA, bufB, scB) && phase(bufB, scB, bufA, scA)) {}
        asm volatile("s_waitcnt vmcnt(0)");
    }
    __syncthreads();
    for (int q = tid; q < a.nq_tile; q += THREADS) a.cand_cnt[size_t(q) * a.seg_stride + blockIdx.x] = scnt[q];
}

// ===========================================================================
// Batched scan, score mode P, append mode only: one pass serves NT query tiles
// (NT*32 queries).  A workgroup walks groups of 4*MW blocks; each wave decodes
// its MW blocks once per chunk and feeds NT tiles' MFMAs from the same decoded
// operand, so the nibble decode -- the VALU cost that bounds the single-tile
// kernel -- is amortised NT times.  The NT tiles' weights (NT * dim bytes) do
// not fit LDS whole, so they stream through it in slices of KC chunks, double
// buffered, shared by the four waves and re-read from L2 once per block group.
// ===========================================================================

template <int NT, int MW, int KC, int OCC>
__global__ __launch_bounds__(kScanThreads, OCC) void k_scan_p4_batched(ScanArgs a) {
    extern __shared__ __align__(16) uint8_t smem[];
    if (launch_switched_off(a.run_if)) return;
    constexpr int kSliceBytes = NT * KC * 2048;           // one slice of all tiles
    constexpr int kStage = kSliceBytes / (kScanThreads * 16);  // uint4 per thread per slice
    static_assert(kSliceBytes % (kScanThreads * 16) == 0, "slice must split evenly over the workgroup");
    uint8_t *sB = smem;                                   // [2][NT][KC][2][1024]
    uint32_t *scnt = reinterpret_cast<uint32_t *>(smem + 2 * kSliceBytes);  // [NT*32]
    const int nch = a.nch;
    const int nslices = nch / KC;                         // host guarantees nch % KC == 0
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int qn = lane & 31, h = lane >> 5;
    const int nt_active = (a.nq_tile + kQTile - 1) / kQTile;
    const uint32_t t0 = a.lv[0], t1 = a.lv[1], t2 = a.lv[2], t3 = a.lv[3];

    for (int i = tid; i < NT * kQTile; i += kScanThreads) scnt[i] = 0u;

    float qs[NT], qb[NT], tau[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int q = t * kQTile + qn;
        const bool act = q < a.nq_tile;
        qs[t] = act ? a.qscale[q] : 0.0f;
        qb[t] = act ? a.qbias[q] : 0.0f;
        tau[t] = act ? order_unkey(a.gtau[q]) : __int_as_float(0x7fc00000);  // NaN: nothing passes
    }

    const uint32_t step = a.b_step;
    const uint32_t nj = (a.n_blocks + step - 1) / step;   // logical blocks
    constexpr uint32_t kGroup = 4 * MW;                   // logical blocks per workgroup iteration
    const uint32_t ngroups = (nj + kGroup - 1) / kGroup;

    // staging of weight slices: thread copies kStage uint4 per slice; slice s of tile t lives at
    // tables + t*nch*2048 + s*KC*2048 (KC*2048 contiguous bytes)
    uint4 stage[kStage];
    auto load_slice = [&](int sl) {
#pragma unroll
        for (int e = 0; e < kStage; ++e) {
            const int idx = e * kScanThreads + tid;               // uint4 index within the slice
            const int t = idx / (KC * 128), r = idx % (KC * 128);
            if (t < nt_active)
                stage[e] = reinterpret_cast<const uint4 *>(a.tables + (size_t(t) * nch + size_t(sl) * KC) * 2048)[r];
            else
                stage[e] = make_uint4(0, 0, 0, 0);
        }
    };
    auto store_slice = [&](int buf) {
        uint4 *dst = reinterpret_cast<uint4 *>(sB + buf * kSliceBytes);
#pragma unroll
        for (int e = 0; e < kStage; ++e) dst[e * kScanThreads + tid] = stage[e];
    };

    const uint4 *codes = reinterpret_cast<const uint4 *>(a.codes) + lane;
    uint32_t g = blockIdx.x;
    if (g >= ngroups) {                                   // whole workgroup leaves together, with empty segments
        for (int q = tid; q < a.nq_tile; q += kScanThreads) a.cand_cnt[size_t(q) * a.seg_stride + blockIdx.x] = 0u;
        return;
    }
    load_slice(0);
    store_slice(0);
    __syncthreads();
    int ring = 0;                                         // buffer holding the slice about to be consumed

    for (; g < ngroups; g += gridDim.x) {
        // this wave's MW logical blocks
        uint32_t jb[MW];
        bool live[MW];
        uint32_t mw[MW];
#pragma unroll
        for (int m = 0; m < MW; ++m) {
            jb[m] = g * kGroup + wave * MW + m;
            live[m] = jb[m] < nj;
            mw[m] = 0xffffffffu;
            if (live[m] && a.mask != nullptr) {
                const uint32_t b = jb[m] * step;
                mw[m] = uint32_t(a.mask[b >> 1] >> ((b & 1) * 32));
                live[m] = mw[m] != 0u;                    // block skip (search.rs:3015-3029)
            }
        }
        v16i acc[MW][NT];
#pragma unroll
        for (int m = 0; m < MW; ++m)
#pragma unroll
            for (int t = 0; t < NT; ++t) acc[m][t] = v16i{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};

        uint4 abuf[MW][KC];                               // codes of the slice being computed
#pragma unroll
        for (int m = 0; m < MW; ++m)
#pragma unroll
            for (int c = 0; c < KC; ++c)
                abuf[m][c] = live[m] ? load_stream16(&codes[(size_t(jb[m]) * step * nch + c) * 64]) : make_uint4(0, 0, 0, 0);

        for (int sl = 0; sl < nslices; ++sl) {
            const bool more = sl + 1 < nslices || g + gridDim.x < ngroups;
            const int next_sl = sl + 1 < nslices ? sl + 1 : 0;
            if (more) load_slice(next_sl);
            uint4 acur[MW][KC];
#pragma unroll
            for (int m = 0; m < MW; ++m)
#pragma unroll
                for (int c = 0; c < KC; ++c) acur[m][c] = abuf[m][c];
            if (sl + 1 < nslices) {
#pragma unroll
                for (int m = 0; m < MW; ++m)
#pragma unroll
                    for (int c = 0; c < KC; ++c)
                        abuf[m][c] = live[m] ? load_stream16(&codes[(size_t(jb[m]) * step * nch + (sl + 1) * KC + c) * 64])
                                             : make_uint4(0, 0, 0, 0);
            }
            const uint4 *bl = reinterpret_cast<const uint4 *>(sB + ring * kSliceBytes) + lane;
#pragma unroll
            for (int c = 0; c < KC; ++c) {
                v4i alo[MW], ahi[MW];
#pragma unroll
                for (int m = 0; m < MW; ++m) {
                    const uint32_t x[4] = {acur[m][c].x, acur[m][c].y, acur[m][c].z, acur[m][c].w};
#pragma unroll
                    for (int d = 0; d < 4; ++d) {
                        alo[m][d] = int(levels_of(x[d] & 0x0f0f0f0fu, t0, t1, t2, t3));
                        ahi[m][d] = int(levels_of((x[d] >> 4) & 0x0f0f0f0fu, t0, t1, t2, t3));
                    }
                }
                // all low-nibble products first, then all high-nibble ones: the two MFMAs that
                // chain on one accumulator end up NT*MW instructions apart instead of back to back
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const uint4 wl = bl[((t * KC + c) * 2) * 64];
                    const v4i blo = {int(wl.x), int(wl.y), int(wl.z), int(wl.w)};
#pragma unroll
                    for (int m = 0; m < MW; ++m)
                        acc[m][t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(alo[m], blo, acc[m][t], 0, 0, 0);
                }
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const uint4 wh = bl[((t * KC + c) * 2 + 1) * 64];
                    const v4i bhi = {int(wh.x), int(wh.y), int(wh.z), int(wh.w)};
#pragma unroll
                    for (int m = 0; m < MW; ++m)
                        acc[m][t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(ahi[m], bhi, acc[m][t], 0, 0, 0);
                }
            }
            if (more) store_slice(ring ^ 1);
            __syncthreads();
            ring ^= 1;
        }

        // ---- epilogue ----
#pragma unroll
        for (int m = 0; m < MW; ++m) {
            if (!live[m]) continue;
            const uint32_t slot0 = jb[m] * step * 32u;
            float vs[16];
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4) {
                const float4 f = *reinterpret_cast<const float4 *>(a.scales + slot0 + 8 * q4 + 4 * h);
                vs[q4 * 4 + 0] = f.x; vs[q4 * 4 + 1] = f.y; vs[q4 * 4 + 2] = f.z; vs[q4 * 4 + 3] = f.w;
            }
#pragma unroll
            for (int t = 0; t < NT; ++t) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const float s = fmaf(float(acc[m][t][r]), qs[t], qb[t]) * vs[r];
                    if (s >= tau[t]) {
                        const int i = 8 * (r >> 2) + 4 * h + (r & 3);
                        const uint32_t slot = slot0 + i;
                        if (slot < a.n && ((mw[m] >> i) & 1u)) {
                            const int q = t * kQTile + qn;
                            const uint32_t pos = atomicAdd(&scnt[q], 1u);
                            if (pos < kSegCap)
                                a.cand[(size_t(q) * a.seg_stride + blockIdx.x) * kSegCap + pos] = sort_key(s, slot);
                        }
                    }
                }
            }
        }
    }
    __syncthreads();
    for (int q = tid; q < a.nq_tile; q += kScanThreads) a.cand_cnt[size_t(q) * a.seg_stride + blockIdx.x] = scnt[q];
}

// ===========================================================================
// Final merge of the per-lane lists of one query tile.
// One workgroup per query: every thread folds a strided subset of the lists
// into a private top-k, then the 256*k survivors are bitonic-sorted.
// ===========================================================================

__global__ __launch_bounds__(256) void k_merge(const float *__restrict__ part_scores,
                                               const uint32_t *__restrict__ part_idx,
                                               const int *__restrict__ part_cnt, int total_threads, int qmod,
                                               int k, int k_eff, int sort_n, float *__restrict__ out_scores,
                                               int64_t *__restrict__ out_idx, int *__restrict__ out_tau) {
    extern __shared__ __align__(16) uint8_t msm[];
    float *ls = reinterpret_cast<float *>(msm);
    uint32_t *li = reinterpret_cast<uint32_t *>(ls + k * 256);
    uint64_t *keys = reinterpret_cast<uint64_t *>(li + k * 256);
    __shared__ int total;
    const int qn = blockIdx.x;
    const int t = threadIdx.x;
    if (t == 0) total = 0;
    LaneList L{0, 0.0f, 0u, 0};
    // lane (gt % 64) of every wave owns query (gt % 64) % qmod
    const int per_wave = 64 / qmod;
    const int n_lists = total_threads / 64 * per_wave;
    for (int l = t; l < n_lists; l += 256) {
        const int gt = (l / per_wave) * 64 + (l % per_wave) * qmod + qn;
        const int cnt = part_cnt[gt];
        for (int e = 0; e < cnt; ++e)
            list_offer(L, ls, li, 256, t, k, part_scores[size_t(e) * total_threads + gt],
                       part_idx[size_t(e) * total_threads + gt]);
    }
    __syncthreads();
    const int base = atomicAdd(&total, L.cnt);
    for (int e = 0; e < L.cnt; ++e) keys[base + e] = sort_key(ls[e * 256 + t], li[e * 256 + t]);
    __syncthreads();
    for (int i = total + t; i < sort_n; i += 256) keys[i] = 0;  // below every real key
    __syncthreads();
    for (int size = 2; size <= sort_n; size <<= 1) {
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            for (int i = t; i < sort_n / 2; i += 256) {
                const int lo = 2 * i - (i & (stride - 1));
                const int hi = lo + stride;
                const bool desc = (lo & size) == 0;
                const uint64_t x = keys[lo], y = keys[hi];
                if ((x < y) == desc) { keys[lo] = y; keys[hi] = x; }
            }
            __syncthreads();
        }
    }
    if (out_tau != nullptr) {
        // sampling pass: publish a floor that at least k_eff scanned slots reach
        if (t == 0) {
            float s = 0.0f; uint32_t idx = 0;
            if (total >= k_eff && k_eff <= sort_n) sort_unkey(keys[k_eff - 1], s, idx);
            out_tau[qn] = (total >= k_eff && k_eff <= sort_n) ? order_key(s == 0.0f ? -0.0f : s) : kTauInit;
        }
        return;
    }
    for (int j = t; j < k_eff; j += 256) {
        float s; uint32_t idx;
        sort_unkey(keys[j], s, idx);
        out_scores[size_t(qn) * k_eff + j] = s;
        out_idx[size_t(qn) * k_eff + j] = int64_t(idx);
    }
}

// ===========================================================================
// Final selection over the candidates an append-mode scan collected: one
// workgroup per query finds the `need` largest keys and emits them in order, or
// takes the last of them as a floor.  A query whose candidates did not fit is
// flagged for the caller to redo.
//
// The work is a few thousand keys in a few hundred short segments, and all of
// it is latency; a thousand queries share the chip.  So: a thread per segment,
// its head requested together with its count -- four threads for one query with many candidates, and
// then the whole of it; up to sixteen leading keys take the need-th largest of groups of threads' best keys
// as a threshold few keys reach (select_top), and more are counted out into 1024 bins, since a few hundred keys in as many segments
// give 256 groups too little to choose from (50K x 3072, 33 queries, k = 100 107 us a search and 92; 20K x 1024 3-bit, 4 queries,
// k = 100 66 and 64); those are collected in LDS and ranked by comparing each with all -- no sort, a handful of
// barriers, 30 KiB of LDS, and workgroups no larger than the segments need.
// Per launch under the profiler, with waves sorting chunks in 64 KiB of LDS (1024 threads per query), with
// every threshold counted out, and now: one query, k = 10, 12, 11, 10.5 us; k = 100, 60 and 33, 21 and 18, 14 and 13; 1000 queries,
// k = 10, 61 to 75, 13 to 19, 11 to 17.
// ===========================================================================
constexpr uint32_t kFinalStage = 2048;     // candidates copied to LDS when some segment is long
constexpr uint32_t kFinalLong = 128;       // ... of which this many segments can be
// One query's segments are read by four threads each where one of them is expected to hold more than the sixteen candidates that a thread
// keeps: it would send all of them through LDS, or, where they are too many for it, have each thread read its segment twice.  us a
// search with one thread a segment and with four: k = 400 700K x 1536 2-bit 230 and 186, 50K x 3072 190 and 156, 10M x 1536 4-bit 1602 and 1567; k = 256
// 2M x 128 166 and 139; k = 100 10M x 1536 2-bit 675 and 665; but with shorter ones 2M x 1536 2-bit, k = 100 182 and 187, 384
// dimensions, k = 100 160 and 168.
constexpr double kFinalLongest = 16.0;
static_assert(kSelectKept > uint32_t(kMaxSampledK) && kFinalStage / 17 < kFinalLong, "k_final's buffers");

// GUESSED: the two-step table scan's selections, with `passed` or keep_floor == 2 (an instance of its own: the others lost 0.4 us a launch to
// it, 1.47M x 128, 7 queries, k = 66 95.5 us a search and, without, 93.9).
template <uint32_t T, uint32_t PARTS, bool GUESSED>
__global__ __launch_bounds__(T) void k_final(const uint64_t *__restrict__ cand,
                                               const uint32_t *__restrict__ cand_cnt, uint32_t n_seg,
                                               uint32_t seg_stride, int k_eff, int k_floor,
                                               float *__restrict__ out_scores, int64_t *__restrict__ out_idx,
                                               uint32_t *__restrict__ overflow, int *__restrict__ tau_out,
                                               int tau_stride_q, int keep_floor, int *__restrict__ raise_out,
                                               const uint32_t *__restrict__ row_map, uint32_t *level_over,
                                               uint32_t *clear_flag, const uint32_t *run_if, const uint32_t *slots, uint64_t *stamp, const int *passed) {
    constexpr uint32_t W = T / 64;
    __shared__ __align__(16) uint64_t kept[kSelectKept + 2];
    __shared__ uint64_t stage[kFinalStage];
    __shared__ SelectShared sh;
    __shared__ TopShared top;
    __shared__ uint32_t any_full, any_long, long_n, n_kept;
    __shared__ uint32_t long_seg[kFinalLong], long_pos[kFinalLong], long_cnt[kFinalLong];
    if (launch_switched_off(run_if)) return;
    const int qn = blockIdx.x;
    const uint32_t t = threadIdx.x, lane = t & 63u, wv = t >> 6;
    const bool sampling = tau_out != nullptr;
    int *tau_slot = sampling ? tau_out + (qn / tau_stride_q) * kQTile + qn % tau_stride_q : nullptr;
    if (clear_flag != nullptr && qn == 0 && t == 0) *clear_flag = 0u;
    if (stamp != nullptr && !sampling && qn == 0 && t == 0) *stamp = wall_clock64();
    if (t == 0) { any_full = 0u; any_long = 0u; long_n = 0u; n_kept = 0u; }
    __syncthreads();
    // every thread owns a contiguous run of this query's segments, or sixteen places of one
    const uint32_t per = (n_seg * PARTS + T - 1) / T;
    const uint32_t s0 = PARTS > 1 ? min(t / PARTS, n_seg) : min(t * per, n_seg), s1 = PARTS > 1 ? min(s0 + 1u, n_seg) : min(s0 + per, n_seg);
    const uint32_t *cnt = cand_cnt + size_t(qn) * seg_stride;
    const uint64_t *segs = cand + size_t(qn) * seg_stride * kSegCap;
    constexpr uint32_t kShort = 16;
    static_assert(PARTS == 1 || PARTS * kShort == kSegCap, "a segment is dealt out whole");
    const uint32_t at0 = PARTS > 1 ? t % PARTS * kShort : 0u;
    // One segment per thread (the usual case): its head is requested together with its count, not
    // after it -- the segment's memory is there whatever the count says.
    const bool one_each = PARTS > 1 || per == 1;
    uint64_t head[kShort];
#pragma unroll
    for (uint32_t e = 0; e < kShort; ++e) head[e] = 0ull;
    uint32_t mine = 0;
    if (one_each) {
        if (s0 < s1) {
            const uint64_t *src = segs + size_t(s0) * kSegCap + at0;
            const uint32_t c = cnt[s0];
#pragma unroll
            for (uint32_t e = 0; e < kShort; ++e) head[e] = src[e];
            if (c > kSegCap) any_full = 1u;
            mine = min(c, uint32_t(kSegCap));
            if (PARTS > 1) mine = min(mine - min(mine, at0), kShort);
            if (mine > kShort) any_long = 1u;
        }
    } else {
        for (uint32_t sg = s0; sg < s1; ++sg) {
            const uint32_t c = cnt[sg];
            if (c > kSegCap) any_full = 1u;
            mine += min(c, uint32_t(kSegCap));
        }
    }
    // exclusive prefix over the threads, and the total
    uint32_t incl = mine;
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t v = __shfl_up(incl, off);
        if (lane >= uint32_t(off)) incl += v;
    }
    if (lane == 63u) sh.w_sum[wv] = incl;
    __syncthreads();
    uint32_t base = incl - mine, total = 0;
    for (uint32_t w = 0; w < W; ++w) { if (w < wv) base += sh.w_sum[w]; total += sh.w_sum[w]; }
    const bool too_many = total > uint32_t(kFinalCap);
    // A sampling level whose candidates did not all fit yields its floor from the subset that was
    // kept: a valid floor, but possibly far below the k_floor-th best of the level.  The flag lets
    // the caller's conditional launches repeat the level from that floor, which then fits.
    if (sampling && level_over != nullptr && t == 0 && (too_many || any_full)) *level_over = 1u;
    // A final pass whose candidates did not fit: flag 1 = the caller repeats the full scan for this
    // query with the raised floor written below (the k_floor-th best of what was kept -- real
    // slots, so a valid lower bound of the true k-th best, and above the floor that let too many
    // through); flag 2 = straight to the exact path (no such floor: fewer than k_eff candidates,
    // or the caller takes no raised floors).
    bool raising = false;
    if (!sampling) {
        const bool redo = too_many || any_full || total < uint32_t(k_eff);
        raising = redo && raise_out != nullptr && total >= uint32_t(k_eff);
        if constexpr (GUESSED) {
            // (floors that were guessed: a query that too few rows reached is repeated from an open one)
            const bool missed = passed != nullptr && !too_many && !any_full && total < uint32_t(k_eff);
            if (t == 0 && missed && raise_out != nullptr) raise_out[qn] = kTauInit;
            if (t == 0 && (redo || passed == nullptr)) overflow[qn] = redo ? (raising || (missed && raise_out != nullptr) ? 1u : 2u) : 0u;
        } else if (t == 0) {
            overflow[qn] = redo ? (raising ? 1u : 2u) : 0u;
        }
        if (redo && !raising) return;
    }
    // (the last query's workgroup is among the last to end)
    auto stamp_end = [&]() {
        if (stamp != nullptr && sampling && qn + 1 == int(gridDim.x) && t == 0) *stamp = wall_clock64();
    };
    if (sampling && total < uint32_t(k_eff)) {
        // Too few allowed slots reached the floor in this sample.  The floor of the level before
        // (k_floor scanned slots reach it) is still a valid lower bound: it stays.  Only the
        // first level, which reads the standing array of open floors, has none to keep.
        if (t == 0 && !keep_floor) *tau_slot = kTauInit;
        stamp_end();
        return;
    }
    const uint32_t need = (sampling || raising) ? min(uint32_t(k_floor), total) : uint32_t(k_eff);   // leading keys wanted
    const bool held = one_each && any_long == 0u;              // every key sits in a register
    const bool staged = !held && total <= kFinalStage;
    if (staged) {
        // A thread copies a short segment itself; long ones (the first sampling level fills a few
        // segments to the brim) go on a list the waves then share, a key per lane.
        uint32_t pos = base;
        for (uint32_t sg = s0; sg < s1; ++sg) {
            const uint32_t c = one_each ? mine : min(cnt[sg], uint32_t(kSegCap));
            if (c <= kShort) {
                const uint64_t *src = segs + size_t(sg) * kSegCap;
                uint64_t v[kShort];
#pragma unroll
                for (uint32_t e = 0; e < kShort; ++e) v[e] = one_each ? head[e] : (e < c ? src[e] : 0ull);
#pragma unroll
                for (uint32_t e = 0; e < kShort; ++e)
                    if (e < c) stage[pos + e] = v[e];
            } else {
                const uint32_t i = atomicAdd(&long_n, 1u);
                long_seg[i] = sg;
                long_pos[i] = pos;
                long_cnt[i] = c;
            }
            pos += c;
        }
        __syncthreads();
        for (uint32_t i = wv; i < long_n; i += W)
            if (lane < long_cnt[i]) stage[long_pos[i] + lane] = segs[size_t(long_seg[i]) * kSegCap + lane];
        __syncthreads();
    }
    // every candidate once, wherever it is
    auto each = [&](auto &&f) {
        if (held) {
#pragma unroll
            for (uint32_t e = 0; e < kShort; ++e)
                if (e < mine) f(head[e]);
        } else if (staged) {
            for (uint32_t i = t; i < total; i += T) f(stage[i]);
        } else {
            for (uint32_t sg = s0; sg < s1; ++sg) {
                const uint32_t c = min(cnt[sg], uint32_t(kSegCap));
                const uint64_t *src = segs + size_t(sg) * kSegCap;
                for (uint32_t e = 0; e < c; ++e) f(src[e]);
            }
        }
    };
    // (256 keys are ranked as they are)
    uint32_t least = 1u;
    const bool counted = total > 256u && need > kSelectTopFew;
    if (total > 256u && !counted) {
        uint32_t most = 0u;
        each([&](uint64_t k) { most = max(most, uint32_t(k >> 32)); });
        least = select_top<T>(most, need, top);
    }
    const uint32_t n = keep_best<T>(each, least, need, kept, n_kept, sh, counted);
    const size_t row = row_map ? size_t(row_map[qn]) : size_t(qn);   // a repeated pass writes to the rows of the queries it repeats
    for (uint32_t i = t; i < n; i += T) {
        const uint64_t k = kept[i];
        const uint32_t rank = rank_in(kept, n, k);
        if (rank >= need) continue;
        float s; uint32_t idx;
        sort_unkey(k, s, idx);
        if (sampling || raising) {
            // the floor: the k_floor-th best sampled score (k_floor >= k_eff steadies the estimate)
            if (rank == need - 1u) {
                const int floor = order_key(s == 0.0f ? -0.0f : s);
                *(sampling ? tau_slot : raise_out + qn) = GUESSED && sampling && keep_floor == 2 ? max(floor, *tau_slot) : floor;
            }
        } else {
            // Of floors that were guessed the highest is the last: what the scans left out lies below it, and the result is whole if its
            // last row does not.  Otherwise that row is a floor k rows do reach.
            if (GUESSED && passed != nullptr && rank == need - 1u) {
                const int last = order_key(s == 0.0f ? -0.0f : s);
                const bool missed = last < passed[(qn / tau_stride_q) * kQTile + qn % tau_stride_q];
                overflow[qn] = missed ? (raise_out != nullptr ? 1u : 2u) : 0u;
                if (missed && raise_out != nullptr) raise_out[qn] = last;
            }
            out_scores[row * k_eff + rank] = s;
            out_idx[row * k_eff + rank] = int64_t(slots != nullptr ? slots[idx] : idx);
        }
    }
    stamp_end();
}

// ===========================================================================
// Bandwidth probes: a pure read (sum) and a plain copy over a caller buffer.
// They calibrate what the scan can hope for on this device and give the
// hardware counters a kernel of known traffic to be scaled against.
// ===========================================================================

// The read probe uses the pattern that reads fastest on this device: every wave takes whole
// 8 KiB runs (eight 16-byte loads per lane in flight), with the non-temporal hint.
__global__ __launch_bounds__(256) void k_probe_read(const uint4 *__restrict__ src, size_t n16, uint32_t *sink) {
    uint32_t acc = 0;
    const size_t wave = (size_t(blockIdx.x) * 256 + threadIdx.x) >> 6, lane = threadIdx.x & 63;
    const size_t n_waves = size_t(gridDim.x) * 4;
    constexpr size_t kRun = 64 * 8;   // 16-byte words per run
    size_t r = wave;
    for (; (r + 1) * kRun <= n16; r += n_waves) {
        uint4 v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = load_stream16(src + r * kRun + u * 64 + lane);
#pragma unroll
        for (int u = 0; u < 8; ++u) acc += v[u].x ^ v[u].y ^ v[u].z ^ v[u].w;
    }
    // the words behind the last whole run
    const size_t done = (n16 / kRun) * kRun;
    for (size_t i = done + size_t(blockIdx.x) * 256 + threadIdx.x; i < n16; i += size_t(gridDim.x) * 256) {
        const uint4 a = src[i];
        acc += a.x ^ a.y ^ a.z ^ a.w;
    }
    if (acc == 0x12345678u) *sink = acc;  // keeps the loads alive; practically never taken
}

__global__ __launch_bounds__(256) void k_probe_copy(const uint4 *__restrict__ src, uint4 *__restrict__ dst, size_t n16) {
    size_t i = size_t(blockIdx.x) * 256 + threadIdx.x;
    const size_t stride = size_t(gridDim.x) * 256;
    for (; i < n16; i += stride) dst[i] = src[i];
}

hipError_t launch_probe(const void *src, void *dst, size_t bytes, int copy, uint32_t *sink, hipStream_t s) {
    const size_t n16 = bytes / 16;
    if (copy) hipLaunchKernelGGL(k_probe_copy, dim3(256 * 8), dim3(256), 0, s, static_cast<const uint4 *>(src),
                                 static_cast<uint4 *>(dst), n16);
    else hipLaunchKernelGGL(k_probe_read, dim3(256 * 8), dim3(256), 0, s, static_cast<const uint4 *>(src), n16, sink);
    return hipGetLastError();
}

// ===========================================================================
// Launchers
// ===========================================================================

hipError_t launch_seq_to_native(const uint8_t *d_seq, uint8_t *d_native, const Geometry &g, size_t first_block,
                                size_t n_blocks, hipStream_t s) {
    if (n_blocks == 0) return hipSuccess;
    hipLaunchKernelGGL(k_seq_to_native, dim3(unsigned(n_blocks * g.nch)), dim3(256), 0, s, d_seq, d_native, g.G,
                       g.nch, first_block);
    return hipGetLastError();
}

hipError_t launch_native_to_seq(const uint8_t *d_native, uint8_t *d_seq, const Geometry &g, size_t first_block,
                                size_t n_blocks, size_t block_bytes, const float *d_scales, hipStream_t s) {
    if (n_blocks == 0) return hipSuccess;
    hipLaunchKernelGGL(k_native_to_seq, dim3(unsigned(n_blocks * g.nch)), dim3(256), 0, s, d_native, d_seq, g.G,
                       g.nch, first_block, block_bytes, d_scales);
    return hipGetLastError();
}

hipError_t launch_append_rows(const uint8_t *d_rows, uint8_t *d_native, const Geometry &g, size_t old_n,
                              size_t n_new, hipStream_t s) {
    const size_t total = n_new * size_t(g.G);
    if (total == 0) return hipSuccess;
    hipLaunchKernelGGL(k_append_rows, dim3(unsigned((total + 255) / 256)), dim3(256), 0, s, d_rows, d_native, g.G,
                       g.nch, old_n, n_new);
    return hipGetLastError();
}

hipError_t launch_move_lane(uint8_t *d_native, float *d_scales, const Geometry &g, size_t src, size_t dst,
                            hipStream_t s) {
    hipLaunchKernelGGL(k_move_lane, dim3(unsigned((g.G + 255) / 256)), dim3(256), 0, s, d_native, d_scales, g.G,
                       g.nch, src, dst);
    return hipGetLastError();
}

hipError_t launch_gather_redo(const float *d_q, const uint32_t *d_rows, const int *d_raised, int dim, int tile_q,
                              size_t n_redo, float *d_q_out, int *d_tau_out, hipStream_t s) {
    if (n_redo == 0) return hipSuccess;
    hipLaunchKernelGGL(k_gather_redo, dim3(unsigned(n_redo)), dim3(256), 0, s, d_q, d_rows, d_raised, dim, tile_q,
                       d_q_out, d_tau_out);
    return hipGetLastError();
}

hipError_t launch_fill_i32(int *p, int v, size_t n, hipStream_t s) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_fill_i32, dim3(unsigned((n + 255) / 256)), dim3(256), 0, s, p, v, n);
    return hipGetLastError();
}

hipError_t launch_lay_tables(const uint32_t *from, uint32_t *to, size_t n, int *floors, int v, size_t n_floors, hipStream_t s) {
    if (n + n_floors == 0) return hipSuccess;
    if (n + n_floors > (size_t(1) << 30)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_lay_tables, dim3(unsigned((n + n_floors + 255) / 256)), dim3(256), 0, s, from, to, uint32_t(n), floors, v, uint32_t(n_floors));
    return hipGetLastError();
}

template <typename K>
static hipError_t allow_lds(K kernel, size_t bytes) {
    if (bytes <= 48 * 1024) return hipSuccess;
    return hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                               int(bytes));
}

static constexpr size_t kLdsBudget = 160 * 1024;

size_t scan_lds_bytes(int mode_p, int nch, int k, int lut_queries) {
    const size_t lists = size_t(k) * kScanThreads * 8 + kQTile * sizeof(int) + (mode_p ? kDecodeBytes : 0);
    if (mode_p) {
        const size_t w = size_t(nch) * 2048;
        return (w + lists <= kLdsBudget ? w : 0) + lists;
    }
    return size_t(nch) * 1024 * lut_queries + lists;
}

// Workgroup size of the append-mode permute-dot scan (sample-then-filter, up to 32 queries).  The
// scan streams fastest with sixteen waves per CU on ONE copy of the query tile's weights in LDS:
// a 1024-thread workgroup of four four-wave groups, each group with a candidate segment of its own
// (the selection kernel reads short segments fastest).  Four-wave workgroups with a copy each (48 KiB
// at 1536 dimensions) reach twelve waves per CU where three copies fit -- one query over 10M x 1536
// bytes of codes at 128 to 1792 dimensions: 0.61-0.93 ms, the large workgroup 0.60-0.91, up to 18 %
// less -- and four waves per CU from 2560 dimensions (0.88 ms against 0.60).  Rows whose weights do
// not fit LDS (beyond 5056 dimensions) read them from global memory in four-wave workgroups.
constexpr int kScanThreadsShared = 4 * kScanThreads;
static int scan_p4_append_threads(int nch) {
    const size_t lds = size_t(nch) * 2048 + kDecodeBytes + (kScanThreadsShared / kScanThreads) * kQTile * sizeof(int);
    return lds <= kLdsBudget ? kScanThreadsShared : kScanThreads;
}

// One attribute, not the whole property record: a search asks several times.
int device_cus(int device) {
    int cus = 0;
    return hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess && cus > 0 ? cus : 256;
}

int scan_grid_blocks(int device, int mode_p, int nch, int k, int nq_tile) {
    const int cus = device_cus(device);
    if (mode_p && k == 0 && scan_p4_append_threads(nch) != kScanThreads)           // (k = 0: the append-mode scans)
        return cus * (kScanThreadsShared / kScanThreads);                         // one workgroup per CU, counted in four-wave groups
    const size_t lds = scan_lds_bytes(mode_p, nch, k, nq_tile);
    int per_cu = int(kLdsBudget / (lds ? lds : 1));
    if (per_cu < 1) per_cu = 1;
    if (per_cu > 4) per_cu = 4;
    // (the instances that read four or eight chunks per burst hold three waves per SIMD: a fourth
    // workgroup per CU would only wait for a place and run as a tail)
    if (mode_p && k == 0 && nch % 4 == 0 && per_cu > 3) per_cu = 3;
    return cus * per_cu;
}

hipError_t launch_scan_p4(const ScanArgs &args, int grid, int mode, hipStream_t s) {
    ScanArgs a = args;
    const int threads = (mode == kModeAppend || mode == kModeBest) ? scan_p4_append_threads(a.nch) : kScanThreads;
    const int groups = threads / kScanThreads;
    a.vgrid = uint32_t(grid);                        // `grid` counts four-wave groups
    const int wgs = (grid + groups - 1) / groups;
    const size_t w = size_t(a.nch) * 2048;
    const size_t lists = kDecodeBytes + groups * kQTile * sizeof(int) + (mode != kModeLists ? 0 : size_t(a.k) * kScanThreads * 8);
    const bool w_lds = w + lists <= kLdsBudget;
    const size_t lds = (w_lds ? w : 0) + lists;
    // (append-mode scans whose weights fit LDS take the large workgroup; four-wave ones read them from global memory)
    if ((mode == kModeAppend || mode == kModeBest) && groups == 1 && w_lds) return hipErrorInvalidValue;
    hipError_t e = hipSuccess;
#define TV_LAUNCH_P4_T(U, D, W, T)                                                              \
    do {                                                                                        \
        e = allow_lds(k_scan_p4<U, D, W, T>, lds);                                              \
        if (e != hipSuccess) return e;                                                          \
        hipLaunchKernelGGL((k_scan_p4<U, D, W, T>), dim3(wgs), dim3(T), lds, s, a);             \
    } while (0)
#define TV_LAUNCH_P4(U, D, W) TV_LAUNCH_P4_T(U, D, W, kScanThreads)
// (sixteen waves per CU leave a wave 128 registers: the large workgroup reads bursts of four chunks
// at most, and its floorless level -- a short launch either way -- of two)
#define TV_PICK_P4(U)                                                                           \
    do {                                                                                        \
        if (groups > 1) { if (mode == kModeAppend) TV_LAUNCH_P4_T((U > 4 ? 4 : U), kModeAppend, true, kScanThreadsShared); else TV_LAUNCH_P4_T((U > 2 ? 2 : U), kModeBest, true, kScanThreadsShared); } \
        else if (mode == kModeDump) { if (w_lds) TV_LAUNCH_P4(U, kModeDump, true); else TV_LAUNCH_P4(U, kModeDump, false); } \
        else if (mode == kModeAppend) TV_LAUNCH_P4(U, kModeAppend, false);                      \
        else if (mode == kModeBest) TV_LAUNCH_P4(U, kModeBest, false);                          \
        else { if (w_lds) TV_LAUNCH_P4(U, kModeLists, true); else TV_LAUNCH_P4(U, kModeLists, false); } \
    } while (0)
    if (a.nch % 8 == 0) TV_PICK_P4(8);          // 8 KiB per wave in flight: +3 % over 4 at 24 chunks, 12 is slower
    else if (a.nch % 4 == 0) TV_PICK_P4(4);
    else if (a.nch % 2 == 0) TV_PICK_P4(2);
    else TV_PICK_P4(1);
#undef TV_PICK_P4
#undef TV_LAUNCH_P4
#undef TV_LAUNCH_P4_T
    return hipGetLastError();
}

// Batched append-mode launches for up to batched_tiles()*32 queries (a.nq_tile counts queries,
// a.tables holds ceil(nq/32) consecutive tiles).  Two kernels: when the weights of at least two
// tiles fit LDS together they stay resident (k_scan_p4_multi); wider rows stream four tiles'
// weights through LDS in slices (k_scan_p4_batched).

// Query tiles whose weights fit LDS together, capped at 4.
// LDS of the resident-weights kernel beside nt tiles' weights: the byte table, the candidate
// counters and the block counter, 24 bytes of constants per query, a block's row scales per wave.
static size_t multi_fixed_lds(int nt) { return kDecodeBytes + (size_t(nt) * kQTile + 4) * sizeof(uint32_t) + size_t(nt) * kQTile * 24 + 16 * 32 * sizeof(float); }
static int resident_tiles(int nch) {
    const size_t per_tile = size_t(nch) * 2048;
    for (int nt = 4; nt >= 1; --nt)
        if (nt * per_tile + multi_fixed_lds(nt) <= kLdsBudget) return nt;
    return 0;
}

// Waves per workgroup of the resident-weights kernel and code bytes per lane and chunk it decodes
// through the table.  Four tiles: three waves per SIMD (measured best of 512 / 768 / 1024 threads),
// eight table bytes.  Two tiles fit 128 registers and run four waves per SIMD (2 to 7 % faster per
// launch, 256 to 2048 dimensions).  Three tiles fit them with four table bytes -- fewer reads in
// flight, fewer registers; by itself that split is 1 % slower -- and gain 1 to 3 % from the fourth wave.
template <int NT> constexpr int kMultiTableBytes = NT == 3 ? 4 : 8;
template <int NT> constexpr int kMultiThreads = NT <= 3 ? 1024 : 768;
constexpr int kStreamTiles = 4, kStreamBlocksPerWave = 2, kStreamSliceChunks = 2, kStreamOccupancy = 2;

// The resident-weights kernel reads its weights in k_scan_p4's split order.
bool batched_weights_split(int nch) { return resident_tiles(nch) >= 2; }

int batched_tiles(int nch) {
    const int nt = resident_tiles(nch);
    if (nt >= 2) return nt;
    return nch % kStreamSliceChunks == 0 ? kStreamTiles : 0;
}

int batched_grid_blocks(int device, int nch) {
    const int cus = device_cus(device);
    if (resident_tiles(nch) >= 2) {
        const size_t lds = size_t(resident_tiles(nch)) * nch * 2048 + multi_fixed_lds(resident_tiles(nch));
        const int per_cu = int(kLdsBudget / lds);
        return cus * (per_cu < 1 ? 1 : (per_cu > 2 ? 2 : per_cu));
    }
    return cus * kStreamOccupancy;
}

template <int NT, int U>
static hipError_t launch_multi_u(const ScanArgs &a, int grid, hipStream_t s) {
    constexpr int LB = kMultiTableBytes<NT>;
    const size_t lds = size_t(NT) * a.nch * 2048 + multi_fixed_lds(NT);
    hipError_t e = allow_lds(k_scan_p4_multi<NT, U, kMultiThreads<NT>, LB>, lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((k_scan_p4_multi<NT, U, kMultiThreads<NT>, LB>), dim3(grid), dim3(kMultiThreads<NT>), lds, s, a);
    return hipGetLastError();
}

template <int NT>
static hipError_t launch_multi(const ScanArgs &a, int grid, hipStream_t s) {
    // (four tiles' accumulators and four-chunk bursts together do not fit the 168 registers three
    // waves per SIMD leave: the compiler would spill, which the hand-placed waits cannot allow)
    if constexpr (NT < 4) {
        if (a.nch % 4 == 0) return launch_multi_u<NT, 4>(a, grid, s);
    }
    if (a.nch % 2 == 0) return launch_multi_u<NT, 2>(a, grid, s);
    return launch_multi_u<NT, 1>(a, grid, s);
}

hipError_t launch_scan_p4_batched(const ScanArgs &a, int grid, hipStream_t s) {
    // the instance for the tiles the launch really has: a third resident tile of padding queries
    // would cost its MFMAs all the same
    const int tiles = std::max(2, (a.nq_tile + kQTile - 1) / kQTile);
    switch (std::min(resident_tiles(a.nch), tiles)) {
        case 4: return launch_multi<4>(a, grid, s);
        case 3: return launch_multi<3>(a, grid, s);
        case 2: return launch_multi<2>(a, grid, s);
        default: break;
    }
    constexpr int MW = kStreamBlocksPerWave, KC = kStreamSliceChunks, OCC = kStreamOccupancy;
    if (a.nch % KC != 0 || a.nq_tile > kStreamTiles * kQTile) return hipErrorInvalidValue;
    auto launch = [&](auto ntc) -> hipError_t {
        constexpr int NT = decltype(ntc)::value;
        const size_t lds = size_t(2) * NT * KC * 2048 + NT * kQTile * sizeof(uint32_t);
        hipError_t e = allow_lds(k_scan_p4_batched<NT, MW, KC, OCC>, lds);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL((k_scan_p4_batched<NT, MW, KC, OCC>), dim3(grid), dim3(kScanThreads), lds, s, a);
        return hipGetLastError();
    };
    static_assert(kStreamTiles == 4, "one instance per tile count up to the stream's four");
    switch (tiles) {        // as above: no tile of padding queries
        case 2: return launch(IntC<2>{});
        case 3: return launch(IntC<3>{});
        default: return launch(IntC<4>{});
    }
}

hipError_t launch_merge(const float *part_scores, const uint32_t *part_idx, const int *part_cnt, int total_threads,
                        int qmod, int k, int k_eff, int nq_tile, float *out_scores, int64_t *out_idx,
                        int *out_tau, hipStream_t s) {
    if (nq_tile == 0 || k_eff == 0) return hipSuccess;
    int sort_n = 2;
    while (sort_n < 256 * k) sort_n <<= 1;
    const size_t lds = size_t(k) * 256 * 8 + size_t(sort_n) * 8;
    hipError_t e = allow_lds(k_merge, lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_merge, dim3(nq_tile), dim3(256), lds, s, part_scores, part_idx, part_cnt, total_threads,
                       qmod, k, k_eff, sort_n, out_scores, out_idx, out_tau);
    return hipGetLastError();
}

hipError_t launch_final(const uint64_t *cand, const uint32_t *cand_cnt, uint32_t n_seg, uint32_t seg_stride,
                        int k_eff, int k_floor, int nq, float *out_scores, int64_t *out_idx, uint32_t *overflow,
                        int *tau_out, int tau_stride_q, int keep_floor, int *raise_out, const uint32_t *row_map,
                        uint32_t *level_over, uint32_t *clear_flag, const uint32_t *run_if, const uint32_t *slots, uint64_t *stamp, double longest, hipStream_t s, const int *passed) {
    if (nq == 0 || k_eff == 0) return hipSuccess;
    auto launch = [&](auto kernel, unsigned threads) {
        hipLaunchKernelGGL(kernel, dim3(nq), dim3(threads), 0, s, cand, cand_cnt, n_seg, seg_stride, k_eff, k_floor, out_scores,
                           out_idx, overflow, tau_out, tau_stride_q, keep_floor, raise_out, row_map, level_over, clear_flag, run_if, slots, stamp, passed);
    };
    if (passed != nullptr || keep_floor == 2) {
        if (n_seg <= 256) launch(k_final<256, 1, true>, 256);
        else if (n_seg <= 512) launch(k_final<512, 1, true>, 512);
        else launch(k_final<1024, 1, true>, 1024);
    } else if (n_seg <= 256 && nq == 1 && longest > kFinalLongest) launch(k_final<1024, 4, false>, 1024);
    else if (n_seg <= 256) launch(k_final<256, 1, false>, 256);
    else if (n_seg <= 512) launch(k_final<512, 1, false>, 512);
    else launch(k_final<1024, 1, false>, 1024);
    return hipGetLastError();
}

}  // namespace tv
