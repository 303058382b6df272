// Scan, score mode L with the u32 epilogue, append mode, batches: the table lookups as a sparse
// contraction on the matrix unit.
//
// acc = sum over nibbles of lut[position][nibble] is, per position, the dot product of a one-hot
// vector (the nibble) with the position's table: a contraction of length 16 per nibble (8 for
// 3-bit codes, whose nibbles stay below 8).  Dense int8 MFMAs would multiply zeros for most of
// it, but a one-hot vector is within the matrix unit's 4:2 structured sparsity: of every four
// consecutive entries at most two are non-zero.  v_smfmac_i32_32x32x64_i8 takes A in that form --
// two stored values per group of four and a 2-bit position for each -- and contracts 64 entries
// in the time a dense instruction takes for 32.  An entry of a nibble's table is selected by
// a 1 in one stored slot of one group, with the group's positions set to (0, 1) or (2, 3); every
// other stored value is zero.  The sums are the same integers
// the lookups would give, in any order.
//
// A operands are built on the vector ALU from the raw codes: per code byte two shifts of a one
// and a byte permute, shared by the NT query tiles the wave works on; B operands -- the tables,
// laid out by k_prep_lut in the order the instruction wants them -- pass through LDS, each
// read feeding the wave's BLK blocks.  A workgroup of eight waves takes 8 * BLK blocks and one
// group of NT query tiles through the whole row, chunk by chunk; the launch's groups work side by
// side, each on its share of the workgroups (dealt so that with eight or sixteen groups an XCD sees
// one or two of them and their tables stay in its L2), and each reads all of the codes.
//
// What bounds it: 192 sparse instructions per (block, tile) at 1536 dimensions and 2 bits, 1.26e14
// stored operations for 10M rows and 1024 queries.  At 32 clocks each they take 32 ms on a matrix unit that does
// nothing else, at the 1.87 GHz the chip holds under them; the scan takes 44 ms, the matrix unit 72 % busy and the
// vector ALU 48 % (by counters), against 64 passes of 1.5 ms of the table lookups, which are bound by LDS reads.  Two
// tiles and four blocks per wave: the operands of a block are built once for two instructions, every
// LDS read feeds four, and the sums (128 registers) still leave room for two waves per SIMD.
//
// Integers and float epilogue: turbovec/src/search.rs:2856-2994, 1174-1177, term for term.
#include <algorithm>

#include "tv_device.h"
#include "tv_internal.h"

namespace tv {

typedef int v8i __attribute__((ext_vector_type(8)));

constexpr int kMxThreads = 512, kMxWaves = kMxThreads / 64;
constexpr int kMxRing = 4;       // LDS slots, one slice of the tables each

__device__ __forceinline__ void mx_dma16(uint32_t lds_addr, const void *sbase, uint32_t lane16) {
    const uint32_t u = uint32_t(__builtin_amdgcn_readfirstlane(int(lds_addr)));
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(u), "v"(lane16), "s"(sbase) : "memory", "m0");
}
__device__ __forceinline__ void mx_load16(u32x4 &dst, const void *sbase, uint32_t lane16) {
    asm volatile("global_load_dwordx4 %0, %1, %2" : "=&v"(dst) : "v"(lane16), "s"(sbase));
}

__device__ __forceinline__ void mx_load4(float &dst, const void *sbase, uint32_t lane4) {
    asm volatile("global_load_dword %0, %1, %2" : "=&v"(dst) : "v"(lane4), "s"(sbase));
}
// Waits for a requested register (at most N younger requests outstanding) and moves its contents on.
// One statement, so that the move cannot come before the wait: tied to a variable that lives on
// around a loop, the wait alone may have its operand copied to the loop's register ahead of it.
template <int N>
__device__ __forceinline__ void mx_take(u32x4 &to, const u32x4 &from) {
    uint32_t x, y, z, w;
    asm volatile("s_waitcnt vmcnt(%8)\n\tv_mov_b32 %0, %4\n\tv_mov_b32 %1, %5\n\tv_mov_b32 %2, %6\n\tv_mov_b32 %3, %7"
                 : "=&v"(x), "=&v"(y), "=&v"(z), "=&v"(w) : "v"(from.x), "v"(from.y), "v"(from.z), "v"(from.w), "n"(N));
    to = u32x4{x, y, z, w};
}
template <int N>
__device__ __forceinline__ void mx_take(float &to, const float &from) {
    asm volatile("s_waitcnt vmcnt(%2)\n\tv_mov_b32 %0, %1" : "=&v"(to) : "v"(from), "n"(N));
}

// What a dword of raw codes (four byte-groups of one vector) turns into before its A operands are
// formed, four bytes at a time: per nibble the bit a one is shifted to, and the byte of 2-bit
// positions its groups get.
struct MxPrep {
    uint32_t sh, sl;        // shift of the high / low nibble's one: 8 * its stored slot
    uint32_t ih, il;        // positions of the high / low nibble's groups: 0x44 = (0, 1), 0xee = (2, 3)
};
template <int ENT>
__device__ __forceinline__ MxPrep mx_prep(uint32_t x) {
    constexpr uint32_t slot = ENT == 16 ? 0x38383838u : 0x18181818u;
    constexpr int top = ENT == 16 ? 3 : 2;
    MxPrep r;
    r.sh = (x >> 1) & slot;
    r.sl = (x << 3) & slot;
    asm("" : "+v"(r.sh), "+v"(r.sl));      // (opaque: shifted and masked again per byte otherwise)
    r.ih = __builtin_amdgcn_perm(0u, 0x0000ee44u, (x >> (4 + top)) & 0x01010101u);
    r.il = __builtin_amdgcn_perm(0u, 0x0000ee44u, (x >> top) & 0x01010101u);
    return r;
}
// The A operand of step J of the lane's 16 code bytes: stored values and positions.
template <int ENT, int J>
__device__ __forceinline__ void mx_operand(const MxPrep &m, v4i &a, int &idx) {
    if constexpr (ENT == 16) {
        constexpr int e = J & 3;
        const uint64_t hi = 1ull << ((m.sh >> (8 * e)) & 63u), lo = 1ull << ((m.sl >> (8 * e)) & 63u);
        a[0] = int(uint32_t(hi)); a[1] = int(uint32_t(hi >> 32));
        a[2] = int(uint32_t(lo)); a[3] = int(uint32_t(lo >> 32));
        idx = int(__builtin_amdgcn_perm(m.il, m.ih, uint32_t((4 + e) << 24 | (4 + e) << 16 | e << 8 | e)));
    } else {
        constexpr int e = (2 * J) & 3;
        a[0] = int(1u << ((m.sh >> (8 * e)) & 31u));
        a[1] = int(1u << ((m.sl >> (8 * e)) & 31u));
        a[2] = int(1u << ((m.sh >> (8 * e + 8)) & 31u));
        a[3] = int(1u << ((m.sl >> (8 * e + 8)) & 31u));
        idx = int(__builtin_amdgcn_perm(m.il, m.ih, uint32_t((5 + e) << 24 | (1 + e) << 16 | (4 + e) << 8 | e)));
    }
}

// Per query, in LDS: a score is ((f32(acc) * qs) + qb) * row_scale; ta, tb give the integer bound
// below which no accumulator can pass (the same derivation and slack as the permute-dot kernel's:
// 1e-5 relative and 2 units, against a few 2^-24 of rounding).
struct MxQuery {
    float ta, tb, qs, qb, tau;
};

// sub (a power of two up to 8): candidate segments a workgroup keeps per query, its waves sharing
// them out.  BEST: no candidates, every (block, query)'s best score (tv_kernels6.hip); an instance of its own, as the
// branch costs the append form 1.4 %.
template <int ENT, int NT, int BLK, bool BEST>
__global__ __launch_bounds__(kMxThreads, 2) void k_scan_lut_mx(ScanArgs a, uint32_t groups, uint32_t sub) {
    extern __shared__ __align__(16) uint8_t smem[];
    if (launch_switched_off(a.run_if)) return;
    constexpr int kSteps = mx_steps(ENT);
    constexpr int kS = kSteps < 16 / NT ? kSteps : 16 / NT;     // steps per slice: a ring slot holds 32 KiB at most
    constexpr int kSpc = kSteps / kS;                           // slices per chunk
    constexpr int kTileSlice = kS * 2048;                       // bytes of one tile in a slice
    constexpr int kSlot = NT * kTileSlice;
    constexpr int kPieces = kSlot / (kMxWaves * 1024);          // direct-to-LDS loads per wave and slice
    static_assert(kSlot % (kMxWaves * 1024) == 0 && kTileSlice % 1024 == 0, "a slice is dealt evenly");
    constexpr int kQ = NT * kQTile;
    const int nch = a.nch;
    const uint32_t group = blockIdx.x % groups, wg = blockIdx.x / groups, wgs = gridDim.x / groups;
    const int n_tiles = (a.nq_tile + kQTile - 1) / kQTile;
    const int q0 = int(group) * kQ;
    MxQuery *sq = reinterpret_cast<MxQuery *>(smem + kMxRing * kSlot);
    uint32_t *scnt = reinterpret_cast<uint32_t *>(sq + kQ);                  // [sub][kQ] candidates appended
    float *s_vs = reinterpret_cast<float *>(scnt + 8 * kQ);                  // [waves][BLK][32] row scales, NaN where not allowed
    uint32_t *snext = reinterpret_cast<uint32_t *>(s_vs + kMxWaves * BLK * 32);
    uint32_t *s_over = snext + 1;                                            // segments of this workgroup that are full
    const uint32_t lds_b = uint32_t(reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) uint8_t *)smem));

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t lane16 = uint32_t(lane) * 16, lane4 = uint32_t(lane & 31) * 4;
    const uint32_t my_sub = uint32_t(wave) & (sub - 1u);
    for (int i = tid; i < kQ; i += kMxThreads) {
        const int q = q0 + i;
        const bool act = q < a.nq_tile;
        const float qs = act ? a.qscale[q] : 0.0f, qb = act ? a.qbias[q] : 0.0f;
        const float tau = act ? order_unkey(a.gtau[q]) : __int_as_float(0x7fc00000);
        const float inf = __int_as_float(0x7f800000);
        const bool bounded = tau >= 1e-30f && tau <= 1e30f && qs >= 1e-30f && qs <= 1e30f && fabsf(qb) <= 1e30f && tau / qs < inf;
        const float rb = qb / qs;
        sq[i] = MxQuery{!act ? inf : bounded ? (tau / qs) * (1.0f - 1e-5f) : -inf,
                        act && bounded ? rb + 1e-5f * fabsf(rb) + 2.0f : 0.0f, qs, qb, tau};
    }
    for (int i = tid; i < 8 * kQ; i += kMxThreads) scnt[i] = 0u;
    if (tid < 5) snext[tid] = 0u;                                            // claims, full segments, three round flags
    __syncthreads();

    const uint32_t step = a.b_step;
    const uint32_t nj = (a.n_blocks + step - 1) / step;
    const int n_slices = nch * kSpc;

    // The group's tables are a periodic stream of slices (steps s * kS .. of the row, for each of its
    // tiles), kept three ahead: in the middle of slice g every wave waits for its own pieces of slice
    // g + 1, meets the others -- after which g + 1 is whole and g - 1 read by nobody -- and requests
    // g + 3 into the slot of g - 1.  (Tiles past the last are stand-ins: the last tile again.)
    static_assert(kTileSlice % (kMxWaves * 1024) == 0, "a round of pieces stays within one tile");
    const uint8_t *tsrc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
        tsrc[t] = a.tables + size_t(min(int(group) * NT + t, n_tiles - 1)) * (size_t(nch) * kSteps * 2048) + size_t(wave) * 1024;
    int req_slice = 0, req_slot = 0;
    auto request_next = [&]() {
        const uint32_t dst = lds_b + uint32_t(req_slot) * kSlot + uint32_t(wave) * 1024;
#pragma unroll
        for (int p = 0; p < kPieces; ++p) {
            constexpr int per_tile = kTileSlice / (kMxWaves * 1024);
            mx_dma16(dst + uint32_t(p) * (kMxWaves * 1024),
                     tsrc[p / per_tile] + (uint32_t(req_slice) * kTileSlice + uint32_t(p % per_tile) * (kMxWaves * 1024)), lane16);
        }
        req_slice = req_slice + 1 == n_slices ? 0 : req_slice + 1;
        req_slot = (req_slot + 1) & (kMxRing - 1);
    };
    // `younger`: vector-memory requests after those of slice g + 1.  The bare barrier is enough: what a
    // wave has read of slice g - 1 it has also waited for, and nothing else passes between waves here.
    auto hand_over = [&](auto younger) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(decltype(younger)::value) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        request_next();
    };

    // Blocks of this workgroup: m * wgs + wg for m = 0, 1, ..., dealt to the waves as they ask, BLK at a
    // time (under a mask one by one, blocks without an allowed row skipped); nj stands for none.
    uint32_t blk[BLK];
    auto claim = [&](uint32_t (&to)[BLK], bool stop) -> uint32_t {      // how many it got
        uint32_t got = 0;
        auto ask = [&](uint32_t count) -> uint32_t {
            uint32_t m = 0;
            if (lane == 0) m = atomicAdd(snext, count);
            return uint32_t(__builtin_amdgcn_readfirstlane(int(m)));
        };
        const uint32_t m0 = (stop || a.mask != nullptr) ? 0u : ask(uint32_t(BLK));
#pragma unroll
        for (int k = 0; k < BLK; ++k) {
            uint32_t j = stop ? nj : min((m0 + uint32_t(k)) * wgs + wg, nj);
            if (!stop && a.mask != nullptr) {
                for (;;) {
                    j = ask(1u) * wgs + wg;
                    if (j >= nj) { j = nj; break; }
                    const uint32_t b = j * step;
                    if (uint32_t(a.mask[b >> 1] >> ((b & 1) * 32)) != 0u) break;
                }
            }
            to[k] = uint32_t(__builtin_amdgcn_readfirstlane(int(j)));      // (uniform, and known to be)
            got += to[k] < nj ? 1u : 0u;
        }
        return uint32_t(__builtin_amdgcn_readfirstlane(int(got)));
    };
    auto block_of = [&](uint32_t j) { return uint32_t(__builtin_amdgcn_readfirstlane(int(j < nj ? j * step : 0u))); };
    // Row scales of a block into this wave's LDS rows, NaN where a row may not be returned; the largest
    // one's reciprocal for the accumulator bound.
    int inv_vmax[BLK];
    uint32_t odd_blocks = 0u;                               // bit k: block k has a row scale no bound can be taken from
    auto take_scales = [&](const float (&raw_sc)[BLK]) {
        odd_blocks = 0u;
        int el = lane;                                      // (opaque, as in the epilogue)
        asm volatile("" : "+v"(el));
#pragma unroll
        for (int k = 0; k < BLK; ++k) {
            const uint32_t b = block_of(blk[k]), slot = b * 32u + uint32_t(el & 31);
            bool ok = blk[k] < nj && slot < a.n;
            if (ok && a.mask != nullptr) ok = (uint32_t(a.mask[b >> 1] >> ((b & 1) * 32)) >> (el & 31)) & 1u;
            const float sc = ok ? raw_sc[k] : __int_as_float(0x7fc00000);
            if (el < 32) s_vs[(wave * BLK + k) * 32 + el] = sc;
            float vmax = ok ? sc : 0.0f;
            const bool odd = ok && !(sc >= 0.0f && sc <= 1e30f);
#pragma unroll
            for (int d = 16; d >= 1; d >>= 1) vmax = fmaxf(vmax, __shfl_xor(vmax, d));
            if (__any(odd || (vmax > 0.0f && vmax < 1e-30f))) odd_blocks |= 1u << k;
            inv_vmax[k] = __builtin_amdgcn_readfirstlane(__float_as_int(1.0f / vmax));
        }
    };

    // "Does any wave have blocks in round r?" is flag[r % 3], set before and read after a barrier that
    // every wave passes in the last slice of round r - 1; the next round's is cleared in between.
    uint32_t *flag = snext + 2;
    uint32_t has = claim(blk, false);
    if (has != 0u && lane == 0) flag[0] = 1u;
    request_next();
    request_next();
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kPieces) : "memory");
    __syncthreads();
    request_next();
    // (read as LDS, not through a generic pointer: a flat load is counted by both memory counters and
    // the compiler would wait for every table request in flight before it)
    auto lds_at = [&](const uint32_t *p) -> uint32_t {
        const uint32_t at = lds_b + uint32_t(reinterpret_cast<const uint8_t *>(p) - smem);
        return uint32_t(__builtin_amdgcn_readfirstlane(int(*reinterpret_cast<const volatile __attribute__((address_space(3))) uint32_t *>(uintptr_t(at)))));
    };
    uint32_t more = lds_at(flag);
    uint32_t round_no = 0;
    int use_slot = 0;
    u32x4 cur[BLK];
    float sc[BLK];
    {
        u32x4 nxt[BLK];
        float nsc[BLK];
#pragma unroll
        for (int k = 0; k < BLK; ++k) {
            mx_load4(nsc[k], a.scales + size_t(block_of(blk[k])) * 32, lane4);
            mx_load16(nxt[k], a.codes + size_t(block_of(blk[k])) * uint32_t(nch * 1024), lane16);
        }
#pragma unroll
        for (int k = 0; k < BLK; ++k) { mx_take<0>(cur[k], nxt[k]); mx_take<0>(sc[k], nsc[k]); }
    }

    while (more != 0u) {
        uint32_t nblk[BLK];
#pragma unroll
        for (int k = 0; k < BLK; ++k) nblk[k] = nj;
        uint32_t nhas = 0u;
        take_scales(sc);
        // In the round's last chunk: the next round's blocks.  Every segment of this workgroup full: every
        // query of the group is certain to be repeated from a raised floor and nothing more would be
        // kept, so no further blocks are taken.
        auto look_ahead = [&]() {
            const bool futile = lds_at(s_over) >= uint32_t(min(kQ, a.nq_tile - q0)) * sub;
            nhas = claim(nblk, futile);
            if (tid == 0) flag[(round_no + 2) % 3u] = 0u;
            if (nhas != 0u && lane == 0) flag[(round_no + 1) % 3u] = 1u;
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");             // there before this wave meets the barrier
        };
        if (has == 0u) {      // (for good: there is nothing left to claim)
            for (int s = 0; s < n_slices; ++s) {
                if (s == n_slices - kSpc) look_ahead();
                hand_over(IntC<kPieces>{});
            }
            use_slot = (use_slot + n_slices) & (kMxRing - 1);
        } else {
        v16i acc[BLK][NT];
#pragma unroll
        for (int k = 0; k < BLK; ++k) {
#pragma unroll
            for (int t = 0; t < NT; ++t) acc[k][t] = v16i{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
        }
        // B operands one step ahead of their use, in two sets of registers
        v4i bl[2][NT][2];
        auto fetch = [&](auto set, auto step_no, const v4i *bt) {
            constexpr int js = decltype(step_no)::value;
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                bl[decltype(set)::value][t][0] = bt[t * (kTileSlice / 16) + js * 128];
                bl[decltype(set)::value][t][1] = bt[t * (kTileSlice / 16) + js * 128 + 64];
            }
        };
        fetch(IntC<0>{}, IntC<0>{}, reinterpret_cast<const v4i *>(smem + use_slot * kSlot) + lane);
        for (int c = 0; c < nch; ++c) {
            // the next chunk's codes -- in the last chunk the next round's first, and its row scales
            const bool last = c + 1 == nch;
            // (always requested, needed or not: the counts waited for are fixed)
            if (last) look_ahead();
            u32x4 nxt[BLK];
            float nsc[BLK];
#pragma unroll
            for (int k = 0; k < BLK; ++k) {
                const uint32_t from = blk[k] ^ ((blk[k] ^ nblk[k]) & (last ? ~0u : 0u));     // (a choice of values: the arrays stay in registers)
                mx_load16(nxt[k], a.codes + size_t(block_of(from)) * uint32_t(nch * 1024) + (last ? 0u : uint32_t(c + 1) * 1024u), lane16);
                mx_load4(nsc[k], a.scales + size_t(block_of(from)) * 32, lane4);
            }
            MxPrep pr[BLK];
            static_for<kSpc>([&](auto pp) {
                constexpr int part = decltype(pp)::value;
                const v4i *bt = reinterpret_cast<const v4i *>(smem + use_slot * kSlot) + lane;
                use_slot = (use_slot + 1) & (kMxRing - 1);
                const v4i *bn = reinterpret_cast<const v4i *>(smem + use_slot * kSlot) + lane;
                static_for<kS>([&](auto jj) {
                    constexpr int js = decltype(jj)::value, j = part * kS + js, set = j & 1;
                    constexpr int dword = ENT == 16 ? j / 4 : j / 2;
                    if constexpr (js == kS / 2) hand_over(IntC<(part < 2 ? kPieces + 2 * BLK : kPieces)>{});
                    __builtin_amdgcn_sched_barrier(0x6);
                    if constexpr (js + 1 < kS) fetch(IntC<1 - set>{}, IntC<js + 1>{}, bt);
                    else fetch(IntC<1 - set>{}, IntC<0>{}, bn);
                    __builtin_amdgcn_sched_barrier(0x6);
                    if constexpr (ENT == 16 ? j % 4 == 0 : j % 2 == 0) {
#pragma unroll
                        for (int k = 0; k < BLK; ++k) pr[k] = mx_prep<ENT>(cur[k][dword]);
                    }
                    v8i b[NT];
#pragma unroll
                    for (int t = 0; t < NT; ++t) {
                        const v4i b0 = bl[set][t][0], b1 = bl[set][t][1];
                        b[t] = v8i{b0[0], b0[1], b0[2], b0[3], b1[0], b1[1], b1[2], b1[3]};
                    }
#pragma unroll
                    for (int k = 0; k < BLK; ++k) {
                        v4i av;
                        int idx;
                        mx_operand<ENT, j>(pr[k], av, idx);
#pragma unroll
                        for (int t = 0; t < NT; ++t) acc[k][t] = __builtin_amdgcn_smfmac_i32_32x32x64_i8(av, b[t], acc[k][t], idx, 0, 0);
                    }
                });
            });
            // (landed before the loop's back edge: no register with a load on its way is carried around it)
#pragma unroll
            for (int k = 0; k < BLK; ++k) { mx_take<kSpc * kPieces>(cur[k], nxt[k]); mx_take<kSpc * kPieces>(sc[k], nsc[k]); }
        }
        // lane: query qn of each tile, rows 8 (r / 4) + 4 h + r % 4.  (The lane number is made opaque here:
        // hoisted out of the rounds, the addresses below would take registers from the loop above.)
        int el = lane;
        asm volatile("" : "+v"(el));
        const int qn = el & 31, h = el >> 5;
        auto bound_of = [&](int i, int inv, int k) {
            int bound;
            const float bf = fmaf(sq[i].ta, __int_as_float(inv), -sq[i].tb) - 1.0f;
            asm("v_cvt_i32_f32 %0, %1" : "=v"(bound) : "v"(bf));      // saturates; NaN gives 0
            return ((odd_blocks >> k) & 1u) ? int(0x80000000) : bound;
        };
        uint32_t hits = 0u;         // bit k * NT + t: some lane of (block k, tile t) reaches its query's bound
        static_for<BLK * NT>([&](auto ii) {
            constexpr int k = decltype(ii)::value / NT, t = decltype(ii)::value % NT;
            const v16i &v = acc[k][t];
            const int bound = bound_of(t * kQTile + qn, inv_vmax[k], k);
            int m0 = max(max(v[0], v[1]), v[2]), m1 = max(max(v[3], v[4]), v[5]);
            int m2 = max(max(v[6], v[7]), v[8]), m3 = max(max(v[9], v[10]), v[11]);
            m0 = max(max(m0, v[12]), v[13]);
            m1 = max(max(m1, v[14]), v[15]);
            if (__any(max(max(m0, m1), max(m2, m3)) >= bound)) hits |= 1u << decltype(ii)::value;
        });
        if constexpr (BEST) hits = (1u << (BLK * NT)) - 1u;
        // (One body for all pairs, on a copy of the sums: unrolled, it would outgrow the instruction cache.)
#pragma unroll 1
        while (hits != 0u) {
            const int kt = __builtin_ctz(hits);
            hits &= hits - 1u;
            v16i v = acc[0][0];
            uint32_t jb = blk[0];
            int inv = inv_vmax[0];
            static_for<BLK * NT>([&](auto ii) {
                constexpr int k = decltype(ii)::value / NT;
                if (decltype(ii)::value > 0 && kt == decltype(ii)::value) { v = acc[k][decltype(ii)::value % NT]; jb = blk[k]; inv = inv_vmax[k]; }
            });
            const int k = kt / NT, i = (kt % NT) * kQTile + qn;
            const int bound = bound_of(i, inv, k);
            const float qs = sq[i].qs, qb = sq[i].qb, tau = sq[i].tau;
            const float *vs = s_vs + (wave * BLK + k) * 32 + 4 * h;
            if constexpr (BEST) {
                float m = -__int_as_float(0x7f800000);
#pragma unroll
                for (int r = 0; r < 16; ++r) m = fmaxf(m, ((float(v[r]) * qs) + qb) * vs[8 * (r >> 2) + (r & 3)]);     // (NaN never wins)
                m = fmaxf(m, __shfl_xor(m, 32));
                if (h == 0 && q0 + i < a.nq_tile && jb < nj) a.best_out[size_t(q0 + i) * a.best_stride + jb] = best_word(m);
                continue;
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                if (v[r] >= bound) {
                    const int row = 8 * (r >> 2) + (r & 3);
                    const float s = ((float(v[r]) * qs) + qb) * vs[row];
                    if (s >= tau) {
                        const uint32_t pos = atomicAdd(&scnt[my_sub * kQ + i], 1u);
                        if (pos < kSegCap)
                            a.cand[(size_t(q0 + i) * a.seg_stride + wg * sub + my_sub) * kSegCap + pos] =
                                sort_key(s, block_of(jb) * 32u + uint32_t(row + 4 * h));
                        else if (pos == kSegCap) atomicAdd(s_over, 1u);      // the one append that finds the segment just full
                    }
                }
            }
        }
        }
        ++round_no;
        more = lds_at(flag + round_no % 3u);
        has = nhas;
#pragma unroll
        for (int k = 0; k < BLK; ++k) blk[k] = nblk[k];
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // requests still in flight write this workgroup's LDS
    if constexpr (BEST) return;
    __syncthreads();
    for (int i = tid; i < kQ * int(sub); i += kMxThreads) {
        const int q = q0 + i % kQ, sb = i / kQ;
        if (q < a.nq_tile) a.cand_cnt[size_t(q) * a.seg_stride + wg * sub + sb] = scnt[sb * kQ + i % kQ];
    }
}

constexpr int kMxBlk = 4;                 // blocks of one wave and round in a long launch
constexpr int kMxSegments = 256;          // candidate segments a query has room for

// A level of few blocks is one round of the grid and as long as a wave's share of it: one or two
// blocks per wave where that covers the level.  Open floors: every row read is appended, and two
// blocks fill a segment -- a segment per wave and at most two blocks each.
MxShape mx_shape(int device, size_t nq, size_t level_blocks, bool open_floors) {
    MxShape m;
    const size_t tiles = (nq + kQTile - 1) / kQTile;
    m.nt = tiles > 1 ? 2 : 1;
    m.groups = unsigned((tiles + m.nt - 1) / m.nt);
    const size_t most = std::min<size_t>(kMxSegments, std::max<size_t>(1, size_t(wide_grid_blocks(device)) / m.groups));
    m.blk = level_blocks <= most * kMxWaves ? 1 : (open_floors || level_blocks <= most * kMxWaves * 2) ? 2 : kMxBlk;
    m.wgs = unsigned(std::min(most, (level_blocks + size_t(kMxWaves * m.blk) - 1) / size_t(kMxWaves * m.blk)));
    m.sub = 1;
    while (m.sub < unsigned(kMxWaves) && size_t(m.sub) * 2 * m.wgs <= size_t(kMxSegments)) m.sub *= 2;
    return m;
}
int mx_segments() { return kMxSegments; }
int mx_round_blocks(int device, size_t nq) {
    const MxShape m = mx_shape(device, nq, size_t(1) << 31, false);
    return int(m.wgs) * kMxWaves * m.blk;
}

template <int ENT, int NT, int BLK, bool BEST>
static hipError_t launch_mx_best(const ScanArgs &a, const MxShape &m, hipStream_t s) {
    constexpr int kS = mx_steps(ENT) < 16 / NT ? mx_steps(ENT) : 16 / NT;
    const size_t lds = size_t(kMxRing) * NT * kS * 2048 + NT * kQTile * (sizeof(MxQuery) + 8 * 4) + kMxWaves * BLK * 32 * 4 + 64;
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(k_scan_lut_mx<ENT, NT, BLK, BEST>), hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((k_scan_lut_mx<ENT, NT, BLK, BEST>), dim3(m.wgs * m.groups), dim3(kMxThreads), lds, s, a, m.groups, m.sub);
    return hipGetLastError();
}
template <int ENT, int NT, int BLK>
static hipError_t launch_mx(const ScanArgs &a, const MxShape &m, hipStream_t s) {
    return a.best_out != nullptr ? launch_mx_best<ENT, NT, BLK, true>(a, m, s) : launch_mx_best<ENT, NT, BLK, false>(a, m, s);
}
template <int ENT, int NT>
static hipError_t launch_mx_blk(const ScanArgs &a, const MxShape &m, hipStream_t s) {
    return m.blk == 1 ? launch_mx<ENT, NT, 1>(a, m, s) : m.blk == 2 ? launch_mx<ENT, NT, 2>(a, m, s) : launch_mx<ENT, NT, kMxBlk>(a, m, s);
}

// One append-mode launch: a.nq_tile = all queries of the chunk, a.tables = their B operands
// (of k_prep_lut), scales, floors and segments by query.
hipError_t launch_scan_lut_mx(const ScanArgs &a, const MxShape &m, int bits, hipStream_t s) {
    if (a.classic != 0 || a.nq_tile <= 0 || (a.best_out == nullptr && size_t(m.wgs) * m.sub > a.seg_stride)) return hipErrorInvalidValue;
    if (bits == 3) return m.nt == 1 ? launch_mx_blk<8, 1>(a, m, s) : launch_mx_blk<8, 2>(a, m, s);
    return m.nt == 1 ? launch_mx_blk<16, 1>(a, m, s) : launch_mx_blk<16, 2>(a, m, s);
}

}  // namespace tv
