// HIP kernels that prepare queries: rotation, TQ+ inverse, int8 weights (permute-dot) or byte tables (u8 LUT),
// one workgroup per query and one launch for all of it.
//
// Compiled with -ffp-contract=off like every file here: the operations, their operands and their order
// are the reference's (turbovec/src/search.rs:3237-3269), so the bits are.
#include "tv_device.h"
#include "tv_internal.h"

#include <cfloat>

namespace tv {

constexpr int kPrepPiece = 1024;     // products of the bias chain in LDS at a time

struct PrepArgs {
    const float *q, *signs;
    const uint32_t *perms;
    const float *shift, *scale;     // null without a TQ+ pair
    float inv_sqrt_block;
    int dim, log_block, G, nch;
    uint8_t *tables, *mx;           // mx: or null
    float *qscale, *qbias;
    int near_nch;                   // chunks of the row there, the last ones zero
    uint8_t *near;                  // or null: int8 weights of the scan that goes before the tables, ...
    float *near_unit, *near_err;    // ... per query what one unit of its sums is in table units, and how far a row's table sum may lie above
    float cs;                       // the codebook over its int8 levels
    uint32_t lv[2];                 // the levels
    float *rot_out;                 // when given: the rotated (and calibrated) rows
    size_t nq;
    uint64_t *stamp;
    uint64_t *cleared;              // when given: a word per query, set to zero
};

// A row lies in LDS with eight floats of padding after every 64: lanes whose elements are 64 apart in
// groups of eight then spread over the banks.
__host__ __device__ constexpr int prep_at(int j) { return j + (j >> 6) * 8; }
__host__ __device__ constexpr int prep_floats(int dim) { return prep_at(dim - 1) + 1 + 7 - (prep_at(dim - 1) & 7); }

// Sixteen bytes of the caller's rows, whose alignment is a float's (the load is the same 16-byte one).
typedef float RowPiece __attribute__((ext_vector_type(4), aligned(4)));

// R butterfly stages from stride 2^S on over the whole row.
template <int T, int R>
__device__ __forceinline__ void prep_pass(float *buf, int dim, int S) {
    constexpr int N = 1 << R;
    for (int g = threadIdx.x; g < dim / N; g += T) {
        const int base = ((g >> S) << (S + R)) + (g & ((1 << S) - 1));
        float v[N];
#pragma unroll
        for (int e = 0; e < N; ++e) v[e] = buf[prep_at(base + (e << S))];
        butterflies<R>(v);
#pragma unroll
        for (int e = 0; e < N; ++e) buf[prep_at(base + (e << S))] = v[e];
    }
    __syncthreads();
}

// turbovec/src/rotation.rs:265-320 (apply_with_scratch) + :964-982 (wht_block_scalar): the rotated row, still
// to be multiplied by inv_sqrt_block, at B's padded places.  Three stages at a time through registers: a
// barrier per pass instead of one per stage (1536 dimensions: 8 instead of 20, which was most of the time
// one query's preparation took).
template <int T>
__device__ __forceinline__ void rotate_row(const float *src, const float *signs, const uint32_t *perms, int dim, int log_block,
                                           float inv_sqrt_block, float *A, float *B) {
    // the row itself first, 16 bytes at a time: it may lie in host memory, where a gather would fetch it piece by piece
    for (int i = threadIdx.x; i < dim / 4; i += T) {
        const RowPiece p = reinterpret_cast<const RowPiece *>(src)[i];
        *reinterpret_cast<float4 *>(B + 4 * i) = float4{p.x, p.y, p.z, p.w};
    }
    __syncthreads();
#pragma unroll
    for (int round = 0; round < 2; ++round) {
        float *buf = round == 0 ? A : B;
        for (int g = threadIdx.x; g < dim / 8; g += T) {
            const uint4 *p4 = reinterpret_cast<const uint4 *>(perms + size_t(round) * dim + 8 * g);
            const float4 *s4 = reinterpret_cast<const float4 *>(signs + size_t(round) * dim + 8 * g);
            const uint4 pa = p4[0], pb = p4[1];
            const float4 sa = s4[0], sb = s4[1];
            const uint32_t p[8] = {pa.x, pa.y, pa.z, pa.w, pb.x, pb.y, pb.z, pb.w};
            const float s[8] = {sa.x, sa.y, sa.z, sa.w, sb.x, sb.y, sb.z, sb.w};
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e)      // the 1/sqrt(B) scale of round 0 rides the round-1 gather: (x * inv) * sign
                v[e] = round == 0 ? B[p[e]] * s[e] : (A[prep_at(int(p[e]))] * inv_sqrt_block) * s[e];
            butterflies<3>(v);
            float4 *dst = reinterpret_cast<float4 *>(buf + prep_at(8 * g));
            dst[0] = float4{v[0], v[1], v[2], v[3]};
            dst[1] = float4{v[4], v[5], v[6], v[7]};
        }
        __syncthreads();
        for (int S = 3; S < log_block; S += 3) {
            if (log_block - S >= 3) prep_pass<T, 3>(buf, dim, S);
            else if (log_block - S == 2) prep_pass<T, 2>(buf, dim, S);
            else prep_pass<T, 1>(buf, dim, S);
        }
    }
}

// The rotated row at A[0 .. dim), its TQ+ inverse where there is a pair (search.rs:3154-3186
// calibrate_queries), and the pair's bias term.  The reference's f64 sum is sequential over d, but only its f32
// rounding is used: all threads add, and where every value within the two orders' distance -- dim roundings at most on the
// way of a term there, dim / 256 + 9 here, and those of the magnitude's sum -- rounds to the same float, that is it.
// Otherwise (one query in 10^5) one thread adds in order.  With the chain always: 3032 dimensions 47 us for one query, now 25.
// late: becomes true there.
template <int T>
__device__ __forceinline__ float calibrated_row(const float *src, const PrepArgs &a, float *A, float *B, double *prod, bool &late) {
    const int t = threadIdx.x, dim = a.dim;
    rotate_row<T>(src, a.signs, a.perms, dim, a.log_block, a.inv_sqrt_block, A, B);
    float bias = 0.0f;
    if (a.scale != nullptr) {
        double sum = 0.0, mass = 0.0;
        for (int i = t; i < dim; i += T) {
            const double p = double(B[prep_at(i)] * a.inv_sqrt_block) * double(a.shift[i]);
            sum -= p;
            mass += fabs(p);
        }
        for (int d = 32; d >= 1; d >>= 1) {
            sum += __shfl_xor(sum, d);
            mass += __shfl_xor(mass, d);
        }
        if ((t & 63) == 0) { prod[t >> 6] = sum; prod[T / 64 + (t >> 6)] = mass; }
        __syncthreads();
        sum = 0.0;
        mass = 0.0;
#pragma unroll
        for (int i = 0; i < T / 64; i += 4) {
            sum += (prod[i] + prod[i + 1]) + (prod[i + 2] + prod[i + 3]);
            mass += (prod[T / 64 + i] + prod[T / 64 + i + 1]) + (prod[T / 64 + i + 2] + prod[T / 64 + i + 3]);
        }
        __syncthreads();
        const double slack = double(2 * dim + 256) * 0x1p-53 * mass;
        bias = float(sum - slack);
        if (__float_as_uint(bias) != __float_as_uint(float(sum + slack)) || !(slack < 1e30)) {     // (uniform over the workgroup)
            late = true;
            double bc = 0.0;
            for (int d0 = 0; d0 < dim; d0 += kPrepPiece) {
                const int m = min(kPrepPiece, dim - d0);      // (a multiple of eight, as dim is)
                for (int i = t; i < m; i += T) prod[i] = double(B[prep_at(d0 + i)] * a.inv_sqrt_block) * double(a.shift[d0 + i]);
                __syncthreads();
                if (t == 0) {
                    for (int i = 0; i < m; i += 8) {
                        double p[8];
#pragma unroll
                        for (int e = 0; e < 8; ++e) p[e] = prod[i + e];
#pragma unroll
                        for (int e = 0; e < 8; ++e) bc -= p[e];
                    }
                }
                __syncthreads();
            }
            bias = float(bc);                                 // (for thread 0, which uses it)
        }
    }
    for (int i = t; i < dim; i += T) {
        float x = B[prep_at(i)] * a.inv_sqrt_block;
        if (a.scale != nullptr) x = x / a.scale[i];
        A[i] = x;
        if (a.rot_out != nullptr) a.rot_out[size_t(blockIdx.x) * dim + i] = x;
    }
    __syncthreads();
    return bias;
}

template <int T>
__device__ __forceinline__ float block_max(float v, float *red) {
    // exact: max is order-free
    for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    v = red[0];
#pragma unroll
    for (int i = 1; i < T / 64; ++i) v = fmaxf(v, red[i]);
    __syncthreads();
    return v;
}

__device__ __forceinline__ float clamp_round_i8(float v) {
    // Rust f32::round is half-away-from-zero, like roundf; then clamp(-127, 127)
    v = roundf(v);
    return v < -127.0f ? -127.0f : (v > 127.0f ? 127.0f : v);
}

// turbovec/src/search.rs:2806-2846 build_permute_dot, emitting the weights in
// the MFMA B-fragment order of the scan.  Plane order (the batched scans, whose
// decode yields one A operand of low nibbles and one of high nibbles per chunk):
// for query tile t, chunk c and nibble plane p (0 = low nibble = odd dimension,
// 1 = high nibble = even dimension) a 1 KiB fragment whose lane (h*32 + n) holds
// the 16 weights of query n for groups 32c + 16h .. +15.  Split order (k_scan_p4,
// which decodes the first 8 code bytes of a lane on the vector ALU, four at a
// time, and looks the other 8 up whole, both levels of a byte side by side):
// fragment 0 of chunk c holds, in lane (h*32 + n), for e = 0..7, the plane-p
// weight of group 32c + 16h + e at byte 8*(e/4) + 4p + e%4; fragment 1 the
// plane-p weight of group 32c + 16h + 8 + e at byte 2e + p.
__device__ __forceinline__ size_t wfrag_offset(int g, int n, int plane, bool split) {
    const size_t lane16 = size_t(((g & 31) >> 4) * 32 + n) * 16;
    if (split) {
        const int e = g & 7;
        const int at = (g & 8) ? 2 * e + plane : 8 * (e >> 2) + 4 * plane + (e & 3);
        return size_t(g >> 5) * 2048 + size_t((g & 15) >> 3) * 1024 + lane16 + size_t(at);
    }
    return size_t(g >> 5) * 2048 + size_t(plane) * 1024 + lane16 + size_t(g & 15);
}

template <int T>
__global__ __launch_bounds__(T) void k_prep_p(PrepArgs a, float cs, bool split) {
    extern __shared__ __align__(16) float prep_lds[];
    __shared__ float red[T / 64];
    __shared__ __align__(16) double prod[kPrepPiece];
    float *A = prep_lds, *B = prep_lds + prep_floats(a.dim);
    const size_t qi = blockIdx.x;
    const int n = int(qi % kQTile), t = threadIdx.x;
    uint8_t *base = a.tables + qi / kQTile * size_t(a.nch) * 2048;
    if (qi >= a.nq) {  // padding query of the last tile: zero weights
        for (int g = t; g < a.nch * 32; g += T) {
            base[wfrag_offset(g, n, 0, split)] = 0;
            base[wfrag_offset(g, n, 1, split)] = 0;
        }
        if (t == 0) { a.qscale[qi] = 0.0f; a.qbias[qi] = 0.0f; }
        return;
    }
    bool late = false;
    const float bias = calibrated_row<T>(a.q + qi * size_t(a.dim), a, A, B, prod, late);
    float m = 0.0f;
    for (int d = t; d < a.dim; d += T) m = fmaxf(m, fabsf(A[d]));
    const float qmax = block_max<T>(m, red);
    float qs = qmax / 127.0f, inv_qs;
    if (qs >= FLT_MIN) inv_qs = 1.0f / qs; else { qs = 1.0f; inv_qs = 1.0f; }
    for (int g = t; g < a.nch * 32; g += T) {
        int8_t lo = 0, hi = 0;
        if (g < a.G) {
            lo = int8_t(clamp_round_i8(A[2 * g + 1] * inv_qs));
            hi = int8_t(clamp_round_i8(A[2 * g] * inv_qs));
        }
        base[wfrag_offset(g, n, 0, split)] = uint8_t(lo);
        base[wfrag_offset(g, n, 1, split)] = uint8_t(hi);
    }
    if (t == 0) {
        a.qscale[qi] = cs * qs;
        a.qbias[qi] = 0.0f + bias;
        if (a.cleared != nullptr) a.cleared[qi] = 0;
        if (a.stamp != nullptr && (late || qi + kStampsBefore >= a.nq)) a.stamp[qi % kStampsBefore] = wall_clock64();      // (among the last to end)
    }
}

// turbovec/src/search.rs:2856-2994 build_query_neon_lut_from_slice.  Output per
// query: nch*32 rows of 32 bytes, row g = [16 entries indexed by the byte's HIGH
// nibble (the group's first dimensions) | 16 entries indexed by the LOW nibble];
// rows of padding groups are zero.
template <int BITS>
__device__ __forceinline__ float lut_entry(const float *q, const float *cen, int dim_start, int sub, int nv) {
    constexpr int cpb = 8 / BITS, cpn = cpb / 2;
    constexpr unsigned code_mask = (1u << BITS) - 1;
    float s = 0.0f;
#pragma unroll
    for (int c = 0; c < cpn; ++c) {
        const int sh = (cpn - 1 - c) * BITS;
        const unsigned code = (unsigned(nv) >> sh) & code_mask;
        s += q[dim_start + sub * cpn + c] * cen[code];
    }
    return s;
}

// A byte-group's two tables as B operands of k_scan_lut_mx.  Piece ((tile, chunk, step j, part p), lane
// (u, n)) is 16 bytes of query 32 tile + n: the 16 lanes-halves p of the A operand meet part p, and
// of that lane's stored bytes 0..7 half u = 0, 8..15 half u = 1.
//   16-entry tables: byte-group 16 p + j of the chunk, its high (u = 0) or low (u = 1) nibble's table
//    8-entry tables: byte-group 16 p + 2 j + u, the 8 entries of its high nibble, then of its low
// A table's entries come in the order the operand's bits are cheapest in: the nibble's low bits are
// the stored slot's number (three of four bits, two of three), its highest the choice of positions, so
// that entry 8 p + 2 g + s (4 p + 2 g + s) is the group g's fourth 2 p + s.
// (In a launch of their own they took 5 us of 37 queries' 219 and the gap in front of it.)
// (An instance of its own writes them: the code for both made the other searches' tables wait, 1024 dimensions 3-bit, 4 queries 11.7 us a
// launch without it and 13.1 with, 1536 14.5 and 16.6.)
__device__ __forceinline__ uint32_t zip_lo(uint32_t a, uint32_t b) { return (a & 0xffffu) | (b << 16); }
__device__ __forceinline__ uint32_t zip_hi(uint32_t a, uint32_t b) { return (a >> 16) | (b & 0xffff0000u); }
template <int BITS>
__device__ __forceinline__ void mx_put(uint8_t *mx, int nch, int qi, int g, uint4 hi, uint4 lo) {
    constexpr int kSteps = mx_steps(BITS == 3 ? 8 : 16);
    const int p = (g & 31) >> 4, in = g & 15, j = BITS == 3 ? in >> 1 : in;
    uint4 *out = reinterpret_cast<uint4 *>(mx) + ((size_t(qi / kQTile) * nch + size_t(g >> 5)) * kSteps + j) * 128 + p * 64 + qi % kQTile;
    if constexpr (BITS == 3) {
        out[(in & 1) * 32] = make_uint4(zip_lo(hi.x, hi.y), zip_hi(hi.x, hi.y), zip_lo(lo.x, lo.y), zip_hi(lo.x, lo.y));
    } else {
        out[0] = make_uint4(zip_lo(hi.x, hi.z), zip_hi(hi.x, hi.z), zip_lo(hi.y, hi.w), zip_hi(hi.y, hi.w));
        out[32] = make_uint4(zip_lo(lo.x, lo.z), zip_hi(lo.x, lo.z), zip_lo(lo.y, lo.w), zip_hi(lo.y, lo.w));
    }
}

// Field f of byte-group g of a query's int8 weights, as the B operands of k_scan_p4_wide's instances for such codes read them: per
// chunk one 1 KiB fragment per field of a code byte (the highest bits first), in it 16 byte-groups to a lane.
__device__ __forceinline__ size_t near_at(int qi, int nch, int fields, int g, int f) {
    return (size_t(qi / kQTile) * nch + size_t(g >> 5)) * size_t(fields) * 1024 + size_t(f) * 1024 + size_t(((g & 31) >> 4) * 32 + qi % kQTile) * 16 + size_t(g & 15);
}
// The int8 weights of one nibble and what they leave out.  A row's table sum is, nibble by nibble, an entry
// T[v] of a table of 16 (8); the scan in front of the tables takes unit * (weights . levels of the codes) in its place, and what
// the entry exceeds that by is at most `over`, over all values of the nibble.  The weights are the query's dimensions in int8, or
// their neighbours where those leave less over the mean (levels may be lifted by a constant): 9 (3) pairs, 1536 dimensions 2-bit 1.10 standard deviations of the score instead of 1.22.
template <int BITS>
__device__ __forceinline__ void near_fit(const uint32_t *w, const float *q, float inv_u, float unit, const PrepArgs &a, int8_t (&out)[2], float &over) {
    constexpr int cpn = BITS == 2 ? 2 : 1, N = BITS == 2 ? 4 : 8;
    float lev[N];
#pragma unroll
    for (int i = 0; i < N; ++i) lev[i] = unit * float(int8_t(a.lv[i / 4] >> (8 * (i & 3))));
    int w0[2] = {0, 0};
#pragma unroll
    for (int c = 0; c < cpn; ++c) w0[c] = int(fminf(fmaxf(rintf(q[c] * inv_u), -127.0f), 127.0f));      // (NaN gives -127: any weights do)
    float best = __int_as_float(0x7f800000);
    over = best;
    for (int d0 = -1; d0 <= 1; ++d0) {
        for (int d1 = cpn == 2 ? -1 : 0; d1 <= (cpn == 2 ? 1 : 0); ++d1) {
            const int a0 = min(max(w0[0] + d0, -127), 127), a1 = cpn == 2 ? min(max(w0[1] + d1, -127), 127) : 0;
            float most = -__int_as_float(0x7f800000);
#pragma unroll
            for (int v = 0; v < (BITS == 2 ? 16 : 8); ++v) {
                const float t = float((w[v / 4] >> (8 * (v & 3))) & 0xffu);
                most = fmaxf(most, BITS == 2 ? (t - float(a0) * lev[v >> 2]) - float(a1) * lev[v & 3] : t - float(a0) * lev[v & 7]);
            }
            const float cost = most + 0.5f * (lev[0] + lev[N - 1]) * float(a0 + a1);
            if (cost < best || (d0 == -1 && d1 <= 0 && best == __int_as_float(0x7f800000))) { best = cost; over = most; out[0] = int8_t(a0); out[1] = int8_t(a1); }
        }
    }
}

template <int T, int BITS, bool MX, bool NEAR>
__global__ __launch_bounds__(T) void k_prep_lut(PrepArgs a, const float *__restrict__ centroids) {
    extern __shared__ __align__(16) float prep_lds[];
    __shared__ float red[T / 64];
    __shared__ __align__(16) double prod[kPrepPiece];
    __shared__ float cen[16];
    __shared__ uint32_t next;
    constexpr int cpb = 8 / BITS;
    constexpr int kEntries = BITS == 3 ? 8 : 16;        // of a nibble that differ
    float *A = prep_lds, *B = prep_lds + prep_floats(a.dim);
    const size_t qi = blockIdx.x;
    uint8_t *dst = a.tables + qi * size_t(a.nch) * 1024;
    const int t = threadIdx.x, G = a.G;
    if (qi >= a.nq) {
        for (int i = t; i < a.nch * 64; i += T) reinterpret_cast<uint4 *>(dst)[i] = make_uint4(0, 0, 0, 0);
        if constexpr (MX)
            for (int g = t; g < a.nch * 32; g += T) mx_put<BITS>(a.mx, a.nch, int(qi), g, make_uint4(0, 0, 0, 0), make_uint4(0, 0, 0, 0));
        if constexpr (NEAR)
            for (int g = t; g < a.near_nch * 32; g += T) {
#pragma unroll
                for (int f = 0; f < cpb; ++f) a.near[near_at(int(qi), a.near_nch, cpb, g, f)] = 0;
            }
        if (t == 0) { a.qscale[qi] = 0.0f; a.qbias[qi] = 0.0f; }
        return;
    }
    if (t < (1 << BITS)) cen[t] = centroids[t];
    if (t == 0) next = 0u;
    bool late = false;
    const float bias_corr = calibrated_row<T>(a.q + qi * size_t(a.dim), a, A, B, prod, late);
    float *mins = B;                                   // two per group: at most a row's length
    float *pairs = reinterpret_cast<float *>(prod);    // their sums, where they fit
    constexpr int kAtOnce = 16;                        // of them in registers, twice
    const int padded = (G + 2 * kAtOnce - 1) / (2 * kAtOnce) * (2 * kAtOnce);      // (zeros behind the last, which change nothing)
    const bool paired = padded <= 2 * kPrepPiece;
    if (paired && t < padded - G) pairs[G + t] = 0.0f;
    float span = 0.0f;
    for (int g = t; g < G; g += T) {
#pragma unroll
        for (int sub = 0; sub < 2; ++sub) {
            float mn = FLT_MAX, mx = -FLT_MAX;
#pragma unroll
            for (int nv = 0; nv < kEntries; ++nv) {
                const float s = lut_entry<BITS>(A, cen, g * cpb, sub, nv);
                if (s < mn) mn = s;
                if (s > mx) mx = s;
            }
            mins[2 * g + sub] = mn;
            span = fmaxf(span, mx - mn);
        }
        if (paired) pairs[g] = mins[2 * g] + mins[2 * g + 1];
    }
    const float max_span = block_max<T>(span, red);   // also orders the writes of mins
    float scale = max_span > 0.0f ? max_span / 127.0f : 1.0f, inv_scale;
    if (scale >= FLT_MIN) inv_scale = 1.0f / scale; else { scale = 1.0f; inv_scale = 1.0f; }
    if (t == 0) {
        // Sequential f32 sum over groups, inner add first (search.rs:2910): one lane's chain of additions, 16 clocks a group with both of them
        // in it, so the inner ones are done before and the other waves work on the tables below meanwhile (3072 dimensions 3-bit, one query 26.4 us a launch and
        // 18.8; 1536 2-bit 12.0 and 10.7; 768 3-bit, 300 queries 13.6 and 10.7).
        float bias = 0.0f;
        int g = 0;
        if (paired) {
            // (the groups after next are on their way from LDS)
            float4 m[2][kAtOnce / 4];
            auto fetch = [&](auto set, int from) {
#pragma unroll
                for (int e = 0; e < kAtOnce / 4; ++e) m[decltype(set)::value][e] = reinterpret_cast<const float4 *>(pairs + from)[e];
                __builtin_amdgcn_sched_barrier(0);
            };
            auto add = [&](auto set) {
#pragma unroll
                for (int e = 0; e < kAtOnce / 4; ++e) {
                    const float4 v = m[decltype(set)::value][e];
                    bias += v.x;
                    bias += v.y;
                    bias += v.z;
                    bias += v.w;
                }
                __builtin_amdgcn_sched_barrier(0);
            };
            fetch(IntC<0>{}, 0);
            for (; g < padded; g += 2 * kAtOnce) {
                fetch(IntC<1>{}, g + kAtOnce);
                add(IntC<0>{});
                fetch(IntC<0>{}, min(g + 2 * kAtOnce, padded - kAtOnce));
                add(IntC<1>{});
            }
        }
        for (; g + 8 <= G; g += 8) {
            float4 m[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) m[e] = reinterpret_cast<const float4 *>(mins + 2 * g)[e];
#pragma unroll
            for (int e = 0; e < 4; ++e) { bias += m[e].x + m[e].y; bias += m[e].z + m[e].w; }
        }
        for (; g < G; ++g) bias += mins[2 * g] + mins[2 * g + 1];
        a.qscale[qi] = scale;
        a.qbias[qi] = bias + bias_corr;      // (+0 without a pair, search.rs:3176-3185)
    }
    float near_inv = 0.0f, unit = 0.0f, over_sum = 0.0f;
    if constexpr (NEAR) {
        float m = 0.0f;
        for (int d = t; d < a.dim; d += T) m = fmaxf(m, fabsf(A[d]));
        float u = block_max<T>(m, red) / 127.0f;
        if (!(u >= FLT_MIN)) u = 1.0f;
        near_inv = 1.0f / u;
        unit = (inv_scale * u) * a.cs;
    }
    // 64 byte-groups at a time, to whichever wave is free: the one with the chain comes late (dealt out beforehand where other
    // workgroups fill the time: 1024 queries of 1536 dimensions 20.3 and, claimed, 21.1 us)
    const bool dealt = gridDim.x > 512u;
    for (uint32_t turn = 0;; ++turn) {
        uint32_t claimed = turn * uint32_t(T) + uint32_t(t & ~63);
        if (!dealt) {
            if ((t & 63) == 0) claimed = atomicAdd(&next, 64u);
            claimed = uint32_t(__builtin_amdgcn_readfirstlane(int(claimed)));
        }
        const int g = int(claimed) + (t & 63);
        if (int(claimed) >= a.nch * 32) break;
        if (g >= a.nch * 32) continue;
        uint32_t w[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        int8_t nw[4] = {0, 0, 0, 0};
        if (g < G) {
#pragma unroll
            for (int sub = 0; sub < 2; ++sub) {
                const float mn = mins[2 * g + sub];
#pragma unroll
                for (int nv = 0; nv < kEntries; ++nv) {
                    float v = roundf((lut_entry<BITS>(A, cen, g * cpb, sub, nv) - mn) * inv_scale);
                    v = v < 0.0f ? 0.0f : (v > 127.0f ? 127.0f : v);
                    w[sub * 4 + nv / 4] |= uint32_t(uint8_t(v)) << (8 * (nv & 3));
                }
                if constexpr (BITS == 3) { w[sub * 4 + 2] = w[sub * 4]; w[sub * 4 + 3] = w[sub * 4 + 1]; }
            }
        }
        const uint4 hi = make_uint4(w[0], w[1], w[2], w[3]), lo = make_uint4(w[4], w[5], w[6], w[7]);
        uint4 *o = reinterpret_cast<uint4 *>(dst + size_t(g) * 32);
        o[0] = hi;
        o[1] = lo;
        if constexpr (MX) mx_put<BITS>(a.mx, a.nch, int(qi), g, hi, lo);
        if constexpr (NEAR) {
            if (g < G) {
#pragma unroll
                for (int sub = 0; sub < 2; ++sub) {
                    int8_t to[2] = {0, 0};
                    float over;
                    near_fit<BITS>(w + 4 * sub, A + g * cpb + sub * (cpb / 2), near_inv, unit, a, to, over);
                    over_sum += over;
#pragma unroll
                    for (int c = 0; c < cpb / 2; ++c) nw[sub * (cpb / 2) + c] = to[c];
                }
            }
#pragma unroll
            for (int f = 0; f < cpb; ++f) a.near[near_at(int(qi), a.near_nch, cpb, g, f)] = uint8_t(nw[f]);
        }
    }
    if constexpr (NEAR) {
        for (int g = a.nch * 32 + t; g < a.near_nch * 32; g += T) {
#pragma unroll
            for (int f = 0; f < cpb; ++f) a.near[near_at(int(qi), a.near_nch, cpb, g, f)] = 0;
        }
        for (int d = 32; d >= 1; d >>= 1) over_sum += __shfl_xor(over_sum, d);
        if ((t & 63) == 0) red[t >> 6] = over_sum;
        __syncthreads();
        if (t == 0) {
            a.near_unit[qi] = unit;
            float all = 0.0f;
            for (int i = 0; i < T / 64; ++i) all += red[i];
            a.near_err[qi] = all;
        }
    }
    if (t == 0 && a.cleared != nullptr) a.cleared[qi] = 0;
    if (t == 0 && a.stamp != nullptr && (late || qi + kStampsBefore >= a.nq)) a.stamp[qi % kStampsBefore] = wall_clock64();      // (among the last to end)
}

static_assert(size_t(2) * prep_floats(16384) * sizeof(float) + kPrepPiece * sizeof(double) + 256 <= 160 * 1024,
              "the longest row the index accepts must fit a workgroup's LDS");

hipError_t launch_prep(const PrepRequest &r, const Geometry &g, size_t nq, size_t nq_padded, hipStream_t s) {
    if (nq_padded == 0) return hipSuccess;
    PrepArgs a;
    a.q = r.q; a.signs = r.signs; a.perms = r.perms; a.shift = r.shift; a.scale = r.scale;
    a.inv_sqrt_block = r.inv_sqrt_block;
    a.dim = g.dim; a.log_block = __builtin_ctz(unsigned(r.block)); a.G = g.G; a.nch = g.nch;
    a.tables = r.tables; a.mx = r.tables_mx; a.qscale = r.qscale; a.qbias = r.qbias; a.rot_out = r.rot_out;
    a.nq = nq; a.stamp = r.stamp; a.cleared = r.cleared;
    a.near_nch = near_nch(g.nch, g.bits); a.near = r.near; a.near_unit = r.near_unit; a.near_err = r.near_err; a.cs = r.near_cs; a.lv[0] = r.lv[0]; a.lv[1] = r.lv[1];
    const size_t lds = size_t(2) * prep_floats(g.dim) * sizeof(float);
    auto launch = [&](auto kernel, int threads, auto... rest) -> hipError_t {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(kernel, dim3(unsigned(nq_padded)), dim3(unsigned(threads)), lds, s, a, rest...);
        return hipGetLastError();
    };
    auto all = [&](auto threads) -> hipError_t {
        constexpr int T = decltype(threads)::value;
        if (r.permute_dot) return launch(k_prep_p<T>, T, r.cs, r.split);
        auto tables = [&](auto mx) -> hipError_t {
            constexpr bool M = decltype(mx)::value != 0;
            return g.bits == 2 ? launch(k_prep_lut<T, 2, M, false>, T, r.centroids) : g.bits == 3 ? launch(k_prep_lut<T, 3, M, false>, T, r.centroids) : launch(k_prep_lut<T, 4, M, false>, T, r.centroids);
        };
        return r.tables_mx != nullptr ? tables(IntC<1>{}) : tables(IntC<0>{});
    };
    if (r.near != nullptr) {
        if (a.near_nch == 0 || r.tables_mx == nullptr) return hipErrorInvalidValue;
        return g.bits == 2 ? launch(k_prep_lut<256, 2, true, true>, 256, r.centroids) : launch(k_prep_lut<256, 3, true, true>, 256, r.centroids);
    }
    // A workgroup's time is latency, pass after pass with a barrier each: where queries leave the chip empty, twice the threads halve a long row's
    // passes.  20K rows, us a search with 256 threads and 512: x 3072 3-bit, one query 73.9 and 69.1, 4-bit 55.4 and 52.1, 64 queries 57.2 and 53.9; x 1536
    // 2-bit 43.3 and 41.3, 4-bit, 200 queries 62.9 and 62.0; x 768 38.1 and 37.9, x 512 level; 1024 threads gain nothing more.
    return nq > 256 || g.dim < 768 ? all(IntC<256>{}) : all(IntC<512>{});
}

}  // namespace tv
