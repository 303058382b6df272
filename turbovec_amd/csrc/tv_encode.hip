// Ingest: encode raw float rows on the device and append them to the index.
//
// Every float operation is the one the reference does,
// in the reference's order, so codes and scales are bit-identical to the CPU
// encoder's (turbovec/src/encode.rs:1418-1476 encode_batch_chunk, :560-664
// quantize, :900-932 norm; turbovec/src/rotation.rs:218-255 apply_scaled_into):
//   * the squared norm runs in 8 interleaved f32 chains (element j feeds chain
//     j % 8), folded pairwise; each chain is sequential, so 8 lanes carry them;
//   * the rotation is the query rotation with the 1/norm folded into the first
//     gather: (x[perm0[i]] * inv) * sign0[i];
//   * the reconstruction inner product runs in 4 interleaved f64 chains
//     (element j feeds chain j % 4), folded pairwise; only its f32 rounding is used, so
//     k_encode_rows adds in an order of its own and falls back to the chains where the
//     rounding could depend on it.
//
// k_encode_rows takes rows of up to 4096 dimensions, a wave (or part of one) per
// row and a group of four waves' rows (eight, up to 512 dimensions) through each step
// together, so that the sequential chains of all of them run side by side in the lanes of
// one or more waves.  k_encode takes one workgroup per row: longer rows, the rotated rows of
// a TQ+ fit, and tables whose signs are not +-1.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "tv_device.h"
#include "tv_internal.h"

namespace tv {

struct EncodeArgs {
    const float *vecs;        // n_new * dim raw rows (device)
    const float *signs;       // 2 * dim
    const uint32_t *perms;    // 2 * dim
    const float *shift;       // dim, or nullptr for the identity pair (encode.rs:578-590)
    const float *scale;       // dim, or nullptr
    float cen[16];
    float bnd[16];
    int dim, bits, G, nch, block;
    float inv_sqrt_block;
    float *rot_out;           // when set: write the rotated unit rows here and stop (TQ+ fit input)
    uint8_t *nat;             // codes in the device layout
    float *scales;
    size_t old_n, n_new;
};

__device__ __forceinline__ size_t enc_byte_index(size_t v, int g, int nch) {
    const size_t b = v >> 5;
    const int i = int(v & 31);
    return ((b * size_t(nch) + size_t(g >> 5)) * 64 + size_t(((g & 31) >> 4) * 32 + i)) * 16 + size_t(g & 15);
}

__device__ __forceinline__ void wht_lds(float *x, int dim, int block, int t) {
    for (int len = 1; len < block; len <<= 1) {
        for (int p = t; p < dim / 2; p += 256) {
            const int j = 2 * p - (p & (len - 1));
            const float a = x[j], b = x[j + len];
            x[j] = a + b;
            x[j + len] = a - b;
        }
        __syncthreads();
    }
}

__global__ __launch_bounds__(256) void k_encode(EncodeArgs a) {
    extern __shared__ __align__(16) float enc_lds[];
    const int dim = a.dim, t = threadIdx.x;
    float *A = enc_lds;
    float *B = enc_lds + dim;
    __shared__ float red[8];
    __shared__ double dred[4];
    __shared__ float s_cen[16];
    const size_t row = blockIdx.x;
    const float *src = a.vecs + row * size_t(dim);
    if (t < 16) s_cen[t] = a.cen[t];
    for (int i = t; i < dim; i += 256) A[i] = src[i];
    __syncthreads();

    // encode.rs:920-932: c[j % 8] += x * x (separate multiply and add), then the pairwise fold
    for (int i = t; i < dim; i += 256) B[i] = A[i] * A[i];
    __syncthreads();
    if (t < 8) {
        float c = 0.0f;
        for (int j = t; j < dim; j += 8) c = c + B[j];
        red[t] = c;
    }
    __syncthreads();
    const float nrm = sqrtf(((red[0] + red[1]) + (red[2] + red[3])) + ((red[4] + red[5]) + (red[6] + red[7])));
    const float inv = nrm > 1e-10f ? 1.0f / nrm : 0.0f;   // lib.rs:163 MIN_INPUT_NORM

    for (int i = t; i < dim; i += 256) B[i] = (A[a.perms[i]] * inv) * a.signs[i];
    __syncthreads();
    wht_lds(B, dim, a.block, t);
    for (int i = t; i < dim; i += 256) A[i] = (B[a.perms[dim + i]] * a.inv_sqrt_block) * a.signs[dim + i];
    __syncthreads();
    wht_lds(A, dim, a.block, t);
    for (int i = t; i < dim; i += 256) B[i] = A[i] * a.inv_sqrt_block;   // B = rotated unit row
    __syncthreads();
    if (a.rot_out != nullptr) {
        float *dst = a.rot_out + row * size_t(dim);
        for (int i = t; i < dim; i += 256) dst[i] = B[i];
        return;
    }

    // encode.rs:600-640: code = number of boundaries below the calibrated value
    uint8_t *codes = reinterpret_cast<uint8_t *>(A);
    const int nb = (1 << a.bits) - 1;
    for (int i = t; i < dim; i += 256) {
        const float sh = a.shift ? a.shift[i] : 0.0f;
        const float sc = a.scale ? a.scale[i] : 1.0f;
        const float calib = (B[i] + sh) * sc;
        int v = 0;
        for (int b = 0; b < nb; ++b) v += calib > a.bnd[b] ? 1 : 0;
        codes[i] = uint8_t(v);
    }
    __syncthreads();

    // encode.rs:1442-1475: inner = <rotated, reconstruction> in f64, four chains by j % 4.
    // The f64 products are parked piece by piece in what is left of A behind the codes
    // (3 * dim bytes), so the kernel needs 8 * dim bytes of LDS whatever the row length; a
    // chain walks its elements in rising order across the pieces, as in one sweep.
    // (rows of 8 dimensions leave no room for one product per chain there: they use the four
    // spare doubles behind B)
    const int piece = dim >= 16 ? (3 * dim / 8) & ~3 : 4;
    double *terms = dim >= 16 ? reinterpret_cast<double *>(reinterpret_cast<uint8_t *>(A) + dim)
                              : reinterpret_cast<double *>(enc_lds + 2 * dim);
    double ch = 0.0;
    for (int j0 = 0; j0 < dim; j0 += piece) {
        const int j1 = min(dim, j0 + piece);
        for (int j = j0 + t; j < j1; j += 256) {
            const float sh = a.shift ? a.shift[j] : 0.0f;
            const float sc = a.scale ? a.scale[j] : 1.0f;
            const float inv_sc = 1.0f / sc;                       // encode.rs:594
            const double recon = double(s_cen[codes[j]]) * double(inv_sc) - double(sh);
            terms[j - j0] = double(B[j]) * recon;
        }
        __syncthreads();
        if (t < 4)
            for (int j = j0 + t; j < j1; j += 4) ch = ch + terms[j - j0];
        __syncthreads();
    }
    if (t < 4) dred[t] = ch;
    __syncthreads();
    if (t == 0) {
        const double inner = (dred[0] + dred[1]) + (dred[2] + dred[3]);
        a.scales[a.old_n + row] = inner > 0.1 ? nrm / float(inner) : 0.0f;   // encode.rs:1194-1200
    }

    // pack.rs:264-282 byte of a group (first dimension in the high bits; 3-bit codes sit in
    // 4-bit fields), written at the row's lane of the device layout (pack.rs:211-233 append_lanes)
    const int cpb = a.bits == 2 ? 4 : 2;
    const int field = a.bits == 2 ? 2 : 4;
    for (int g = t; g < a.G; g += 256) {
        unsigned byte = 0;
        for (int c = 0; c < cpb; ++c) byte |= unsigned(codes[g * cpb + c]) << ((cpb - 1 - c) * field);
        a.nat[enc_byte_index(a.old_n + row, g, a.nch)] = uint8_t(byte);
    }
}

// ---- rows of up to 4096 dimensions ------------------------------------------------------------
// A row of L lanes lies in LDS as its lanes hold it, L groups of eight elements at a time: the groups' first four
// elements side by side, then their last four, four floats of padding behind each.  A lane's two 16-byte pieces then go to
// neighbouring places of their neighbours', and with rows at a stride of 8 modulo 64 floats the norm's chains, eight
// of a row side by side and rows apart, spread over all banks.
__host__ __device__ constexpr int enc_half(int L) { return 4 * L + 4; }
__host__ __device__ constexpr int enc_at(int j, int L) { return ((j >> 3) / L) * 2 * enc_half(L) + ((j >> 2) & 1) * enc_half(L) + ((j >> 3) % L) * 4 + (j & 3); }
// Lanes per row: a power of two, 8 to 64.
static int enc_lanes(int dim) {
    int lanes = 8;
    while (lanes < 64 && lanes * 8 < dim) lanes *= 2;
    return lanes;
}
// (a row's place also holds the f64 products of one run of its groups, 16 lanes floats, where enc_in_order needs it)
__host__ __device__ constexpr int enc_row_stride(int dim, int lanes) {
    int s = enc_at(dim - 1, lanes) + 1;
    if (s < 16 * lanes + 16) s = 16 * lanes + 16;
    while (s % 64 != 8) ++s;
    return s;
}
// The butterfly stages between lanes whose numbers differ in one of the four lowest bits leave their upper element negated
// (enc_lane_stage): the group g of a row comes out of a round with this sign.
constexpr int kEncNegating = 4;
__host__ __device__ inline bool enc_negated(int g, int log_block) {
    const int stages = log_block - 3 < kEncNegating ? log_block - 3 : kEncNegating;
#ifdef __HIP_DEVICE_COMPILE__
    return __popc(unsigned(g) & ((1u << stages) - 1u)) & 1;
#else
    return __builtin_popcount(unsigned(g) & ((1u << stages) - 1u)) & 1;
#endif
}
// Where the first round leaves element j: the stages between lanes 16 and 32 apart exchange an element's two lowest
// bits with those of the lane (enc_swap_stage), and only the last round changes them back.
__host__ __device__ constexpr int enc_at_swapped(int j, int L, int log_block) {
    const int l = (j >> 3) % L, from4 = log_block > 7 ? ((l >> 4) ^ j) & 1 : 0, from5 = log_block > 8 ? ((l >> 5) ^ (j >> 1)) & 1 : 0;
    return enc_at(j ^ (from4 | from5 << 1) ^ (from4 << 4 | from5 << 5) * 8, L);
}
// The packed rotation tables, a word per round and position: where the round's gather reads (the place in bytes) in the lower
// half, the sign in the highest bit -- the second round's with the sign that the first leaves the element it reads with.
constexpr int kEncMaxDim = 4096;
static_assert(enc_at(kEncMaxDim - 1, 64) * 4 < (1 << 16), "a place takes half a word");
bool encode_pack_tables(const float *signs, const uint32_t *perms, int dim, int block, uint32_t *packed) {
    if (dim > kEncMaxDim) return false;
    // (a rotation keeps a row's length, which enc_slack counts on: both gathers must be permutations)
    for (int r = 0; r < 2; ++r) {
        std::vector<bool> seen(size_t(dim), false);
        for (int j = 0; j < dim; ++j) {
            if (seen[perms[size_t(r) * dim + j]]) return false;
            seen[perms[size_t(r) * dim + j]] = true;
        }
    }
    const int lanes = enc_lanes(dim), log_block = __builtin_ctz(unsigned(block));
    for (int j = 0; j < 2 * dim; ++j) {
        const int from = int(perms[j]);
        const bool second = j >= dim;
        if (signs[j] != 1.0f && signs[j] != -1.0f) return false;
        const bool minus = (signs[j] < 0.0f) != (second && enc_negated(from >> 3, log_block));
        packed[j] = uint32_t(second ? enc_at_swapped(from, lanes, log_block) : enc_at(from, lanes)) * 4 | (minus ? 0x80000000u : 0u);
    }
    return true;
}

// A butterfly stage between lanes, on eight elements of each: lanes whose numbers differ in bit S hold the two ends.
// The lower lane gets the sum, the upper one its own element less the lower lane's -- the difference, negated -- in one
// fused operation by +1 or -1 (`side`, by the lane's bit S), whose product is exact.
// Bit 2 of a lane's number in the row is the mirror image within eight lanes (enc_lane), which is what one step of the
// data-parallel path can reach.  The wait states are those between a write and a read through that path.
__device__ __forceinline__ int enc_lane(int t, int L) { return (t ^ ((t & 4) ? 3 : 0)) & (L - 1); }
#define TV_LANE_STAGE(CTRL)                                                                                              \
    asm volatile("s_nop 1\n\t"                                                                                          \
                 "v_fmac_f32_dpp %0, %0, %8 " CTRL " row_mask:0xf bank_mask:0xf\n\t"                                    \
                 "v_fmac_f32_dpp %1, %1, %8 " CTRL " row_mask:0xf bank_mask:0xf\n\t"                                    \
                 "v_fmac_f32_dpp %2, %2, %8 " CTRL " row_mask:0xf bank_mask:0xf\n\t"                                    \
                 "v_fmac_f32_dpp %3, %3, %8 " CTRL " row_mask:0xf bank_mask:0xf\n\t"                                    \
                 "v_fmac_f32_dpp %4, %4, %8 " CTRL " row_mask:0xf bank_mask:0xf\n\t"                                    \
                 "v_fmac_f32_dpp %5, %5, %8 " CTRL " row_mask:0xf bank_mask:0xf\n\t"                                    \
                 "v_fmac_f32_dpp %6, %6, %8 " CTRL " row_mask:0xf bank_mask:0xf\n\t"                                    \
                 "v_fmac_f32_dpp %7, %7, %8 " CTRL " row_mask:0xf bank_mask:0xf"                                         \
                 : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]), "+v"(v[6]), "+v"(v[7])         \
                 : "v"(side))
template <int S>
__device__ __forceinline__ void enc_lane_stage(float (&v)[8], float side) {
    static_assert(S < kEncNegating, "the lanes of a row of sixteen");
    if constexpr (S == 0) TV_LANE_STAGE("quad_perm:[1,0,3,2]");
    if constexpr (S == 1) TV_LANE_STAGE("quad_perm:[2,3,0,1]");
    if constexpr (S == 2) TV_LANE_STAGE("row_half_mirror");
    if constexpr (S == 3) TV_LANE_STAGE("row_ror:8");
}
#undef TV_LANE_STAGE
// The same between lanes 16 (S = 4) or 32 (S = 5) apart: elements that differ in their number's bit S - 4 exchange halves,
// so that a lane holds both ends of one of them, and unless the order they then have will do, change back (nothing is
// negated).  Written out because the compiler copies the operands of every exchange.
#define TV_SWAP_STAGE(SWAP, A0, A1, A2, A3, B0, B1, B2, B3)                                                              \
    asm volatile("s_nop 1\n\t"                                                                                          \
                 SWAP " %4, %8\n\t" SWAP " %5, %9\n\t" SWAP " %6, %10\n\t" SWAP " %7, %11\n\t"                        \
                 "v_add_f32 %0, %4, %8\n\t" "v_sub_f32 %8, %4, %8\n\t"                                                 \
                 "v_add_f32 %1, %5, %9\n\t" "v_sub_f32 %9, %5, %9\n\t"                                                 \
                 "v_add_f32 %2, %6, %10\n\t" "v_sub_f32 %10, %6, %10\n\t"                                              \
                 "v_add_f32 %3, %7, %11\n\t" "v_sub_f32 %11, %7, %11"                                                   \
                 : "=&v"(s0), "=&v"(s1), "=&v"(s2), "=&v"(s3), "+v"(v[A0]), "+v"(v[A1]), "+v"(v[A2]), "+v"(v[A3]),       \
                   "+v"(v[B0]), "+v"(v[B1]), "+v"(v[B2]), "+v"(v[B3]));                                                  \
    if (back)                                                                                                            \
        asm volatile("s_nop 1\n\t"                                                                                      \
                     SWAP " %0, %4\n\t" SWAP " %1, %5\n\t" SWAP " %2, %6\n\t" SWAP " %3, %7"                          \
                     : "+v"(s0), "+v"(s1), "+v"(s2), "+v"(s3), "+v"(v[B0]), "+v"(v[B1]), "+v"(v[B2]), "+v"(v[B3]));      \
    v[A0] = s0; v[A1] = s1; v[A2] = s2; v[A3] = s3
template <int S>
__device__ __forceinline__ void enc_swap_stage(float (&v)[8], bool back) {
    float s0, s1, s2, s3;
    if constexpr (S == 4) {
        TV_SWAP_STAGE("v_permlane16_swap_b32", 0, 2, 4, 6, 1, 3, 5, 7);
    } else {
        TV_SWAP_STAGE("v_permlane32_swap_b32", 0, 1, 4, 5, 2, 3, 6, 7);
    }
}
#undef TV_SWAP_STAGE
// The sum of a row's lanes, in every one of them.
__device__ __forceinline__ double enc_lane_sum(double x, int L) {
    auto other = [](double y, auto ctrl) {
        constexpr int c = decltype(ctrl)::value;
        return __hiloint2double(__builtin_amdgcn_update_dpp(0, __double2hiint(y), c, 0xf, 0xf, false),
                                __builtin_amdgcn_update_dpp(0, __double2loint(y), c, 0xf, 0xf, false));
    };
    x += other(x, IntC<0xB1>{});                      // quad_perm [1,0,3,2]
    x += other(x, IntC<0x4E>{});                      // quad_perm [2,3,0,1]
    x += other(x, IntC<0x141>{});                     // row_half_mirror
    if (L > 8) x += other(x, IntC<0x128>{});          // row_ror:8
    if (L > 16) x += __shfl_xor(x, 16);
    if (L > 32) x += __shfl_xor(x, 32);
    return x;
}

// Sixteen bytes of the caller's rows: a row starts where the caller's pointer says, so four-byte alignment is all
// that is known (the load is the same 16-byte one).
typedef float RowPiece __attribute__((ext_vector_type(4), aligned(4)));

struct EncodeRowsArgs {
    const float *vecs;
    const uint32_t *packed;   // 2 * dim entries (encode_pack_tables)
    const float *shift;       // nullptr for the identity pair
    const float *scale;       // dim, and their reciprocals behind them
    float cen[16];
    float bnd[16];
    int dim, bits, nch, log_block;
    int lanes;                // lanes per row: a power of two, 8 to 64
    int row_stride;           // floats
    int cells;                // boundaries found by cell (enc_cells) instead of one by one
    float cell_mul, cell_add;
    double slack;             // no TQ+ pair: how far the two orders of inner's additions can lie apart
    float inv_sqrt_block;
    uint8_t *nat;
    float *scales;
    size_t old_n, n_new;
};

// Orders a wave's LDS accesses with each other (the LDS serves a wave's requests in order; this keeps
// the compiler from reordering them).
__device__ __forceinline__ void enc_wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// The number of boundaries below a value, from the cell it falls into: a rising map of values to kEncCells cells
// leaves the boundaries of earlier cells below it and those of later cells not, so where no cell holds two
// boundaries one comparison is left (15 boundaries: four levels of three comparisons before).
// (The cell is the integer part of a float at which consecutive integers are neighbours: one fused operation rounds to it.
// NaN goes to cell 0, where it exceeds nothing.)
constexpr int kEncCells = 64;
constexpr float kEncCellZero = 12582912.0f;
struct EncCell { float bound; uint32_t below; };
__host__ __device__ __forceinline__ uint32_t enc_cell_bits(float x, float mul, float add) {
    const float cell = fmaf(x, mul, add), last = kEncCellZero + float(kEncCells - 1);
#ifdef __HIP_DEVICE_COMPILE__
    return __float_as_uint(__builtin_amdgcn_fmed3f(cell, kEncCellZero, last));
#else
    const float in = std::fmin(std::fmax(cell, kEncCellZero), last);
    uint32_t bits;
    std::memcpy(&bits, &in, sizeof bits);
    return bits;
#endif
}
constexpr uint32_t kEncCellZeroBits = 0x4b400000u;
// How far two orders of adding dim terms of the given total magnitude in f64 lie apart at most: dim / 4 + 3
// roundings on the way of any term in the four chains (its product's among them), 8 NG + 6 in k_encode_rows, and the
// few of the magnitude itself and of stepping this far to either side.
__host__ __device__ __forceinline__ double enc_slack(int dim, double mass) { return double(dim + 256) * 0x1p-53 * mass; }

// The row scale with the additions of inner in the reference's order: element j feeds chain j % 4, each chain
// sequential, folded pairwise.  Met by the whole wave; L lanes per row, lane l of them holding groups l, l + L, ...
template <int NG, typename Recon>
__device__ __forceinline__ float enc_in_order(const float (&v)[NG][8], const Recon &recon_of, float *row, int dim, int l, int L, float nrm) {
    const int ng = dim / 8;
    double *terms = reinterpret_cast<double *>(row);               // a run's products: [group of the run][8]
    double chain[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int i = 0; i < NG; ++i) {
        enc_wave_sync();                                           // the run before has been read
        if (l + i * L < ng) {
#pragma unroll
            for (int e = 0; e < 8; ++e) terms[l * 8 + e] = double(v[i][e]) * recon_of(i, e);
        }
        enc_wave_sync();
        const int n_here = 8 * min(L, ng - i * L);
        for (int j = 0; j < n_here; j += 4) {
#pragma unroll
            for (int c = 0; c < 4; ++c) chain[c] = chain[c] + terms[j + c];
        }
    }
    const double inner = (chain[0] + chain[1]) + (chain[2] + chain[3]);
    return inner > 0.1 ? nrm / float(inner) : 0.0f;
}

// NG = groups of eight elements per lane.  The float work of a row is 1220 vector instructions of its wave at 1536 dimensions,
// half of them butterflies, and its norm is a chain of 192 dependent f32 additions: a workgroup
// per row spent most of its time waiting for chains.  Here the norm chains of a workgroup's rows run in one wave, while
// other workgroups of the CU are in their parallel part; the f64 sum needs no chain (enc_slack).  A row is held in
// registers and all stages of a round are done there (the same additions in the same pairs), between lanes through the
// data-parallel path; it is in LDS for the norm and for the two gathers alone.  Its codes leave as
// 16-byte stores that consecutive rows complete to whole lines.  The vector ALU bounds it, busy for 80 % of the clocks.  100K
// rows of 1536 dimensions: 2.02 ms with a workgroup per row, 0.39 with the stages through LDS three at a time, 1.75K instructions a
// row, 0.28 now (2.5 TB/s, every byte once); an add of 100K x 1024: 320 us before, 217 now, 30K x 4096: 1020 and 370, 77K x 1000 with a pair 420 and 205.
// CAL: there is a TQ+ pair.  FULL: rows of NG * 512 dimensions, in blocks as large as they can be: every lane has NG groups and
// all the stages are there, known at compile time.
// Waves per workgroup: four, so that the workgroups of a CU are in different steps and the registers of a SIMD are dealt out
// evenly (us an add with four and eight: 100K x 1536 315 and 319, 200K x 768 387 and 432, 100K x 1024 217 and 238; with six: 40K x 3072
// 351 and 462; with two: 60K x 2048 264 and 270); eight where a lane has one group of elements, rows of up to 512 dimensions (400K x 128 120 and 121).
constexpr int enc_waves(int ng) { return ng == 1 ? 8 : 4; }
constexpr int enc_waves_per_simd(int ng, bool full) { return ng == 1 ? 6 : ng == 2 ? 5 : ng <= 4 ? 4 : ng <= 6 && !full ? 3 : 2; }    // what their registers leave room for
template <int NG, bool CAL, bool FULL>
__global__ __launch_bounds__(enc_waves(NG) * 64, enc_waves_per_simd(NG, FULL)) void k_encode_rows(EncodeRowsArgs a) {
    extern __shared__ __align__(16) float enc_lds[];
    int t = threadIdx.x;
    const int dim = FULL ? NG * 512 : a.dim, ng = dim / 8, L = FULL ? 64 : a.lanes;
    const int rs = FULL ? enc_row_stride(NG * 512, 64) : a.row_stride, lb = FULL ? 9 + __builtin_ctz(NG) : a.log_block;
    constexpr int kThreads = enc_waves(NG) * 64;
    const int R = kThreads / L;                                      // rows of a workgroup
    uint32_t *s_codes = reinterpret_cast<uint32_t *>(enc_lds + R * rs);   // [R][ng] eight codes each, packed as in the index
    float2 *s_norm = reinterpret_cast<float2 *>(enc_lds + (R * rs + R * ng + 1) / 2 * 2);   // [R] norm and what rows are multiplied by
    double *s_cen = reinterpret_cast<double *>(s_norm + R);        // centroids in f64
    int r = t / L;                                                 // this thread's row of the group ...
    int l = enc_lane(t, L);                                        // ... and its lane in the row
    const int half = enc_half(L);
    EncCell *s_cell = reinterpret_cast<EncCell *>(s_cen + 16);
    if (t < 16) s_cen[t] = double(a.cen[t]);
    if (t < kEncCells) {
        // (the boundary of this cell, if it has one, and how many lie in the cells before it)
        EncCell cell{__int_as_float(0x7f800000), 0u};
        for (int b = 0; b < (1 << a.bits) - 1; ++b) {
            const int k = int(enc_cell_bits(a.bnd[b], a.cell_mul, a.cell_add) - kEncCellZeroBits);
            if (k < t) ++cell.below;
            if (k == t) cell.bound = a.bnd[b];
        }
        s_cell[t] = cell;
    }

    constexpr bool kFetchEarly = NG <= 3 && !(CAL && NG == 2);      // (longer rows, and a pair, leave no registers for it)
    const size_t n_groups = (a.n_new + R - 1) / R;
    RowPiece pre[NG][2];
    auto fetch = [&](size_t grp) {
        // (lanes without a row or a group of their own read the last one's)
        const uint8_t *rows = reinterpret_cast<const uint8_t *>(a.vecs + grp * R * size_t(dim));
        const int rr = int(min(size_t(r), a.n_new - 1 - grp * R));
#pragma unroll
        for (int i = 0; i < NG; ++i) {
            const RowPiece *src = reinterpret_cast<const RowPiece *>(rows + uint32_t(rr * dim + (FULL ? l + i * L : min(l + i * L, ng - 1)) * 8) * 4u);
            pre[i][0] = src[0];
            pre[i][1] = src[1];
        }
    };
    // All butterfly stages of a round on the row's groups, in registers.  (Lanes without a group take part.)
    const float side[4] = {l & 1 ? -1.0f : 1.0f, l & 2 ? -1.0f : 1.0f, l & 4 ? -1.0f : 1.0f, l & 8 ? -1.0f : 1.0f};
    auto stages = [&](float (&v)[NG][8], bool back) {
        auto each = [&](auto &&f) {
#pragma unroll
            for (int i = 0; i < NG; ++i) f(v[i]);
            __builtin_amdgcn_sched_barrier(0);      // (one stage after the other, nothing loaded ahead: it would spill)
        };
        each([](float (&x)[8]) { butterflies<3>(x); });
        if (lb > 3) each([&](float (&x)[8]) { enc_lane_stage<0>(x, side[0]); });
        if (lb > 4) each([&](float (&x)[8]) { enc_lane_stage<1>(x, side[1]); });
        if (lb > 5) each([&](float (&x)[8]) { enc_lane_stage<2>(x, side[2]); });
        if (lb > 6) each([&](float (&x)[8]) { enc_lane_stage<3>(x, side[3]); });
        if (lb > 7) each([&](float (&x)[8]) { enc_swap_stage<4>(x, back); });
        if (lb > 8) each([&](float (&x)[8]) { enc_swap_stage<5>(x, back); });
        static_for<3>([&](auto bb) {      // between a lane's groups
            constexpr int far = 1 << decltype(bb)::value;
            if constexpr (NG > far) {
                if (lb > 9 + decltype(bb)::value) {
#pragma unroll
                    for (int i = 0; i < NG; ++i) {
                        if ((i & far) != 0 || i + far >= NG) continue;
#pragma unroll
                        for (int e = 0; e < 8; ++e) {
                            const float x = v[i][e], y = v[i + far][e];
                            v[i][e] = x + y;
                            v[i + far][e] = x - y;
                        }
                    }
                }
            }
        });
    };

    const float last_factor = enc_negated(l, lb) ? -a.inv_sqrt_block : a.inv_sqrt_block;
    size_t grp = blockIdx.x;
    if (grp < n_groups) fetch(grp);
    for (; grp < n_groups; grp += gridDim.x) {
        // (opaque in every turn and step: the addresses derived from it, kept in registers from one to
        // the next, would spill)
        asm volatile("" : "+v"(l), "+v"(r), "+v"(t));
        float *row = enc_lds + r * rs;
        const uint32_t row_at = uint32_t(reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) float *)row));
        uint32_t tab[NG][8];
        auto fetch_table = [&](int round) {
#pragma unroll
            for (int i = 0; i < NG; ++i) {
                const uint4 *src = reinterpret_cast<const uint4 *>(reinterpret_cast<const uint8_t *>(a.packed + round * dim) + uint32_t(FULL ? l + i * L : min(l + i * L, ng - 1)) * 32u);
                const uint4 x = src[0], y = src[1];
                tab[i][0] = x.x; tab[i][1] = x.y; tab[i][2] = x.z; tab[i][3] = x.w;
                tab[i][4] = y.x; tab[i][5] = y.y; tab[i][6] = y.z; tab[i][7] = y.w;
            }
        };
        fetch_table(0);
        auto put = [&](int i, float4 x, float4 y) {
            float *at = row + 4 * l + 2 * i * half;
            if (FULL || l + i * L < ng) {
                *reinterpret_cast<float4 *>(at) = x;
                *reinterpret_cast<float4 *>(at + half) = y;
            }
        };
#pragma unroll
        for (int i = 0; i < NG; ++i)
            put(i, float4{pre[i][0].x, pre[i][0].y, pre[i][0].z, pre[i][0].w}, float4{pre[i][1].x, pre[i][1].y, pre[i][1].z, pre[i][1].w});
        __syncthreads();
        // encode.rs:920-932: c[j % 8] += x * x (separate multiply and add), then the pairwise fold
        for (int idx = t; idx < 8 * R; idx += kThreads) {
            const float *x = enc_lds + (idx >> 3) * rs + ((idx >> 2) & 1) * half + (idx & 3);
            auto group = [&](int g) { return x + g / L * 2 * half + g % L * 4; };      // (eight from a multiple of eight on lie side by side)
            float c = 0.0f;
            int i = 0;
            if (ng >= 8) {
                // eight groups of eight at a time, the next ones on their way
                float v[2][8];
                auto load = [&](float (&to)[8], int g) {
                    const float *from = group(g);
#pragma unroll
                    for (int e = 0; e < 8; ++e) to[e] = from[4 * e];
                };
                auto add = [&](const float (&from)[8]) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) c = c + from[e] * from[e];
                };
                load(v[0], 0);
#pragma unroll 1
                for (; i + 24 <= ng; i += 16) {
                    load(v[1], i + 8);
                    add(v[0]);
                    load(v[0], i + 16);
                    add(v[1]);
                }
                add(v[0]);
                i += 8;
                if (i + 8 <= ng) { load(v[1], i); add(v[1]); i += 8; }
            }
            for (; i < ng; ++i) { const float v = *group(i); c = c + v * v; }
            // (a row's eight chains lie side by side; a + b is b + a)
            c += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(c), 0xB1, 0xf, 0xf, false));
            c += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(c), 0x4E, 0xf, 0xf, false));
            c += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(c), 0x141, 0xf, 0xf, false));
            const float nrm = sqrtf(c);
            if ((idx & 7) == 0) s_norm[idx >> 3] = float2{nrm, nrm > 1e-10f ? 1.0f / nrm : 0.0f};   // lib.rs:163 MIN_INPUT_NORM
        }
        __syncthreads();
        const float2 norm = s_norm[r];
        const float nrm = norm.x, inv = norm.y;

        // rotation (rotation.rs:218-255): gather, sign, stages; the factor rides the gather
        float v[NG][8];
#pragma unroll
        for (int round = 0; round < 2; ++round) {
            asm volatile("" : "+v"(l));
            const uint32_t factor = __float_as_uint(round == 0 ? inv : a.inv_sqrt_block);
#pragma unroll
            for (int i = 0; i < NG; ++i) {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const uint32_t w = tab[i][e];
                    uint32_t at;      // (the row's address and the word's lower half)
                    asm("v_add_u32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:WORD_0" : "=v"(at) : "v"(row_at), "v"(w));
                    const float x = *reinterpret_cast<const __attribute__((address_space(3))) float *>(uintptr_t(at));
                    v[i][e] = x * __uint_as_float((factor & 0x7fffffffu) | (w & 0x80000000u));      // (x * factor) * +-1; no factor is negative
                }
            }
            enc_wave_sync();                                       // every lane has gathered before any overwrites
            __builtin_amdgcn_sched_barrier(0);
            if (round == 0) fetch_table(1);
            if (kFetchEarly && round == 1 && grp + gridDim.x < n_groups) fetch(grp + gridDim.x);
            __builtin_amdgcn_sched_barrier(0);
            stages(v, round == 1);
            if (round == 0) {
#pragma unroll
                for (int i = 0; i < NG; ++i) put(i, float4{v[i][0], v[i][1], v[i][2], v[i][3]}, float4{v[i][4], v[i][5], v[i][6], v[i][7]});
                enc_wave_sync();
            }
        }
#pragma unroll
        for (int i = 0; i < NG; ++i) {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[i][e] = v[i][e] * last_factor;
        }

        // encode.rs:600-640: code = number of boundaries below the calibrated value
        asm volatile("" : "+v"(l));
        uint32_t code4[NG];
        // encode.rs:1442-1475: inner = <rotated, reconstruction> in f64, four chains by j % 4.  The row scale takes
        // float(inner), so the order of the additions shows only where it moves inner across a rounding boundary: the
        // lanes add their own elements, then each other's sums, and where every value within the two orders' distance
        // gives the same row scale, that is it.
        auto recon_of = [&](uint32_t code, int j) -> double {
            double recon = s_cen[code];                                                        // (no TQ+ pair: * 1 - 0)
            if constexpr (CAL) recon = recon * double(a.scale[dim + j]) - double(a.shift[j]);  // encode.rs:594
            return recon;
        };
        double inner = 0.0, mass = 0.0;                            // the sum, and (for a pair) the sum of the terms' magnitudes
#pragma unroll
        for (int i = 0; i < NG; ++i) {
            const int g = l + i * L;
            if (!FULL && g >= ng) continue;
            uint32_t c[8];
            auto calibrated = [&](int e) {
                float x = v[i][e];
                if constexpr (CAL) x = (x + a.shift[8 * g + e]) * a.scale[8 * g + e];
                return x;
            };
            if (a.cells) {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float x = calibrated(e);
                    const EncCell cell = s_cell[enc_cell_bits(x, a.cell_mul, a.cell_add) - kEncCellZeroBits];
                    c[e] = cell.below + (x > cell.bound ? 1u : 0u);
                    if (CAL && e == 3) __builtin_amdgcn_sched_barrier(0);
                }
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float x = calibrated(e);
                    c[e] = 0u;
#pragma unroll 1
                    for (int b = 0; b < (1 << a.bits) - 1; ++b) c[e] += x > a.bnd[b] ? 1u : 0u;
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            if (CAL) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const double recon = recon_of(c[e], 8 * g + e), x = double(v[i][e]);
                inner = fma(x, recon, inner);
                if constexpr (CAL) mass = fma(fabs(x), fabs(recon), mass);
                if (e == 3) __builtin_amdgcn_sched_barrier(0);
            }
            code4[i] = c[0] | c[1] << 4 | c[2] << 8 | c[3] << 12 | c[4] << 16 | c[5] << 20 | c[6] << 24 | c[7] << 28;
            // pack.rs:264-282: first dimension in the high bits; 3-bit codes sit in 4-bit fields
            s_codes[r * ng + g] = a.bits == 2 ? (c[0] << 6 | c[1] << 4 | c[2] << 2 | c[3]) | (c[4] << 6 | c[5] << 4 | c[6] << 2 | c[7]) << 8
                                              : ((code4[i] >> 4) & 0x0f0f0f0fu) | ((code4[i] & 0x0f0f0f0fu) << 4);
            __builtin_amdgcn_sched_barrier(0);      // (one group after the other: several at once would spill)
        }
        inner = enc_lane_sum(inner, L);
        if constexpr (CAL) mass = enc_lane_sum(mass, L);
        const double slack = CAL ? enc_slack(dim, mass) : a.slack;
        const double lo = inner - slack, hi = inner + slack;
        float scale = lo > 0.1 ? nrm / float(lo) : 0.0f;                                       // encode.rs:1194-1200
        const bool settled = lo > 0.1 ? float(lo) == float(hi) : hi <= 0.1;                    // (NaN: not settled)
        if (__any(!settled)) {                                                                 // one row in 10^5
            // (opaque: what the sum above was made of, kept in registers for this, would spill)
            asm volatile("" : "+v"(l));
#pragma unroll
            for (int i = 0; i < NG; ++i) {
                asm volatile("" : "+v"(code4[i]));
#pragma unroll
                for (int e = 0; e < 8; ++e) asm volatile("" : "+v"(v[i][e]));
            }
            scale = enc_in_order<NG>(v, [&](int i, int e) { return recon_of((code4[i] >> (4 * e)) & 15u, 8 * (l + i * L) + e); }, row, dim, l, L, nrm);
        }
        if (l == 0 && grp * R + r < a.n_new) a.scales[a.old_n + grp * R + r] = scale;
        __syncthreads();                                           // every row's codes are there
        // the rows' code bytes, 16 at a time, into their lanes of the device layout (pack.rs:211-233
        // append_lanes), the bytes past a row's last group zero: nothing need have been cleared for a row
        const int per = a.bits == 2 ? 8 : 4, pieces = 2 * a.nch;
        for (int idx = t; idx < R * pieces; idx += kThreads) {
            const int rr = idx % R, p = idx / R;
            const size_t vec = grp * R + rr;
            if (vec >= a.n_new) continue;
            uint32_t o[4] = {0u, 0u, 0u, 0u};
            const uint32_t *src = s_codes + rr * ng + p * per;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                if (e >= per || p * per + e >= ng) continue;
                if (a.bits == 2) o[e >> 1] |= src[e] << (16 * (e & 1));
                else o[e & 3] = src[e];
            }
            *reinterpret_cast<uint4 *>(a.nat + enc_byte_index(a.old_n + vec, 16 * p, a.nch)) = uint4{o[0], o[1], o[2], o[3]};
        }
        if (!kFetchEarly && grp + gridDim.x < n_groups) fetch(grp + gridDim.x);
    }
}

template <int NG, bool CAL, bool FULL>
static hipError_t launch_encode_rows_full(const EncodeRowsArgs &a, int device, hipStream_t s) {
    constexpr int kThreads = enc_waves(NG) * 64;
    const int R = kThreads / a.lanes, ng = a.dim / 8;
    const size_t lds = size_t(R * a.row_stride + R * ng + 2 * R + 2) * 4 + 16 * 8 + kEncCells * sizeof(EncCell);
    if (lds > 160 * 1024) return hipErrorInvalidValue;
    const void *kernel = reinterpret_cast<const void *>(k_encode_rows<NG, CAL, FULL>);
    hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
    if (e != hipSuccess) return e;
    // a workgroup keeps its tables for all its turns: as many as are resident at once, by registers and LDS
    const size_t groups = (a.n_new + R - 1) / R;
    const size_t resident = size_t(device_cus(device)) * std::max<size_t>(1, std::min<size_t>(size_t(4 * enc_waves_per_simd(NG, FULL)) / enc_waves(NG), 160 * 1024 / lds));
    hipLaunchKernelGGL((k_encode_rows<NG, CAL, FULL>), dim3(unsigned(std::min(groups, resident))), dim3(kThreads), lds, s, a);
    return hipGetLastError();
}
template <int NG, bool CAL>
static hipError_t launch_encode_rows_cal(const EncodeRowsArgs &a, int device, hipStream_t s) {
    // (with a pair the straight-line code would spill)
    if constexpr (!CAL)
        if (a.dim == NG * 512 && a.log_block == 9 + __builtin_ctz(NG)) return launch_encode_rows_full<NG, CAL, true>(a, device, s);
    return launch_encode_rows_full<NG, CAL, false>(a, device, s);
}
template <int NG>
static hipError_t launch_encode_rows_n(const EncodeRowsArgs &a, int device, hipStream_t s) {
    return a.scale != nullptr ? launch_encode_rows_cal<NG, true>(a, device, s) : launch_encode_rows_cal<NG, false>(a, device, s);
}

// A and B, one float row each; codes and the f64 products overlay A.  128 KiB at the largest
// row the index accepts (16384 dimensions), inside the 160 KiB a workgroup may have.
static_assert(size_t(2) * 16384 * sizeof(float) + 4 * sizeof(double) <= 160 * 1024,
              "the longest row the index accepts (lib.rs:101 MAX_DIM) must fit a workgroup's LDS");
size_t encode_lds_bytes(int dim) { return size_t(2) * size_t(dim) * sizeof(float) + 4 * sizeof(double); }

hipError_t launch_encode(const float *d_vecs, size_t n_new, size_t old_n, const float *d_signs,
                         const uint32_t *d_perms, const uint32_t *d_packed, const float *d_shift, const float *d_scale,
                         const float *centroids, const float *boundaries, const Geometry &g, int block,
                         float inv_sqrt_block, uint8_t *d_native, float *d_scales, float *d_rot_out,
                         int device, hipStream_t s) {
    if (n_new == 0) return hipSuccess;
    if (d_packed != nullptr && d_rot_out == nullptr) {
        EncodeRowsArgs a;
        a.vecs = d_vecs; a.packed = d_packed; a.shift = d_shift; a.scale = d_scale;
        const int nl = 1 << g.bits;
        for (int i = 0; i < 16; ++i) { a.cen[i] = i < nl ? centroids[i] : 0.0f; a.bnd[i] = i < nl - 1 ? boundaries[i] : 0.0f; }
        a.dim = g.dim; a.bits = g.bits; a.nch = g.nch;
        a.log_block = __builtin_ctz(unsigned(block));
        a.lanes = enc_lanes(g.dim);
        a.row_stride = enc_row_stride(g.dim, a.lanes);
        // cells of equal width from the first boundary to the last; no two boundaries may share one, and handed-over
        // centroids may be in any order, equal, infinite or NaN
        const int nb = nl - 1;
        a.cell_mul = float(kEncCells - 2) / (a.bnd[nb - 1] - a.bnd[0]);
        a.cell_add = 1.0f - a.bnd[0] * a.cell_mul + kEncCellZero;
        a.cells = a.cell_mul > 0.0f && a.cell_mul < 1e30f && std::fabs(a.cell_add) < 1e30f;
        for (int i = 0; a.cells && i + 1 < nb; ++i)
            a.cells = a.bnd[i] < a.bnd[i + 1] && enc_cell_bits(a.bnd[i], a.cell_mul, a.cell_add) < enc_cell_bits(a.bnd[i + 1], a.cell_mul, a.cell_add);
        // without a pair the terms are x * centroid over a row of length 1: |x c| <= (x^2 + c^2) / 2
        double c_max = 0.0;
        for (int i = 0; i < nl; ++i) c_max = std::fabs(double(centroids[i])) >= c_max ? std::fabs(double(centroids[i])) : c_max;
        a.slack = enc_slack(g.dim, (1.01 + double(g.dim) * c_max * c_max) / 2.0);
        a.inv_sqrt_block = inv_sqrt_block;
        a.nat = d_native; a.scales = d_scales; a.old_n = old_n; a.n_new = n_new;
        switch ((g.dim / 8 + a.lanes - 1) / a.lanes) {
            case 1: return launch_encode_rows_n<1>(a, device, s);
            case 2: return launch_encode_rows_n<2>(a, device, s);
            case 3: return launch_encode_rows_n<3>(a, device, s);
            case 4: return launch_encode_rows_n<4>(a, device, s);
            case 5: case 6: return launch_encode_rows_n<6>(a, device, s);
            default: return launch_encode_rows_n<8>(a, device, s);
        }
    }
    EncodeArgs a;
    a.vecs = d_vecs; a.signs = d_signs; a.perms = d_perms; a.shift = d_shift; a.scale = d_scale;
    const int nl = 1 << g.bits;
    for (int i = 0; i < 16; ++i) { a.cen[i] = i < nl ? centroids[i] : 0.0f; a.bnd[i] = i < nl - 1 ? boundaries[i] : 0.0f; }
    a.dim = g.dim; a.bits = g.bits; a.G = g.G; a.nch = g.nch; a.block = block;
    a.inv_sqrt_block = inv_sqrt_block;
    a.nat = d_native; a.scales = d_scales; a.old_n = old_n; a.n_new = n_new;
    a.rot_out = d_rot_out;
    const size_t lds = encode_lds_bytes(g.dim);
    if (lds > 48 * 1024) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(k_encode),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(k_encode, dim3(unsigned(n_new)), dim3(256), lds, s, a);
    return hipGetLastError();
}

}  // namespace tv
