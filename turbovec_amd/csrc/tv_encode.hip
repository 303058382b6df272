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
// row and a group of eight waves' rows through each step together, so that the
// sequential chains of all of them run side by side in the lanes of one or two
// waves.  k_encode takes one workgroup per row: longer rows, the rotated rows of
// a TQ+ fit, and tables whose signs are not +-1.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
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
// A row lies in LDS with eight floats of padding after every 64, and rows follow each other at a
// stride of 8 modulo 64 floats: the passes below, whose lanes are 64 floats apart in groups of eight,
// and the chains, whose lanes are a row apart, then spread over all banks.
__host__ __device__ constexpr int enc_at(int j) { return j + (j >> 6) * 8; }
// (and a row's place holds the f64 products of one run of its groups, 16 lanes floats, where enc_in_order needs it)
static int enc_row_stride(int dim, int lanes) {
    int s = std::max(enc_at(dim - 1) + 1, 16 * lanes + 16);
    while (s % 64 != 8) ++s;
    return s;
}
// A position's entry of the packed rotation tables: where each round's gather reads (the padded place),
// and the round's sign above it.
constexpr int kEncMaxDim = 4096;
static_assert(enc_at(kEncMaxDim - 1) < (1 << 15), "a padded place takes fifteen bits");
bool encode_pack_tables(const float *signs, const uint32_t *perms, int dim, uint32_t *packed) {
    if (dim > kEncMaxDim) return false;
    // (a rotation keeps a row's length, which enc_slack counts on: both gathers must be permutations)
    for (int r = 0; r < 2; ++r) {
        std::vector<bool> seen(size_t(dim), false);
        for (int j = 0; j < dim; ++j) {
            if (seen[perms[size_t(r) * dim + j]]) return false;
            seen[perms[size_t(r) * dim + j]] = true;
        }
    }
    for (int j = 0; j < dim; ++j) {
        uint32_t w = 0;
        for (int r = 0; r < 2; ++r) {
            const float s = signs[size_t(r) * dim + j];
            if (s != 1.0f && s != -1.0f) return false;
            w |= (uint32_t(enc_at(int(perms[size_t(r) * dim + j]))) | (s < 0.0f ? 0x8000u : 0u)) << (16 * r);
        }
        packed[j] = w;
    }
    return true;
}

// Sixteen bytes of the caller's rows: a row starts where the caller's pointer says, so four-byte alignment is all
// that is known (the load is the same 16-byte one).
typedef float RowPiece __attribute__((ext_vector_type(4), aligned(4)));

struct EncodeRowsArgs {
    const float *vecs;
    const uint32_t *packed;   // dim entries (encode_pack_tables)
    const float *shift;       // nullptr for the identity pair
    const float *scale;
    float cen[16];
    float bnd[16];
    int dim, bits, G, nch, log_block;
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
constexpr int kEncCells = 64;
struct EncCell { float bound; uint32_t below; };
__host__ __device__ __forceinline__ int enc_cell(float x, float mul, float add) {
#ifdef __HIP_DEVICE_COMPILE__
    uint32_t c;
    asm("v_cvt_u32_f32 %0, %1" : "=v"(c) : "v"(fmaf(x, mul, add)));               // saturates; NaN: cell 0, where it exceeds nothing
    return int(min(c, uint32_t(kEncCells - 1)));
#else
    return int(std::fmin(std::fmax(std::fmaf(x, mul, add), 0.0f), float(kEncCells - 1)));
#endif
}
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

// NG = groups of eight elements per lane; W = waves per workgroup.  The float work of a row is a few
// thousand instructions of its wave, but its norm is a chain of 192 dependent f32 additions (1536 dimensions): a workgroup
// per row spent most of its time waiting for chains.  Here the norm chains of a workgroup's rows run in one wave, while
// other workgroups of the CU are in their parallel part; the f64 sum needs no chain (enc_slack).  A row's rotation
// goes through LDS three stages at a time in registers (the same additions in the same pairs), and its codes leave as
// 16-byte stores that consecutive rows complete to whole lines.  100K rows of 1536 dimensions: 2.02 ms with a workgroup per
// row, 0.50 with the f64 chains too in one wave and four levels of three comparisons per value, 0.39 now (1.8 TB/s, every
// byte once); of 2048: 1.15 -> 0.62.
// CAL: there is a TQ+ pair.
constexpr int enc_waves_per_simd(int ng) { return ng == 1 ? 6 : ng == 2 ? 5 : ng <= 4 ? 4 : 2; }    // what their registers leave room for
template <int NG, int W, bool CAL>
__global__ __launch_bounds__(W * 64, enc_waves_per_simd(NG)) void k_encode_rows(EncodeRowsArgs a) {
    extern __shared__ __align__(16) float enc_lds[];
    const int dim = a.dim, t = threadIdx.x, ng = dim / 8, rs = a.row_stride, L = a.lanes;
    const int R = W * 64 / L;                                      // rows of a workgroup
    uint32_t *s_codes = reinterpret_cast<uint32_t *>(enc_lds + R * rs);   // [R][ng] eight codes each, packed as in the index
    float *s_part = reinterpret_cast<float *>(s_codes + R * ng);   // [R][8] chains of the squared norm
    double *s_cen = reinterpret_cast<double *>(enc_lds + (R * rs + R * ng + 8 * R + 3) / 4 * 4);   // centroids in f64
    const int r = t / L;                                           // this thread's row of the group ...
    int l = t % L;                                                 // ... and its lane in the row
    float *row = enc_lds + r * rs;
    EncCell *s_cell = reinterpret_cast<EncCell *>(s_cen + 16);
    if (t < 16) s_cen[t] = double(a.cen[t]);
    if (t < kEncCells) {
        // (the boundary of this cell, if it has one, and how many lie in the cells before it)
        EncCell cell{__int_as_float(0x7f800000), 0u};
        for (int b = 0; b < (1 << a.bits) - 1; ++b) {
            const int k = enc_cell(a.bnd[b], a.cell_mul, a.cell_add);
            if (k < t) ++cell.below;
            if (k == t) cell.bound = a.bnd[b];
        }
        s_cell[t] = cell;
    }

    const size_t n_groups = (a.n_new + R - 1) / R;
    RowPiece pre[NG][2];
    auto fetch = [&](size_t grp) {
        const size_t rr = grp * R + r;
#pragma unroll
        for (int i = 0; i < NG; ++i) {
            const int g = l + i * L;
            pre[i][0] = pre[i][1] = RowPiece{0.0f, 0.0f, 0.0f, 0.0f};
            if (rr < a.n_new && g < ng) {
                const RowPiece *src = reinterpret_cast<const RowPiece *>(a.vecs + rr * size_t(dim)) + 2 * g;
                pre[i][0] = src[0];
                pre[i][1] = src[1];
            }
        }
    };
    // R stages from stride 2^S on, over this wave's rows; `last`: the scale is applied on the way out.
    // Elements 2^S apart are a fixed distance apart in the padded row: 8 within a run of 64, nine
    // eighths of their distance beyond.
    auto pass = [&](auto ss, auto rr_, bool last) {
        constexpr int S = decltype(ss)::value, N = 1 << decltype(rr_)::value, per = 8 / N;
        constexpr int apart = S == 3 ? 8 : (1 << S) / 8 * 9;
        asm volatile("" : "+v"(l));
        enc_wave_sync();
#pragma unroll
        for (int i = 0; i < per * NG; ++i) {
            const int g = l + i * L;
            if (g >= per * ng) continue;
            float *at = row + enc_at(((g >> S) << S) * N + (g & ((1 << S) - 1)));
            float v[N];
#pragma unroll
            for (int e = 0; e < N; ++e) v[e] = at[e * apart];
            butterflies<decltype(rr_)::value>(v);
            if (last) {
#pragma unroll
                for (int e = 0; e < N; ++e) v[e] = v[e] * a.inv_sqrt_block;
            }
#pragma unroll
            for (int e = 0; e < N; ++e) at[e * apart] = v[e];
        }
    };
    auto passes = [&](bool scaled) {
        const int lb = a.log_block;
        auto from = [&](auto ss) {
            constexpr int S = decltype(ss)::value;
            if (lb >= S + 3) pass(ss, IntC<3>{}, scaled && lb == S + 3);
            else if (lb == S + 2) pass(ss, IntC<2>{}, scaled);
            else if (lb == S + 1) pass(ss, IntC<1>{}, scaled);
        };
        from(IntC<3>{});
        if (NG * 64 * 8 > 64) from(IntC<6>{});
        if (lb > 9) from(IntC<9>{});
        enc_wave_sync();
    };

    size_t grp = blockIdx.x;
    if (grp < n_groups) fetch(grp);
    for (; grp < n_groups; grp += gridDim.x) {
        // (opaque in every turn and step: the addresses derived from it, kept in registers from one to
        // the next, would spill)
        asm volatile("" : "+v"(l));
        uint32_t tab[NG][8];
#pragma unroll
        for (int i = 0; i < NG; ++i) {
            const uint4 *src = reinterpret_cast<const uint4 *>(a.packed) + 2 * min(l + i * L, ng - 1);
            const uint4 x = src[0], y = src[1];
            tab[i][0] = x.x; tab[i][1] = x.y; tab[i][2] = x.z; tab[i][3] = x.w;
            tab[i][4] = y.x; tab[i][5] = y.y; tab[i][6] = y.z; tab[i][7] = y.w;
        }
#pragma unroll
        for (int i = 0; i < NG; ++i) {
            const int g = l + i * L;
            if (g < ng) {
                float4 *dst = reinterpret_cast<float4 *>(row + enc_at(8 * g));
                dst[0] = float4{pre[i][0].x, pre[i][0].y, pre[i][0].z, pre[i][0].w};
                dst[1] = float4{pre[i][1].x, pre[i][1].y, pre[i][1].z, pre[i][1].w};
            }
        }
        __syncthreads();
        // encode.rs:920-932: c[j % 8] += x * x (separate multiply and add), then the pairwise fold
        for (int idx = t; idx < 8 * R; idx += W * 64) {
            const float *x = enc_lds + (idx >> 3) * rs + (idx & 7);
            float c = 0.0f;
            int i = 0;
            if (ng >= 8) {
                // eight groups of eight -- 64 floats and their padding -- at a time, the next ones on their way
                float v[2][8];
                auto load = [&](float (&to)[8], int at) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) to[e] = x[9 * at + 8 * e];
                };
                auto add = [&](const float (&from)[8]) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) c = c + from[e] * from[e];
                };
                load(v[0], 0);
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
            for (; i < ng; ++i) { const float v = x[8 * i + (i >> 3) * 8]; c = c + v * v; }
            s_part[idx] = c;
        }
        __syncthreads();
        const float *p8 = s_part + r * 8;
        const float nrm = sqrtf(((p8[0] + p8[1]) + (p8[2] + p8[3])) + ((p8[4] + p8[5]) + (p8[6] + p8[7])));
        const float inv = nrm > 1e-10f ? 1.0f / nrm : 0.0f;   // lib.rs:163 MIN_INPUT_NORM

        // rotation (rotation.rs:218-255): gather, sign, stages; the factor rides the gather
#pragma unroll
        for (int round = 0; round < 2; ++round) {
            asm volatile("" : "+v"(l));
            const float factor = round == 0 ? inv : a.inv_sqrt_block;
            float v[NG][8];
#pragma unroll
            for (int i = 0; i < NG; ++i) {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const uint32_t w = tab[i][e];
                    const uint32_t at = round == 0 ? w & 0x7fffu : (w >> 16) & 0x7fffu;
                    const uint32_t sign = (round == 0 ? w << 16 : w) & 0x80000000u;
                    v[i][e] = __uint_as_float(__float_as_uint(row[at] * factor) ^ sign);     // (x * factor) * +-1
                }
            }
            enc_wave_sync();                                       // every lane has gathered before any overwrites
            if (NG <= 3 && round == 1 && grp + gridDim.x < n_groups) fetch(grp + gridDim.x);    // (longer rows leave no registers for it)
#pragma unroll
            for (int i = 0; i < NG; ++i) {
                const int g = l + i * L;
                butterflies<3>(v[i]);
                if (round == 1 && a.log_block == 3) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) v[i][e] = v[i][e] * a.inv_sqrt_block;
                }
                if (g < ng) {
                    float4 *dst = reinterpret_cast<float4 *>(row + enc_at(8 * g));
                    dst[0] = float4{v[i][0], v[i][1], v[i][2], v[i][3]};
                    dst[1] = float4{v[i][4], v[i][5], v[i][6], v[i][7]};
                }
            }
            passes(round == 1);
        }

        // encode.rs:600-640: code = number of boundaries below the calibrated value
        asm volatile("" : "+v"(l));
        float v[NG][8];
        uint32_t code4[NG];
#pragma unroll
        for (int i = 0; i < NG; ++i) {
            const int g = l + i * L;
            if (g >= ng) continue;
            const float4 *src = reinterpret_cast<const float4 *>(row + enc_at(8 * g));
            const float4 x = src[0], y = src[1];
            v[i][0] = x.x; v[i][1] = x.y; v[i][2] = x.z; v[i][3] = x.w;
            v[i][4] = y.x; v[i][5] = y.y; v[i][6] = y.z; v[i][7] = y.w;
            uint32_t c[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                float x = v[i][e];
                if constexpr (CAL) x = (x + a.shift[8 * g + e]) * a.scale[8 * g + e];
                if (a.cells) {
                    const EncCell cell = s_cell[enc_cell(x, a.cell_mul, a.cell_add)];
                    c[e] = cell.below + (x > cell.bound ? 1u : 0u);
                } else {
                    c[e] = 0u;
                    for (int b = 0; b < (1 << a.bits) - 1; ++b) c[e] += x > a.bnd[b] ? 1u : 0u;
                }
            }
            code4[i] = c[0] | c[1] << 4 | c[2] << 8 | c[3] << 12 | c[4] << 16 | c[5] << 20 | c[6] << 24 | c[7] << 28;
            // pack.rs:264-282: first dimension in the high bits; 3-bit codes sit in 4-bit fields
            s_codes[r * ng + g] = a.bits == 2 ? (c[0] << 6 | c[1] << 4 | c[2] << 2 | c[3]) | (c[4] << 6 | c[5] << 4 | c[6] << 2 | c[7]) << 8
                                              : ((code4[i] >> 4) & 0x0f0f0f0fu) | ((code4[i] & 0x0f0f0f0fu) << 4);
            __builtin_amdgcn_sched_barrier(0);      // (one group after the other: several at once would spill)
        }
        // encode.rs:1442-1475: inner = <rotated, reconstruction> in f64, four chains by j % 4.  The row scale takes
        // float(inner), so the order of the additions shows only where it moves inner across a rounding boundary: the
        // lanes add their own elements, then each other's sums, and where every value within the two orders' distance
        // gives the same row scale, that is it.
        auto recon_of = [&](int i, int e) -> double {
            double recon = s_cen[(code4[i] >> (4 * e)) & 15u];                                 // (no TQ+ pair: * 1 - 0)
            if constexpr (CAL) {
                const int j = 8 * (l + i * L) + e;
                recon = recon * double(1.0f / a.scale[j]) - double(a.shift[j]);                // encode.rs:594
            }
            return recon;
        };
        double inner = 0.0, mass = 0.0;                            // the sum, and (for a pair) the sum of the terms' magnitudes
#pragma unroll
        for (int i = 0; i < NG; ++i) {
            if (l + i * L >= ng) continue;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const double recon = recon_of(i, e), x = double(v[i][e]);
                inner = fma(x, recon, inner);
                if constexpr (CAL) mass = fma(fabs(x), fabs(recon), mass);
                if (e == 3) __builtin_amdgcn_sched_barrier(0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        for (int d = 1; d < L; d <<= 1) {
            inner += __shfl_xor(inner, d);
            if constexpr (CAL) mass += __shfl_xor(mass, d);
        }
        const double slack = CAL ? enc_slack(dim, mass) : a.slack;
        const double lo = inner - slack, hi = inner + slack;
        float scale = lo > 0.1 ? nrm / float(lo) : 0.0f;                                       // encode.rs:1194-1200
        const bool settled = lo > 0.1 ? float(lo) == float(hi) : hi <= 0.1;                    // (NaN: not settled)
        if (__any(!settled)) scale = enc_in_order<NG>(v, recon_of, row, dim, l, L, nrm);       // one row in 10^5
        if (l == 0 && grp * R + r < a.n_new) a.scales[a.old_n + grp * R + r] = scale;
        __syncthreads();                                           // every row's codes are there
        // the rows' code bytes, 16 at a time, into their lanes of the device layout (pack.rs:211-233
        // append_lanes); the bytes past a row's last group are zero there and stay so
        const int per = a.bits == 2 ? 8 : 4, pieces = (a.G + 15) / 16;
        for (int idx = t; idx < R * pieces; idx += W * 64) {
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
        if (NG > 3 && grp + gridDim.x < n_groups) fetch(grp + gridDim.x);
    }
}

template <int NG, int W, bool CAL>
static hipError_t launch_encode_rows_cal(const EncodeRowsArgs &a, int device, hipStream_t s) {
    const int R = W * 64 / a.lanes, ng = a.dim / 8;
    const size_t lds = size_t(R * a.row_stride + R * ng + 8 * R + 4) * 4 + 16 * 8 + kEncCells * sizeof(EncCell);
    if (lds > 160 * 1024) return hipErrorInvalidValue;
    const void *kernel = reinterpret_cast<const void *>(k_encode_rows<NG, W, CAL>);
    hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
    if (e != hipSuccess) return e;
    // a workgroup keeps its tables for all its turns: as many as are resident at once, by registers and LDS
    const size_t groups = (a.n_new + R - 1) / R;
    const size_t resident = size_t(device_cus(device)) * std::max<size_t>(1, std::min<size_t>(size_t(4 * enc_waves_per_simd(NG)) / W, 160 * 1024 / lds));
    hipLaunchKernelGGL((k_encode_rows<NG, W, CAL>), dim3(unsigned(std::min(groups, resident))), dim3(W * 64), lds, s, a);
    return hipGetLastError();
}
template <int NG, int W>
static hipError_t launch_encode_rows_n(const EncodeRowsArgs &a, int device, hipStream_t s) {
    return a.scale != nullptr ? launch_encode_rows_cal<NG, W, true>(a, device, s) : launch_encode_rows_cal<NG, W, false>(a, device, s);
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
        a.dim = g.dim; a.bits = g.bits; a.G = g.G; a.nch = g.nch;
        a.log_block = __builtin_ctz(unsigned(block));
        a.lanes = 8;
        while (a.lanes < 64 && a.lanes * 8 < g.dim) a.lanes *= 2;
        a.row_stride = enc_row_stride(g.dim, a.lanes);
        // cells of equal width from the first boundary to the last; no two boundaries may share one, and handed-over
        // centroids may be in any order, equal, infinite or NaN
        const int nb = nl - 1;
        a.cell_mul = float(kEncCells - 2) / (a.bnd[nb - 1] - a.bnd[0]);
        a.cell_add = 1.0f - a.bnd[0] * a.cell_mul;
        a.cells = a.cell_mul > 0.0f && a.cell_mul < 1e30f && std::fabs(a.cell_add) < 1e30f;
        for (int i = 0; a.cells && i + 1 < nb; ++i)
            a.cells = a.bnd[i] < a.bnd[i + 1] && enc_cell(a.bnd[i], a.cell_mul, a.cell_add) < enc_cell(a.bnd[i + 1], a.cell_mul, a.cell_add);
        // without a pair the terms are x * centroid over a row of length 1: |x c| <= (x^2 + c^2) / 2
        double c_max = 0.0;
        for (int i = 0; i < nl; ++i) c_max = std::fabs(double(centroids[i])) >= c_max ? std::fabs(double(centroids[i])) : c_max;
        a.slack = enc_slack(g.dim, (1.01 + double(g.dim) * c_max * c_max) / 2.0);
        a.inv_sqrt_block = inv_sqrt_block;
        a.nat = d_native; a.scales = d_scales; a.old_n = old_n; a.n_new = n_new;
        // Waves per workgroup: a wave's worth of norm chains (eight rows) where two such workgroups fit a CU's LDS and
        // registers, fewer where one would (ms for 300K x 2048 rows in three adds: 3.1 with eight, 2.23 with four, 2.13
        // with two; 400K x 1024: 1.98 with six, 1.45 with four, 1.48 with two; 200K x 3072: 2.78 with four, 4.2 with two).
        switch ((g.dim / 8 + a.lanes - 1) / a.lanes) {
            case 1: return launch_encode_rows_n<1, 8>(a, device, s);
            case 2: return launch_encode_rows_n<2, 4>(a, device, s);
            case 3: return launch_encode_rows_n<3, 8>(a, device, s);
            case 4: return launch_encode_rows_n<4, 2>(a, device, s);
            case 5: case 6: return launch_encode_rows_n<6, 4>(a, device, s);
            default: return launch_encode_rows_n<8, 4>(a, device, s);
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
