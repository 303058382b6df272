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
//     (element j feeds chain j % 4), folded pairwise; 4 lanes carry them.
//
// k_encode_rows takes rows of up to 4096 dimensions, a wave (or part of one) per
// row and a group of eight waves' rows through each step together, so that the
// sequential chains of all of them run side by side in the lanes of one or two
// waves.  k_encode takes one workgroup per row: longer rows, the rotated rows of
// a TQ+ fit, and tables whose signs are not +-1.
#include <hip/hip_runtime.h>

#include <algorithm>

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
// (and a row's place holds the f64 products of one run of its groups, 16 lanes + 16 floats, later on)
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
    int by_quarters;          // fifteen boundaries, in rising order
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

// NG = groups of eight elements per lane; W = waves per workgroup.  The float work of a row is a few
// thousand instructions of its wave, but the two chains are 192 dependent f32 and 384 f64 additions
// (1536 dimensions): a workgroup per row spent 40 us on a row, nearly all of it waiting for them.
// Here the chains of a workgroup's rows run in one or two waves, while the other workgroup of the CU is
// in its parallel part.  A row's rotation goes through LDS three stages at a time in registers
// (the same additions in the same pairs), and its codes leave as 16-byte stores that consecutive
// rows complete to whole lines.  100K rows of 1536 dimensions: 2.02 ms with a workgroup per row, 0.50 now (1.4 TB/s,
// every byte once).  By counters the vector ALU issues in 60 % of the clocks (1750 instructions a row) and a wave
// waits 56 % of its time, for the steps of its row that follow one another: barriers, chains, LDS.
template <int NG, int W>
__global__ __launch_bounds__(W * 64, NG <= 3 ? 4 : 2) void k_encode_rows(EncodeRowsArgs a) {
    extern __shared__ __align__(16) float enc_lds[];
    const int dim = a.dim, t = threadIdx.x, ng = dim / 8, rs = a.row_stride, L = a.lanes;
    const int R = W * 64 / L;                                      // rows of a workgroup
    uint32_t *s_codes = reinterpret_cast<uint32_t *>(enc_lds + R * rs);   // [R][ng] eight codes each, packed as in the index
    float *s_nrm = reinterpret_cast<float *>(s_codes + R * ng);
    float *s_part = s_nrm + R;                                     // [R][8] chains of the squared norm
    double *s_cen = reinterpret_cast<double *>(enc_lds + (R * rs + R * ng + 9 * R + 3) / 4 * 4);   // centroids in f64
    double *s_chain = s_cen + 16;                                  // [R][4]
    const int r = t / L;                                           // this thread's row of the group ...
    int l = t % L;                                                 // ... and its lane in the row
    float *row = enc_lds + r * rs;
    float4 *s_quarter = reinterpret_cast<float4 *>(s_chain + 4 * R);       // [4] the boundaries inside each quarter
    if (t < 16) s_cen[t] = double(a.cen[t]);
    if (t < 4) s_quarter[t] = float4{a.bnd[4 * t], a.bnd[4 * t + 1], a.bnd[4 * t + 2], 0.0f};

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
            for (; i + 8 <= ng; i += 8) {                          // eight groups of eight: 64 floats and their padding
                float v[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = x[9 * i + 8 * e];
#pragma unroll
                for (int e = 0; e < 8; ++e) c = c + v[e] * v[e];
            }
            for (; i < ng; ++i) { const float v = x[8 * i + (i >> 3) * 8]; c = c + v * v; }
            s_part[idx] = c;
        }
        __syncthreads();
        const float *p8 = s_part + r * 8;
        const float nrm = sqrtf(((p8[0] + p8[1]) + (p8[2] + p8[3])) + ((p8[4] + p8[5]) + (p8[6] + p8[7])));
        const float inv = nrm > 1e-10f ? 1.0f / nrm : 0.0f;   // lib.rs:163 MIN_INPUT_NORM
        if (l == 0) s_nrm[r] = nrm;

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
                if (a.scale != nullptr) x = (x + a.shift[8 * g + e]) * a.scale[8 * g + e];
                if (a.by_quarters) {
                    // fifteen boundaries in rising order: the quarter first, then its three
                    const uint32_t q = (x > a.bnd[3] ? 1u : 0u) + (x > a.bnd[7] ? 1u : 0u) + (x > a.bnd[11] ? 1u : 0u);
                    const float4 b = s_quarter[q];
                    c[e] = 4u * q + (x > b.x ? 1u : 0u) + (x > b.y ? 1u : 0u) + (x > b.z ? 1u : 0u);
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
        enc_wave_sync();                                           // every lane has its elements: their places are free
        // encode.rs:1442-1475: inner = <rotated, reconstruction> in f64, four chains by j % 4, NG runs of L
        // groups one after the other: the products by all lanes, in pairs at (element pair, lane) ...
        const int pair = 16 * L + 16;                              // bytes from one element pair's line to the next
#pragma unroll
        for (int i = 0; i < NG; ++i) {
            const int g = l + i * L;
            if (g < ng) {
#pragma unroll
                for (int e = 0; e < 8; e += 2) {
                    double p[2];
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        double recon = s_cen[(code4[i] >> (4 * (e + u))) & 15u];          // (no TQ+ pair: * 1 - 0)
                        if (a.scale != nullptr)
                            recon = recon * double(1.0f / a.scale[8 * g + e + u]) - double(a.shift[8 * g + e + u]);   // encode.rs:594
                        p[u] = double(v[i][e + u]) * recon;
                    }
                    *reinterpret_cast<double2 *>(reinterpret_cast<uint8_t *>(row) + (e / 2) * pair + l * 16) = double2{p[0], p[1]};
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            __syncthreads();
            // ... and the additions by the chains: elements 8 g + c and 8 g + 4 + c of every group in turn
            const int n_here = min(L, ng - i * L);
            for (int idx = t; idx < 4 * R; idx += W * 64) {
                const int c = idx & 3;
                const uint8_t *x = reinterpret_cast<const uint8_t *>(enc_lds + (idx >> 2) * rs) + (c >> 1) * pair + (c & 1) * 8;
                double sum = i == 0 ? 0.0 : s_chain[idx];
                int k = 0;
                for (; k + 8 <= n_here; k += 8) {
                    double y[16];
#pragma unroll
                    for (int u = 0; u < 8; ++u) {
                        y[2 * u] = *reinterpret_cast<const double *>(x + (k + u) * 16);
                        y[2 * u + 1] = *reinterpret_cast<const double *>(x + (k + u) * 16 + 2 * pair);
                    }
#pragma unroll
                    for (int u = 0; u < 16; ++u) sum = sum + y[u];
                }
                for (; k < n_here; ++k) {
                    sum = sum + *reinterpret_cast<const double *>(x + k * 16);
                    sum = sum + *reinterpret_cast<const double *>(x + k * 16 + 2 * pair);
                }
                s_chain[idx] = sum;
            }
            if (i == 0) {
                // the rows' code bytes, 16 at a time, into their lanes of the device layout (pack.rs:211-233
                // append_lanes); the bytes past a row's last group are zero there and stay so
                const int per = a.bits == 2 ? 8 : 4, pieces = (a.G + 15) / 16;
                for (int idx = W * 64 - 1 - t; idx < R * pieces; idx += W * 64) {     // (the last waves first: the first one carries the chains)
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
            }
            if (i + 1 < NG) __syncthreads();
        }
        __syncthreads();
        if (t < R && grp * R + t < a.n_new) {
            const double *d = s_chain + 4 * t;
            const double inner = (d[0] + d[1]) + (d[2] + d[3]);
            a.scales[a.old_n + grp * R + t] = inner > 0.1 ? s_nrm[t] / float(inner) : 0.0f;   // encode.rs:1194-1200
        }
        if (NG > 3 && grp + gridDim.x < n_groups) fetch(grp + gridDim.x);
    }
}

template <int NG, int W>
static hipError_t launch_encode_rows_n(EncodeRowsArgs &a, int device, hipStream_t s) {
    const int R = W * 64 / a.lanes, ng = a.dim / 8;
    const size_t lds = size_t(R * a.row_stride + R * ng + 9 * R + 4) * 4 + (16 + 4 * size_t(R)) * 8 + 64;
    if (lds > 160 * 1024) return hipErrorInvalidValue;
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(k_encode_rows<NG, W>), hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
    if (e != hipSuccess) return e;
    const size_t groups = (a.n_new + R - 1) / R;
    const size_t resident = size_t(device_cus(device)) * std::max<size_t>(1, std::min<size_t>(size_t(2048) / (W * 64), 160 * 1024 / lds));   // (a workgroup keeps its tables for all its turns)
    hipLaunchKernelGGL((k_encode_rows<NG, W>), dim3(unsigned(std::min(groups, resident))), dim3(W * 64), lds, s, a);
    return hipGetLastError();
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
        // (each no larger than the next: handed-over centroids may be out of order, or NaN, which is in no order)
        a.by_quarters = g.bits == 4 && std::adjacent_find(a.bnd, a.bnd + 15, [](float x, float y) { return !(x <= y); }) == a.bnd + 15;
        a.inv_sqrt_block = inv_sqrt_block;
        a.nat = d_native; a.scales = d_scales; a.old_n = old_n; a.n_new = n_new;
        switch ((g.dim / 8 + a.lanes - 1) / a.lanes) {
            case 1: return launch_encode_rows_n<1, 8>(a, device, s);
            case 2: return launch_encode_rows_n<2, 8>(a, device, s);
            case 3: return launch_encode_rows_n<3, 8>(a, device, s);
            case 4: return launch_encode_rows_n<4, 8>(a, device, s);
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
