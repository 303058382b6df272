// Internal declarations shared by the HIP kernels and the C-ABI host code.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <condition_variable>
#include <mutex>
#include <vector>

#include "host_tables.h"

namespace tv {

constexpr int kVecBlock = 32;    // vectors per block (turbovec/src/lib.rs:89)
constexpr int kChunkGroups = 32; // byte-groups per native chunk
constexpr int kQTile = 32;       // queries per MFMA column tile
constexpr int kScanThreads = 256;
constexpr int kMaxListK = 32;    // largest k served by the per-lane lists
constexpr int kSegCap = 64;      // candidate keys one workgroup may append per query and launch
constexpr int kFinalCap = 8192;  // candidate keys per query the final sort holds (64 KiB of LDS)
constexpr int kMaxSampledK = 512;   // largest k served by sample-then-filter
constexpr int kTimedLaunches = 32;  // scan launches of one search that are timed with events

// What a scan launch does with the scores it computes.
enum { kModeLists = 0,   // per-lane top-k lists (written out for k_merge)
       kModeDump = 1,    // every score (and accumulator) to dense rows
       kModeAppend = 2,  // every allowed slot scoring >= the query's fixed floor to a candidate buffer
       kModeBest = 3     // per scanned block and query, the best allowed slot to the candidate buffer (no floor)
};

// Native device layout of the codes ("vm32"): the byte of (block b, group g,
// vector i) lives at ((b*nch + g/32)*64 + ((g%32)/16)*32 + i)*16 + g%16, groups
// padded with zero bytes to a multiple of 32.  One 64-lane wave reads a chunk
// (32 vectors x 32 groups = 1 KiB) with one 16-byte load per lane, and the 16
// bytes a lane receives are 16 consecutive groups of ONE vector -- the operand
// shape of the i8 MFMA and of the per-vector LUT walk alike.
struct Geometry {
    int dim = 0, bits = 0;
    int G = 0;    // byte groups per vector = dim*bits/8 (3-bit: dim/2)
    int nch = 0;  // chunks per block: ceil(G/32), plus padding chunks for some 4-bit row lengths (tv_index_create)
    size_t block_bytes() const { return size_t(nch) * 1024; }
};

// A part of an index that k_scan_p4_wide (its instances for 2- and 3-bit codes) and k_near_rescore pass over together: `groups` groups of
// eight blocks, from number `first` of a fixed order of all `total` groups, in which any run of consecutive ones lies spread over the whole index: number x
// is group x * mul % total, and group g the blocks g, g + total, ... (the last of them may lie beyond the index): neighbouring rows, often neighbours
// of one query, are of groups that lie apart in that order.
constexpr int kNearBlocks = 8;
struct NearStage {
    uint32_t first, groups, total, mul;
    uint16_t *masks;           // [tile][group][query of the tile][block][lane half]: bit 15 - r for row 8 (r / 4) + 4 half + r % 4
    uint8_t *rows;             // the stage's rows one after the other, nch * 32 bytes each
};
__host__ __device__ constexpr uint32_t near_group(const NearStage &n, uint32_t x) { return uint32_t(uint64_t(x) * n.mul % n.total); }
__host__ __device__ constexpr uint32_t near_block(const NearStage &n, uint32_t group, uint32_t w) { return group + w * n.total; }
struct ScanArgs {
    const uint8_t *codes;
    const float *scales;       // padded to a multiple of 32 entries
    const uint64_t *mask;      // nullptr = unfiltered
    const uint8_t *tables;     // this tile's weight fragments (mode P) or LUTs (mode L)
    const float *qscale;       // this tile's per-query scale (kQTile entries)
    const float *qbias;
    int nq_tile;
    uint32_t n;
    uint32_t n_blocks;
    int nch;
    int k;
    uint32_t lv[4];            // the 16 int8 codebook levels, little-endian packed
    int *gtau;                 // kQTile running thresholds (orderable ints)
    float *part_scores;        // [k][total_threads]
    uint32_t *part_idx;
    int *part_cnt;             // [total_threads]
    int32_t *acc_out;          // dump mode: [nq_tile][n] (may be null)
    float *score_out;          // dump mode: [nq_tile][n]
    int classic;               // mode L: 0 = u32 epilogue, 1 = fma flush per 256 groups, 2 = the scalar definition's chain of adds
    int n_groups;              // byte groups of a row that carry codes (the rest of the last chunks is padding)
    uint32_t b_step;           // 1, or a sampling stride: only blocks j*b_step are scanned
    int share_tau;             // lists mode: waves share and raise gtau while scanning
    uint64_t *cand;            // append mode: [nq_tile][seg_stride][kSegCap] sort keys, one segment per workgroup (per four-wave group in the single-tile permute-dot scan)
    uint32_t *cand_cnt;        // append mode: [nq_tile][seg_stride] counts (above kSegCap: that segment overflowed)
    uint32_t seg_stride;       // segments allocated per query (>= grid of the launch)
    uint32_t vgrid;            // single-tile permute-dot scan: four-wave groups of the launch (set by its launcher)
    int best_of_block;         // all-queries-per-pass kernel: no floor, per scanned block and query the best allowed slot (kModeBest)
    uint32_t *best_out;        // when given: [nq_tile][best_stride] score words, per query and scanned block the best allowed row's (tv_kernels6.hip)
    uint32_t best_stride;
    int best_rows;             // (of launch_scan_p4_best) ... every row's score as a float instead, NaN for rows that may not be returned: [nq_tile][best_stride], by row
    const uint32_t *rows;      // all-queries-per-pass kernel: when given, the slot of each of the n rows to scan, in order, 32 neighbours of them within 4 GiB
    // Instances of the all-queries-per-pass kernel for 2- and 3-bit codes (NearStage): tables and lv are int8 weights and levels, and
    // nothing is scored; per (tile, block of the stage, query) a bit for each row whose table sum may reach the floor.
    const float *near_unit, *near_err;
    NearStage near;
    const uint32_t *run_if;    // append mode: when given and *run_if == 0 the launch does nothing (a level's conditional repeat)
};

// ---- launchers (tv_kernels.hip) ----
hipError_t launch_seq_to_native(const uint8_t *d_seq, uint8_t *d_native, const Geometry &g, size_t first_block,
                                size_t n_blocks, hipStream_t s);
// d_seq takes a block's codes every block_bytes, and behind them its row scales when d_scales is given.
hipError_t launch_native_to_seq(const uint8_t *d_native, uint8_t *d_seq, const Geometry &g, size_t first_block,
                                size_t n_blocks, size_t block_bytes, const float *d_scales, hipStream_t s);
hipError_t launch_append_rows(const uint8_t *d_rows, uint8_t *d_native, const Geometry &g, size_t old_n,
                              size_t n_new, hipStream_t s);
// With d_packed every byte of the rows' lanes is written, and their scales; without, the padding behind a row's last group is not.
hipError_t launch_encode(const float *d_vecs, size_t n_new, size_t old_n, const float *d_signs,
                         const uint32_t *d_perms, const uint32_t *d_packed, const float *d_shift, const float *d_scale,
                         const float *centroids, const float *boundaries, const Geometry &g, int block,
                         float inv_sqrt_block, uint8_t *d_native, float *d_scales, float *d_rot_out,
                         int device, hipStream_t s);
size_t encode_lds_bytes(int dim);
// The rotation tables of both rounds in one word per position for the several-rows-per-workgroup
// encoder; false where it does not apply (long rows, signs other than +-1, gathers that are no permutations).
bool encode_pack_tables(const float *signs, const uint32_t *perms, int dim, int block, uint32_t *packed);
hipError_t launch_move_lane(uint8_t *d_native, float *d_scales, const Geometry &g, size_t src, size_t dst,
                            hipStream_t s);

// Query preparation in one launch (tv_prep.hip).  `stamp` here and below, when given: a word that takes the
// device clock as the last query's workgroup ends (of the preparation and of a sampling level's selection) or the
// first one's starts (of a last selection): the full scan between two of them, gaps between launches included, is
// timed without events, whose packets the launches behind them wait for, 5 to 6 us each.
// (Of the preparation, the last kStampsBefore queries' workgroups, one to a die, and those that add a bias in order take one of as
// many words each, and the latest counts.)
constexpr int kStampsBefore = 8;
struct PrepRequest {
    const float *q, *signs;
    const uint32_t *perms;
    int block;
    float inv_sqrt_block;
    const float *shift, *scale;     // the TQ+ pair, or null
    bool permute_dot;               // int8 weights (cs, split: k_scan_p4's order) or u8 tables (centroids)
    bool split;
    float cs, near_cs;
    const float *centroids;
    uint8_t *tables;
    uint8_t *tables_mx;             // or null: u8 tables also as the operands of k_scan_lut_mx
    float *qscale, *qbias;
    uint8_t *near;                  // or null: u8 tables also as int8 weights (with tables_mx; near_cs and lv are read) ...
    float *near_unit, *near_err;    // ... and per query what they leave out (tv_prep.hip: near_fit)
    uint32_t lv[2];                 // the int8 levels of up to eight codes
    float *rot_out;                 // or null
    uint64_t *stamp;                // or null: kStampsBefore words
    uint64_t *cleared;              // or null: a word per query to set to zero
};
hipError_t launch_prep(const PrepRequest &r, const Geometry &g, size_t nq, size_t nq_padded, hipStream_t s);

int device_cus(int device);   // compute units
int scan_grid_blocks(int device, int mode_p, int nch, int k, int lut_queries);
size_t scan_lds_bytes(int mode_p, int nch, int k, int lut_queries);
// Queries one launch of the LUT scan serves (1, 2 or 4), from the LDS budget.
int lut_tile_queries(int nch, int k);
// Queries per LDS entry (1, 2 or 4) the LUT scan launch picks for nq_tile queries.
int lut_launch_ql(int nch, int k, int nq_tile);
int lut_append_queries(int nch);
int lut_append_grid(int device, int nch);
bool lut_single_uses_byte_tables(int nch, int grid);
// Sixteen queries per append-mode pass, score mode L with the u32 or the classic epilogue (tv_kernels4.hip): the
// tables entry-major, 16 bytes per entry, two chunks (32 KiB) after another; chunks padded to even.
constexpr int kLut16Queries = 16;
size_t lut16_table_bytes(int nch, size_t nq);
hipError_t launch_lut_interleave16(const uint8_t *d_src, uint8_t *d_dst, int nch, size_t nq, hipStream_t s);
hipError_t launch_scan_lut16(const ScanArgs &a, int grid, int tiles, hipStream_t s);
int lut16_blocks_per_workgroup(bool classic);   // blocks one workgroup carries through a round of the row's chunks
// Batches in score mode L with the u32 epilogue, on the sparse matrix instructions (tv_kernels5.hip).
struct MxShape {
    unsigned groups, wgs, sub;   // query groups, workgroups per group, segments per workgroup and query
    int nt, blk;                 // query tiles per group, blocks per wave and round
};
// Steps (code bytes per lane half, or pairs of them) in a chunk of 32 byte-groups.
__host__ __device__ constexpr int mx_steps(int entries) { return entries == 16 ? 16 : 8; }
constexpr size_t mx_table_bytes(int nch, int bits, size_t nq) { return (nq + kQTile - 1) / kQTile * size_t(nch) * size_t(mx_steps(bits == 3 ? 8 : 16)) * 2048; }
MxShape mx_shape(int device, size_t nq, size_t level_blocks, bool open_floors);
int mx_segments();
int mx_round_blocks(int device, size_t nq);   // blocks a launch over nq queries works through per round
hipError_t launch_scan_lut_mx(const ScanArgs &a, const MxShape &m, int bits, hipStream_t s);
hipError_t launch_scan_p4(const ScanArgs &a, int grid, int mode, hipStream_t s);
// Small indexes without sampling (tv_kernels6.hip): the best row of every block, then the best blocks' rows.
constexpr int kMaxPickK = 128;             // most results k_pick ranks
constexpr size_t kMaxPickBlocks = 32768;   // most blocks it chooses from
constexpr size_t kPickLds = 144 * 1024;    // rows' keys and sums and the query's tables, beside its 15 KiB of fixed buffers
bool best_serves(int nch);
hipError_t launch_scan_p4_best(const ScanArgs &a, bool split, int device, hipStream_t s);
// The same where blocks are few: a block's chunks over `parts` waves (tv_kernels8.hip); 1 where that does not pay.
int p4_parts(int nch, size_t n_blocks, int tiles, int cus);
hipError_t launch_scan_p4_parts(const ScanArgs &a, bool split, int parts, int device, hipStream_t s);
int lut_parts(int nch, int nq, size_t n_blocks, int cus);      // u8 tables, u32 epilogue
hipError_t launch_scan_lut_parts(const ScanArgs &a, int parts, int device, hipStream_t s);
// The k_floor-th best of n score words per query as its floor, to tau_out like launch_final.
constexpr uint32_t kMaxFloorBlocks = 8192;
hipError_t launch_floor(const uint32_t *words, uint32_t stride, uint32_t n, int k_floor, int nq, int *tau_out, int tau_stride_q, uint64_t *stamp,
                        hipStream_t s);
// The k_eff best of n row scores per query (ScanArgs::best_rows): the last step of a search of so few rows.
constexpr uint32_t kMaxPickRows = 4096;
hipError_t launch_pick_rows(const float *scores, uint32_t stride, uint32_t n, int k_eff, int nq, float *out_scores, int64_t *out_idx, const uint32_t *slots,
                            uint32_t *overflow, uint64_t *stamp, hipStream_t s);
size_t pick_lds_bytes(int nch, size_t k_eff, bool lut);
// Workgroups that share a query's work in launch_pick; more than one need pick_shared_bytes of it, the first nq words zero.
int pick_shares(int device, int nch, size_t k_eff, size_t nq, bool lut);
size_t pick_shared_bytes(size_t k_eff, size_t nq);
hipError_t launch_pick(const ScanArgs &a, bool lut, bool split, int k_eff, float *out_scores, int64_t *out_idx, const uint32_t *slots, uint32_t *overflow,
                       int shares, uint64_t *shared, uint64_t *stamp, hipStream_t s);
hipError_t launch_scan_lut(const ScanArgs &a, int grid, int mode, hipStream_t s);
// Query tiles one batched permute-dot launch serves for this geometry (0: not available).
int batched_tiles(int nch);
int batched_grid_blocks(int device, int nch);
hipError_t launch_scan_p4_batched(const ScanArgs &a, int grid, hipStream_t s);
bool batched_weights_split(int nch);   // which weight order launch_scan_p4_batched's kernel reads
// out_tau == nullptr: write the k_eff best of the merged lists; else write only the
// order key of the k_eff-th best (a floor at least k_eff scanned slots reach) per query.
// Wide batched scan (every query of a chunk in one pass; tv_kernels3.hip).
int wide_min_queries(int nch);
int wide_grid_blocks(int device);
hipError_t launch_scan_p4_wide(const ScanArgs &a, int grid, hipStream_t s);
int wide_blocks_per_workgroup(int nch);
bool wide_serves_best_of_block(int nch);
int wide_max_queries(int nch);
bool wide_weights_split(int nch);
bool wide_reads_rows(int nch, int nq);

// The same over 2- and 3-bit codes, in front of their u8 tables (tv_kernels7.hip): an int8 scan that tells the rows whose table sum cannot reach
// the floor, and the rest scored from the tables.
int near_chunks(int nch, int bits);                    // chunks of 64 dimensions of the scan's instance; 0 = there is none
int near_nch(int nch, int bits);                       // chunks of 32 byte-groups there: a row's, or more, with weights of zero
int near_blocks_per_workgroup(int nch, int bits);
hipError_t launch_scan_near(const ScanArgs &a, int bits, int grid, hipStream_t s);
struct NearRescore {
    NearStage stage;
    const uint8_t *tables;     // launch_prep's u8 tables
    const float *scales, *qscale, *qbias;
    const int *gtau;
    uint64_t *cand;            // as in ScanArgs; this stage's segments are numbers seg0 .. seg0 + splits * sub - 1, `sub` (a power of two) to a workgroup
    uint32_t *cand_cnt;
    uint32_t seg_stride, seg0, splits, sub, n;
    int nq, nch;
};
int near_rescore_queries(int nch);                     // of one workgroup; 0: the tables do not fit
hipError_t launch_near_rescore(const NearRescore &a, hipStream_t s);

hipError_t launch_merge(const float *part_scores, const uint32_t *part_idx, const int *part_cnt, int total_threads,
                        int qmod, int k, int k_eff, int nq_tile, float *out_scores, int64_t *out_idx,
                        int *out_tau, hipStream_t s);
// Gathers each query's candidate segments (n_seg of them, seg_stride allocated), sorts, and either
// emits the k_eff best (tau_out == nullptr; a query that did not fit is flagged in overflow) or, for a
// sampling level, writes the order key of the k_floor-th best as the query's next floor to
// tau_out[(q / tau_stride_q) * kQTile + q % tau_stride_q] (keep_floor: a level that gathers fewer than k_eff
// candidates leaves the floor already there in place instead of opening it).  A final pass that
// overflows writes flag 1 and a raised floor to raise_out[q] when raise_out is given (flag 2 and
// nothing otherwise); row_map, when given, names the output row of each query.
// level_over (sampling levels): set to 1 when some query's candidates of this level did not all fit
// (its floor then comes from a subset and may be far too low); clear_flag: a word this launch resets
// to 0 (the flag of the level after); run_if: when given and *run_if == 0 the launch does nothing; slots: when
// given, the slot of each row, for out_idx; passed: (a final pass) floors laid out as tau_out that may be above the result's last row -- such a
// query is flagged 1, and that row is its raised floor (open with fewer rows than k_eff); keep_floor == 2: no floor is lowered; longest: about how many candidates a query's longest segment holds.
hipError_t launch_final(const uint64_t *cand, const uint32_t *cand_cnt, uint32_t n_seg, uint32_t seg_stride,
                        int k_eff, int k_floor, int nq, float *out_scores, int64_t *out_idx, uint32_t *overflow,
                        int *tau_out, int tau_stride_q, int keep_floor, int *raise_out, const uint32_t *row_map,
                        uint32_t *level_over, uint32_t *clear_flag, const uint32_t *run_if, const uint32_t *slots, uint64_t *stamp, double longest, hipStream_t s,
                        const int *passed = nullptr);
// Packs the queries rows[0..n_redo) of a chunk and their raised floors for one more full scan.
hipError_t launch_gather_redo(const float *d_q, const uint32_t *d_rows, const int *d_raised, int dim, int tile_q,
                              size_t n_redo, float *d_q_out, int *d_tau_out, hipStream_t s);
hipError_t launch_fill_i32(int *p, int v, size_t n, hipStream_t s);
hipError_t launch_lay_tables(const uint32_t *from, uint32_t *to, size_t n, int *floors, int v, size_t n_floors, hipStream_t s);
hipError_t launch_probe(const void *src, void *dst, size_t bytes, int copy, uint32_t *sink, hipStream_t s);
hipError_t launch_probe_mfma(int device, int iters, uint32_t *sink, double *ops, hipStream_t s);
// Exact top-k of a dense score row per query (NaN = excluded slot).
hipError_t launch_select_topk(const float *d_scores, size_t n, int nq_tile, size_t k_eff, uint64_t *d_keys_tmp,
                              uint32_t *d_hist, float *out_scores, int64_t *out_idx, hipStream_t s);
size_t select_tmp_keys(size_t k_eff);
// Filtered searches on the allowed rows alone (tv_filter.hip).  How many of the mask's bits below n are set and in how many blocks
// of 32, piece by piece to counts (two words for each of mask_counts(n) pieces) and, unless null, in all to the words totals[0 .. mask_totals(n))
// (host memory): those with the bit kMaskCounted are there, and their sum counts both.
constexpr uint64_t kMaskCounted = uint64_t(1) << 63;
constexpr size_t kMaxMaskTotals = 256;
__host__ __device__ constexpr uint64_t mask_total(uint32_t rows, uint32_t blocks) { return uint64_t(blocks) << 31 | rows; }     // (rows below 2^31, of all words too)
size_t mask_counts(size_t n);
size_t mask_totals(size_t n);
hipError_t launch_mask_count(const uint64_t *mask, size_t n, uint32_t *counts, uint64_t *totals, hipStream_t s);
// The rows of those bits, in order, to slots[0 .. room).
hipError_t launch_mask_slots(const uint64_t *mask, size_t n, const uint32_t *counts, uint32_t *slots, size_t room, hipStream_t s);
// *far becomes 1 (host memory; cleared by the caller) where the rows of a block of 32 among slots[0 .. n) lie 4 GiB of codes or more apart.
hipError_t launch_rows_apart(const uint32_t *slots, size_t n, size_t block_bytes, uint32_t *far, hipStream_t s);
// The rows slots[0 .. n) into blocks of their own, the last one's missing rows zero.
hipError_t launch_gather_rows(const uint8_t *codes, const float *scales, int nch, const uint32_t *slots, size_t n, uint8_t *out, float *out_scales, hipStream_t s);
// idx[i] = slots[idx[i]] where idx[i] is below n.
hipError_t launch_map_slots(int64_t *idx, size_t count, const uint32_t *slots, size_t n, hipStream_t s);

}  // namespace tv

struct tv_request;   // a search call waiting for the index (tv_api.hip)

// Pinned host memory that the indexes of a device share: one block at a time is lent to a call on host arrays.
struct tv_pinned {
    uint8_t *host = nullptr, *dev = nullptr;   // the same bytes, as the host and as the device address them
    size_t bytes = 0;
    bool lent = false;
};

// What a search reads: n rows in blocks of 32, scales padded to whole blocks.
struct tv_rows {
    const uint8_t *codes = nullptr;
    const float *scales = nullptr;
    size_t n = 0;
    const uint32_t *slots = nullptr;   // the index's slot of each row, when that is not its place
    size_t live = 0;                   // ... and the index's blocks with such a row
    bool in_place = false;             // ... and codes and scales are the index's own: the rows lie at their slots
};

// Device memory that an index keeps between searches and does without where an allocation of the device needs it (tv_api.hip:
// device_alloc takes it then, unless a search is using it).
struct tv_spare {
    void *p = nullptr;
    size_t bytes = 0;
    bool in_use = false;
};

// The opaque handle of the C ABI.
struct tv_index {
    tv::Geometry geo;
    int device = 0;
    int score_mode = 0;
    tv::RotationTables rot;
    tv::Codebook cb;
    std::vector<float> tq_shift, tq_scale;
    int8_t levels[16] = {0};
    float cs = 1.0f;
    int8_t near_levels[8] = {0};       // the same for 2- and 3-bit codes, as the scan in front of the tables takes them
    float near_cs = 1.0f;

    hipStream_t stream = nullptr;
    hipEvent_t ev_start[tv::kTimedLaunches] = {}, ev_stop[tv::kTimedLaunches] = {};
    bool events_ready = false;
    float *d_signs = nullptr;
    uint32_t *d_perms = nullptr;
    uint32_t *d_packed = nullptr;  // both rounds' gathers and signs in one word per position (encode_pack_tables) ...
    bool packed_ok = false;        // ... when the tables in use have that form
    float *d_centroids = nullptr;
    float *d_tq_shift = nullptr, *d_tq_scale = nullptr;
    int *d_tau_open = nullptr;     // order key of -inf per query: the floors before any level has run

    uint8_t *d_codes = nullptr;
    float *d_scales = nullptr;
    size_t codes_bytes = 0, scales_bytes = 0;   // allocated
    size_t ahead = 0;              // ... of it beyond growing by half (guarded as the device's pool of blocks is)
    size_t cap_blocks = 0;
    size_t n = 0;

    // Search calls that arrived while another held the index: whoever takes `mu` next serves every
    // waiting call that asks for the same k under the same mask together with its own, as one batch.
    std::mutex waiting_mu;
    std::condition_variable waiting_cv;   // a call registered, or a batch was served
    std::vector<tv_request *> waiting;
    bool serving = false;          // some caller is serving a batch right now ...
    const tv_request *served = nullptr;   // ... this call's and what could join it
    size_t last_batch_calls = 0;   // calls in the batch served last: how many callers to expect again shortly
    size_t merged_calls = 0;       // calls that were served by another caller's launch

    // per-search workspace, grown on demand, guarded by mu
    mutable std::mutex mu;
    void *ws = nullptr;
    void *io = nullptr;            // staging for tv_search's host buffers (queries, mask, results); grows, never shrinks
    size_t io_bytes = 0;
    size_t ws_bytes = 0;
    bool ws_fixed = false;         // ws is a lent buffer of fixed size (tv_search_dev_noalloc): never reallocated
    tv_spare slots, gathered;      // a filtered search's allowed rows: their slots, and their codes and scales (tv_api.hip: gather_allowed)
    tv_index *older = nullptr, *newer = nullptr;   // the device's indexes, linked (guarded as their pool of blocks is)
    tv_rows allowed;               // for the length of such a search: what it reads in place of the index's rows (codes null otherwise)
    tv_rows rows() const { return allowed.codes ? allowed : tv_rows{d_codes, d_scales, n, nullptr, 0, false}; }
    void *scratch = nullptr;       // this device's copy of the library's static scratch array
    uint32_t *h_tables = nullptr;  // in the allocation of h_flags: the tables on their way to the device
    uint32_t *h_flags = nullptr;   // pinned host memory: the overflow flags of one group of chunks, then the rows to repeat (before a search: a mask's totals)
    uint32_t *d_flags_host = nullptr;   // the device's address of h_flags
    uint64_t *h_stamps = nullptr, *d_stamps = nullptr;   // in the same allocation: the device clock before and after a full scan
    size_t exact_redos = 0;        // queries that went on to the exact path
    float last_scan_ms = 0.0f;
    int last_scan_launches = 0;
    int last_queries_per_launch = 0;   // queries one full-scan launch of the last search served
    int force_robust = 0;          // test hook: skip sample-then-filter
    int no_batched = 0;            // test hook: one query tile per scan launch even for large batches
    int no_lut16 = 0;              // test hook: mode L batches stay on the scan with whole tables in LDS (8 queries per pass at most)
    bool no_lut_mx = false;        // for the length of a call: the scratch array holds only the sixteen-query passes' working set
    int no_wide = 0;               // test hook: large batches go through the tile-group kernels, not the wide one
    int no_direct = 0;             // test hook: small indexes are sampled, those of up to 16384 blocks by levels of rows where there are such
    int force_near = 0;            // test hook: u8-LUT batches take the two-step scan wherever it has an instance for the row length
    int no_gather = 0;             // test hook: filtered searches read the mask as they scan ...
    int force_gather = 0;          // ... or gather their allowed rows whatever their number
    size_t gathered_searches = 0, in_place_searches = 0;   // searches that ran on the allowed rows alone, and those of them that read all of their queries' rows in place
    size_t overflow_redos = 0;     // queries redone because their candidate buffer overflowed
    // The floorless first level (best row per block) misjudges the floor when a query's neighbours
    // sit together in a few blocks (a clustered corpus in insertion order): after a search in which
    // it made an eighth of the queries overflow, the next searches run the ladder of row-level
    // samples instead, and the floorless level gets another try afterwards.  When the row-level
    // ladder then fails the same way (rows laid out against its strides), the floorless level comes
    // back at once and stays for as many searches: its failure costs less.
    int row_ladder_left = 0;
    int floorless_kept_left = 0;
    int near_sure_left = 0;        // the two-step table scan guessed floors too high for many queries: so many searches take floors that are sure
    int track_levels = 0;          // test hook: read the per-level flags back with the overflow flags and count them
    size_t level_repeats = 0;      // sampling levels that ran a second time because their candidates did not fit
};
