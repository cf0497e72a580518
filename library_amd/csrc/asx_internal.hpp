// Internal declarations shared by the HIP translation units of libalphasparse_amd.so.
#pragma once
#include <algorithm>
#include <cmath>
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "../../include/alphasparse_amd.h"
#include "asx_device.hpp"
#include "asx_pool.hpp"

namespace asx {

// Tile geometry of the SpMV kernels (one workgroup of 256 threads per tile).
constexpr int kBlock = 256;
constexpr int kXcds = 8;  // workgroups are dealt to the 8 XCDs round-robin (workgroup b runs on XCD b % 8)
constexpr int kMergeItemsPerThread = 8;
constexpr int kMergeTile = kBlock * kMergeItemsPerThread;  // rows + stored elements per tile
constexpr int kStreamTile = 1024;                          // stored elements per row block
constexpr int kFlatTile = 1024;                            // stored elements per flat tile
// Plans made without columns and values go from the flat to the merge-path kernel above this row length; with them the
// estimates (estimate_kernels) leave the flat kernel out there.
constexpr int kLongRow = 8192;
// SpMM: merge items (rows + stored elements) per wave
constexpr int kSpmmSegmentSmall = 128, kSpmmSegmentMedium = 256, kSpmmSegmentLarge = 512;
// SpMM chunk kernel: threads of a workgroup, what it can stage, and merge items per segment - where rows may be cut (a segment
// then holds up to twice as many elements) and where none is longer than kChunkLongest.  kChunkItemsMost: the shortest segments
// that are within 1 % of the fastest (8 M elements, 5 to 48 per row within 3000 of the diagonal, 4 and 8 columns fp64, 4 and 16
// fp32, on average: 1664 items 8 % behind, 2048 3 %, 2368 1.5 %, 3008 and 3392 alike; 24 per row, 8 columns fp64 58.0, 55.5, 55.4, 2688
// items 55.5, 53.3, 53.3; 20 per row 59.9, 57.1, 56.1, 54.7, 55.2, 55.1).
constexpr int kChunkThreads = 512, kChunkElems = 2880, kChunkRows = 2689;
constexpr int kChunkWideLeast = 64;  // longer rows are taken by all waves where a wave has four groups or fewer
constexpr int kChunkItems = 1344, kChunkItemsMost = 2688, kChunkLongest = kChunkElems - kChunkItemsMost;
constexpr int kChunkItemsWide = 640;      // the most where rows of B are wide
constexpr int64_t kChunkRound = 768;      // three workgroups on each of 256 compute units
static_assert(2 * kChunkItems <= kChunkElems && kChunkItemsMost < kChunkRows, "a segment fits what is staged");
// Which calls it takes.  Rows of B of up to 32 bytes unless rows of A are short: 66 such cases of all families 9 %
// faster on average (3 columns fp64, 56 per row 16.7 -> 7.4 us; 2 columns fp32, 5 per row 21.0 -> 16.0), but with 4 per row,
// 2 columns fp32 8.2 -> 10.1, with 7, 3 columns fp64 4.7 -> 5.1.  spmm_chunked_unplanned and spmm_plan_chunked say when; what it
// takes beside these: spmm_chunked_mid, spmm_chunked_wide.
inline bool spmm_chunked_narrow(int32_t m, int32_t nnz, int64_t ncols, size_t sv)
{
    return ncols * (int64_t)sv <= 32 && 2 * (int64_t)nnz >= (sv == 4 ? 9 : 16) * (int64_t)m;
}
// One round of workgroups takes all of A: then in any case (8 to 50 per row, 0.5 to 1 M items, both types: merge takes 1 to 2.2 times
// as long).  With more rounds only where a plan knows that no row of A is long: rows that are cut leave carries, and segments
// of few long rows have no work for most lane groups (planned, power-law rows of up to 4000: 4 columns fp64, 14 per row, 3 M items
// 39.6 us with merge, 43.4 here; 45 per row, 5 M 50.7 and 66.3; 8 fp32 44.6 and 62.0; 2 fp64, 25 per row, 8 M 86.7 and 109.8), and
// without a plan every workgroup looks its segment up before it loads any of it (1.1 to 5 M items, 8 to 20 per row: merge takes
// 0.84 to 1.01 of the time for 3 columns fp64, 0.81 to 1.01 for 8 fp32, 0.82 to 1.03 for 2 fp64).  Rows of B of up to 16 bytes in fp32
// come here all the same: merge takes 0.9 to 1.4 of the time with 8 to 30 per row, 1.2 to 1.7 with 50, 0.9 to 1.3 with power-law rows.
inline bool spmm_chunk_one_round(int32_t m, int32_t nnz) { return (int64_t)m + nnz <= kChunkRound * kChunkItems; }
inline bool spmm_chunked_unplanned(int32_t m, int32_t nnz, int64_t ncols, size_t sv)
{
    return spmm_chunked_narrow(m, nnz, ncols, sv) && (spmm_chunk_one_round(m, nnz) || (sv == 4 && ncols <= 4));
}
// Rows of B of 33 to 128 bytes while one round of workgroups takes all of A, planned or not: 57 such cases of all families 6 %
// faster on average (7 columns fp64, 61 per row, 462624 elements 12.1 -> 8.1 us; 31 fp32, 5-point stencil of 642649 14.4 -> 11.9;
// 24 fp32, power-law rows of 699314 19.3 -> 17.0), none slower by more than calls of 6 us differ; with several rounds they gain and lose
// alike (18 columns fp32 27.3 -> 29.6, 12 columns fp64 86.8 -> 83.0).
inline bool spmm_chunked_mid(int32_t m, int32_t nnz, int64_t ncols, size_t sv)
{
    return ncols * (int64_t)sv > 32 && ncols * (int64_t)sv <= 128 && spmm_chunk_one_round(m, nnz);
}
// Wider rows of B while one round of workgroups takes all of A: the merge kernel's few waves then walk 128 items each, one or two
// rows of A at a time, where eight waves share them here.  40 such cases of all families, planned or not, take 0.7 of their time
// (37 columns fp64, 5-point stencil of 26353 elements 12.3 -> 5.6 us; 80 columns fp32, power-law rows of 77812 37.6 -> 18.5; 57,
// 12543 rows of 5 16.4 -> 8.3); none is slower, except where four groups share rows of more than 32 elements (20 columns fp64, 64
// per row 8.6 -> 9.6).  Not rows of B that end on lines, which are cut into tiles that keep the merge kernel's groups at work: 120 such
// calls (256, 512 and 1024 bytes, 2000 to 30000 rows of 8 to 20) would take 1.13 times as long on average (128 columns fp32, 6000
// uniform rows of 12 without a plan 10.7 -> 19.0 us, 12000 planned rows of 20 11.3 -> 12.9), though 18 of power-law rows up to 0.3
// less (64 columns fp32, 2000 rows of 8 13.2 -> 9.4).
inline int64_t spmm_chunk_wide_work(int32_t m, int32_t nnz, int64_t row_bytes) { return ((int64_t)m + nnz) * ceil_div64(row_bytes, 512); }
inline bool spmm_chunked_wide(int32_t m, int32_t nnz, int64_t ncols, size_t sv)
{
    const int64_t bytes = ncols * (int64_t)sv;
    return bytes > 128 && bytes % 128 != 0 && (bytes > 256 || nnz <= 32 * (int64_t)m) &&
           spmm_chunk_wide_work(m, nnz, bytes) <= kChunkRound * kChunkItemsWide;
}
inline bool spmm_chunked(int32_t m, int32_t nnz, int64_t ncols, size_t sv)  // without a plan
{
    return spmm_chunked_unplanned(m, nnz, ncols, sv) || spmm_chunked_mid(m, nnz, ncols, sv) || spmm_chunked_wide(m, nnz, ncols, sv);
}
// Under a plan also rows of B of up to 64 bytes (those of up to 32 that spmm_chunked_narrow leaves out among them) where no row of A
// is long, rows hold 3.5 elements or more on average, and there are several rounds of workgroups (16 columns fp32, 23 per row,
// 8 M elements 60.9 -> 52.2 us; 9 per row, 5 M 50.5 and 50.5; but 14 columns, 27 per row, 2.2 M 23.3 -> 24.3; rows of up to
// 1510 57.4 -> 73.5).  With 3 per row, 2 to 16 columns, both types, near and scattered, merge is 5 % ahead on average (2 columns
// fp32 15.5 against 14.5, 6 columns 68.8 against 61.9, 16 columns 61.2 against 55.8); from 4 on they differ by 1 % on average.
//
// And scattered columns where 32 lanes or more (tile_lanes) take a row of B: the merge kernel's waves, whose
// LDS leaves room for 20 a compute unit, wait for one or two rows of B at a time, and its short segments leave more carries: 36 such
// cases of 0.5 to 13 M items 3 % faster, none more than 1 % slower (91 columns fp64, power-law rows of 5 178 -> 155 us; 34,
// 6 per row 264 -> 240; 113 fp32, rows of up to 75394 127 -> 113).  Near columns gain and lose alike (199 fp32 29.6 -> 27.7,
// 248 49.1 -> 50.5).
inline bool spmm_plan_chunked(int32_t m, int32_t nnz, int64_t ncols, size_t sv, int64_t longest, bool scattered, int tile_lanes)
{
    if (spmm_chunked(m, nnz, ncols, sv)) return true;  // a plan's segments are never more than a call's without one
    if (spmm_chunked_narrow(m, nnz, ncols, sv)) return longest <= kChunkLongest;
    if (ncols * (int64_t)sv <= 64)
        return longest <= kChunkLongest && 2 * (int64_t)nnz >= 7 * (int64_t)m && (int64_t)m + nnz >= 4000000;
    return scattered && tile_lanes >= 32;
}
// Segments of wide rows of B fill whole rounds (527000 items, rows of B of 520 bytes: in 1030 workgroups, a round and a third, 70 us, in 687 59).
inline int32_t spmm_chunk_wide_items(int64_t work)
{
    const int64_t rounds = ceil_div64(work, kChunkRound * kChunkItemsWide), items = ceil_div64(work, kChunkRound * rounds);
    return (int32_t)(items < kSpmmSegmentSmall ? kSpmmSegmentSmall : items);
}
// Where rows may be cut: one round, if its segments are neither short (448 to 896 items are alike up
// to 500000 items; at 1 M 896 take 20 % longer than 1344) nor more than a workgroup can stage.
inline int32_t spmm_chunk_items(int64_t items)
{
    return (int32_t)std::min<int64_t>(std::max<int64_t>(ceil_div64(items, kChunkRound), kChunkItems / 2), kChunkItems);
}
// Where a plan knows that none is: segments that fill one round of workgroups or two, with more rounds the longest.  A round that is
// only begun leaves the chip idle: 16 per row, 2.0 M elements within 20000 of the diagonal, in 800 workgroups and in 1536 (3 columns
// fp64 17.3 and 15.2 us, 8 fp32 15.7 and 14.0); 12 per row, 2.6 M (4 columns fp64 19.6 and 18.3); 66 such cases of 2 and 2.6 M
// elements 3 % faster on average, of 4 M and more alike.
inline int32_t spmm_chunk_uncut_items(int64_t items)
{
    const int64_t rounds = std::max<int64_t>(ceil_div64(items, kChunkRound * kChunkItemsMost), 1);
    if (rounds > 2) return kChunkItemsMost;
    return (int32_t)std::max<int64_t>(ceil_div64(items, kChunkRound * rounds), kChunkItems / 2);
}
constexpr double kScatteredMinSpread = 0.5;  // of a column sample: from here on the columns count as scattered

inline int status_of(hipError_t e)
{
    switch (e) {
    case hipSuccess: return ASX_STATUS_SUCCESS;
    case hipErrorOutOfMemory: return ASX_STATUS_ALLOC_FAILED;
    case hipErrorInvalidValue: return ASX_STATUS_INVALID_VALUE;
    case hipErrorInvalidDevicePointer: return ASX_STATUS_INVALID_POINTER;
    case hipErrorInvalidDevice:
    case hipErrorInvalidResourceHandle: return ASX_STATUS_INVALID_HANDLE;
    default: return ASX_STATUS_INTERNAL_ERROR;
    }
}
inline int check_launch() { return status_of(hipGetLastError()); }

inline size_t align_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

// ---- analysis launchers (asx_analysis.hip) ----
int launch_row_histogram(const int32_t *d_row_ptr, int32_t m, int64_t *d_hist, int64_t *d_stats,
                         hipStream_t s);
int launch_partition_rows_by_nnz(const int32_t *d_row_ptr, int32_t m, int32_t nparts, int32_t *d_out,
                                 hipStream_t s);
int launch_nnz_split_rows(const int32_t *d_row_ptr, int32_t m, int32_t nnz, int32_t items,
                          int32_t *d_out, hipStream_t s);
int launch_nnz_split_rows_n(const int32_t *d_row_ptr, int32_t m, int32_t nseg, int32_t items, int32_t *d_out,
                            hipStream_t s);
int launch_flat_seg_rows(const int32_t *d_row_ptr, int32_t m, int32_t nnz, int32_t *d_seg_row, hipStream_t s);
int launch_merge_path_search(const int32_t *d_row_ptr, int32_t m, int32_t nnz, int32_t items,
                             int32_t *d_xs, int32_t *d_ys, hipStream_t s);
int launch_loadbalance_partition(const int32_t *d_row_ptr, int32_t m, int32_t nnz, int32_t warp_size,
                                 int32_t nwarps, int32_t *d_out, hipStream_t s);
int launch_stream_row_blocks(const int32_t *d_row_ptr, int32_t m, int32_t nnz, int32_t *d_blocks,
                             hipStream_t s);
int launch_copy_bytes(const void *d_src, void *d_dst, size_t bytes, hipStream_t s);
int launch_fill_i32(int32_t *d_dst, int64_t n, int32_t value, hipStream_t s);
// d_now[0..1] = two 64-bit checksums of `bytes` bytes (a multiple of 4, from a 16-byte boundary);
// d_partials: 2 * checksum_parts() words of scratch
int checksum_parts();
int launch_checksum(const void *d_data, size_t bytes, unsigned long long *d_partials, unsigned long long *d_now, hipStream_t s);
// kept = now
int launch_checksum_commit(const unsigned long long *d_now, unsigned long long *d_kept, hipStream_t s);
int launch_sample_columns(const int32_t *d_col, int64_t stride, int shift, const int32_t *d_row_ptr, int32_t m,
                          int32_t width, int32_t samples, int32_t *d_out, hipStream_t s);
// what launch_row_histogram and launch_sample_columns count (samples = 0: no sample), in one launch and one that adds up: the histogram,
// the stats and, from word `sampled` on, the sample, in d_counters, the other words 0, and the same in h_counters (page-locked);
// d_scratch: plan_stats_bytes; d_row_blocks: the nb row blocks of launch_stream_row_blocks too (null: not wanted)
size_t plan_stats_bytes(int32_t m);
int launch_plan_stats(const int32_t *d_row_ptr, int32_t m, int64_t *d_counters, int ncounters, int sampled, int64_t *h_counters,
                      const int32_t *d_col, int64_t stride, int shift, int32_t width, int32_t samples, void *d_scratch, int32_t nb,
                      int32_t *d_row_blocks, hipStream_t s);
int launch_gather_lines(const void *d_buf, size_t bytes, int group_lanes, int per_lane, void *d_out, int *nthreads,
                        hipStream_t s);

// ---- SpMV launchers (asx_spmv.hip) ----
// Rows that the vector kernel gives more than a lane group: nwide rows a workgroup each, then nlong rows a wave each, all of
// long_len elements or more (rows == nullptr: none).
struct LongRows {
    const int32_t *rows;
    int32_t nwide, nlong, long_len;
};
int launch_long_rows(const int32_t *d_row_ptr, int32_t m, int32_t long_len, int32_t wide_len, int32_t nwide, int32_t *d_at,
                     int32_t *d_out, hipStream_t s);
template <typename T>
int launch_spmv_vector(int32_t m, int32_t nnz, T alpha, const int32_t *row_ptr, const int32_t *col,
                       const T *val, const T *x, T beta, T *y, const LongRows &long_rows, hipStream_t s);
template <typename T>
int launch_spmv_merge(int32_t m, int32_t nnz, T alpha, const int32_t *row_ptr, const int32_t *col,
                      const T *val, const T *x, T beta, T *y, const int32_t *xs, const int32_t *ys,
                      T *carry, hipStream_t s);
template <typename T>
int launch_spmv_stream(int32_t m, int32_t nnz, T alpha, const int32_t *row_ptr, const int32_t *col,
                       const T *val, const T *x, T beta, T *y, const int32_t *blocks, hipStream_t s);

template <typename T>
int launch_spmv_flat(int32_t m, int32_t nnz, T alpha, const int32_t *row_ptr, const int32_t *col,
                     const T *val, const T *x, T beta, T *y, int32_t *seg_row, bool search, T *carry,
                     bool carry_pass, hipStream_t s);  // search: seg_row is written by the call
int launch_flat_has_carry(const int32_t *d_row_ptr, int32_t m, int32_t nnz, const int32_t *d_seg_row,
                          int32_t *d_flag, hipStream_t s);

// ---- SpMM launchers (asx_spmm.hip) ----
template <typename T>
int launch_spmm_row(int32_t m, int32_t ncols, T alpha, const int32_t *row_ptr, const int32_t *col,
                    const T *val, const T *B, int64_t ldb, T beta, T *C, int64_t ldc, hipStream_t s);
// Where the device decides whether the sweep kernel takes a call: what it has to know, and where it leaves its answer.
struct SweepAsk {
    int32_t n;          // columns of A
    int32_t longest;    // row the sweep takes
    int32_t blocks;     // its workgroups
    int32_t *answer;    // 1: taken (null: nobody asks)
    uint8_t *too_long;  // of each workgroup: it left rows of more than `longest` elements out
};
template <typename T>
int launch_spmm_merge(bool chunked, int32_t rows, int32_t m, int32_t nnz, int32_t items, int32_t ncols, T alpha, const int32_t *row_ptr,
                      const int32_t *col, const T *val, const T *B, int64_t ldb, T beta, T *C,
                      int64_t ldc, const int32_t *xs, const int32_t *ys, T *carry, int32_t *carry_row,
                      bool carry_pass, int tile_bytes, const SweepAsk &ask, hipStream_t s);

// ---- SpMM of columns that lie all over B (asx_spmm_sweep.hip) ----
struct SpmmSweep {
    int32_t slots;   // sums of rows of C a lane group has registers for (0: not taken)
    int32_t rows;    // rows it is given, `chains` sums each
    int32_t cap;     // elements of A a wave stages at once
    uint32_t width;  // columns a window
    int log_lanes;   // of a group
    int64_t tiles;   // of columns of B
    int32_t chains;  // sums of stretches that a row of more than 32 elements is made of: 1, 2 or 4
};
template <typename T>
int launch_spmm_sweep(const SpmmSweep &sw, const SweepAsk *ask, int32_t m, int32_t n, int32_t nnz, int32_t ncols, T alpha,
                      const int32_t *row_ptr, const int32_t *col, const T *val, const T *B, int64_t ldb, T beta, T *C, int64_t ldc,
                      hipStream_t s);

// merge-path split points of SpMM, `items` apart, moved to the ends of the short rows they cut; *has_carry (may be null)
// is set to 1 if a row stays cut
int launch_spmm_splits(int32_t m, int32_t nnz, int32_t items, const int32_t *row_ptr, int32_t *xs, int32_t *ys,
                       int32_t *has_carry, hipStream_t s);

// ---- blocked (MFMA) SpMM (asx_blocked.hip) ----
struct BlockedMatrix {
    int32_t nbrows;     // ceil(m / 16)
    int32_t nblocks;    // non-empty 16x4 blocks
    int32_t *brow_ptr;  // nbrows + 1
    int32_t *bcol;      // column quad of each block
    void *bval;         // nblocks * 64 values, lane order of the MFMA A operand
    int32_t nnz;        // stored elements of A
    int32_t *upd_src;   // nnz: position in A's values of every stored element, in block order
    int64_t *upd_dst;   // nnz: its slot in bval; sign bit = repeats the (row, column) before it
};
template <typename T>
int build_blocked(int32_t m, int32_t k, int32_t nnz, const int32_t *row_ptr, const int32_t *col,
                  const T *val, BlockedMatrix *out, hipStream_t s);
void free_blocked(BlockedMatrix *b, bool idle);  // idle: as for pool_free
template <typename T>
int blocked_update_values(const BlockedMatrix *bm, const T *val, hipStream_t s);
template <typename T>
int launch_spmm_blocked(int32_t m, int32_t k, int32_t ncols, T alpha, const BlockedMatrix *bm, const T *B,
                        int64_t ldb, T beta, T *C, int64_t ldc, hipStream_t s);

// out[r] = first i with sorted[i] >= r, r in [0, n]
int launch_offsets_from_sorted(const int32_t *sorted, int32_t count, int32_t n, int32_t *out, hipStream_t s);

// ---- column-sliced SpMV (asx_sliced.hip) ----
// The stored elements regrouped by column slice (slice = col / width), a slice of x being small
// enough to sit in the LDS of one compute unit, so that the gathers of x never reach the L2.
// Pass 1: one workgroup per (slice, range of tiles) loads the slice of x into LDS and streams
// the slice's stored elements, kSlicedTile per wave and step, in row order; it writes one partial
// sum per run of elements of the same row (a run is also cut at every tile start, so tiles are
// independent).  Pass 2: one wave per block of `rows_per_wave` rows of A adds the partial sums of
// its rows, slice after slice, into LDS accumulators and writes y.  The partial sums of one row
// block inside one slice are a contiguous range (`chunk_lo`).
constexpr int kSlicedTile = 256;  // stored elements per wave and step: 4 per lane
constexpr int kSlicedMaxSlices = 1024;  // the plan build ranks stored elements by slice in LDS
struct SlicedMatrix {
    int32_t width;          // columns per slice
    int32_t nslices;
    int32_t ntiles;         // all slices; every slice starts a new tile and is padded to whole tiles
    int32_t npartials;      // partial sums written per call
    int32_t nwg;            // workgroups of pass 1
    int32_t npieces;        // what they work off: runs of tiles inside one slice
    int32_t rows_per_wave;  // pass 2
    int32_t nrb;            // ceil(m / rows_per_wave)
    void *store;            // one allocation: val, perm, cf, tile_base, wg_tab, chunk_lo, pstep_ptr
    void *val;              // ntiles * kSlicedTile values (a copy of A's, in slice order; pads are 0)
    void *partial;          // npartials + kSlicedReducePad values: the partial sums of one call, for callers
                            // that bring no buffer of their own (null once released)
    uint16_t *cf;           // ntiles * kSlicedTile: column inside the slice, bit 15 = first element of a run
    int32_t *perm;          // where each stored copy comes from in A's val (-1 for pads)
    int32_t *tile_base;     // ntiles + 1: index of the first partial sum of each tile
    int32_t *wg_tab;        // npieces x 4: slice, first tile, end tile, 0
    int32_t nnz, nsort_blocks;  // stored elements; blocks of 4096 of them, as the build sorted them
    uint16_t *pos;          // nnz: position of each stored element among its block's elements in slice order
    int32_t *block_base;    // (nsort_blocks + 1) x nslices: slot of a block's first element of each slice (last row: the slices' ends)
    int32_t *wg_pieces;     // nwg x 8: first piece, end piece of each workgroup, 0, 0, then the first piece's four
                            // words again
    uint16_t *prow;         // npartials + kSlicedReducePad: row of each partial sum inside its row block
    int32_t *chunk_lo;      // (nrb + 1) x nslices: first partial sum of row block b in slice s
    int32_t npsteps;        // steps of pass 2, all row blocks
    int32_t *pstep_ptr;     // nrb + 1: first step of each row block
    int32_t *psteps;        // npsteps (+ kSlicedStepPad) x 4: up to 64 partial sums from up to 3 pieces of ranges
};
constexpr int kSlicedStepPad = 64;     // readable step descriptors past the last one
constexpr int kSlicedReducePad = 256;  // entries of prow / partial that pass 2 may read past the last partial sum
// the most steps there can be (k_sliced_pack)
inline int64_t sliced_steps_most(int64_t npartials, int64_t nrb, int64_t nslices) { return npartials / kWave + nrb * (nslices / 3 + 2); }
template <typename T>
int build_sliced(int32_t m, int32_t n, int32_t nnz, int32_t width, int32_t rows_per_wave, int32_t target_wgs,
                 const int32_t *row_ptr, const int32_t *col, const T *val, SlicedMatrix *out, hipStream_t s);
void free_sliced(SlicedMatrix *p, bool idle);
template <typename T>
int sliced_update_values(const SlicedMatrix *sm, const T *val, hipStream_t s, const unsigned long long *unless_equal = nullptr);
template <typename T>
int launch_spmv_sliced(int32_t m, int32_t n, T alpha, const SlicedMatrix *sm, const T *x, T beta, T *y, T *partial,
                       hipStream_t s);
inline size_t sliced_scratch_bytes(const SlicedMatrix *sm, size_t sv) { return ((size_t)sm->npartials + kSlicedReducePad) * sv; }

// ---- row blocks with sliding windows of x in LDS (asx_window.hip) ----
// Blocks of `rows_per_block` consecutive rows whose columns all lie inside at most kWindowBands
// bands that together span fewer than 16384 columns, chained: a workgroup walks a chain of blocks
// with a ring in LDS per band and fetches, per block, only the columns that are new.  The stored
// elements stream as tiles (16-bit LDS slot + row-start flag, as the sliced kernel's); every row
// owns at least one slot, so a tile's runs are consecutive rows and go straight to y.
constexpr int kWindowBands = 4;
struct WindowMatrix {
    int32_t rows_per_block;
    int32_t nblocks;
    int32_t nchains;         // workgroups
    int32_t npieces;         // entries of `pieces`
    int32_t ntiles;
    int32_t nbands;          // 1: one window per block; 2..kWindowBands: bands of diagonals
    int32_t stack_rows;      // > 0: three bands on stacked planes of this many rows, the blocks stored column by column
    int has_carry;           // some tile starts inside a row: the ordered carry pass is needed
    int by_reference;        // every row holds two stored elements or more: the stored elements of a tile are consecutive in
                             // A's val, which the kernel reads in place (no val, no perm)
    void *store;             // one allocation: val, perm (unless by_reference), cf, tile_info
    void *tables;            // one allocation: blocks, pieces, chains
    void *val;               // ntiles * kSlicedTile values (a copy of A's; pads are 0)
    void *carry;             // ntiles values: the carries of one call, for callers that bring no buffer (null once released)
    uint16_t *cf;            // ntiles * kSlicedTile: LDS slot of the column, bit 15 = first slot of a row (or tile)
    int32_t *perm;           // where each stored copy comes from in A's val (-1 for pads)
    int32_t *tile_info;      // ntiles x 4: row of the tile's first slot (bit 31: the tile starts inside it), rows in the tile,
                             // by_reference: index of the tile's first stored element in A's val, stored elements in the tile
    int32_t *blocks;         // nblocks x 4: first tile, end tile, first piece, end piece
    int32_t *pieces;         // x 4: columns of x to fetch before a block (from, to), first LDS slot and size of their ring
    int32_t *chains;         // nchains x 2: first block, end block
};
// in_place: where no row holds fewer than two stored elements, keep no copy of the values and read A's in every call
template <typename T>
int build_window(int32_t m, int32_t n, int32_t nnz, int32_t target_wgs, bool in_place, const int32_t *row_ptr,
                 const int32_t *col, const T *val, WindowMatrix *out, hipStream_t s);
void free_window(WindowMatrix *p, bool idle);
template <typename T>
int window_update_values(const WindowMatrix *wm, const T *val, hipStream_t s, const unsigned long long *unless_equal = nullptr);
template <typename T>
int launch_spmv_window(int32_t m, int32_t n, T alpha, const WindowMatrix *wm, const T *val, const T *x, T beta, T *y, T *carry,
                       hipStream_t s);
inline size_t window_scratch_bytes(const WindowMatrix *wm, size_t sv) { return wm->has_carry ? (size_t)wm->ntiles * sv : 0; }

// lanes per row of the vector kernel: the power of two that holds a mean row
inline int vector_lanes(int32_t m, int32_t nnz)
{
    int l = 2;
    while (l < 64 && (double)nnz > (double)l * (double)m) l *= 2;
    return l;
}
inline int32_t merge_tiles(int32_t m, int32_t nnz) { return (int32_t)ceil_div64((int64_t)m + nnz, kMergeTile); }
// Without a plan the flat kernel's tiles look up their own rows up to this many tiles; beyond it the search's latency at the
// start of every workgroup costs more than a launch of its own (12 per row, within 3000 of the diagonal, tiles' own search and the
// launch: 2000 tiles fp64 16.8 and 17.8 us, fp32 13.3 and 14.7; 4700 28.1 and 28.3, 22.8 and 22.0; 6500 37.7 and 36.4, 28.3 and
// 27.2; 8192 47.9 and 46.8, 33.3 and 30.8; 16400 91.5 and 87.0, 65.3 and 59.1; scattered columns, fp32 2000 18.3 and 19.1, 8192
// 53.7 and 50.3).
constexpr int32_t kFlatSelfSearchMost = 4096;
inline int32_t flat_tiles(int32_t nnz) { int32_t t = (int32_t)ceil_div64(nnz, kFlatTile); return t < 1 ? 1 : t; }
inline int32_t stream_blocks(int32_t nnz) { return (int32_t)ceil_div64(nnz, kStreamTile); }
// What an SpMM plan knows of A's columns: nothing; that neighbouring rows share most of them (stencils, narrow bands); that
// they share few, but a stretch of rows stays within a part of B that an L2 can keep; that they lie all over B.
enum { kColumnsUnknown = 0, kColumnsNear = 1, kColumnsScattered = 2, kColumnsSpread = 3 };
// How many bytes of a row of B a wave takes at once; the tiles of columns are worked off one after the other, so what an
// L2 (4 MB, one per XCD) or L1 (32 KB) can keep of B is the narrower the more rows of it.
//   Rows of B that start on 128-byte lines can be cut between lines: 128 bytes while all of B's tile is small
//   (k = 30000, 256 columns fp32: 58 us against 77 with 256 bytes and 102 with 1 KB; k = 100000: 173 / 197 / 228;
//   k = 200000: 459 / 446 / 499) or the part of it that a stretch of rows needs is, unless that fits 256 bytes wide as well
//   (64 columns fp64, 20 per row within 30000 of the diagonal: 187 us against 232; within 1000, 128 columns: 128 against
//   118), else 256 (fewer reads of A; near columns: 2-D stencil 193 us against 214).
//   Other rows begin and end inside lines wherever they are cut, 100 columns fp32 are 4.1 lines in one piece and 5.1 in
//   two: 1 KB for scattered columns, 512 bytes for near ones (7-point stencil, 200 columns: 223 us against 244) or
//   when nothing is known.
constexpr int64_t kSmallTileOfB = 16 << 20;
inline int spmm_tile_bytes(int columns, int64_t k, const void *B, size_t pitch)
{
    if (pitch % 128 == 0 && (uintptr_t)B % 128 == 0)
        return columns == kColumnsSpread || (columns != kColumnsNear && k * 128 <= kSmallTileOfB) ? 128 : 256;
    return columns == kColumnsScattered ? 1024 : 512;
}
// spread: distinct 128-byte lines of a vector of the value type per stored element of a sample tile; span: columns between a
// tile's first and last; mean: elements per row.  Rows that share little touch more than 4 new columns each, counting whole
// lines (2-D stencils 3.4, 20 per row within 300 and 1000 of the diagonal 13 and 40); shorter ones than 8 do not repay the
// second read of A (4 per row within 10000: 66 us against 64), longer ones than 30 leave lane groups idle (32: 352 / 352).
inline int spmm_columns(double spread, double span, double mean, size_t sv)
{
    if (mean >= 8.0 && mean <= 30.0 && spread * mean * (128 / sv) > 4.0 && span * 256 > (4 << 20) && span * 128 <= kSmallTileOfB)
        return kColumnsSpread;
    return spread < kScatteredMinSpread ? kColumnsNear : kColumnsScattered;
}

// Merge items per wave of the SpMM merge kernel.  Longer segments leave fewer carries and keep the
// lane groups of narrow N busy, shorter ones leave room for more waves (LDS) and spread small
// matrices: 128 while 256 a wave would leave fewer than 16 waves per compute unit.  Where a row of B
// takes 16 lanes or more of fp32 (at most four groups a wave, 8 bytes staged per element) 512 measured
// 2 % ahead of 256 on 17 M items, elsewhere 256 is up to 16 % ahead (8 columns of fp64: 46.4 / 55.2 us).
inline int32_t spmm_segment_items(int32_t m, int32_t nnz, int32_t ncols, size_t sv)
{
    const int64_t items = (int64_t)m + nnz;
    if (spmm_chunked_unplanned(m, nnz, ncols, sv)) return spmm_chunk_items(items);
    if (spmm_chunked_mid(m, nnz, ncols, sv)) return (int32_t)std::max<int64_t>(kSpmmSegmentMedium, ceil_div64(items, kChunkRound));
    if (spmm_chunked_wide(m, nnz, ncols, sv)) return spmm_chunk_wide_items(spmm_chunk_wide_work(m, nnz, ncols * (int64_t)sv));
    if (items < (int64_t)kSpmmSegmentMedium * 4096) return kSpmmSegmentSmall;
    return sv == 4 && ncols > 32 && items >= (int64_t)kSpmmSegmentLarge * 4096 ? kSpmmSegmentLarge : kSpmmSegmentMedium;
}
// Columns of B a lane takes, tiles of columns, and lane groups of a wave (which take a row of A each) when a wave takes at most
// tile_bytes of a row of B.
struct SpmmTiling {
    int vec;
    int64_t tiles;
    int log_lanes, groups;
};
inline SpmmTiling spmm_tiling(int64_t ncols, int tile_bytes, size_t sv)
{
    SpmmTiling t;
    t.vec = ncols >= (int64_t)(16 / sv) ? (int)(16 / sv) : ncols >= 2 ? 2 : 1;
    const int64_t most = tile_bytes / (int64_t)sv;
    t.tiles = ceil_div64(ncols, most > t.vec ? most : t.vec);
    const int64_t lanes = ceil_div64(ceil_div64(ncols, t.tiles), t.vec);
    for (t.log_lanes = 0; ((int64_t)1 << t.log_lanes) < lanes;) ++t.log_lanes;
    t.groups = kWave >> t.log_lanes;
    return t;
}
// Rows of up to this many elements are taken by one lane group each, longer ones by all groups together.  32 against 16 with
// up to 4 groups: 40 columns fp64, 20 per row within 2000 of the diagonal 170 -> 148 us, 64 columns fp32 over scattered rows
// of 25 141 -> 135 us, power-law rows 207.7 -> 204.1 us.
constexpr int spmm_dealt(int groups) { return groups == 1 ? 1 << 30 : groups <= 4 ? 32 : 64; }
// Where a wave's groups take a row each and its segment holds fewer than five eighths as many, most groups have nothing to do: then the
// segment is twice as long, up to 256 items, or 512 of fp32 that several tiles of columns read (one tile: 21 columns, 55 per row 29.5 us with 256
// and 35.3 with 512).  Never shorter than usual, so that the carries fit.  The merge kernel with
// rows of B on lines, 128 bytes of them at a time, 0.9 M elements, uniform columns and within 1500 of the diagonal, segments of 128 items
// against 256 and 512: 28 per row 256 columns fp32 91.8 and 78.5, 83.0 and 60.1; 48 88.3 and 61.5, 83.6 and 56.9; 61 94.8, 78.1 and 66.1, 91.7,
// 76.1 and 57.7; 96 columns fp64, 36 per row 34.9 and 25.2; but 20 per row, 6 of 8 groups, 60.0 and 64.0, 34.2 and 36.8.  Twelve
// waves a compute unit have to be left (27 columns fp64, 3144 rows of 62 17.4 us in 1550 waves, 20.4 in 775).
inline int32_t spmm_filled_items(int32_t usual, const SpmmTiling &tiling, int32_t m, int32_t nnz, size_t sv)
{
    const int32_t most = sv == 4 && tiling.tiles > 1 ? kSpmmSegmentLarge : kSpmmSegmentMedium;
    const int64_t all = (int64_t)m + nnz;
    int32_t items = usual;
    while (items < most && 8 * (int64_t)items * m < 5 * tiling.groups * all && all / (2 * items) * tiling.tiles >= 12 * 256) items *= 2;
    return items;
}
// Segments of a plan whose columns are near or spread, where they leave no row cut (carries of more segments would not fit the
// workspace that callers size without a plan).  They are short, so that fewer rows of B are in use at a time, and where rows are
// of one length (the longest at most a quarter above the mean) they hold as many as the wave's groups take in full turns.
// 64 columns fp32, 20 per row within 1000 of the diagonal: 94.9 us with segments of 512 items, 54.2 with two turns of 84;
// 7-point stencil 78.7 -> 59.7, 5-point stencil 128.7 -> 85.7; 13 per row 50.2 -> 42.3.
// Chunk kernel: where rows are too long for the longest segments, but none for one of the usual length, no row is cut (a carry
// pass is a launch more: longest row 913 of 82000 elements 8.8 -> 5.9 us).  In more than two rounds even rows do without a last turn
// of a workgroup's groups that would not be half full (8 columns fp64 within 3000 of the diagonal, 8 M elements, whole turns against
// segments of 2688 items: 15 per row 62.1 against 66.5 us, 17 59.5 and 64.3, 19 57.7 and 61.7; 16 columns fp32, 19 per row 54.2
// and 56.0; a last turn that is half full is kept: 10 per row 71.9 without and 68.7 with), in one or two without one of a sixteenth
// (5 per row, 6 columns fp32, 2 M 20.0 -> 18.1).  Rounding up would make fewer and longer segments: 9 per row, 350000 elements, 3
// columns fp64 152 workgroups 7.0 us, 579 6.2; 5 per row, 8 fp32 7.6 and 6.5; 9 per row, 3 columns fp64, 800000 10.3 and 8.9, 1.4 M
// 14.2 and 13.0.  Wide rows of B (row_bytes): never more segments than usual, so that their carries fit.
inline int32_t spmm_plan_items(int32_t usual, int columns, const SpmmTiling &tiling, int32_t m, int32_t nnz, int64_t longest, bool chunked,
                               int64_t row_bytes, size_t sv)
{
    const int groups = tiling.groups;
    if (chunked && spmm_chunked_mid(m, nnz, row_bytes, 1)) return usual;
    if (chunked && row_bytes > 64) return std::max(usual, spmm_chunk_wide_items(spmm_chunk_wide_work(m, nnz, row_bytes)));
    if (chunked) {
        const int32_t cut = spmm_chunk_items((int64_t)m + nnz);  // usual or more
        if (longest > kChunkLongest) return longest > kChunkItems || longest <= cut ? cut : (int32_t)longest;
        const int32_t items = spmm_chunk_uncut_items((int64_t)m + nnz);
        if (4 * (longest + 1) * m > 5 * ((int64_t)m + nnz)) return items;
        const int64_t turn = (int64_t)groups * (kChunkThreads / kWave) * (longest + 1), over = items % turn;
        return turn <= items && (items < kChunkItemsMost ? 16 : 2) * over <= turn ? (int32_t)(items - over) : items;
    }
    if (columns != kColumnsNear && columns != kColumnsSpread) return spmm_filled_items(usual, tiling, m, nnz, sv);
    const int32_t least = usual == kSpmmSegmentLarge ? kSpmmSegmentSmall : usual;
    const int64_t turn = groups * (longest + 1);
    const int32_t most = usual == kSpmmSegmentLarge && turn > kSpmmSegmentSmall ? kSpmmSegmentMedium : least;
    if (longest > spmm_dealt(groups) || turn > most || 4 * (longest + 1) * m > 5 * ((int64_t)m + nnz)) return least;
    return (int32_t)(most / turn * turn);
}
// Columns lie all over B and ascend in a row, as a sample's tiles of 1024 elements tell: first and last column of a tile nearly as
// far apart as B has rows (uniform columns: 0.998 of them); about as many different lines as uniform columns would touch, of
// `lines` on average lines (1 - exp(-1024 / lines)); and about one fall a row (unsorted rows: one every other element, two a row and
// more from four elements on).
inline bool spmm_everywhere(double spread, double span, double falls, double mean, int64_t k, size_t sv)
{
    const double lines = (double)k * (double)sv / 128.0 + 1.0;
    return span >= 0.9 * (double)k && spread * kFlatTile >= 0.7 * lines * (1.0 - exp(-kFlatTile / lines)) && falls * mean <= 1.25 * kFlatTile;
}
// The sweep kernel, where its sizes suit it (slots 0: not).  What its caller has to know beside these: that columns ascend in a row
// and lie all over B, and that no row is longer than spmm_sweep_longest.
//   Sixteen waves a compute unit share 160 KB of LDS, in which a wave stages its part of A; a group takes as many rows as that and
//   its registers allow, evened out over the rounds of waves.
//   Windows: the more, the less of B a window needs (a wave ahead or behind does less harm), but every window costs its
//   instructions whether rows have an element in it or not: 1.24 MB(B)^0.35 mean^-0.3 windows an element of a mean row, between 1
//   and 2.5, fitted to 110 uniform matrices (both types, rows of B of 72 to 2000 bytes, 4 to 64 per row, B of 14 to 317 MB)
//   timed with 1 to 6, all with one sum a row: 0.5 % behind the best of these on average; then a tenth less where a group has 16 lanes or more, which inputs that
//   are not in the Infinity Cache want (74 such matrices, three sets of inputs in turn: 0.986 of the time with the tenth; 100
//   columns fp32, 150001 rows of 25 150 us and 141).
//   On those 110 it took 0.78 of the row-ordered kernels' time on average (100 columns fp32, 160000 rows of 25 270 us against
//   130; 96, 94796 of 49 316 and 136; 64, 573065 of 9 204 and 191; 22, 1 M of 4 138 and 133).  Not taken: a B that the L2s keep
//   between them (9 MB, 14 where rows of A are short) - where rows of B start on lines the row-ordered kernels work through it
//   in tiles of one line, which they can keep up to 40000 rows or 20 MB (192 columns fp32, 27903 rows of 8 22.6 us there, 23.4 here;
//   32, 101110 of 8 17.3 and 18.4; 448, 28456 of 9 52.3 and 59.8) -; rows of fewer than 4; and where an XCD's waves meet a row of B
//   only every fourth round or less (kSweepSharedLeast; 74 columns fp32, 525797 x 1032224, 13 per row 406 and 429).
//   Long rows: in fp32 a row's error grows with the elements that one sum runs over, and the row-ordered kernels sum rows of more than
//   spmm_dealt elements in as many sums as a wave has groups.  So does the sweep (chains), and a group then has registers for
//   1 / chains of the rows; rows that those kernels cut, or give to a whole workgroup, are not taken.  49 per row, 100 columns: rms error 1.34
//   times theirs with one sum, as theirs with two.
constexpr int kSweepWaves = 16;
constexpr double kSweepSharedLeast = 0.25;
// sums a row for rows of up to `longest` elements, none of which is cut; 0: more than the sweep has
inline int spmm_sweep_chains(int64_t longest, int groups, bool chunked)
{
    if (longest <= (chunked ? std::min(spmm_dealt(groups), kChunkWideLeast) : spmm_dealt(groups))) return 1;
    return groups > 1 && groups <= 4 && (!chunked || longest <= kChunkWideLeast) ? groups : 0;
}
inline int64_t spmm_sweep_longest(int32_t m, int32_t nnz) { return 2 * ((int64_t)nnz / (m > 0 ? m : 1)) + 8; }
constexpr int32_t spmm_sweep_cap(size_t sv) { return (int32_t)(160 * 1024 / kSweepWaves / (4 + sv)) & ~1; }
// what does not depend on the number of columns
inline SpmmSweep spmm_sweep_shape(int32_t m, int32_t nnz, int64_t ncols, size_t sv, int chains)
{
    SpmmSweep sw{};
    if (m <= 0 || ncols * (int64_t)sv <= 64 || nnz / m < 4 || chains < 1) return sw;
    const double mean = (double)nnz / m;
    const SpmmTiling t = spmm_tiling(ncols, 1024, sv);
    const int32_t cap = spmm_sweep_cap(sv);
    int64_t rows = std::min<int64_t>((t.log_lanes < 5 ? 1 << t.log_lanes : 20) / chains, (int64_t)(cap / (1.05 * mean * t.groups)));
    if (t.log_lanes < 3 || rows < 1 || t.tiles > 65535) return sw;
    const int64_t round = (int64_t)kSweepWaves * 256 * t.groups;
    rows = ceil_div64(m, round * ceil_div64(m, round * rows));
    sw.rows = (int32_t)rows;
    sw.chains = chains;
    const int64_t slots = rows * chains;
    sw.slots = slots <= 4 ? 4 : slots <= 8 ? 8 : slots <= 12 ? 12 : slots <= 16 ? 16 : 20;
    sw.cap = std::min(cap, ((int32_t)(1.1 * mean * (double)(rows * t.groups)) + 2) & ~1);
    sw.log_lanes = t.log_lanes;
    sw.tiles = t.tiles;
    return sw;
}
inline int64_t spmm_sweep_blocks(const SpmmSweep &sw, int32_t m)
{
    const int64_t waves = ceil_div64(m, (int64_t)sw.rows * (kWave >> sw.log_lanes));
    return ceil_div64(ceil_div64(waves, kBlock / kWave), kXcds) * kXcds;
}
// elements an XCD's waves hold at a time for each row of B
inline double spmm_sweep_shared(const SpmmSweep &sw, int32_t m, int32_t n, int32_t nnz)
{
    const int64_t round = (int64_t)kSweepWaves * 256 * (kWave >> sw.log_lanes);
    return (double)std::min<int64_t>(round * sw.rows, m) * ((double)nnz / m) / kXcds / n;
}
inline SpmmSweep spmm_sweep(int32_t m, int32_t n, int32_t nnz, int64_t ncols, size_t sv, int chains)
{
    const int64_t bytes = ncols * (int64_t)sv;
    SpmmSweep sw = spmm_sweep_shape(m, nnz, ncols, sv, chains);
    if (sw.slots == 0 || n <= 0) return SpmmSweep{};
    const double mean = (double)nnz / m, mb = 1e-6 * (double)bytes * n;
    if (bytes % 128 == 0 ? mb < 20.0 || n < 40000 : mb < (mean < 14.0 ? 14.0 : 9.0)) return SpmmSweep{};
    if (spmm_sweep_shared(sw, m, n, nnz) < kSweepSharedLeast) return SpmmSweep{};
    const double windows = (sw.log_lanes >= 4 ? 0.9 : 1.0) * mean * std::min(std::max(1.24 * pow(mb, 0.35) * pow(mean, -0.3), 1.0), 2.5);
    sw.width = (uint32_t)std::max((double)n / windows, 1.0) + 1;
    return sw;
}
// Calls whose columns nobody has looked at: whether asking pays (slots 0: not).  Where the answer is no, the launch is spent: 4.6 us with
// one round of workgroups (100 columns fp32, 160001 power-law rows of 20: 264 us before), 5.8 with two, 8 with three (250 columns, 100003 rows
// of 36 within 3000 of the diagonal: 274 us before).  So it is for calls whose rows of B, each fetched by itself, take 240 us and more,
// for two rounds at most (three where a row is several sums), and where an XCD's waves meet a row of B often: 100 columns fp32, 150001
// uniform rows of 25, 3.1 times, 257 us without and 150 with; 250 columns, 80000 rows of 25 and 400000 columns of A, 0.62 times, 359 and 278
// - below 0.6 a yes still gains (500000, 0.5 times, 359 and 289), but less, for the same price of a no.  Rows of B that start on lines,
// which the merge kernel takes a line or two at a time, gain less (256 columns fp32, 60001 uniform rows of 30, 173 us without and 157 with; 128 fp64, 20 per row
// within 3000 of the diagonal 165 and 171): from twice as many lines on.  Rows that the merge kernel cuts have to be longer than
// the sweep takes: it looks at whole rows only.
constexpr double kSweepAskLines = 240e-6 * 58e9, kSweepAskShared = 0.6;
constexpr int64_t kSweepAskBlocks = 3 * 1024;
constexpr int64_t spmm_sweep_ask_blocks(int chains) { return chains > 1 ? kSweepAskBlocks : 2 * 1024; }
// The longest row it takes then: rows of up to spmm_dealt elements where the mean is no longer, so that they need one sum each; longer
// means with two or four sums, but no row that eight groups would share.
inline int32_t spmm_sweep_ask_longest(int32_t m, int32_t nnz, int groups)
{
    const int64_t longest = spmm_sweep_longest(m, nnz), dealt = spmm_dealt(groups);
    return (int32_t)(nnz <= dealt * m || groups > 4 ? std::min(longest, dealt) : longest);
}
inline bool spmm_sweep_askable(const SpmmSweep &sw, int32_t m, int32_t nnz, int64_t ncols, size_t sv, int32_t items)
{
    const int64_t bytes = ncols * (int64_t)sv;
    return sw.slots > 0 && (double)nnz * ((double)bytes / 128.0 + (bytes % 128 ? 1.0 : 0.0)) >= kSweepAskLines &&
           (bytes % 128 || (double)nnz * (double)bytes / 128.0 >= 2.0 * kSweepAskLines) &&
           spmm_sweep_longest(m, nnz) <= items && spmm_sweep_blocks(sw, m) <= spmm_sweep_ask_blocks(1);
}
inline int32_t spmm_segments(int32_t m, int32_t nnz, int32_t items) { return (int32_t)ceil_div64((int64_t)m + nnz, items); }

}  // namespace asx

constexpr int kPlanCounters = 128;
// Plan: analysis results kept on the device across calls.
struct asx_plan {
    int is_spmm;
    int alg;  // resolved kernel
    int value_type;
    int32_t m, n, nnz, ncols;
    const int32_t *row_ptr;  // the device array the plan was built from (identity check only)
    int64_t *d_counters;     // kPlanCounters words on the device: histogram (33), stats (4), a flag (40), counts of long rows (41),
                             // checksums of the values: of this call (44, 45) and of the copy the plan holds (46, 47),
                             // 64 sample counts (64..95)
    int checked;             // the plan holds a copy of A's values and a checksum of them (asx_spmv_plan_create_checked)
    unsigned long long *d_checksum_parts;  // checked plans: the workgroups' partial sums of one checksum run
    int32_t nmarked;         // row blocks of the stream kernel behind the counters (0: none)
    int32_t *d_meta;         // split points / row blocks (layout depends on alg)
    size_t meta_bytes;
    int32_t nunits;  // tiles / row blocks / segments
    int carry_pass;  // flat and SpMM merge kernel: 0 when no row is cut between units of work
    int32_t nwide, nlong, long_len;  // vector kernel: d_meta lists the long rows (asx::LongRows)
    int columns;     // SpMM merge kernel: kColumns*
    int32_t items;   // SpMM merge and chunk kernels: merge items per segment
    int chunked;     // SpMM: the chunk kernel
    int sweep;       // SpMM: rows and columns of A suit the sweep kernel
    int asks;        // SpMM: DEFAULT without a look at the columns
    int64_t hist[33];
    int64_t stats[4];
    size_t workspace_bytes;
    asx::BlockedMatrix blocked;  // only for ASX_SPMM_BLOCKED plans
    asx::SlicedMatrix sliced;    // only for ASX_SPMV_SLICED plans
    asx::WindowMatrix window;    // only for ASX_SPMV_WINDOW plans
};
