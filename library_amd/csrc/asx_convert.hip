// Operand conversions around the CSR kernels, all on the device:
//   asx_csr_transpose   A -> A^T as zero-based CSR (what opA = TRANSPOSE runs on).  The reference
//                       does this on the host with two copies across PCIe per call and writes the
//                       result over the caller's arrays (hip/format/transpose_csr.h:9-71).
//   asx_csr_rebase      one-based row offsets / column indices -> zero-based copies.
//   asx_dense_transpose out[c][r] = in[r][c] for a strided dense matrix (column-major B and C of
//                       SpMM; the reference: hip/format/transpose_dn_mat.h:4-35, one element per
//                       thread with uncoalesced writes).
#include <rocprim/device/device_radix_sort.hpp>

#include <algorithm>
#include <cstring>
#include <type_traits>

#include "asx_internal.hpp"
#include "asx_rank.hpp"
#include "asx_scan.hpp"

namespace asx {

// For matrices of so many columns that the bucket passes below do not take them:
// key = (zero-based column << 32) | row, payload = position of the stored element.  A stable sort
// of the keys orders the elements of each column by row, duplicates in their stored order: the
// order the reference's counting transpose produces.
__global__ __launch_bounds__(kBlock) void k_transpose_keys(const int32_t *__restrict__ row_ptr,
                                                           const int32_t *__restrict__ col, int32_t m,
                                                           int32_t nnz, int32_t base,
                                                           uint64_t *__restrict__ keys,
                                                           int32_t *__restrict__ idx)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nnz) return;
    const int32_t e = (int32_t)i + base;  // position in the numbering row_ptr uses
    int32_t lo = 0, hi = m;               // largest r with row_ptr[r] <= e
    while (lo < hi) {
        const int32_t mid = lo + (hi - lo + 1) / 2;
        if (row_ptr[mid] <= e)
            lo = mid;
        else
            hi = mid - 1;
    }
    keys[i] = ((uint64_t)(uint32_t)(col[i] - base) << 32) | (uint32_t)lo;
    idx[i] = (int32_t)i;
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_transpose_apply(const uint64_t *__restrict__ keys,
                                                            const int32_t *__restrict__ idx,
                                                            const T *__restrict__ val, int32_t nnz,
                                                            int32_t *__restrict__ trow,
                                                            int32_t *__restrict__ col_t,
                                                            T *__restrict__ val_t)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nnz) return;
    const uint64_t k = keys[i];
    trow[i] = (int32_t)(k >> 32);
    col_t[i] = (int32_t)(k & 0xFFFFFFFFu);
    val_t[i] = val[idx[i]];
}

// row_ptr_t[r] = first i with trow[i] >= r, r in [0, n]
__global__ __launch_bounds__(kBlock) void k_offsets_from_sorted(const int32_t *__restrict__ trow, int32_t nnz,
                                                                int32_t n, int32_t *__restrict__ row_ptr_t)
{
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r > n) return;
    int32_t lo = 0, hi = nnz;
    while (lo < hi) {
        const int32_t mid = (lo + hi) / 2;
        if (trow[mid] < r)
            lo = mid + 1;
        else
            hi = mid;
    }
    row_ptr_t[r] = lo;
}

int launch_offsets_from_sorted(const int32_t *sorted, int32_t count, int32_t n, int32_t *out, hipStream_t s)
{
    hipLaunchKernelGGL(k_offsets_from_sorted, dim3((unsigned)ceil_div64((int64_t)n + 1, kBlock)), dim3(kBlock), 0, s,
                       sorted, count, n, out);
    return check_launch();
}

namespace {

// ---- transpose: two passes -----------------------------------------------------------------
// A stable counting sort of the stored elements by column, in two passes over them.  Buckets are
// ranges of 2^shift columns, at most kBuckets of them, of about kSortElems elements each.
//   1. k_transpose_count: every block of 4096 elements counts its elements per bucket (and looks up
//      the row its waves' elements start in); an exclusive scan over (bucket, block) gives each block
//      its place in every bucket.
//   2. k_transpose_bucket: the block's elements are ranked inside their buckets (stable: row order
//      survives), ordered by bucket in LDS and written - row, column inside the bucket, value - in runs
//      of consecutive places.
//   3. k_transpose_rows: one workgroup per bucket orders its elements by column through LDS and writes the columns' row
//      offsets: up to 8 elements a thread in one turn, larger buckets 4096 elements at a time behind a
//      count of their columns.  Buckets far above the average follow in pieces.
// 3.6 M elements, fp32, 250013 columns: 97 us with the CSR multiply that follows it; a radix sort of
// 64-bit (column, row) keys moved 24 bytes an element five times and took 316 us of kernels alone.
constexpr int kBuckets = 1024;
constexpr int kBucketColumns = 4096;  // the most columns a bucket may span: 16-bit counters per wave in LDS

__global__ __launch_bounds__(kSortThreads) void k_transpose_count(const int32_t *__restrict__ row_ptr,
                                                                  const int32_t *__restrict__ col, int32_t m, int32_t nnz,
                                                                  int32_t base, int shift, int32_t nbuckets, int32_t nblocks,
                                                                  int32_t *__restrict__ counts, int32_t *__restrict__ seg_row)
{
    __shared__ int32_t hist[kBuckets];
    const int32_t b = block_of_xcd();
    if (b >= nblocks) return;  // the whole workgroup leaves
    int32_t c[kSortPerLane];
    load_columns(col, nnz, b, c);
    for (int s = threadIdx.x; s < nbuckets; s += kSortThreads) hist[s] = 0;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kSortPerLane; ++k)
        if ((int64_t)b * kSortElems + k * kSortThreads + threadIdx.x < nnz)
            atomicAdd(&hist[(c[k] - base) >> shift], 1);  // integer counts: the order does not matter
    block_seg_rows(row_ptr, m, nnz, base, b, nblocks, seg_row);
    __syncthreads();
    for (int s = threadIdx.x; s < nbuckets; s += kSortThreads) counts[(int64_t)s * nblocks + b] = hist[s];
    if (b == 0 && threadIdx.x == 0) counts[(int64_t)nbuckets * nblocks] = 0;
}

// Four workgroups a compute unit in fp32 (37 KB of LDS, 64 registers), three in fp64 (53 KB): its chain of dependent steps
// is long, and 3.6 M elements are 879 workgroups - two rounds with 57 KB.  Transpose and multiply:
// 120.1 -> 114.5 us.
template <typename T>
__global__ __launch_bounds__(kSortThreads, sizeof(T) == 4 ? 8 : 6) void k_transpose_bucket(const int32_t *__restrict__ row_ptr,
                                                                   const int32_t *__restrict__ col, const T *__restrict__ val,
                                                                   const int32_t *__restrict__ seg_row, int32_t nnz, int32_t base,
                                                                   int shift, int32_t nbuckets, int nbits, int32_t nblocks,
                                                                   const int32_t *__restrict__ offs, int32_t *__restrict__ brow,
                                                                   uint16_t *__restrict__ bcol, T *__restrict__ bval)
{
    // per wave and bucket: count, then first rank of the wave's elements; when those are used up, the columns in bucket order
    __shared__ __align__(16) unsigned char lds[kSortElems * sizeof(int32_t)];
    static_assert(sizeof(uint16_t) * kSortWaves * kBuckets <= sizeof(lds), "the counters lie where the columns go");
    __shared__ int32_t lofs[kBuckets];  // per bucket: the block's count, then its first position in bucket order, then its place minus that
    __shared__ int32_t wave_tot[kSortWaves];
    __shared__ __align__(16) unsigned char stage[kSortElems * (sizeof(T) > 4 ? sizeof(T) : 4)];
    uint16_t *cnt = reinterpret_cast<uint16_t *>(lds);
    int32_t *col_s = reinterpret_cast<int32_t *>(lds);
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    // consecutive blocks write neighbouring places of every bucket: keep them on one XCD, whose L2
    // then merges their pieces of a cache line (the grid is a multiple of kXcds workgroups)
    const int32_t per_xcd = (int32_t)gridDim.x / kXcds;
    const int32_t b = ((int32_t)blockIdx.x % kXcds) * per_xcd + (int32_t)blockIdx.x / kXcds;
    if (b >= nblocks) return;  // the whole workgroup leaves
    for (int i = tid; i < kSortWaves * nbuckets; i += kSortThreads) cnt[i] = 0;
    const int64_t wbase = (int64_t)b * kSortElems + (int64_t)wave * kSortWaveElems;
    int32_t c[kSortPerLane], p[kSortPerLane];
    T v[kSortPerLane];
#pragma unroll
    for (int k = 0; k < kSortPerLane; ++k) {
        const int64_t i = wbase + k * kWave + lane, at = i < nnz ? i : nnz - 1;
        c[k] = col[at] - base;
        v[k] = val[at];
    }
    const int64_t g = (int64_t)b * kSortWaves + wave;
    const int32_t r_lo = __builtin_amdgcn_readfirstlane(seg_row[g]), r_hi = __builtin_amdgcn_readfirstlane(seg_row[g + 1]);
    int32_t *row_s = reinterpret_cast<int32_t *>(stage);
    int32_t *my_rows = row_s + wave * kSortWaveElems;
    int32_t r[kSortPerLane];
    wave_rows(row_ptr, base, r_lo, r_hi, wbase, nnz, my_rows, r);
    // the rows wait in LDS: in registers they would cost waves
#pragma unroll
    for (int k = 0; k < kSortPerLane; ++k) my_rows[k * kWave + lane] = r[k];
    __syncthreads();
    uint16_t *mycnt = cnt + wave * nbuckets;
#pragma unroll
    for (int k = 0; k < kSortPerLane; ++k) p[k] = wave_rank(c[k] >> shift, wbase + k * kWave + lane < nnz, nbits, mycnt);
    __syncthreads();
    constexpr int kPer = kBuckets / kSortThreads;
    int32_t place[kPer];  // of the block's first element in buckets tid, tid + kSortThreads, ...
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
        const int s = tid + q * kSortThreads;
        if (s >= nbuckets) break;
        place[q] = offs[(int64_t)s * nblocks + b];
        int32_t run = 0;
#pragma unroll
        for (int w = 0; w < kSortWaves; ++w) {
            const int32_t t = cnt[w * nbuckets + s];
            cnt[w * nbuckets + s] = (uint16_t)run;
            run += t;
        }
        lofs[s] = run;
    }
    __syncthreads();
    block_exclusive_sum(lofs, nbuckets, wave_tot);
#pragma unroll
    for (int k = 0; k < kSortPerLane; ++k) {
        if (wbase + k * kWave + lane < nnz) p[k] += lofs[c[k] >> shift] + mycnt[c[k] >> shift];
        r[k] = my_rows[k * kWave + lane];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
        const int s = tid + q * kSortThreads;
        if (s < nbuckets) lofs[s] = place[q] - lofs[s];
    }
    const int32_t *to = lofs;
#pragma unroll
    for (int k = 0; k < kSortPerLane; ++k) {
        if (wbase + k * kWave + lane < nnz) {
            col_s[p[k]] = c[k];
            row_s[p[k]] = r[k];
        }
    }
    __syncthreads();
    const int64_t left = (int64_t)nnz - (int64_t)b * kSortElems;
    const int32_t count = left < kSortElems ? (int32_t)left : kSortElems;
    const int32_t inside = (1 << shift) - 1;
    for (int j = tid; j < count; j += kSortThreads) {
        const int32_t q = col_s[j], d = to[q >> shift] + j;
        brow[d] = row_s[j];
        bcol[d] = (uint16_t)(q & inside);
    }
    __syncthreads();
    T *val_s = reinterpret_cast<T *>(stage);
#pragma unroll
    for (int k = 0; k < kSortPerLane; ++k)
        if (wbase + k * kWave + lane < nnz) val_s[p[k]] = v[k];
    __syncthreads();
    for (int j = tid; j < count; j += kSortThreads) bval[to[col_s[j] >> shift] + j] = val_s[j];
}

// in-place exclusive sum of a[0 .. COLS) by the whole workgroup, COLS a multiple of THREADS or the other way round (barriers inside)
template <int COLS, int THREADS = kSortThreads>
__device__ __forceinline__ void columns_exclusive_sum(int32_t *a, int32_t *wave_tot)
{
    constexpr int Q = COLS > THREADS ? COLS / THREADS : 1;
    const bool has = (int)threadIdx.x * Q < COLS;
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    int32_t v[Q], mine = 0;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        v[q] = has ? a[tid * Q + q] : 0;
        mine += v[q];
    }
    int32_t incl = mine;
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
        const int32_t t = __shfl_up(incl, d, kWave);
        if (lane >= d) incl += t;
    }
    if (lane == kWave - 1) wave_tot[wave] = incl;
    __syncthreads();
    int32_t run = incl - mine;
    for (int w = 0; w < wave; ++w) run += wave_tot[w];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        if (has) a[tid * Q + q] = run;
        run += v[q];
    }
    __syncthreads();
}

// COLS: columns of a bucket, rounded up to a multiple of kSortThreads
template <typename T, int COLS, int THREADS = kSortThreads>
struct RowsShared {
    alignas(16) uint16_t cnt[THREADS / kWave * COLS];  // per wave and column: count, then first rank of the wave's elements
    int32_t first[COLS];                          // per column: next free place in A^T
    int32_t lofs[COLS];                           // per column: count, then first position in column order
    int32_t wave_tot[THREADS / kWave];
    int32_t row_s[kSortElems];
    uint16_t col_s[kSortElems];
    T val_s[kSortElems];
};

// Elements [s0, s1) of a bucket to their places in A^T, sh.first[c] being that of the first one of column c.
template <typename T, int COLS, int THREADS = kSortThreads>
__device__ __forceinline__ void place_by_column(RowsShared<T, COLS, THREADS> &sh, int32_t s0, int32_t s1, int nbits,
                                                const int32_t *__restrict__ brow, const uint16_t *__restrict__ bcol,
                                                const T *__restrict__ bval, int32_t *__restrict__ col_t, T *__restrict__ val_t)
{
    constexpr int WAVES = THREADS / kWave, PER = kSortElems / THREADS;
    uint16_t *cnt = sh.cnt, *col_s = sh.col_s;
    int32_t *first = sh.first, *lofs = sh.lofs, *row_s = sh.row_s;
    T *val_s = sh.val_s;
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    uint16_t *mycnt = cnt + wave * COLS;
    for (int32_t e0 = s0; e0 < s1; e0 += kSortElems) {  // uniform; one turn where the bucket fits
        __syncthreads();
        for (int i = tid; i < WAVES * COLS / 2; i += THREADS) reinterpret_cast<uint32_t *>(cnt)[i] = 0;
        const int32_t wbase = e0 + wave * (kSortElems / WAVES);
        int32_t c[PER], p[PER], r[PER];
        T v[PER];
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            const int32_t i = wbase + k * kWave + lane, at = i < s1 ? i : s1 - 1;
            c[k] = bcol[at];
            r[k] = brow[at];
            v[k] = bval[at];
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < PER; ++k) p[k] = wave_rank(c[k], wbase + k * kWave + lane < s1, nbits, mycnt);
        __syncthreads();
        for (int i = tid; i < COLS; i += THREADS) {
            int32_t run = 0;
#pragma unroll
            for (int w = 0; w < WAVES; ++w) {
                const int32_t t = cnt[w * COLS + i];
                cnt[w * COLS + i] = (uint16_t)run;
                run += t;
            }
            lofs[i] = run;
        }
        __syncthreads();
        columns_exclusive_sum<COLS, THREADS>(lofs, sh.wave_tot);
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            if (wbase + k * kWave + lane < s1) {
                const int32_t q = lofs[c[k]] + mycnt[c[k]] + p[k];
                col_s[q] = (uint16_t)c[k];
                row_s[q] = r[k];
                val_s[q] = v[k];
            }
        }
        __syncthreads();
        const int32_t count = s1 - e0 < kSortElems ? s1 - e0 : kSortElems;
        for (int j = tid; j < count; j += THREADS) {
            const int32_t q = col_s[j], d = first[q] + (j - lofs[q]);
            col_t[d] = row_s[j];
            val_t[d] = val_s[j];
        }
        if (e0 + kSortElems < s1) {  // uniform: where the next elements of every column go
            __syncthreads();
            for (int i = tid; i < COLS; i += THREADS) first[i] += (i + 1 < COLS ? lofs[i + 1] : count) - lofs[i];
        }
    }
}

// Buckets of more than kLargeBucket elements - a column that very many rows share - are left to k_transpose_large_*, which
// cut them into pieces: one workgroup takes 10 us for 4096 elements of one column, so that alone it would keep the device
// waiting (transpose of 8 M elements fp32, 6 M of them in one column: 14.7 ms, in pieces 0.30; of 400000, 68000 of them in
// one: 208 us and 153).  large[2 b], large[2 b + 1]: where the elements of such a bucket start and end, for the host
// (page-locked, cleared).
constexpr int32_t kLargeBucket = 16 * kSortElems, kLargePiece = 8 * kSortElems;

// A bucket of up to PER elements a thread is sorted in one turn: its elements are loaded once, ranked, and what the waves have counted
// per column gives the row offsets of A^T as well as the places, which are consecutive then.  Where buckets of up to 512 columns hold
// more than 4096 elements on average, all take 1024 threads instead of a count and two turns of 512, one workgroup behind the other on a
// compute unit being what bounds the kernel; counters and staged elements share LDS and values are loaded late, so that two such
// workgroups fit (64 registers).  Larger averages take them as well: most of their buckets need several turns either way, and 512
// threads came out alike (transpose and multiply, 300000 columns, 1024 and 512 threads: 6 M elements fp32 172 and 173 us, fp64 195 and
// 192; 16 M 415 and 415, 542 and 541; 32 M 921 and 927, 1235 and 1230).
// 3.6 M elements of 489 buckets, fp32: 25.9 -> 19.6 us.  Transpose and multiply, 4 M uniform elements into 200013 rows: fp32 127 -> 112
// us, fp64 149 -> 134; 1 M in one turn of 512 threads 62 -> 59.
template <typename T, int COLS, int THREADS>
struct OneTurn {
    static constexpr int PER = 8, WAVES = THREADS / kWave;
    static constexpr size_t kCounters = sizeof(uint16_t) * WAVES * COLS, kStage = sizeof(T) * PER * THREADS;
    alignas(16) unsigned char lds[kCounters > kStage ? kCounters : kStage];
    int32_t lofs[COLS];  // per column: count, then first position in column order
    int32_t wave_tot[WAVES];
};
template <typename T, int COLS, int THREADS>
__device__ __forceinline__ void rows_in_one_turn(OneTurn<T, COLS, THREADS> &sh, int32_t s0, int32_t s1, int nbits, int64_t c0, int32_t ncols,
                                                 const int32_t *__restrict__ brow, const uint16_t *__restrict__ bcol, const T *__restrict__ bval,
                                                 int32_t *__restrict__ row_ptr_t, int32_t *__restrict__ col_t, T *__restrict__ val_t)
{
    constexpr int PER = OneTurn<T, COLS, THREADS>::PER, WAVES = THREADS / kWave;
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    uint16_t *cnt = reinterpret_cast<uint16_t *>(sh.lds), *mycnt = cnt + wave * COLS;
    int32_t *lofs = sh.lofs;
    const int32_t count = s1 - s0, wbase = s0 + wave * (PER * kWave);
    const int32_t from = wbase < s1 ? wbase : s1 - 1;  // uniform; elements past the bucket's last repeat it
    const uint32_t most = (uint32_t)(s1 - 1 - from);
    const auto at = [&](int k) { return (uint32_t)(k * kWave + lane) < most ? (uint32_t)(k * kWave + lane) : most; };
    brow += from, bcol += from, bval += from;
    int32_t c[PER], p[PER], r[PER];
    T v[PER];
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        c[k] = bcol[at(k)];
        r[k] = brow[at(k)];
    }
    for (int i = tid; i < WAVES * COLS / 2; i += THREADS) reinterpret_cast<uint32_t *>(cnt)[i] = 0;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < PER; ++k) p[k] = wave_rank(c[k], wbase + k * kWave + lane < s1, nbits, mycnt);
    // ahead of the ranks the values would take the registers of a second workgroup, 64-bit ones ahead of the rows' places as well
    const auto values = [&]() {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < PER; ++k) v[k] = bval[at(k)];
    };
    if constexpr (sizeof(T) == 4) values();
    __syncthreads();
    for (int i = tid; i < COLS; i += THREADS) {
        int32_t run = 0;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            const int32_t t = cnt[w * COLS + i];
            cnt[w * COLS + i] = (uint16_t)run;
            run += t;
        }
        lofs[i] = run;
    }
    __syncthreads();
    columns_exclusive_sum<COLS, THREADS>(lofs, sh.wave_tot);
    for (int i = tid; i < ncols; i += THREADS) row_ptr_t[c0 + i] = s0 + lofs[i];
#pragma unroll
    for (int k = 0; k < PER; ++k)
        if (wbase + k * kWave + lane < s1) p[k] += lofs[c[k]] + mycnt[c[k]];
    __syncthreads();
    int32_t *row_s = reinterpret_cast<int32_t *>(sh.lds);
    T *val_s = reinterpret_cast<T *>(sh.lds);
#pragma unroll
    for (int k = 0; k < PER; ++k)
        if (wbase + k * kWave + lane < s1) row_s[p[k]] = r[k];
    if constexpr (sizeof(T) == 8) values();
    __syncthreads();
    for (int j = tid; j < count; j += THREADS) col_t[s0 + j] = row_s[j];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < PER; ++k)
        if (wbase + k * kWave + lane < s1) val_s[p[k]] = v[k];
    __syncthreads();
    for (int j = tid; j < count; j += THREADS) val_t[s0 + j] = val_s[j];
}

template <typename T, int COLS, int THREADS>
__global__ __launch_bounds__(THREADS, THREADS > kSortThreads ? 8 : 1) void k_transpose_rows(const int32_t *__restrict__ offs, int32_t nblocks, int shift,
                                                            int nbits, int32_t n, int32_t nnz,
                                                            const int32_t *__restrict__ brow,
                                                            const uint16_t *__restrict__ bcol, const T *__restrict__ bval,
                                                            int32_t *__restrict__ row_ptr_t, int32_t *__restrict__ col_t,
                                                            T *__restrict__ val_t, int32_t *__restrict__ large)
{
    __shared__ union Lds {
        RowsShared<T, COLS, THREADS> turns;
        OneTurn<T, COLS, THREADS> one;
        __device__ Lds() {}
    } lds;
    RowsShared<T, COLS, THREADS> &sh = lds.turns;
    const int tid = threadIdx.x;
    const int32_t b = blockIdx.x;
    const int32_t s0 = offs[(int64_t)b * nblocks], s1 = offs[(int64_t)(b + 1) * nblocks];
    const int64_t c0 = (int64_t)b << shift;
    if (b == (int32_t)gridDim.x - 1 && tid == 0) row_ptr_t[n] = nnz;
    if (s1 - s0 > kLargeBucket) {  // the whole workgroup leaves
        if (tid == 0) large[2 * b] = s0, large[2 * b + 1] = s1;
        return;
    }
    if (s1 > s0 && s1 - s0 <= OneTurn<T, COLS, THREADS>::PER * THREADS) {  // uniform
        const int64_t ncols = n - c0 < (int64_t)1 << shift ? n - c0 : (int64_t)1 << shift;
        rows_in_one_turn<T, COLS, THREADS>(lds.one, s0, s1, nbits, c0, (int32_t)ncols, brow, bcol, bval, row_ptr_t, col_t, val_t);
        return;
    }
    // column counts of the whole bucket -> row offsets of A^T
    constexpr int PER = kSortElems / THREADS;
    for (int i = tid; i < COLS; i += THREADS) sh.first[i] = 0;
    __syncthreads();
    for (int32_t i0 = s0; i0 < s1; i0 += kSortElems) {  // uniform; a turn's loads together (28.0 -> 26.1 us), past the end the last one
        int32_t c[PER];
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            const int32_t i = i0 + k * THREADS + tid;
            c[k] = bcol[i < s1 ? i : s1 - 1];
        }
#pragma unroll
        for (int k = 0; k < PER; ++k)
            if (i0 + k * THREADS + tid < s1) atomicAdd(&sh.first[c[k]], 1);
    }
    __syncthreads();
    columns_exclusive_sum<COLS, THREADS>(sh.first, sh.wave_tot);
    for (int i = tid; i < (1 << shift); i += THREADS) {
        const int32_t at = s0 + sh.first[i];
        sh.first[i] = at;
        if (c0 + i < n) row_ptr_t[c0 + i] = at;
    }
    place_by_column<T, COLS, THREADS>(sh, s0, s1, nbits, brow, bcol, bval, col_t, val_t);
}

// ---- large buckets: pieces of kLargePiece elements, a workgroup each ----
// A large bucket: its number, the number of its first piece, its elements.  A call has at most kBuckets of them.
struct LargeBucket {
    int32_t bucket, piece, from, to;
};
// the bucket of piece p: the last one that starts at or before it (uniform)
__device__ __forceinline__ LargeBucket bucket_of_piece(const LargeBucket *__restrict__ large, int32_t nlarge, int32_t p)
{
    int32_t lo = 0, hi = nlarge - 1;
    while (lo < hi) {
        const int32_t mid = lo + (hi - lo + 1) / 2;
        if (large[mid].piece <= p)
            lo = mid;
        else
            hi = mid - 1;
    }
    return large[lo];
}

// table[p][c] = elements of column c in piece p
template <int COLS>
__global__ __launch_bounds__(kSortThreads) void k_transpose_large_count(const LargeBucket *__restrict__ large, int32_t nlarge,
                                                                        const uint16_t *__restrict__ bcol,
                                                                        int32_t *__restrict__ table)
{
    __shared__ int32_t count[COLS];
    const LargeBucket q = bucket_of_piece(large, nlarge, blockIdx.x);
    for (int i = threadIdx.x; i < COLS; i += kSortThreads) count[i] = 0;
    __syncthreads();
    const int64_t from = q.from + (int64_t)((int32_t)blockIdx.x - q.piece) * kLargePiece;
    const int64_t to = from + kLargePiece < q.to ? from + kLargePiece : q.to;
    for (int64_t i = from + threadIdx.x; i < to; i += kSortThreads) atomicAdd(&count[bcol[i]], 1);
    __syncthreads();
    for (int i = threadIdx.x; i < COLS; i += kSortThreads) table[(int64_t)blockIdx.x * COLS + i] = count[i];
}

// A workgroup per large bucket: row offsets of A^T, and in the table the place of every piece's first element of every column
template <int COLS>
__global__ __launch_bounds__(kSortThreads) void k_transpose_large_places(const LargeBucket *__restrict__ large, int shift,
                                                                         int32_t n, int32_t *__restrict__ table,
                                                                         int32_t *__restrict__ row_ptr_t)
{
    __shared__ int32_t first[COLS];
    __shared__ int32_t wave_tot[kSortWaves];
    const LargeBucket q = large[blockIdx.x];
    const int32_t pieces = (q.to - q.from + kLargePiece - 1) / kLargePiece;
    int32_t *mine = table + (int64_t)q.piece * COLS;
    for (int i = threadIdx.x; i < COLS; i += kSortThreads) {
        int32_t sum = 0;
#pragma unroll 8
        for (int32_t p = 0; p < pieces; ++p) sum += mine[(int64_t)p * COLS + i];
        first[i] = sum;
    }
    __syncthreads();
    columns_exclusive_sum<COLS>(first, wave_tot);
    const int64_t c0 = (int64_t)q.bucket << shift;
    for (int i = threadIdx.x; i < COLS; i += kSortThreads) {
        int32_t at = q.from + first[i];
        if (i < (1 << shift) && c0 + i < n) row_ptr_t[c0 + i] = at;
#pragma unroll 8
        for (int32_t p = 0; p < pieces; ++p) {
            const int32_t count = mine[(int64_t)p * COLS + i];
            mine[(int64_t)p * COLS + i] = at;
            at += count;
        }
    }
}

template <typename T, int COLS>
__global__ __launch_bounds__(kSortThreads) void k_transpose_large_rows(const LargeBucket *__restrict__ large, int32_t nlarge,
                                                                       int nbits, const int32_t *__restrict__ brow,
                                                                       const uint16_t *__restrict__ bcol,
                                                                       const T *__restrict__ bval,
                                                                       const int32_t *__restrict__ table,
                                                                       int32_t *__restrict__ col_t, T *__restrict__ val_t)
{
    __shared__ RowsShared<T, COLS> sh;
    const LargeBucket q = bucket_of_piece(large, nlarge, blockIdx.x);
    const int64_t from = q.from + (int64_t)((int32_t)blockIdx.x - q.piece) * kLargePiece;
    const int64_t to = from + kLargePiece < q.to ? from + kLargePiece : q.to;
    for (int i = threadIdx.x; i < COLS; i += kSortThreads) sh.first[i] = table[(int64_t)blockIdx.x * COLS + i];
    place_by_column<T, COLS>(sh, (int32_t)from, (int32_t)to, nbits, brow, bcol, bval, col_t, val_t);
}

// Columns of a bucket, as a power of two: buckets of up to two turns of kSortElems elements (a run of 8 elements per
// block and bucket in pass 2; 3.6 M elements: 33 us there against 40 with buckets of one turn), fewer where that
// leaves less than a workgroup per compute unit, more where kBuckets of them are not enough.  -1: the sort by keys takes the
// matrix, because a bucket would span more than kBucketColumns columns, or because so few columns hold so much that most
// buckets would be large ones.
int bucket_shift(int32_t n, int32_t nnz)
{
    if (nnz > 0x7fff0000) return -1;  // element numbers past the last one have to fit as well
    const double per_bucket = std::min<double>(7600.0, std::max<double>(1024.0, nnz / 256.0));
    int shift = 0;
    while ((1 << (shift + 1)) <= kBucketColumns && (double)nnz / (double)ceil_div64(n, (int64_t)1 << (shift + 1)) <= per_bucket) ++shift;
    while (ceil_div64(n, (int64_t)1 << shift) > kBuckets) ++shift;
    if ((1 << shift) > kBucketColumns) return -1;
    const int64_t buckets = ceil_div64(n, (int64_t)1 << shift);
    return buckets >= 128 || nnz / buckets <= 65536 ? shift : -1;
}

int bits_for(int64_t v)
{
    int b = 1;
    while (b < 32 && ((int64_t)1 << b) < v) ++b;
    return b;
}

template <typename T>
int csr_transpose_buckets(int shift, int32_t m, int32_t n, int32_t nnz, int32_t base, const int32_t *row_ptr, const int32_t *col,
                          const T *val, int32_t *row_ptr_t, int32_t *col_t, T *val_t, hipStream_t s)
{
    const int32_t nbuckets = (int32_t)ceil_div64(n, (int64_t)1 << shift), nblocks = (int32_t)ceil_div64(nnz, kSortElems);
    const int64_t ncount = (int64_t)nbuckets * nblocks + 1;  // at most 2^29: 1024 buckets, 2^19 blocks
    size_t off = 0;
    const auto take = [&off](size_t bytes) {
        const size_t at = off;
        off += align_up(bytes, 256);
        return at;
    };
    const size_t o_counts = take(4 * (size_t)ncount), o_seg = take(4 * ((size_t)nblocks * kSortWaves + 1));
    const size_t o_tmp = take(4 * scan_scratch_ints(ncount)), o_row = take(4 * (size_t)nnz), o_col = take(2 * (size_t)nnz);
    const size_t o_val = take(sizeof(T) * (size_t)nnz);
    Scratch scratch(s);
    char *arena = nullptr;
    int st = status_of(scratch.take(&arena, off));
    if (st) return st;
    int32_t *counts = (int32_t *)(arena + o_counts), *seg = (int32_t *)(arena + o_seg), *brow = (int32_t *)(arena + o_row);
    uint16_t *bcol = (uint16_t *)(arena + o_col);
    T *bval = (T *)(arena + o_val);
    const int bbits = nbuckets > 1 ? bits_for(nbuckets) : 0;
    hipLaunchKernelGGL(k_transpose_count, dim3(count_grid(nblocks)), dim3(kSortThreads), 0, s, row_ptr, col, m, nnz, base, shift,
                       nbuckets, nblocks, counts, seg);
    st = launch_exclusive_scan_i32(counts, counts, ncount, (int32_t *)(arena + o_tmp), s);
    if (st) return st;
    hipLaunchKernelGGL((k_transpose_bucket<T>), dim3((unsigned)(ceil_div64(nblocks, kXcds) * kXcds)), dim3(kSortThreads), 0, s,
                       row_ptr, col, val, seg, nnz, base, shift, nbuckets, bbits, nblocks, counts, brow, bcol, bval);
    int32_t *found = static_cast<int32_t *>(scratch.pinned());
    static_assert(2 * kBuckets * sizeof(int32_t) <= kPinnedBytes, "large buckets are reported through page-locked memory");
    if (!found) return ASX_STATUS_ALLOC_FAILED;
    std::memset(found, 0, 2 * sizeof(int32_t) * (size_t)nbuckets);
    const auto rows = [&](auto cols_, auto threads_) {
        constexpr int COLS = decltype(cols_)::value, THREADS = decltype(threads_)::value;
        hipLaunchKernelGGL((k_transpose_rows<T, COLS, THREADS>), dim3((unsigned)nbuckets), dim3(THREADS), 0, s, counts, nblocks, shift,
                           shift, n, nnz, brow, bcol, bval, row_ptr_t, col_t, val_t, found);
        int rc = check_launch();
        if (!rc) rc = status_of(hipStreamSynchronize(s));
        if (rc) return rc;
        LargeBucket large[kBuckets];
        int32_t nlarge = 0, pieces = 0;
        for (int32_t b = 0; b < nbuckets; ++b) {
            const int32_t from = found[2 * b], to = found[2 * b + 1];
            if (to == 0) continue;
            large[nlarge++] = LargeBucket{b, pieces, from, to};
            pieces += (int32_t)ceil_div64((int64_t)to - from, kLargePiece);
        }
        if (nlarge == 0) return rc;
        LargeBucket *d_large = nullptr;
        int32_t *table = nullptr;
        rc = status_of(scratch.take(&d_large, sizeof(LargeBucket) * (size_t)nlarge));
        if (!rc) rc = status_of(scratch.take(&table, sizeof(int32_t) * COLS * (size_t)pieces));
        if (!rc) rc = status_of(hipMemcpyAsync(d_large, large, sizeof(LargeBucket) * (size_t)nlarge, hipMemcpyHostToDevice, s));
        if (rc) return rc;
        const dim3 per_piece((unsigned)pieces), threads(kSortThreads);
        hipLaunchKernelGGL(k_transpose_large_count<COLS>, per_piece, threads, 0, s, d_large, nlarge, bcol, table);
        hipLaunchKernelGGL(k_transpose_large_places<COLS>, dim3((unsigned)nlarge), threads, 0, s, d_large, shift, n, table, row_ptr_t);
        hipLaunchKernelGGL((k_transpose_large_rows<T, COLS>), per_piece, threads, 0, s, d_large, nlarge, shift, brow, bcol, bval, table,
                           col_t, val_t);
        rc = check_launch();
        return rc ? rc : status_of(hipStreamSynchronize(s));
    };
    const std::integral_constant<int, kSortThreads> usual;
    const bool wide = nnz / nbuckets > kSortElems;  // most buckets would take a second turn of 512 threads
    st = shift <= 9    ? wide ? rows(std::integral_constant<int, 512>{}, std::integral_constant<int, 2 * kSortThreads>{})
                              : rows(std::integral_constant<int, 512>{}, usual)
         : shift == 10 ? rows(std::integral_constant<int, 1024>{}, usual)
                       : rows(std::integral_constant<int, kBucketColumns>{}, usual);
    scratch.idle = st == ASX_STATUS_SUCCESS;
    return st;
}

}  // namespace

template <typename T>
int csr_transpose(int32_t m, int32_t n, int32_t nnz, int32_t base, const int32_t *row_ptr, const int32_t *col,
                  const T *val, int32_t *row_ptr_t, int32_t *col_t, T *val_t, hipStream_t s)
{
    int st = ASX_STATUS_SUCCESS;
    if (nnz == 0) {
        hipLaunchKernelGGL(k_offsets_from_sorted, dim3((unsigned)ceil_div64((int64_t)n + 1, kBlock)), dim3(kBlock), 0,
                           s, (const int32_t *)nullptr, 0, n, row_ptr_t);
        return check_launch();
    }
    const int shift = bucket_shift(n, nnz);
    if (shift >= 0) return csr_transpose_buckets<T>(shift, m, n, nnz, base, row_ptr, col, val, row_ptr_t, col_t, val_t, s);
    uint64_t *keys = nullptr, *keys2 = nullptr;
    int32_t *idx = nullptr, *idx2 = nullptr, *trow = nullptr;
    void *tmp = nullptr;
    size_t tmp_bytes = 0;
    const unsigned grid = (unsigned)ceil_div64(nnz, kBlock);
    const int end_bit = 32 + bits_for(n);
    Scratch scratch(s);
#define ASX_TRY(expr)             \
    do {                          \
        st = status_of(expr);     \
        if (st) return st;        \
    } while (0)
    ASX_TRY(scratch.take(&keys, sizeof(uint64_t) * (size_t)nnz));
    ASX_TRY(scratch.take(&keys2, sizeof(uint64_t) * (size_t)nnz));
    ASX_TRY(scratch.take(&idx, sizeof(int32_t) * (size_t)nnz));
    ASX_TRY(scratch.take(&idx2, sizeof(int32_t) * (size_t)nnz));
    ASX_TRY(scratch.take(&trow, sizeof(int32_t) * (size_t)nnz));
    ASX_TRY(rocprim::radix_sort_pairs(nullptr, tmp_bytes, keys, keys2, idx, idx2, (size_t)nnz, 0u, (unsigned)end_bit, s));
    ASX_TRY(scratch.take(&tmp, tmp_bytes));
    hipLaunchKernelGGL(k_transpose_keys, dim3(grid), dim3(kBlock), 0, s, row_ptr, col, m, nnz, base, keys, idx);
    ASX_TRY(rocprim::radix_sort_pairs(tmp, tmp_bytes, keys, keys2, idx, idx2, (size_t)nnz, 0u, (unsigned)end_bit, s));
    hipLaunchKernelGGL((k_transpose_apply<T>), dim3(grid), dim3(kBlock), 0, s, keys2, idx2, val, nnz, trow, col_t,
                       val_t);
    hipLaunchKernelGGL(k_offsets_from_sorted, dim3((unsigned)ceil_div64((int64_t)n + 1, kBlock)), dim3(kBlock), 0, s,
                       trow, nnz, n, row_ptr_t);
    ASX_TRY(hipGetLastError());
    ASX_TRY(hipStreamSynchronize(s));
#undef ASX_TRY
    scratch.idle = true;
    return st;
}

__global__ __launch_bounds__(kBlock) void k_rebase(const int32_t *__restrict__ in, int64_t count, int32_t base,
                                                   int32_t *__restrict__ out)
{
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count;
         i += (int64_t)gridDim.x * blockDim.x)
        out[i] = in[i] - base;
}

// 64 x 64 tiles through LDS: reads are coalesced along the input rows, writes along the output
// rows.  256 threads = 64 columns x 4 row groups, 16 rows each.
constexpr int kTrTile = 64;
template <typename T>
__global__ __launch_bounds__(kBlock) void k_dense_transpose(int64_t rows, int64_t cols, const T *__restrict__ in,
                                                            int64_t ld_in, T *__restrict__ out, int64_t ld_out)
{
    __shared__ T tile[kTrTile][kTrTile + 1];
    const int tx = threadIdx.x & (kTrTile - 1), ty = threadIdx.x / kTrTile;
    const int64_t r0 = (int64_t)blockIdx.y * kTrTile, c0 = (int64_t)blockIdx.x * kTrTile;
#pragma unroll 4
    for (int i = ty; i < kTrTile; i += kBlock / kTrTile) {
        const int64_t r = r0 + i, c = c0 + tx;
        if (r < rows && c < cols) tile[i][tx] = in[r * ld_in + c];
    }
    __syncthreads();
#pragma unroll 4
    for (int i = ty; i < kTrTile; i += kBlock / kTrTile) {
        const int64_t c = c0 + i, r = r0 + tx;
        if (r < rows && c < cols) out[c * ld_out + r] = tile[tx][i];
    }
}

template <typename T>
int dense_transpose(int64_t rows, int64_t cols, const T *in, int64_t ld_in, T *out, int64_t ld_out, hipStream_t s)
{
    if (rows == 0 || cols == 0) return ASX_STATUS_SUCCESS;
    const int64_t gx = ceil_div64(cols, kTrTile), gy = ceil_div64(rows, kTrTile);
    if (gy > 65535) {  // grid y limit: walk the rows in slabs
        const int64_t slab = (int64_t)65535 * kTrTile;
        for (int64_t r = 0; r < rows; r += slab) {
            const int64_t nr = rows - r < slab ? rows - r : slab;
            hipLaunchKernelGGL((k_dense_transpose<T>), dim3((unsigned)gx, (unsigned)ceil_div64(nr, kTrTile)),
                               dim3(kBlock), 0, s, nr, cols, in + r * ld_in, ld_in, out + r, ld_out);
        }
    } else {
        hipLaunchKernelGGL((k_dense_transpose<T>), dim3((unsigned)gx, (unsigned)gy), dim3(kBlock), 0, s, rows, cols,
                           in, ld_in, out, ld_out);
    }
    return check_launch();
}

}  // namespace asx

extern "C" int asx_csr_transpose(int value_type, int32_t m, int32_t n, int32_t nnz, int32_t idx_base,
                                 const int32_t *d_row_ptr, const int32_t *d_col, const void *d_val,
                                 int32_t *d_row_ptr_t, int32_t *d_col_t, void *d_val_t, void *stream)
{
    if (m < 0 || n < 0 || nnz < 0) return ASX_STATUS_INVALID_SIZE;
    if (idx_base != 0 && idx_base != 1) return ASX_STATUS_INVALID_VALUE;
    if (!d_row_ptr_t || (m > 0 && !d_row_ptr)) return ASX_STATUS_INVALID_POINTER;
    if (nnz > 0 && (!d_row_ptr || !d_col || !d_val || !d_col_t || !d_val_t)) return ASX_STATUS_INVALID_POINTER;
    if (value_type == ASX_R_64F)
        return asx::csr_transpose<double>(m, n, nnz, idx_base, d_row_ptr, d_col, (const double *)d_val, d_row_ptr_t,
                                          d_col_t, (double *)d_val_t, (hipStream_t)stream);
    if (value_type == ASX_R_32F)
        return asx::csr_transpose<float>(m, n, nnz, idx_base, d_row_ptr, d_col, (const float *)d_val, d_row_ptr_t,
                                         d_col_t, (float *)d_val_t, (hipStream_t)stream);
    return ASX_STATUS_NOT_SUPPORTED;
}

extern "C" int asx_csr_rebase(int32_t m, int32_t nnz, int32_t idx_base, const int32_t *d_row_ptr,
                              const int32_t *d_col, int32_t *d_row_ptr_out, int32_t *d_col_out, void *stream)
{
    if (m < 0 || nnz < 0) return ASX_STATUS_INVALID_SIZE;
    if (!d_row_ptr || !d_row_ptr_out || (nnz > 0 && (!d_col || !d_col_out))) return ASX_STATUS_INVALID_POINTER;
    hipStream_t s = (hipStream_t)stream;
    const auto grid_for = [](int64_t count) {
        int64_t g = asx::ceil_div64(count, asx::kBlock);
        return (unsigned)(g > 8192 ? 8192 : g);
    };
    hipLaunchKernelGGL(asx::k_rebase, dim3(grid_for((int64_t)m + 1)), dim3(asx::kBlock), 0, s, d_row_ptr,
                       (int64_t)m + 1, idx_base, d_row_ptr_out);
    if (nnz > 0)
        hipLaunchKernelGGL(asx::k_rebase, dim3(grid_for(nnz)), dim3(asx::kBlock), 0, s, d_col, (int64_t)nnz, idx_base,
                           d_col_out);
    return asx::check_launch();
}

extern "C" int asx_dense_transpose(int value_type, int64_t rows, int64_t cols, const void *d_in, int64_t ld_in,
                                   void *d_out, int64_t ld_out, void *stream)
{
    if (rows < 0 || cols < 0 || ld_in < cols || ld_out < rows) return ASX_STATUS_INVALID_SIZE;
    if (rows > 0 && cols > 0 && (!d_in || !d_out)) return ASX_STATUS_INVALID_POINTER;
    if (value_type == ASX_R_64F)
        return asx::dense_transpose<double>(rows, cols, (const double *)d_in, ld_in, (double *)d_out, ld_out,
                                            (hipStream_t)stream);
    if (value_type == ASX_R_32F)
        return asx::dense_transpose<float>(rows, cols, (const float *)d_in, ld_in, (float *)d_out, ld_out,
                                           (hipStream_t)stream);
    return ASX_STATUS_NOT_SUPPORTED;
}
