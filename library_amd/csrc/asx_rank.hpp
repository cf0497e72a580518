// Stable ranks and small sums inside a workgroup of kSortThreads, for counting sorts of stored elements: blocks of
// kSortElems consecutive elements, kSortWaveElems a wave, 64 at a time.
#pragma once
#include "asx_internal.hpp"

namespace asx {

constexpr int kSortThreads = 512;
constexpr int kSortWaves = kSortThreads / kWave;
constexpr int kSortElems = 4096;  // per block
constexpr int kSortPerLane = kSortElems / kSortThreads;
constexpr int kSortWaveElems = kSortElems / kSortWaves;


// The block of kSortElems that workgroup blockIdx.x of a grid of count_grid(nblocks) counts; at or past nblocks there is none.
// Consecutive blocks write neighbouring counts of every key: on one XCD its L2 merges their pieces of a line.
__device__ __forceinline__ int32_t block_of_xcd()
{
    return (int32_t)(blockIdx.x % kXcds) * (int32_t)(gridDim.x / kXcds) + (int32_t)(blockIdx.x / kXcds);
}
inline unsigned count_grid(int64_t nblocks) { return (unsigned)(ceil_div64(nblocks, kXcds) * kXcds); }

// Columns of block b's elements, all requested together: behind a branch on the lane each load would be waited for before the
// next is issued.  Past the last element it repeats.  With the order above: transpose's counts of 3.6 M elements 13.1 -> 10.4 us,
// the sliced plan's of 33.6 M 97 -> 77.
__device__ __forceinline__ void load_columns(const int32_t *__restrict__ col, int32_t nnz, int32_t b, int32_t (&c)[kSortPerLane])
{
#pragma unroll
    for (int k = 0; k < kSortPerLane; ++k) {
        const int64_t i = (int64_t)b * kSortElems + k * kSortThreads + threadIdx.x;
        c[k] = col[i < nnz ? i : nnz - 1];
    }
}

__device__ __forceinline__ int lanes_below(unsigned long long mask)
{
    return __builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0));
}

// Rank of this lane's element among the elements its wave has ranked with `mycnt` so far, in element
// order: lanes of one key find each other by ballots over the key's `nbits` bits (and one more of an odd number, 0 in all keys).
// mycnt: one counter per key, private to the wave.
// The kernels that sort spend half of their time issuing instructions, most of them here: five a bit (a bit spread over a word, the
// ballot, and half a three-operand OR of what differs for either half of the lanes); selecting the ballot or its
// complement was nine (k_transpose_bucket and _rows of 3.6 M elements 26.5 and 25.9 us).
template <typename C>
__device__ __forceinline__ int32_t wave_rank(int32_t key, bool valid, int nbits, C *mycnt)
{
    uint32_t lo = 0, hi = 0;  // lanes of other keys
    for (int bit = 0; bit < nbits; bit += 2) {
        const uint32_t one = (uint32_t)__builtin_amdgcn_sbfe(key, bit, 1), two = (uint32_t)__builtin_amdgcn_sbfe(key, bit + 1, 1);
        const unsigned long long b1 = __ballot(one != 0), b2 = __ballot(two != 0);
        lo |= (one ^ (uint32_t)b1) | (two ^ (uint32_t)b2);
        hi |= (one ^ (uint32_t)(b1 >> 32)) | (two ^ (uint32_t)(b2 >> 32));
    }
    const unsigned long long same = ~((unsigned long long)hi << 32 | lo) & __ballot(valid);
    const int below = lanes_below(same);  // lanes of this key before this one
    const int32_t prev = valid ? (int32_t)mycnt[key] : 0;
    if (valid && below == 0) mycnt[key] = (C)(prev + __popcll(same));
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    return prev + below;
}

// largest r in [lo, hi] with row_ptr[r] <= i
__device__ __forceinline__ int32_t row_holding(const int32_t *__restrict__ row_ptr, int32_t lo, int32_t hi, int32_t i)
{
    while (lo < hi) {
        const int32_t mid = lo + (hi - lo + 1) / 2;
        if (row_ptr[mid] <= i)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

// The same for one i, by the whole wave: 64 probes at a time, so that a million rows take four
// dependent reads instead of twenty (every lane gets the answer; lo, hi, i uniform).
__device__ __forceinline__ int32_t wave_row_holding(const int32_t *__restrict__ row_ptr, int32_t lo, int32_t hi, int32_t i)
{
    const int lane = threadIdx.x & (kWave - 1);
    while (lo < hi) {
        const int32_t step = (int32_t)(((uint32_t)(hi - lo) + kWave - 1) / kWave);  // unsigned: hi may be 2^31 - 1
        const int64_t p = lo + (int64_t)(lane + 1) * step;
        const int n = __popcll(__ballot(p <= hi && row_ptr[p <= hi ? p : hi] <= i));
        lo += n * step;
        hi = hi - lo < step - 1 ? hi : lo + step - 1;
    }
    return lo;
}

// seg_row[g] = the row holding stored element g * kSortWaveElems (m - 1 behind the last element), written by the workgroup
// of block b of nblocks for its kSortWaves segments, one a wave, and the last block's for the end of the array.
__device__ __forceinline__ void block_seg_rows(const int32_t *__restrict__ row_ptr, int32_t m, int32_t nnz, int32_t base,
                                               int32_t b, int32_t nblocks, int32_t *__restrict__ seg_row)
{
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x & (kWave - 1);
    const int64_t g = (int64_t)b * kSortWaves + wave, e = g * kSortWaveElems;
    const int32_t r = e < nnz ? wave_row_holding(row_ptr, 0, m - 1, (int32_t)e + base) : m - 1;
    if (lane == 0) seg_row[g] = r;
    if (b == nblocks - 1 && threadIdx.x == 0) seg_row[(int64_t)nblocks * kSortWaves] = m - 1;
}

// Rows of the wave's kSortWaveElems consecutive elements from wbase on: rr[k] = row of element
// wbase + k * 64 + lane, all of them in rows r_lo .. r_hi (uniform; r_lo holds element wbase).  The starts
// of the rows are marked in `mark` (kSortWaveElems ints of LDS, the wave's own) and a running maximum
// spreads them: one read of row_ptr per row instead of a binary search per element.  A long run of
// empty rows falls back to the search.
__device__ __forceinline__ void wave_rows(const int32_t *__restrict__ row_ptr, int32_t base, int32_t r_lo, int32_t r_hi,
                                          int64_t wbase, int64_t nnz, int32_t *mark, int32_t (&rr)[kSortPerLane])
{
    const int lane = threadIdx.x & (kWave - 1);
    if (r_hi - r_lo > 8 * kSortWaveElems) {  // uniform
#pragma unroll
        for (int k = 0; k < kSortPerLane; ++k) {
            const int64_t i = wbase + k * kWave + lane;
            rr[k] = row_holding(row_ptr, r_lo, r_hi, (int32_t)(i < nnz ? i : nnz - 1) + base);
        }
        return;
    }
#pragma unroll
    for (int k = 0; k < kSortPerLane; ++k) mark[k * kWave + lane] = 0;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    for (int32_t d = 1 + lane; d <= r_hi - r_lo; d += kWave) {  // counted from r_lo: r_hi may be close to 2^31
        const int64_t at = (int64_t)row_ptr[(int64_t)r_lo + d] - base - wbase;
        if (at >= 0 && at < kSortWaveElems) atomicMax(&mark[at], d);  // of rows that start alike the last one holds the element
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    int32_t before = 0;
#pragma unroll
    for (int k = 0; k < kSortPerLane; ++k) {
        int32_t v = mark[k * kWave + lane];
#define ASX_MAX_STEP(CTRL, ROW_MASK)                     \
    {                                                    \
        const int32_t u = dpp0_i32<CTRL, ROW_MASK>(v);   \
        v = v > u ? v : u;                               \
    }
        ASX_MAX_STEP(0x111, 0xF)  // row_shr:1
        ASX_MAX_STEP(0x112, 0xF)  // row_shr:2
        ASX_MAX_STEP(0x114, 0xF)  // row_shr:4
        ASX_MAX_STEP(0x118, 0xF)  // row_shr:8
        ASX_MAX_STEP(0x142, 0xA)  // row_bcast15 into rows 1 and 3
        ASX_MAX_STEP(0x143, 0xC)  // row_bcast31 into rows 2 and 3
#undef ASX_MAX_STEP
        v = v > before ? v : before;
        rr[k] = r_lo + v;
        before = __builtin_amdgcn_readlane(v, kWave - 1);
    }
}

// in-place exclusive sum of a[0 .. n), n <= 2 * kSortThreads, by the whole workgroup (barriers inside)
__device__ __forceinline__ void block_exclusive_sum(int32_t *a, int n, int32_t *wave_tot)
{
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    const int32_t v0 = 2 * tid < n ? a[2 * tid] : 0, v1 = 2 * tid + 1 < n ? a[2 * tid + 1] : 0;
    int32_t incl = v0 + v1;
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
        const int32_t t = __shfl_up(incl, d, kWave);
        if (lane >= d) incl += t;
    }
    if (lane == kWave - 1) wave_tot[wave] = incl;
    __syncthreads();
    int32_t before = 0;
    for (int w = 0; w < wave; ++w) before += wave_tot[w];
    const int32_t excl = before + incl - (v0 + v1);
    if (2 * tid < n) a[2 * tid] = excl;
    if (2 * tid + 1 < n) a[2 * tid + 1] = excl + v0;
    __syncthreads();
}

}  // namespace asx
