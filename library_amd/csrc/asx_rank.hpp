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


__device__ __forceinline__ int lanes_below(unsigned long long mask)
{
    return __builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0));
}

// Rank of this lane's element among the elements its wave has ranked with `mycnt` so far, in element
// order: lanes of one key find each other by ballots over the key's `nbits` bits.  mycnt: one counter
// per key, private to the wave.
template <typename C>
__device__ __forceinline__ int32_t wave_rank(int32_t key, bool valid, int nbits, C *mycnt)
{
    unsigned long long same = __ballot(valid);
    for (int bit = 0; bit < nbits; ++bit) {
        const bool one = (key >> bit) & 1;
        const unsigned long long bal = __ballot(one);
        same &= one ? bal : ~bal;
    }
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
