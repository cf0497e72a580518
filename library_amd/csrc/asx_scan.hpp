// Exclusive prefix sum of int32 arrays on the device, for the plan builders: one launch up to 65536 items, beyond that two or three
// (sums of blocks of 4096, scan of those sums by one workgroup unless there are few, scan inside every block plus its
// offset).  The arrays scanned here are per-tile, per-block or per-(slice, block) counts, a few MB
// at most: two passes over them cost microseconds.
#pragma once
#include "asx_internal.hpp"

namespace asx {

typedef int32_t scan_i32x4 __attribute__((ext_vector_type(4), aligned(4)));
constexpr int kScanThreads = 256;
constexpr int kScanPerThread = 16;
constexpr int kScanBlock = kScanThreads * kScanPerThread;

// sum over the workgroup; every thread receives the total (barriers inside)
__device__ __forceinline__ int32_t scan_block_total(int32_t v, int32_t *wave_tot)
{
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) v += __shfl_xor(v, d, kWave);
    if (lane == 0) wave_tot[wave] = v;
    __syncthreads();
    int32_t t = 0;
    for (int w = 0; w < kScanThreads / kWave; ++w) t += wave_tot[w];
    __syncthreads();
    return t;
}

// exclusive sum of one value per thread over the workgroup (barriers inside)
__device__ __forceinline__ int32_t scan_block_exclusive(int32_t v, int32_t *wave_tot, int32_t *total)
{
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    int32_t incl = v;
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
        const int32_t t = __shfl_up(incl, d, kWave);
        if (lane >= d) incl += t;
    }
    if (lane == kWave - 1) wave_tot[wave] = incl;
    __syncthreads();
    int32_t before = 0, all = 0;
    for (int w = 0; w < kScanThreads / kWave; ++w) {
        const int32_t t = wave_tot[w];
        before += w < wave ? t : 0;
        all += t;
    }
    __syncthreads();
    *total = all;
    return before + incl - v;
}

static __global__ __launch_bounds__(kScanThreads) void k_scan_block_sums(const int32_t *__restrict__ in, int64_t n,
                                                                          int32_t *__restrict__ sums)
{
    __shared__ int32_t wave_tot[kScanThreads / kWave];
    const int64_t base = (int64_t)blockIdx.x * kScanBlock;
    int32_t v = 0;
#pragma unroll
    for (int k = 0; k < kScanPerThread; ++k) {
        const int64_t i = base + k * kScanThreads + threadIdx.x;
        v += i < n ? in[i] : 0;
    }
    const int32_t t = scan_block_total(v, wave_tot);
    if (threadIdx.x == 0) sums[blockIdx.x] = t;
}

// in-place exclusive scan of sums[0 .. nb) by one workgroup, kScanThreads at a time
static __global__ __launch_bounds__(kScanThreads) void k_scan_sums(int32_t *__restrict__ sums, int32_t nb)
{
    __shared__ int32_t wave_tot[kScanThreads / kWave];
    int32_t carry = 0;
    for (int32_t i0 = 0; i0 < nb; i0 += kScanThreads) {  // uniform
        const int32_t i = i0 + threadIdx.x;
        const int32_t v = i < nb ? sums[i] : 0;
        int32_t total;
        const int32_t e = scan_block_exclusive(v, wave_tot, &total);
        if (i < nb) sums[i] = carry + e;
        carry += total;
    }
}

// Up to so many blocks (4 M items) each adds up the sums before its own by itself, four a thread, where a scan of them was
// a launch between two others (transpose and multiply of 1.2 M elements 87 -> 71 us, of 2.7 M 120 -> 107).
constexpr int64_t kScanOwnSums = 4 * kScanThreads;

// out[i] = sums of the blocks before (OWN: sums[] as they are, else their scan) + sum of in[block start .. i); a thread owns
// kScanPerThread consecutive items
template <bool OWN>
static __global__ __launch_bounds__(kScanThreads) void k_scan_apply(const int32_t *__restrict__ in, int64_t n,
                                                                     const int32_t *__restrict__ sums,
                                                                     int32_t *__restrict__ out)
{
    __shared__ int32_t wave_tot[kScanThreads / kWave];
    const int64_t base = (int64_t)blockIdx.x * kScanBlock + (int64_t)threadIdx.x * kScanPerThread;
    int32_t v[kScanPerThread];
    int32_t mine = 0;
    if (base + kScanPerThread <= n) {  // 16-byte loads (unaligned ones allowed: in may be any int32 array)
#pragma unroll
        for (int k = 0; k < kScanPerThread; k += 4) {
            const scan_i32x4 q = *reinterpret_cast<const scan_i32x4 *>(in + base + k);
            v[k] = q.x, v[k + 1] = q.y, v[k + 2] = q.z, v[k + 3] = q.w;
        }
    } else {
#pragma unroll
        for (int k = 0; k < kScanPerThread; ++k) v[k] = base + k < n ? in[base + k] : 0;
    }
#pragma unroll
    for (int k = 0; k < kScanPerThread; ++k) mine += v[k];
    int32_t before = 0;
    if (OWN) {
        for (int k = threadIdx.x; k < (int)blockIdx.x; k += kScanThreads) before += sums[k];
        before = scan_block_total(before, wave_tot);
    } else {
        before = sums[blockIdx.x];
    }
    int32_t total;
    int32_t run = before + scan_block_exclusive(mine, wave_tot, &total);
#pragma unroll
    for (int k = 0; k < kScanPerThread; ++k) {
        const int32_t t = v[k];
        v[k] = run;
        run += t;
    }
    if (base + kScanPerThread <= n) {
#pragma unroll
        for (int k = 0; k < kScanPerThread; k += 4)
            *reinterpret_cast<scan_i32x4 *>(out + base + k) = scan_i32x4{v[k], v[k + 1], v[k + 2], v[k + 3]};
    } else {
#pragma unroll
        for (int k = 0; k < kScanPerThread; ++k)
            if (base + k < n) out[base + k] = v[k];
    }
}

// Small arrays: one workgroup, one launch, 16 items a thread and turn (29 000 counts: 4 us against 9 and two more gaps
// between kernels).
constexpr int kScanOneThreads = 1024;
constexpr int64_t kScanOneMax = 65536;
static __global__ __launch_bounds__(kScanOneThreads) void k_scan_one(const int32_t *__restrict__ in, int32_t n,
                                                                      int32_t *__restrict__ out)
{
    __shared__ int32_t wave_tot[kScanOneThreads / kWave];
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    int32_t carry = 0;
    for (int32_t b = 0; b < n; b += kScanOneThreads * kScanPerThread) {  // uniform
        const int32_t base = b + (int32_t)threadIdx.x * kScanPerThread;
        int32_t v[kScanPerThread], mine = 0;
        if (base + kScanPerThread <= n) {
#pragma unroll
            for (int k = 0; k < kScanPerThread; k += 4) {
                const scan_i32x4 q = *reinterpret_cast<const scan_i32x4 *>(in + base + k);
                v[k] = q.x, v[k + 1] = q.y, v[k + 2] = q.z, v[k + 3] = q.w;
            }
        } else {
#pragma unroll
            for (int k = 0; k < kScanPerThread; ++k) v[k] = base + k < n ? in[base + k] : 0;
        }
#pragma unroll
        for (int k = 0; k < kScanPerThread; ++k) mine += v[k];
        int32_t incl = mine;
#pragma unroll
        for (int d = 1; d < kWave; d <<= 1) {
            const int32_t t = __shfl_up(incl, d, kWave);
            if (lane >= d) incl += t;
        }
        if (lane == kWave - 1) wave_tot[wave] = incl;
        __syncthreads();
        int32_t before = 0, all = 0;
        for (int w = 0; w < kScanOneThreads / kWave; ++w) {
            const int32_t t = wave_tot[w];
            before += w < wave ? t : 0;
            all += t;
        }
        __syncthreads();
        int32_t run = carry + before + incl - mine;
#pragma unroll
        for (int k = 0; k < kScanPerThread; ++k) {
            const int32_t t = v[k];
            v[k] = run;
            run += t;
        }
        if (base + kScanPerThread <= n) {
#pragma unroll
            for (int k = 0; k < kScanPerThread; k += 4)
                *reinterpret_cast<scan_i32x4 *>(out + base + k) = scan_i32x4{v[k], v[k + 1], v[k + 2], v[k + 3]};
        } else {
#pragma unroll
            for (int k = 0; k < kScanPerThread; ++k)
                if (base + k < n) out[base + k] = v[k];
        }
        carry += all;
    }
}

// ints of scratch the scan of n items needs
inline size_t scan_scratch_ints(int64_t n) { return (size_t)ceil_div64(n > 0 ? n : 1, kScanBlock); }

// out[i] = in[0] + ... + in[i - 1], i in [0, n); in == out is allowed; `scratch`: scan_scratch_ints(n) ints
inline int launch_exclusive_scan_i32(const int32_t *in, int32_t *out, int64_t n, int32_t *scratch, hipStream_t s)
{
    if (n <= 0) return ASX_STATUS_SUCCESS;
    if (n <= kScanOneMax) {
        hipLaunchKernelGGL(k_scan_one, dim3(1), dim3(kScanOneThreads), 0, s, in, (int32_t)n, out);
        return check_launch();
    }
    const int64_t nb = ceil_div64(n, kScanBlock);
    if (nb > 0x7fffffff) return ASX_STATUS_INVALID_SIZE;
    hipLaunchKernelGGL(k_scan_block_sums, dim3((unsigned)nb), dim3(kScanThreads), 0, s, in, n, scratch);
    if (nb <= kScanOwnSums) {
        hipLaunchKernelGGL(k_scan_apply<true>, dim3((unsigned)nb), dim3(kScanThreads), 0, s, in, n, scratch, out);
        return check_launch();
    }
    hipLaunchKernelGGL(k_scan_sums, dim3(1), dim3(kScanThreads), 0, s, scratch, (int32_t)nb);
    hipLaunchKernelGGL(k_scan_apply<false>, dim3((unsigned)nb), dim3(kScanThreads), 0, s, in, n, scratch, out);
    return check_launch();
}

}  // namespace asx
