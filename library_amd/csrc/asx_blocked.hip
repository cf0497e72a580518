// Blocked SpMM variant for matrices with dense sub-blocks: A is re-tiled into 16x4 blocks
// (16 rows x 4 consecutive columns, zero filled) and each block meets the matching 4 rows of B
// in one MFMA (v_mfma_f32_16x16x4_f32 / v_mfma_f64_16x16x4_f64), 16 columns of C at a time.
//
// It pays only where blocks are dense: per stored element it streams 4/fill bytes of A (fp32)
// instead of 8, and reads 4 rows of B per block instead of one row per stored element
// (16/fill vs 256 bytes per element at N = 64).  fill = nnz / (64 * blocks); below about 1/8 (0.2, 0.3
// and 0.4 where rows of B are down to 128, 64 and fewer bytes) the merge kernel is ahead, so DEFAULT
// picks this variant only above that.
//
// The reference's counterpart (hip/kernel/level3/alphasparse_spmm_tc4csr.h:38-256) builds the
// blocks on the host through a dense ceil(M/16) x ceil(K/4) bitmap, keeps them in a global, and
// multiplies with Hygon `mmac` builtins.  Here the blocks are built on the device by sorting
// (block row, column quad) keys; they live in the plan.
//
// The zero fill of a block is multiplied with real rows of B: a non-finite value in a row of B
// that some row of the block does not reference reaches that row of C as NaN (0 * Inf), where a
// row-wise kernel would not have read it.  As for any padded block format, B must be finite.  (What
// a batch fetches past the last block or past B's last row counts as zeros and is not multiplied.)
#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>

#include "asx_internal.hpp"

namespace asx {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef double doublex4 __attribute__((ext_vector_type(4)));

// key = block row (28 bits) | column quad (30 bits) | row in block (4) | column in quad (2)
__global__ __launch_bounds__(kBlock) void k_block_keys(const int32_t *__restrict__ row_ptr,
                                                       const int32_t *__restrict__ col, int32_t m,
                                                       int32_t nnz, uint64_t *__restrict__ keys,
                                                       int32_t *__restrict__ idx)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nnz) return;
    int32_t lo = 0, hi = m;  // row holding stored element i: largest r with row_ptr[r] <= i
    while (lo < hi) {
        const int32_t mid = lo + (hi - lo + 1) / 2;
        if (row_ptr[mid] <= i)
            lo = mid;
        else
            hi = mid - 1;
    }
    const uint32_t r = (uint32_t)lo, c = (uint32_t)col[i];
    keys[i] = ((uint64_t)(r >> 4) << 36) | ((uint64_t)(c >> 2) << 6) | ((uint64_t)(r & 15) << 2) | (c & 3);
    idx[i] = (int32_t)i;
}

__global__ __launch_bounds__(kBlock) void k_block_heads(const uint64_t *__restrict__ keys, int32_t nnz,
                                                        int32_t *__restrict__ head)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nnz) return;
    head[i] = (i == 0 || (keys[i] >> 6) != (keys[i - 1] >> 6)) ? 1 : 0;
}

// Where every stored element goes: upd_src[i] = its position in A's arrays, upd_dst[i] = its slot
// in bval (lane order of the MFMA A operand), sign bit set when the element repeats the (row,
// column) of the element before it (CSR may hold duplicates; they are summed, as every other
// kernel here and the reference do).
__global__ __launch_bounds__(kBlock) void k_block_slots(const uint64_t *__restrict__ keys,
                                                        const int32_t *__restrict__ idx,
                                                        const int32_t *__restrict__ block_of, int32_t nnz,
                                                        uint64_t *__restrict__ bkey, int32_t *__restrict__ upd_src,
                                                        int64_t *__restrict__ upd_dst)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nnz) return;
    const uint64_t key = keys[i];
    const int64_t b = block_of[i] - 1;  // inclusive scan of the head flags
    if (i == 0 || (key >> 6) != (keys[i - 1] >> 6)) bkey[b] = key >> 6;
    const int r16 = (int)((key >> 2) & 15), c4 = (int)(key & 3);
    const bool repeat = i > 0 && keys[i - 1] == key;
    upd_src[i] = idx[i];
    upd_dst[i] = (b * 64 + c4 * 16 + r16) | (repeat ? (int64_t)1 << 63 : 0);
}

// bval[slot] = sum of the values stored for that (row, column), in stored order
template <typename T>
__global__ __launch_bounds__(kBlock) void k_block_values(const int32_t *__restrict__ upd_src,
                                                         const int64_t *__restrict__ upd_dst, int32_t nnz,
                                                         const T *__restrict__ val, T *__restrict__ bval)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nnz) return;
    const int64_t dst = upd_dst[i];
    if (dst < 0) return;  // summed by the first element of its run
    T sum = val[upd_src[i]];
    for (int64_t j = i + 1; j < nnz && upd_dst[j] < 0; ++j) sum += val[upd_src[j]];
    bval[dst] = sum;
}

__global__ __launch_bounds__(kBlock) void k_block_rows(const uint64_t *__restrict__ bkey, int32_t nblocks,
                                                       int32_t nbrows, int32_t *__restrict__ brow_ptr,
                                                       int32_t *__restrict__ bcol)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < nblocks) bcol[t] = (int32_t)(bkey[t] & ((1u << 30) - 1));
    if (t > nbrows) return;
    const uint64_t target = (uint64_t)t << 30;  // first block whose block row is >= t
    int32_t lo = 0, hi = nblocks;
    while (lo < hi) {
        const int32_t mid = (lo + hi) / 2;
        if (bkey[mid] < target)
            lo = mid + 1;
        else
            hi = mid;
    }
    brow_ptr[t] = lo;
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_fill_zero(T *p, int64_t n)
{
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        p[i] = T(0);
}

#define ASX_TRY(expr)                      \
    do {                                   \
        int _s = status_of(expr);          \
        if (_s) {                          \
            st = _s;                       \
            goto done;                     \
        }                                  \
    } while (0)

// Builds the blocked copy of A.  Synchronises the stream (reads the block count back).
template <typename T>
int build_blocked(int32_t m, int32_t k, int32_t nnz, const int32_t *row_ptr, const int32_t *col,
                  const T *val, BlockedMatrix *out, hipStream_t s)
{
    (void)k;
    int st = ASX_STATUS_SUCCESS;
    uint64_t *keys = nullptr, *keys2 = nullptr, *bkey = nullptr;
    int32_t *idx = nullptr, *idx2 = nullptr, *head = nullptr, *block_of = nullptr;
    void *tmp = nullptr;
    size_t tmp_sort = 0, tmp_scan = 0, tmp_bytes = 0;
    int32_t nblocks = 0;
    Scratch scratch(s);
    const int32_t nbrows = (int32_t)ceil_div64(m, 16);
    out->nbrows = nbrows;
    out->nblocks = 0;
    out->brow_ptr = nullptr;
    out->bcol = nullptr;
    out->bval = nullptr;
    out->upd_src = nullptr;
    out->upd_dst = nullptr;
    out->nnz = nnz;
    const unsigned g_nnz = (unsigned)ceil_div64(nnz > 0 ? nnz : 1, kBlock);
    if (nnz > 0) {
        ASX_TRY(scratch.take(&keys, sizeof(uint64_t) * (size_t)nnz));
        ASX_TRY(scratch.take(&keys2, sizeof(uint64_t) * (size_t)nnz));
        ASX_TRY(scratch.take(&idx, sizeof(int32_t) * (size_t)nnz));
        ASX_TRY(scratch.take(&idx2, sizeof(int32_t) * (size_t)nnz));
        ASX_TRY(scratch.take(&head, sizeof(int32_t) * (size_t)nnz));
        ASX_TRY(scratch.take(&block_of, sizeof(int32_t) * (size_t)nnz));
        ASX_TRY(rocprim::radix_sort_pairs(nullptr, tmp_sort, keys, keys2, idx, idx2, (size_t)nnz, 0u, (unsigned)64, s));
        ASX_TRY(rocprim::inclusive_scan(nullptr, tmp_scan, head, block_of, (size_t)nnz, rocprim::plus<int32_t>(), s));
        tmp_bytes = tmp_sort > tmp_scan ? tmp_sort : tmp_scan;
        ASX_TRY(scratch.take(&tmp, tmp_bytes));
        hipLaunchKernelGGL(k_block_keys, dim3(g_nnz), dim3(kBlock), 0, s, row_ptr, col, m, nnz, keys, idx);
        ASX_TRY(rocprim::radix_sort_pairs(tmp, tmp_sort, keys, keys2, idx, idx2, (size_t)nnz, 0u, (unsigned)64, s));
        hipLaunchKernelGGL(k_block_heads, dim3(g_nnz), dim3(kBlock), 0, s, keys2, nnz, head);
        ASX_TRY(rocprim::inclusive_scan(tmp, tmp_scan, head, block_of, (size_t)nnz, rocprim::plus<int32_t>(), s));
        ASX_TRY(hipMemcpyAsync(&nblocks, block_of + (nnz - 1), sizeof(int32_t), hipMemcpyDeviceToHost, s));
        ASX_TRY(hipStreamSynchronize(s));
    }
    out->nblocks = nblocks;
    ASX_TRY(pool_malloc(&out->brow_ptr, sizeof(int32_t) * ((size_t)nbrows + 1), false));
    ASX_TRY(pool_malloc(&out->bcol, sizeof(int32_t) * (size_t)(nblocks > 0 ? nblocks : 1), false));
    ASX_TRY(pool_malloc(&out->bval, sizeof(T) * 64 * (size_t)(nblocks > 0 ? nblocks : 1), false));
    ASX_TRY(scratch.take(&bkey, sizeof(uint64_t) * (size_t)(nblocks > 0 ? nblocks : 1)));
    if (nblocks > 0) {
        ASX_TRY(pool_malloc(&out->upd_src, sizeof(int32_t) * (size_t)nnz, false));
        ASX_TRY(pool_malloc(&out->upd_dst, sizeof(int64_t) * (size_t)nnz, false));
        hipLaunchKernelGGL((k_fill_zero<T>), dim3(4096), dim3(kBlock), 0, s, (T *)out->bval, (int64_t)nblocks * 64);
        hipLaunchKernelGGL(k_block_slots, dim3(g_nnz), dim3(kBlock), 0, s, keys2, idx2, block_of, nnz, bkey,
                           out->upd_src, out->upd_dst);
        hipLaunchKernelGGL((k_block_values<T>), dim3(g_nnz), dim3(kBlock), 0, s, out->upd_src, out->upd_dst, nnz, val,
                           (T *)out->bval);
    }
    {
        const int64_t span = (int64_t)(nblocks > nbrows + 1 ? nblocks : nbrows + 1);
        hipLaunchKernelGGL(k_block_rows, dim3((unsigned)ceil_div64(span, kBlock)), dim3(kBlock), 0, s, bkey,
                           nblocks, nbrows, out->brow_ptr, out->bcol);
    }
    ASX_TRY(hipGetLastError());
    ASX_TRY(hipStreamSynchronize(s));
    scratch.idle = true;
done:
    if (st) free_blocked(out, scratch.settle());
    return st;
}
#undef ASX_TRY

void free_blocked(BlockedMatrix *b, bool idle)
{
    for (void *q : {(void *)b->brow_ptr, (void *)b->bcol, b->bval, (void *)b->upd_src, (void *)b->upd_dst}) pool_free(q, idle);
    b->brow_ptr = nullptr;
    b->bcol = nullptr;
    b->bval = nullptr;
    b->upd_src = nullptr;
    b->upd_dst = nullptr;
}

// Refreshes the blocks' values from A's (same sparsity pattern); the zero fill is untouched.
template <typename T>
int blocked_update_values(const BlockedMatrix *bm, const T *val, hipStream_t s)
{
    if (bm->nblocks <= 0 || bm->nnz <= 0) return ASX_STATUS_SUCCESS;
    hipLaunchKernelGGL((k_block_values<T>), dim3((unsigned)ceil_div64(bm->nnz, kBlock)), dim3(kBlock), 0, s, bm->upd_src,
                       bm->upd_dst, bm->nnz, val, (T *)bm->bval);
    return check_launch();
}

// ---- MFMA wrappers: A 16x4 (lane l: row l%16, k l/16), B 4x16 (lane l: k l/16, col l%16),
// ---- D 16x16 in 4 registers per lane, col l%16; the row of register r differs by type:
// ----   fp32: 4*(l/16) + r        fp64: 4*r + l/16
__device__ __forceinline__ floatx4 mfma16x16x4(float a, float b, floatx4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ doublex4 mfma16x16x4(double a, double b, doublex4 c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
template <typename T>
struct Acc4;
template <>
struct Acc4<float> {
    typedef floatx4 type;
    static __device__ __forceinline__ int row(int lane_hi, int r) { return lane_hi * 4 + r; }
};
template <>
struct Acc4<double> {
    typedef doublex4 type;
    static __device__ __forceinline__ int row(int lane_hi, int r) { return r * 4 + lane_hi; }
};

// VEC consecutive columns of a lane as one access that needs no more alignment than an element has
template <typename T, int VEC>
struct ColsOf {
    typedef T type __attribute__((ext_vector_type(VEC), aligned(sizeof(T))));
};

// Waves a SIMD by the bytes of a row of B that a lane holds: two batches of wide rows want the registers (two waves, 200
// columns fp64: 29 us against 38 with one), and where 16 bytes a lane leave room for eight waves, six keep the rows of B
// that neighbours share longer in the L2 (65 per row, N = 64, fp32: 226 us against 230).
constexpr int blocked_waves(size_t bytes) { return bytes > 32 ? 2 : bytes > 16 ? 3 : bytes == 16 ? 6 : 8; }

// One wave per (block row, tile of up to 16 * VEC * NT columns of C).  Lane (kq, j) = (lane / 16, lane % 16) loads, of row
// kq of a block's four rows of B, the VEC columns from j * VEC on (16 bytes where N allows: one instruction
// fetches the four rows of 64 fp32 columns, where 4 bytes a lane took four) and feeds its v-th column to the v-th
// MFMA: accumulator v holds columns v, VEC + v, 2 VEC + v, ..., so a lane ends up with VEC consecutive columns of
// four rows of C.
// U blocks are in flight while the U before them are multiplied; every load is unconditional (past the end the
// last block is fetched again, a quad that reaches over B's last row repeats that row).  What is fetched so is not
// multiplied, or an infinity in B would meet other zeros of A than those that fill its own block: the last batch leaves
// out blocks past the end, and in the last block, the only one that can hold the partial quad, rows past B's end are zeros.
// Lanes past the last column repeat the last VEC columns and store nothing; where the width is no multiple of
// VEC the last lane overlaps the one before it (same bits, same wave).
// Consecutive block rows run on one XCD: they share most of their rows of B, which its L2 then fetches once.
// Bound by memory: 65 per row, N = 64, fp32 (1.2 GB past the L2s with C read and written): 312 -> 228 us.
template <typename T, int VEC, int NT>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(2, blocked_waves(VEC * NT * sizeof(T)))))
void k_spmm_blocked(int32_t m, int32_t kdim, int32_t ncols, int32_t nbrows, T alpha, const int32_t *__restrict__ brow_ptr,
                    const int32_t *__restrict__ bcol, const T *__restrict__ bval, const T *__restrict__ B, int64_t ldb,
                    T beta, T *__restrict__ C, int64_t ldc)
{
    typedef typename Acc4<T>::type acc_t;
    typedef typename ColsOf<T, VEC>::type V;
    constexpr int U = VEC * NT * sizeof(T) > 32 ? 2 : 4;
    const int lane = threadIdx.x & (kWave - 1);
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const uint32_t per_xcd = gridDim.x / kXcds;
    const int64_t br = ((int64_t)(blockIdx.x % kXcds) * per_xcd + blockIdx.x / kXcds) * (kBlock / kWave) + w;
    if (br >= nbrows) return;  // wave-uniform
    const int kq = lane >> 4, j16 = lane & 15;
    const int64_t t0 = (int64_t)blockIdx.y * ncols / gridDim.y, t1 = (int64_t)(blockIdx.y + 1) * ncols / gridDim.y;
    int64_t col[NT];
    bool active[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int64_t n = t0 + (t * 16 + j16) * VEC;
        active[t] = n < t1;
        col[t] = n < t1 - VEC ? n : t1 - VEC;
    }
    acc_t acc[NT * VEC];
#pragma unroll
    for (int t = 0; t < NT * VEC; ++t) acc[t] = acc_t{0, 0, 0, 0};
    const int32_t b0 = brow_ptr[br], b1 = brow_ptr[br + 1], last = b1 - 1;
    struct Batch {
        T a[U];
        V b[U][NT];
    } cur, next;
    const auto fetch = [&](Batch &q, int32_t first) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int32_t b = first + u < last ? first + u : last;  // scalar
            q.a[u] = bval[(int64_t)b * 64 + lane];
            const int32_t quad = bcol[b] * 4 + kq;
            const T *row = B + (int64_t)(quad < kdim ? quad : kdim - 1) * ldb;
#pragma unroll
            for (int t = 0; t < NT; ++t) q.b[u][t] = *(const V *)(row + col[t]);
        }
    };
    const auto multiply = [&](T a, const V (&bq)[NT]) {
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int v = 0; v < VEC; ++v) acc[t * VEC + v] = mfma16x16x4(a, bq[t][v], acc[t * VEC + v]);
    };
    const auto multiply_all = [&](const Batch &q) {
#pragma unroll
        for (int u = 0; u < U; ++u) multiply(q.a[u], q.b[u]);
    };
    const auto multiply_last = [&](Batch &q, int32_t first) {
        const bool there = bcol[last] * 4 + kq < kdim;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const bool counts = first + u < last || (first + u == last && there);
#pragma unroll
            for (int t = 0; t < NT; ++t) q.b[u][t] = counts ? q.b[u][t] : (V)T(0);
            multiply(counts ? q.a[u] : T(0), q.b[u]);
        }
    };
    if (b0 < b1) {
        fetch(cur, b0);
        int32_t b = b0;
        for (; b + 2 * U < b1; b += 2 * U) {  // uniform
            fetch(next, b + U);
            multiply_all(cur);
            fetch(cur, b + 2 * U);
            multiply_all(next);
        }
        if (b + U < b1) {
            fetch(next, b + U);
            multiply_all(cur);
            multiply_last(next, b + U);
        } else {
            multiply_last(cur, b);
        }
    }
    // every old value before the first store: the overlapping columns may belong to two tiles t of one lane row
    V old[NT][4];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int64_t row = br * 16 + Acc4<T>::row(kq, r);
            old[t][r] = T(0);
            if (beta != T(0)) old[t][r] = *(const V *)(C + (row < m ? row : m - 1) * ldc + col[t]);
        }
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int64_t row = br * 16 + Acc4<T>::row(kq, r);
            V out;
#pragma unroll
            for (int v = 0; v < VEC; ++v) {
                const T s = acc[t * VEC + v][r];
                out[v] = beta == T(0) ? alpha * s : fma_t<T>(alpha, s, beta * old[t][r][v]);
            }
            if (row < m && active[t]) *(V *)(C + row * ldc + col[t]) = out;
        }
}

// Columns per lane and wave: up to 16 and 32 columns take one and two columns a lane, wider ones 16 bytes a lane; beyond
// 64 columns a wave takes 128 (half the reads of A), beyond 128 equal tiles of up to 128.
template <typename T>
int launch_spmm_blocked(int32_t m, int32_t k, int32_t ncols, T alpha, const BlockedMatrix *bm, const T *B,
                        int64_t ldb, T beta, T *C, int64_t ldc, hipStream_t s)
{
    if (m <= 0 || ncols <= 0) return ASX_STATUS_SUCCESS;
    constexpr int kFull = 16 / sizeof(T);
    const unsigned gx = (unsigned)(ceil_div64(ceil_div64(bm->nbrows, kBlock / kWave), kXcds) * kXcds);
#define ASX_BLOCKED(VEC, NT)                                                                                              \
    hipLaunchKernelGGL((k_spmm_blocked<T, VEC, NT>), dim3(gx, (unsigned)ceil_div64(ncols, 16 * (VEC) * (NT))), dim3(kBlock), 0, s, \
                       m, k, ncols, bm->nbrows, alpha, bm->brow_ptr, bm->bcol, (const T *)bm->bval, B, ldb, beta, C, ldc)
    if (ncols <= 16)
        ASX_BLOCKED(1, 1);
    else if (ncols <= 32)
        ASX_BLOCKED(2, 1);
    else if (ncols <= 64)
        ASX_BLOCKED(kFull, 4 / kFull);
    else
        ASX_BLOCKED(kFull, 8 / kFull);
#undef ASX_BLOCKED
    return check_launch();
}

template int build_blocked<float>(int32_t, int32_t, int32_t, const int32_t *, const int32_t *, const float *,
                                  BlockedMatrix *, hipStream_t);
template int build_blocked<double>(int32_t, int32_t, int32_t, const int32_t *, const int32_t *, const double *,
                                   BlockedMatrix *, hipStream_t);
template int blocked_update_values<float>(const BlockedMatrix *, const float *, hipStream_t);
template int blocked_update_values<double>(const BlockedMatrix *, const double *, hipStream_t);
template int launch_spmm_blocked<float>(int32_t, int32_t, int32_t, float, const BlockedMatrix *, const float *,
                                        int64_t, float, float *, int64_t, hipStream_t);
template int launch_spmm_blocked<double>(int32_t, int32_t, int32_t, double, const BlockedMatrix *, const double *,
                                         int64_t, double, double *, int64_t, hipStream_t);

}  // namespace asx
