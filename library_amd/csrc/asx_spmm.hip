// CSR x dense SpMM for gfx950, C = alpha*A*B + beta*C with B (k x N) and C (m x N) row-major.
//
// Every access to a row of B or C covers consecutive columns: 64 lanes of one element in the row kernel, whose stored elements
// are read 64 at a time and broadcast through v_readlane (the address of the row of B is then wave-uniform), 16 bytes a lane
// in the merge and chunk kernels, whose lane groups work on different rows of A.
//
//   row   : one wave per (row, column tile).  Simple; long rows serialise.
//   merge : one wave per segment of consecutive items of the merge path over
//           (row ends, stored elements): bounded work per wave whatever the row lengths.
//           Rows that end inside a segment are written by that segment, and so is a row
//           that starts in it and ends in the next; of a longer row the part that runs past
//           a segment end is kept as a carry row and added by an ordered pass afterwards.  No atomics (the reference's default SpMM,
//           hip/kernel/level3/alphasparse_spmm_csr_nnz_split.h:283-409, scales C in a
//           separate pass and joins segments with atomicAdd).
//   chunk : the same with a workgroup per (longer) segment, for narrow rows of B, and for wide ones of small or scattered matrices.
#include <algorithm>
#include <type_traits>

#include "asx_internal.hpp"

namespace asx {

template <typename T>
__device__ __forceinline__ T readlane_t(T v, int l);
template <>
__device__ __forceinline__ float readlane_t<float>(float v, int l)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
template <>
__device__ __forceinline__ double readlane_t<double>(double v, int l)
{
    int lo = __builtin_amdgcn_readlane(__double2loint(v), l);
    int hi = __builtin_amdgcn_readlane(__double2hiint(v), l);
    return __hiloint2double(hi, lo);
}

#ifndef ASX_SPMM_IN_FLIGHT
#define ASX_SPMM_IN_FLIGHT 8
#endif
constexpr int kSpmmInFlight = ASX_SPMM_IN_FLIGHT;  // rows of B a wave has in flight

// acc += sum over stored elements [k_begin, k_end) of one row: a * B[col, c]
template <typename T>
__device__ __forceinline__ T spmm_accumulate(T acc, int32_t k_begin, int32_t k_end, int lane, bool col_ok,
                                             int64_t c, const int32_t *__restrict__ col,
                                             const T *__restrict__ val, const T *__restrict__ B,
                                             int64_t ldb)
{
    int64_t at = (int64_t)k_begin + lane;
    for (int32_t left = k_end - k_begin; left > 0; left -= kWave, at += kWave) {  // counted down: k_end may be 2^31 - 1
        const int32_t cl = lane < left ? col[at] : 0;
        const T vl = lane < left ? val[at] : T(0);
        const int cnt = left < kWave ? left : kWave;
        // kSpmmInFlight rows of B at a time
        int j = 0;
        for (; j + kSpmmInFlight <= cnt; j += kSpmmInFlight) {
            int32_t cc[kSpmmInFlight];
            T b[kSpmmInFlight];
#pragma unroll
            for (int u = 0; u < kSpmmInFlight; ++u) cc[u] = __builtin_amdgcn_readlane(cl, j + u);
#pragma unroll
            for (int u = 0; u < kSpmmInFlight; ++u) b[u] = col_ok ? B[(int64_t)cc[u] * ldb + c] : T(0);
#pragma unroll
            for (int u = 0; u < kSpmmInFlight; ++u) acc = fma_t<T>(readlane_t<T>(vl, j + u), b[u], acc);
        }
        if (j < cnt) {  // the last, partial batch: all its loads are issued before the first use
            int32_t cc[kSpmmInFlight];
            T b[kSpmmInFlight];
#pragma unroll
            for (int u = 0; u < kSpmmInFlight; ++u) cc[u] = __builtin_amdgcn_readlane(cl, (j + u) & (kWave - 1));
#pragma unroll
            for (int u = 0; u < kSpmmInFlight; ++u) b[u] = (col_ok && j + u < cnt) ? B[(int64_t)cc[u] * ldb + c] : T(0);
#pragma unroll
            for (int u = 0; u < kSpmmInFlight; ++u)
                if (j + u < cnt) acc = fma_t<T>(readlane_t<T>(vl, (j + u) & (kWave - 1)), b[u], acc);
        }
    }
    return acc;
}

template <typename T>
__device__ __forceinline__ T scaled_out(T alpha, T acc, T beta, const T *C, int64_t idx)
{
    return beta == T(0) ? alpha * acc : fma_t<T>(alpha, acc, beta * C[idx]);
}

// ===========================================================================================
// row: one wave per (row, column tile)
// ===========================================================================================
template <typename T>
__global__ __launch_bounds__(kBlock) void k_spmm_row(int32_t m, int32_t ncols, T alpha,
                                                     const int32_t *__restrict__ row_ptr,
                                                     const int32_t *__restrict__ col,
                                                     const T *__restrict__ val, const T *__restrict__ B,
                                                     int64_t ldb, T beta, T *__restrict__ C,
                                                     int64_t ldc)
{
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t row = (int64_t)blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave;
    if (row >= m) return;  // wave-uniform
    const int64_t c = (int64_t)blockIdx.y * kWave + lane;
    const bool col_ok = c < ncols;
    const int32_t s = __builtin_amdgcn_readfirstlane(row_ptr[row]);
    const int32_t e = __builtin_amdgcn_readfirstlane(row_ptr[row + 1]);
    T acc = spmm_accumulate<T>(T(0), s, e, lane, col_ok, c, col, val, B, ldb);
    if (col_ok) C[row * ldc + c] = scaled_out<T>(alpha, acc, beta, C, row * ldc + c);
}

template <typename T>
int launch_spmm_row(int32_t m, int32_t ncols, T alpha, const int32_t *row_ptr, const int32_t *col,
                    const T *val, const T *B, int64_t ldb, T beta, T *C, int64_t ldc, hipStream_t s)
{
    if (m <= 0 || ncols <= 0) return ASX_STATUS_SUCCESS;
    dim3 grid((unsigned)ceil_div64(m, kBlock / kWave), (unsigned)ceil_div64(ncols, kWave));
    hipLaunchKernelGGL((k_spmm_row<T>), grid, dim3(kBlock), 0, s, m, ncols, alpha, row_ptr, col, val, B,
                       ldb, beta, C, ldc);
    return check_launch();
}

// ===========================================================================================
// merge: one wave per segment of merge items
// ===========================================================================================
// Boundary g of the merge path lies between segments g-1 and g, at row x, element y (least row of
// the diagonal g * items whose end is not behind it).  The row cut by a boundary is SHORT there if
// it starts inside segment g-1 and ends inside segment g: then the boundary moves to the end of
// that row, so segment g-1 takes the whole row (running up to `items` past its nominal end) and
// segment g starts after it.  Only rows long enough to cover a whole segment are still cut and
// leave carries.  A segment so holds at most 2 * items elements and items + 1 row ends.
__device__ __forceinline__ void merge_point(const int32_t *__restrict__ row_ptr, int32_t m, int32_t nnz, int64_t d,
                                            int32_t &x, int32_t &y)
{
    const int64_t total = (int64_t)m + nnz;
    d = d < 0 ? 0 : d > total ? total : d;
    int32_t lo = (int32_t)(d > nnz ? d - nnz : 0), hi = (int32_t)(d < m ? d : m);
    while (lo < hi) {
        const int32_t p = lo + (hi - lo) / 2;
        if ((int64_t)row_ptr[p + 1] < d - p)
            lo = p + 1;
        else
            hi = p;
    }
    x = lo;
    y = (int32_t)(d - lo);
}

// One thread per boundary searches it and its two neighbours (three independent chains of loads:
// the latency of one) and applies the rule above; *has_carry (when wanted) is set if a row stays cut.
__global__ __launch_bounds__(kBlock) void k_spmm_splits(int32_t m, int32_t nnz, int32_t items, int32_t nseg,
                                                        const int32_t *__restrict__ row_ptr, int32_t *__restrict__ xs,
                                                        int32_t *__restrict__ ys, int32_t *__restrict__ has_carry)
{
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g > nseg) return;
    int32_t x, y, xp, yp, xn, yn;
    merge_point(row_ptr, m, nnz, (g - 1) * items, xp, yp);
    merge_point(row_ptr, m, nnz, g * items, x, y);
    merge_point(row_ptr, m, nnz, (g + 1) * items, xn, yn);
    if (g > 0 && g < nseg && x < m) {
        const int32_t b = row_ptr[x], e = row_ptr[x + 1];
        if (b < y && b >= yp && e <= yn && x < xn) {
            x += 1;
            y = e;
        } else if (has_carry && b < y) {
            *has_carry = 1;
        }
    }
    xs[g] = x;
    ys[g] = y;
}

// Boundaries seg and seg + 1 by the wave that owns the segment, for calls without a plan (a launch of k_spmm_splits
// before it: 13.9 us against 10.0 with 85000 elements and 8 columns, 271 against 266 with 3.8 M and 100): four groups of 16
// lanes search the points seg - 1 .. seg + 2 side by side, 16 probes at a time.  rest() runs once, behind the first probes' requests; where
// it says that nothing is left to do, false comes back.
struct NothingAsked {
    __device__ bool operator()() const { return true; }
};
template <typename F>
__device__ __forceinline__ bool segment_ends(const int32_t *__restrict__ row_ptr, int32_t m, int32_t nnz, int32_t items,
                                             int32_t nseg, int64_t seg, int32_t &x0, int32_t &y0, int32_t &x1, int32_t &y1,
                                             const F &rest)
{
    const int lane = threadIdx.x & (kWave - 1), q = lane >> 4, l = lane & 15;
    const int64_t total = (int64_t)m + nnz;
    int64_t d = (seg - 1 + q) * items;
    d = d < 0 ? 0 : d > total ? total : d;
    int64_t lo = d > nnz ? d - nnz : 0, hi = d < m ? d : m;
    bool first = true;
    while (__ballot(lo < hi)) {  // uniform; a group that is done repeats its answer
        const int64_t step = (hi - lo + 15) / 16, p = lo + l * step;
        bool before;  // the point lies behind p
        if constexpr (std::is_same<F, NothingAsked>::value) {
            before = lo < hi && p < hi && (int64_t)row_ptr[p + 1] < d - p;
        } else {
            const bool in = lo < hi && p < hi;
            const int32_t end = row_ptr[in ? p + 1 : 0];
            if (first && !rest()) return false;
            first = false;
            before = in && (int64_t)end < d - p;
        }
        const int n = __popc((unsigned)(__ballot(before) >> (q * 16)) & 0xffffu);
        const int64_t at = lo + (n > 0 ? (n - 1) * step + 1 : 0), to = lo + n * step;
        lo = lo < hi ? at : lo;
        hi = to < hi ? to : hi;
    }
    if (first && !rest()) return false;  // nothing to search
    int32_t x[4], y[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        x[k] = __builtin_amdgcn_readlane((int32_t)lo, k * 16);
        y[k] = __builtin_amdgcn_readlane((int32_t)(d - lo), k * 16);
    }
    const auto snap = [&](int64_t g, int k, int32_t &xo, int32_t &yo) {  // as k_spmm_splits does
        xo = x[k], yo = y[k];
        if (g > 0 && g < nseg && x[k] < m) {
            const int32_t b = row_ptr[x[k]], e = row_ptr[x[k] + 1];
            if (b < y[k] && b >= y[k - 1] && e <= y[k + 1] && x[k] < x[k + 1]) xo = x[k] + 1, yo = e;
        }
    };
    snap(seg, 1, x0, y0);
    snap(seg + 1, 2, x1, y1);
    return true;
}

int launch_spmm_splits(int32_t m, int32_t nnz, int32_t items, const int32_t *row_ptr, int32_t *xs, int32_t *ys,
                       int32_t *has_carry, hipStream_t s)
{
    const int32_t nseg = spmm_segments(m, nnz, items);
    hipLaunchKernelGGL(k_spmm_splits, dim3((unsigned)ceil_div64((int64_t)nseg + 1, kBlock)), dim3(kBlock), 0, s, m, nnz,
                       items, nseg, row_ptr, xs, ys, has_carry);
    return check_launch();
}

// VEC consecutive columns of a lane, loaded and stored as one access that needs no more alignment
// than an element has (ldb and ldc may be anything)
template <typename T, int VEC>
struct VecOf {
    typedef T type __attribute__((ext_vector_type(VEC), aligned(sizeof(T))));
};

template <int N>
struct Int {
    static constexpr int value = N;
};

// Sum over staged elements i0, i0 + ST, ... below e: a * (the lane's columns of the row of B that row_of_b fetches for what is
// staged of the element's column).  Batches of U, then at most one of U / 2, then one of U / 2 that is not full.
template <typename T, int VEC, int ST, int U, typename F>
__device__ __forceinline__ typename VecOf<T, VEC>::type spmm_staged(int32_t i0, int32_t e, const int32_t *s_col, const T *s_val,
                                                                    const F &row_of_b)
{
    typedef typename VecOf<T, VEC>::type V;
    V acc = T(0);
    int32_t i = i0;
    const auto batch = [&](auto n_, auto partial_) {  // n elements; partial: those from e on repeat the first
        constexpr int N = decltype(n_)::value;
        constexpr bool PARTIAL = decltype(partial_)::value;
        V b[N];
        T a[N];
#pragma unroll
        for (int u = 0; u < N; ++u) {
            const int32_t iu = !PARTIAL || i + u * ST < e ? i + u * ST : i;
            b[u] = row_of_b(s_col[iu]);
            a[u] = s_val[iu];
        }
#pragma unroll
        for (int u = 0; u < N; ++u) {
            const V sum = __builtin_elementwise_fma((V)a[u], b[u], acc);
            acc = !PARTIAL || i + u * ST < e ? sum : acc;
        }
        i += N * ST;
    };
    while (i + (U - 1) * ST < e) batch(Int<U>{}, Int<0>{});
    if (i + (U / 2 - 1) * ST < e) batch(Int<U / 2>{}, Int<0>{});
    if (i < e) batch(Int<U / 2>{}, Int<1>{});
    return acc;
}

// One wave per segment (of `items` merge items, at most SEG) and tile of columns.  A lane holds VEC columns (16 bytes where N allows), so
// G = 2^LOGG lanes span a tile and the wave's NG = 64 / G groups work on different stored elements at
// once: one load instruction fetches NG rows of B.  (A row of B per instruction, 4 bytes per lane,
// gets 110 G lines/s from an L2, 16 bytes per lane 240 G; with 8 columns in fp64 such a kernel left 56
// lanes of 64 idle.)
//   * the segment's columns, values and row ends are staged in LDS in one round trip;
//   * rows of up to kDealt elements are dealt to the groups, one row each;
//   * longer rows, and the row that goes on past the segment end, are taken by all groups together,
//     element by element in turn, and joined by a butterfly over the groups.
// A lane past the last column of the tile repeats the last VEC columns and stores nothing; a tile
// whose width is no multiple of VEC has its last lane overlap the one before it (both compute the same
// bits from the same old values of C, in one wave).
// Consecutive segments run on one XCD, whose L2 then fetches the rows of B that neighbouring rows
// of A share once.
// ASK: the sweep kernel has been launched ahead; where it answered that it takes the call, what is left are rows longer than it takes.
// That is a kernel of its own, and the usual one has no argument more: with one kernel for both, fp32 calls took 0.3 to 0.5 us
// longer (5-point stencil of 22680 rows, 64 columns 8.1 us and 8.5, 160 columns 12.1 and 12.5), with an argument that nobody reads, and
// so the grid's sizes on a third line of arguments, still 0.15.
template <typename T, int VEC, int LOGG, int SEG, bool ASK>
__device__ __forceinline__ void spmm_merge_segment(int32_t m, int32_t nnz, int32_t items, int32_t nseg, int32_t ncols, T alpha,
                                                   const int32_t *__restrict__ row_ptr,
                                                   const int32_t *__restrict__ col, const T *__restrict__ val,
                                                   const T *__restrict__ B, int64_t ldb, T beta,
                                                   T *__restrict__ C, int64_t ldc,
                                                   const int32_t *__restrict__ xs, const int32_t *__restrict__ ys,
                                                   T *__restrict__ carry, int32_t *__restrict__ carry_row, const SweepAsk &ask)
{
    typedef typename VecOf<T, VEC>::type V;
    constexpr int G = 1 << LOGG, NG = kWave / G;
    constexpr int U = 8;  // rows of B a lane has in flight
    constexpr int kDealt = spmm_dealt(NG);
    constexpr int kElems = 2 * SEG, kEnds = SEG + kWave;
    __shared__ int32_t s_col_all[kBlock / kWave][kElems];
    __shared__ T s_val_all[kBlock / kWave][kElems];
    __shared__ int32_t s_end_all[kBlock / kWave][kEnds + 1];
    const int lane = threadIdx.x & (kWave - 1);
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const uint32_t per_xcd = gridDim.x / kXcds;
    const int64_t blk = (int64_t)(blockIdx.x % kXcds) * per_xcd + blockIdx.x / kXcds;
    const int64_t seg = blk * (kBlock / kWave) + w;
    if (seg >= nseg) return;  // wave-uniform
    int32_t least = -1;  // only rows of more elements are left to do
    int32_t swept = 0;
    if constexpr (ASK) swept = *ask.answer;
    const int grp = lane >> LOGG, gl = lane & (G - 1);
    const int64_t t0 = (int64_t)blockIdx.y * ncols / gridDim.y, t1 = (int64_t)(blockIdx.y + 1) * ncols / gridDim.y;
    int64_t c = t0 + gl * VEC;
    const bool active = c < t1;
    c = c < t1 - VEC ? c : t1 - VEC;
    const char *Bc = (const char *)(B + c);
    const uint64_t ldb_bytes = (uint64_t)ldb * sizeof(T);
    int32_t x0, y0, x1, y1;
    if (xs)  // uniform
        x0 = xs[seg], y0 = ys[seg], x1 = xs[seg + 1], y1 = ys[seg + 1];
    if constexpr (ASK) {
        const auto rest = [&]() {
            if (!swept) return true;
            bool any = false;
            for (int i = lane * 8; i < ask.blocks; i += kWave * 8) any |= *(const uint64_t *)(ask.too_long + i) != 0;
            if (__ballot(any) == 0) return false;
            least = ask.longest;
            return true;
        };
        if (xs ? !rest() : !segment_ends(row_ptr, m, nnz, items, nseg, seg, x0, y0, x1, y1, rest)) {
            if (carry_row && lane == 0 && blockIdx.y == 0) carry_row[seg] = -1;
            return;
        }
    } else if (!xs) {
        segment_ends(row_ptr, m, nnz, items, nseg, seg, x0, y0, x1, y1, NothingAsked{});
    }
    const int32_t nel = y1 - y0 < kElems ? y1 - y0 : kElems, nrow = x1 - x0 < kEnds ? x1 - x0 : kEnds;
    int32_t *s_col = s_col_all[w];
    T *s_val = s_val_all[w];
    int32_t *s_end = s_end_all[w];  // s_end[r + 1]: end of row x0 + r, relative to y0
    // What most segments hold - up to SEG elements and 128 rows - is requested at once, past-the-end
    // lanes repeating the last entry; the rest follows only where there is more.
    const auto stage = [&](auto from_, auto to_, auto rows_from_, auto rows_to_) {
        constexpr int E0 = decltype(from_)::value, E1 = decltype(to_)::value, R0 = decltype(rows_from_)::value,
                      R1 = decltype(rows_to_)::value;
        constexpr int NE = (E1 - E0) / kWave, NR = (R1 - R0) / kWave;
        int32_t tc[NE > 0 ? NE : 1], te[NR > 0 ? NR : 1];
        T tv[NE > 0 ? NE : 1];
#pragma unroll
        for (int j = 0; j < NR; ++j) {
            const int i = R0 + j * kWave + lane;
            te[j] = row_ptr[x0 + (i < nrow ? i + 1 : nrow)];
        }
#pragma unroll
        for (int j = 0; j < NE; ++j) {
            const int i = E0 + j * kWave + lane;
            const int64_t k = (int64_t)y0 + (i < nel ? i : nel - 1);
            tc[j] = col[k];
            tv[j] = val[k];
        }
#pragma unroll
        for (int j = 0; j < NR; ++j) s_end[1 + R0 + j * kWave + lane] = te[j] - y0;
#pragma unroll
        for (int j = 0; j < NE; ++j) {
            s_col[E0 + j * kWave + lane] = tc[j];
            s_val[E0 + j * kWave + lane] = tv[j];
        }
    };
    if (nel > 0)
        stage(Int<0>{}, Int<SEG>{}, Int<0>{}, Int<128>{});
    else
        stage(Int<0>{}, Int<0>{}, Int<0>{}, Int<128>{});
    if (nel > SEG) stage(Int<SEG>{}, Int<kElems>{}, Int<0>{}, Int<0>{});
    if (nrow > 128) stage(Int<0>{}, Int<0>{}, Int<128>{}, Int<kEnds>{});
    if (lane == 0) s_end[0] = 0;
    // the staged data is private to this wave: order its LDS writes before its LDS reads
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

    const auto row_of_b = [&](int32_t column) -> V {
        const uint32_t at = (uint32_t)(NG == 1 ? __builtin_amdgcn_readfirstlane(column) : column);
        return *(const V *)(Bc + at * ldb_bytes);
    };
    const auto together = [&](int32_t k, int32_t e) {  // the row's sum over all groups, in every group
        V acc = spmm_staged<T, VEC, NG, U>(k + grp, e, s_col, s_val, row_of_b);
#pragma unroll
        for (int d = G; d < kWave; d <<= 1)
#pragma unroll
            for (int v = 0; v < VEC; ++v) acc[v] += __shfl_xor(acc[v], d, kWave);
        return acc;
    };
    const bool stores = active && grp == 0;
    // a row that is cut covers a segment, which holds `least` elements or more
    const bool first_cut = ASK && least >= 0 && row_ptr[x0] != y0;
    for (int32_t r0 = 0; r0 < nrow; r0 += NG) {
        const int32_t r = r0 + grp;
        const int32_t k = r < nrow ? s_end[r] : 0, e = r < nrow ? s_end[r + 1] : 0;
        const bool wanted = r < nrow && (!ASK || e - k > least || (first_cut && r == 0));
        const bool dealt = (ASK && !wanted) || e - k <= kDealt;
        if (wanted && dealt) {
            V *out = (V *)(C + (int64_t)(x0 + r) * ldc + c);
            V c_old = T(0);
            if (beta != T(0)) c_old = *out;  // requested before the row's loads of B
            const V acc = spmm_staged<T, VEC, 1, U>(k, e, s_col, s_val, row_of_b);
            const V y = beta == T(0) ? (V)(alpha * acc) : __builtin_elementwise_fma((V)alpha, acc, (V)(beta * c_old));
            if (active) *out = y;
        }
        if (NG > 1) {
            unsigned long long todo = __ballot(!dealt && gl == 0);
            while (todo) {  // wave-uniform
                const int src = __builtin_ctzll(todo);
                todo &= todo - 1;
                const int32_t rr = r0 + (src >> LOGG);
                const int32_t kk = __builtin_amdgcn_readlane(k, src), ee = __builtin_amdgcn_readlane(e, src);
                V *out = (V *)(C + (int64_t)(x0 + rr) * ldc + c);
                V c_old = T(0);
                if (beta != T(0) && stores) c_old = *out;
                const V acc = together(kk, ee);
                const V y = beta == T(0) ? (V)(alpha * acc) : __builtin_elementwise_fma((V)alpha, acc, (V)(beta * c_old));
                if (stores) *out = y;
            }
        }
    }
    const int32_t k = __builtin_amdgcn_readfirstlane(s_end[nrow]);
    // row x1 continues past the segment end (without a carry pass: elements behind the last row's end, which count nowhere)
    const bool has_tail = nel > k && carry_row;
    if (has_tail) {
        const V acc = together(k, nel);
        if (stores) *(V *)(carry + seg * ncols + c) = acc;
    }
    if (carry_row && lane == 0 && blockIdx.y == 0) carry_row[seg] = has_tail ? x1 : -1;
}

template <typename T, int VEC, int LOGG, int SEG>
__global__ __launch_bounds__(kBlock) void k_spmm_merge(int32_t m, int32_t nnz, int32_t items, int32_t nseg, int32_t ncols, T alpha,
                                                       const int32_t *__restrict__ row_ptr,
                                                       const int32_t *__restrict__ col, const T *__restrict__ val,
                                                       const T *__restrict__ B, int64_t ldb, T beta,
                                                       T *__restrict__ C, int64_t ldc,
                                                       const int32_t *__restrict__ xs, const int32_t *__restrict__ ys,
                                                       T *__restrict__ carry, int32_t *__restrict__ carry_row)
{
    spmm_merge_segment<T, VEC, LOGG, SEG, false>(m, nnz, items, nseg, ncols, alpha, row_ptr, col, val, B, ldb, beta, C, ldc, xs, ys, carry,
                                                 carry_row, SweepAsk{});
}

template <typename T, int VEC, int LOGG, int SEG>
__global__ __launch_bounds__(kBlock) void k_spmm_merge_rest(int32_t m, int32_t nnz, int32_t items, int32_t nseg, int32_t ncols, T alpha,
                                                            const int32_t *__restrict__ row_ptr,
                                                            const int32_t *__restrict__ col, const T *__restrict__ val,
                                                            const T *__restrict__ B, int64_t ldb, T beta,
                                                            T *__restrict__ C, int64_t ldc,
                                                            const int32_t *__restrict__ xs, const int32_t *__restrict__ ys,
                                                            T *__restrict__ carry, int32_t *__restrict__ carry_row, SweepAsk ask)
{
    spmm_merge_segment<T, VEC, LOGG, SEG, true>(m, nnz, items, nseg, ncols, alpha, row_ptr, col, val, B, ldb, beta, C, ldc, xs, ys, carry,
                                                carry_row, ask);
}

// ===========================================================================================
// chunk: one workgroup per segment
// ===========================================================================================
// Where a row of B takes four lanes or fewer, rows of B that the L2s could serve wait for stored elements of A on their way from
// memory: a compute unit's L1 answers in order (64-byte rows from an L2 beside a stream from memory 175 G/s wave by wave,
// 217 behind barriers, 259 alone).  So a workgroup of 512 stages one long segment, all of it requested at once, and no wave
// fetches a row of B before the barrier: three workgroups a compute unit that each meet memory once a segment, where the
// merge kernel's twenty waves meet it every 256 items.  Longer segments also give narrow rows enough rows of A to deal out.  Eight
// rows of B in flight a group (four, and the four workgroups that then fit: 103.5 us where eight take 91.9).  Merge kernel and
// this one, three matrices in turn: 8 columns fp64, 20 per row within 3000 of the diagonal 65.4 -> 56.5 us, 2 columns
// 54.1 -> 39.8; 16 columns fp32, 50 per row within 20000 122 -> 91.9; 4 columns fp32, 8 per row within 300 29.3 -> 20.2; band of
// 11, 2 columns fp64 24.3 -> 16.7.
//
// Rows of B of more than 128 bytes (spmm_chunked_wide says which) come here for another reason: too few waves.  Eight waves deal the
// segment's rows out, and one of more than 64 elements is cut between them, in which eight rows of B are then in flight a group.
//
// How a row of B is found (REACH).  kRowsNear: a 32-bit pitch, a multiply-add into 64 bits, however many rows there are: without a
// plan a caller's k is no more than the width of a tile to the kernels that work row by row.  kRowsFar: rows of B of 4 GB and
// more.  kOffsets: where a lane takes a whole row of B, its byte offset is staged in place of the column and fits 32 bits; a
// plan says so, whose number of columns is the matrix's own.  Registers for eight of them in flight then leave room for
// four workgroups a compute unit in fp32.  Planned, 8 M elements within 3000 of the diagonal, kRowsNear and kOffsets: 4 columns fp32, 8 per
// row 40.9 and 37.4 us, 16 29.8 and 28.0, 60 23.7 and 22.8; 2 columns fp64 within 2 %; wider rows of B no faster (8 columns fp64, 20 per
// row 53.7 and 54.9, 40 53.7 and 54.7).
enum { kRowsFar = 0, kRowsNear = 1, kOffsets = 2 };
template <typename T, int VEC, int LOGG, int REACH>
__global__ __launch_bounds__(kChunkThreads, REACH == kRowsFar ? 4 : 6) void k_spmm_chunk(
    int32_t m, int32_t nnz, int32_t items, int32_t nseg, int32_t ncols, T alpha, const int32_t *__restrict__ row_ptr,
    const int32_t *__restrict__ col, const T *__restrict__ val, const T *__restrict__ B, int64_t ldb, T beta, T *__restrict__ C, int64_t ldc,
    const int32_t *__restrict__ xs, const int32_t *__restrict__ ys, T *__restrict__ carry, int32_t *__restrict__ carry_row)
{
    typedef typename VecOf<T, VEC>::type V;
    constexpr int G = 1 << LOGG, NG = kWave / G;
    // Rows of B a lane has in flight.  Where a lane takes a whole one, fp32, six of them and their 64-bit addresses leave room for the
    // registers of four workgroups a compute unit, eight of three (no plan, 4 columns, 20 per row 49.7 us with eight, 44.1 with six,
    // 43.9 with four; 40 per row 50.1, 47.2, 47.1; 60 52.9, 48.2, 50.9).
    constexpr int U = REACH == kRowsNear && sizeof(T) == 4 && VEC == 4 && LOGG == 0 ? 6 : 8;
    constexpr int kWide = NG > 4 ? 256 : kChunkWideLeast;  // longer rows are taken by all waves (elements)
    constexpr int kDealt = spmm_dealt(NG) < kWide ? spmm_dealt(NG) : kWide;
    constexpr int kWaves = kChunkThreads / kWave, NE = (kChunkElems + kChunkThreads - 1) / kChunkThreads;
    __shared__ int32_t s_col[kChunkElems];
    __shared__ T s_val[kChunkElems];
    __shared__ uint16_t s_end[kChunkRows + 1];  // s_end[r + 1]: end of row x0 + r, relative to y0
    __shared__ int32_t s_cut[4], s_long[kChunkElems / kDealt], s_wide[kChunkElems / kWide], s_nlong, s_nwide;
    __shared__ V s_part[kWaves][G];
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int w = __builtin_amdgcn_readfirstlane(tid / kWave);
    const uint32_t per_xcd = gridDim.x / kXcds;  // consecutive segments on one XCD, as in the merge kernel
    const int64_t seg = (int64_t)(blockIdx.x % kXcds) * per_xcd + blockIdx.x / kXcds;
    if (seg >= nseg) return;  // the whole workgroup leaves
    const int grp = lane >> LOGG, gl = lane & (G - 1);
    const int32_t t0 = (int32_t)((int64_t)blockIdx.y * ncols / gridDim.y), t1 = (int32_t)((int64_t)(blockIdx.y + 1) * ncols / gridDim.y);
    int32_t c = t0 + gl * VEC;  // as in the merge kernel
    const bool active = c < t1;
    c = c < t1 - VEC ? c : t1 - VEC;
    const uint64_t ldb_bytes = (uint64_t)ldb * sizeof(T);
    int32_t x0, y0, x1, y1;
    if (xs) {  // uniform
        x0 = xs[seg], y0 = ys[seg], x1 = xs[seg + 1], y1 = ys[seg + 1];
    } else {
        if (w == 0) {
            segment_ends(row_ptr, m, nnz, items, nseg, seg, x0, y0, x1, y1, NothingAsked{});
            if (lane == 0) s_cut[0] = x0, s_cut[1] = y0, s_cut[2] = x1, s_cut[3] = y1;
        }
        __syncthreads();
        x0 = s_cut[0], y0 = s_cut[1], x1 = s_cut[2], y1 = s_cut[3];
    }
    x0 = __builtin_amdgcn_readfirstlane(x0), y0 = __builtin_amdgcn_readfirstlane(y0);
    const int32_t nel = __builtin_amdgcn_readfirstlane(y1 - y0 < kChunkElems ? y1 - y0 : kChunkElems);
    const int32_t nrow = __builtin_amdgcn_readfirstlane(x1 - x0 < kChunkRows ? x1 - x0 : kChunkRows);
    {
        int32_t tc[NE];
        T tv[NE];
#pragma unroll
        for (int j = 0; j < NE; ++j)
            if (j * kChunkThreads < nel) {  // uniform; lanes past the end repeat the last element
                const int i = j * kChunkThreads + tid;
                const int64_t k = (int64_t)y0 + (i < nel ? i : nel - 1);
                tc[j] = col[k];
                tv[j] = val[k];
            }
        if (tid == 0) s_end[0] = 0, s_nlong = s_nwide = 0;
        for (int i = tid; i < nrow; i += kChunkThreads) s_end[i + 1] = (uint16_t)(row_ptr[x0 + i + 1] - y0);
#pragma unroll
        for (int j = 0; j < NE; ++j)
            if (j * kChunkThreads < nel) {
                const int i = j * kChunkThreads + tid;
                if (i < kChunkElems) {
                    s_col[i] = REACH == kOffsets ? (int32_t)((uint32_t)tc[j] * (uint32_t)ldb_bytes) : tc[j];
                    s_val[i] = tv[j];
                }
            }
    }
    __syncthreads();

    const uint64_t pitch = REACH == kRowsFar ? ldb_bytes : (uint32_t)ldb_bytes;
    const uint32_t c_bytes = (uint32_t)c * (uint32_t)sizeof(T);
    const auto row_of_b = [&](int32_t staged) -> V {
        return REACH == kOffsets ? *(const V *)((const char *)B + ((uint32_t)staged + c_bytes))
                                 : *(const V *)((const char *)(B + c) + (uint32_t)staged * pitch);
    };
    const auto together = [&](int32_t k, int32_t e) {  // the sum over the wave's groups, in every group
        V acc = spmm_staged<T, VEC, NG, (NG > 4 ? U / 2 : U)>(k + grp, e, s_col, s_val, row_of_b);
#pragma unroll
        for (int d = G; d < kWave; d <<= 1)
#pragma unroll
            for (int v = 0; v < VEC; ++v) acc[v] += __shfl_xor(acc[v], d, kWave);
        return acc;
    };
    const bool stores = active && grp == 0;
    for (int32_t r0 = w * NG; r0 < nrow; r0 += kWaves * NG) {
        const int32_t r = r0 + grp;
        const int32_t k = r < nrow ? s_end[r] : 0, e = r < nrow ? s_end[r + 1] : 0;
        const bool dealt = e - k <= kDealt;
        if (r < nrow && dealt) {
            V *out = (V *)(C + (int64_t)(x0 + r) * ldc + c);
            V c_old = T(0);
            if (beta != T(0)) c_old = *out;  // requested before the row's loads of B
            const V acc = spmm_staged<T, VEC, 1, U>(k, e, s_col, s_val, row_of_b);
            const V y = beta == T(0) ? (V)(alpha * acc) : __builtin_elementwise_fma((V)alpha, acc, (V)(beta * c_old));
            if (active) *out = y;
        }
        if (!dealt && gl == 0) {  // in any order: each is a sum of its own
            if (e - k > kWide)
                s_wide[atomicAdd(&s_nwide, 1)] = r;
            else
                s_long[atomicAdd(&s_nlong, 1)] = r;
        }
    }
    __syncthreads();
    // Rows longer than a group takes, from a list, one a wave: taken by the wave that they were dealt to, which has up to 64 groups,
    // they left the other waves idle (128 per row, 11 columns fp32 96 -> 53 us; 115 per row, 2 columns fp64 46 -> 19).
    const int32_t nlong = s_nlong;
    for (int32_t i = w; i < nlong; i += kWaves) {  // wave-uniform
        const int32_t r = __builtin_amdgcn_readfirstlane(s_long[i]);
        const int32_t k = __builtin_amdgcn_readfirstlane(s_end[r]), e = __builtin_amdgcn_readfirstlane(s_end[r + 1]);
        V *out = (V *)(C + (int64_t)(x0 + r) * ldc + c);
        V c_old = T(0);
        if (beta != T(0) && stores) c_old = *out;
        const V acc = together(k, e);
        const V y = beta == T(0) ? (V)(alpha * acc) : __builtin_elementwise_fma((V)alpha, acc, (V)(beta * c_old));
        if (stores) *out = y;
    }
    // Rows wider than kWide, and what the segment holds of a row that goes on past its end: a stretch a wave, added up in the
    // order of the waves.
    const int32_t last = s_end[nrow], nwide = s_nwide;
    const bool tail = carry_row && nel > last;
    for (int32_t i = 0; i < nwide + (tail ? 1 : 0); ++i) {  // uniform
        const int32_t r = i < nwide ? s_wide[i] : nrow;
        const int32_t from = s_end[r], to = i < nwide ? s_end[r + 1] : nel, share = (to - from + kWaves - 1) / kWaves;
        const int32_t k = from + w * share, e = k + share < to ? k + share : to;
        const V acc = together(k, e);
        if (grp == 0) s_part[w][gl] = acc;
        __syncthreads();
        if (w == 0 && stores) {
            V sum = s_part[0][gl];
#pragma unroll
            for (int q = 1; q < kWaves; ++q) sum += s_part[q][gl];
            if (i < nwide) {
                V *out = (V *)(C + (int64_t)(x0 + r) * ldc + c);
                *out = beta == T(0) ? (V)(alpha * sum) : __builtin_elementwise_fma((V)alpha, sum, (V)(beta * *out));
            } else {
                *(V *)(carry + seg * ncols + c) = sum;
            }
        }
        __syncthreads();
    }
    if (carry_row && tid == 0 && blockIdx.y == 0) carry_row[seg] = tail ? x1 : -1;
}

// Every wave looks at kFixupSegs consecutive segments (one lane each) for the first segment of a run
// of segments that left carries for the same row; each such run is then summed by the whole wave
// (lanes = columns), one after the other: few segments per wave, because a run costs three or four
// dependent memory round trips and the runs of a wave are taken in turn (64 segments per wave left
// the pass with 2000 waves, each with five runs in a row: 22 us on the Zipf matrix, 19 us with 8; what
// remains is the longest rows, whose hundreds of carry rows one wave adds 64 at a time).  The run length
// comes from ballots over carry_row (64 segments per step), the carry rows are added in segment
// order with a counted, unrolled loop (many independent loads in flight; a loop that tests
// carry_row before every add would pay one memory round trip per segment).
constexpr int kFixupSegs = 8;
template <typename T>
__global__ __launch_bounds__(kBlock) void k_spmm_merge_fixup(int32_t m, int32_t nseg, int32_t ncols,
                                                             T alpha, const T *__restrict__ carry,
                                                             const int32_t *__restrict__ carry_row,
                                                             T *__restrict__ C, int64_t ldc)
{
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t wave = ((int64_t)blockIdx.x * kBlock + threadIdx.x) / kWave;
    const int64_t t = wave * kFixupSegs + lane;
    int32_t my_row = -1;
    bool head = false;
    if (lane < kFixupSegs && t < nseg) {
        my_row = carry_row[t];
        head = my_row >= 0 && my_row < m && (t == 0 || carry_row[t - 1] != my_row);
    }
    unsigned long long todo = __ballot(head);
    while (todo) {  // wave-uniform
        const int src = __ffsll(todo) - 1;
        todo &= todo - 1;
        const int64_t seg = t - lane + src;
        const int32_t row = __shfl(my_row, src, kWave);
        int64_t len = 1;
        for (int64_t base = seg + 1;; base += kWave) {
            const int64_t idx = base + lane;
            const bool same = idx < nseg && carry_row[idx] == row;
            const unsigned long long mask = __ballot(same);
            const int n = mask == ~0ull ? kWave : __ffsll((unsigned long long)~mask) - 1;
            len += n;
            if (n < kWave) break;
        }
        for (int64_t c = lane; c < ncols; c += kWave) {
            const T *p = carry + seg * ncols + c;
            T sum = T(0);
            int64_t j = 0;
            for (; j + 64 <= len; j += 64) {  // a 50 000-element row leaves 390 carry rows
                T v[64];
#pragma unroll
                for (int u = 0; u < 64; ++u) v[u] = p[(j + u) * ncols];
#pragma unroll
                for (int u = 0; u < 64; ++u) sum += v[u];
            }
            for (; j + 8 <= len; j += 8) {
                T v[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) v[u] = p[(j + u) * ncols];
#pragma unroll
                for (int u = 0; u < 8; ++u) sum += v[u];
            }
            for (; j < len; ++j) sum += p[j * ncols];
            const int64_t idx = (int64_t)row * ldc + c;
            C[idx] = fma_t<T>(alpha, sum, C[idx]);
        }
    }
}

// N is cut into equal tiles of at most tile_bytes of a row of B (every tile at least VEC wide); lanes per row of B: the
// smallest power of two that spans a tile at VEC columns each.
template <typename T, int VEC, int SEG>
static void launch_merge_width(const SpmmTiling &tiling, int32_t m, int32_t nnz, int32_t items, int32_t nseg, int32_t ncols, T alpha,
                               const int32_t *row_ptr, const int32_t *col, const T *val, const T *B, int64_t ldb, T beta, T *C, int64_t ldc,
                               const int32_t *xs, const int32_t *ys, T *carry, int32_t *carry_row, const SweepAsk &ask, hipStream_t s)
{
    const dim3 grid((unsigned)(ceil_div64(ceil_div64(nseg, kBlock / kWave), kXcds) * kXcds), (unsigned)tiling.tiles);
#define ASX_WIDTH(LOGG)                                                                                              \
    if (tiling.log_lanes <= LOGG) {                                                                                      \
        if constexpr (VEC == 16 / sizeof(T) && LOGG >= 3) /* the sweep's calls: rows of B of more than 64 bytes */       \
            if (ask.answer) {                                                                                            \
                hipLaunchKernelGGL((k_spmm_merge_rest<T, VEC, LOGG, SEG>), grid, dim3(kBlock), 0, s, m, nnz, items, nseg, ncols, alpha,  \
                                   row_ptr, col, val, B, ldb, beta, C, ldc, xs, ys, carry, carry_row, ask);          \
                return;                                                                                                  \
            }                                                                                                            \
        hipLaunchKernelGGL((k_spmm_merge<T, VEC, LOGG, SEG>), grid, dim3(kBlock), 0, s, m, nnz, items, nseg, ncols, alpha, row_ptr, col, \
                           val, B, ldb, beta, C, ldc, xs, ys, carry, carry_row);                                     \
        return;                                                                                                      \
    }
    ASX_WIDTH(0)
    ASX_WIDTH(1)
    if constexpr (VEC * sizeof(T) == 16) {  // fewer columns per lane only where N is smaller than 16 bytes
        ASX_WIDTH(2)
        ASX_WIDTH(3)
        ASX_WIDTH(4)
        ASX_WIDTH(5)
        ASX_WIDTH(6)
    }
#undef ASX_WIDTH
}

template <typename T, int SEG>
static void launch_merge_seg(const SpmmTiling &tiling, int32_t m, int32_t nnz, int32_t items, int32_t nseg, int32_t ncols, T alpha,
                             const int32_t *row_ptr, const int32_t *col, const T *val, const T *B, int64_t ldb, T beta, T *C, int64_t ldc,
                             const int32_t *xs, const int32_t *ys, T *carry, int32_t *carry_row, const SweepAsk &ask, hipStream_t s)
{
    constexpr int kFull = 16 / sizeof(T);
    if (tiling.vec == kFull)
        launch_merge_width<T, kFull, SEG>(tiling, m, nnz, items, nseg, ncols, alpha, row_ptr, col, val, B, ldb, beta, C, ldc,
                                         xs, ys, carry, carry_row, ask, s);
    else if (tiling.vec == 2)
        launch_merge_width<T, 2, SEG>(tiling, m, nnz, items, nseg, ncols, alpha, row_ptr, col, val, B, ldb, beta, C, ldc,
                                     xs, ys, carry, carry_row, ask, s);
    else
        launch_merge_width<T, 1, SEG>(tiling, m, nnz, items, nseg, ncols, alpha, row_ptr, col, val, B, ldb, beta, C, ldc,
                                     xs, ys, carry, carry_row, ask, s);
}

// As many lanes a group as span the columns.  rows: of B where a plan knows them, else 0.
template <typename T>
static void launch_chunk(const SpmmTiling &tiling, int32_t rows, int32_t m, int32_t nnz, int32_t items, int32_t nseg, int32_t ncols,
                         T alpha, const int32_t *row_ptr, const int32_t *col, const T *val, const T *B, int64_t ldb, T beta, T *C, int64_t ldc,
                         const int32_t *xs, const int32_t *ys, T *carry, int32_t *carry_row, hipStream_t s)
{
    constexpr int kFull = 16 / sizeof(T);
    const dim3 grid((unsigned)(ceil_div64(nseg, kXcds) * kXcds), (unsigned)tiling.tiles);
    const auto launch = [&](auto vec_, auto log_) {
        const auto with = [&](auto reach_) {
            hipLaunchKernelGGL((k_spmm_chunk<T, decltype(vec_)::value, decltype(log_)::value, decltype(reach_)::value>), grid,
                               dim3(kChunkThreads), 0, s, m, nnz, items, nseg, ncols, alpha, row_ptr, col, val, B, ldb, beta, C, ldc, xs,
                               ys, carry, carry_row);
        };
        if constexpr (decltype(log_)::value == 0)
            if (rows > 0 && (uint64_t)rows * (uint64_t)ldb <= 0xffffffffull / sizeof(T)) return with(Int<kOffsets>{});
        if ((uint64_t)ldb > 0xffffffffull / sizeof(T))
            with(Int<kRowsFar>{});
        else
            with(Int<kRowsNear>{});
    };
    if (tiling.vec == kFull) {
        if (tiling.log_lanes == 0)
            launch(Int<kFull>{}, Int<0>{});
        else if (tiling.log_lanes == 1)
            launch(Int<kFull>{}, Int<1>{});
        else if (tiling.log_lanes == 2)
            launch(Int<kFull>{}, Int<2>{});
        else if (tiling.log_lanes == 3)
            launch(Int<kFull>{}, Int<3>{});
        else if (tiling.log_lanes == 4)
            launch(Int<kFull>{}, Int<4>{});
        else if (tiling.log_lanes == 5)
            launch(Int<kFull>{}, Int<5>{});
        else
            launch(Int<kFull>{}, Int<6>{});
    } else if (tiling.vec == 1) {
        launch(Int<1>{}, Int<0>{});
    } else if constexpr (kFull > 2) {  // two or three columns of fp32
        if (tiling.log_lanes == 0)
            launch(Int<2>{}, Int<0>{});
        else
            launch(Int<2>{}, Int<1>{});
    }
}

template <typename T>
int launch_spmm_merge(bool chunked, int32_t rows, int32_t m, int32_t nnz, int32_t items, int32_t ncols, T alpha, const int32_t *row_ptr,
                      const int32_t *col, const T *val, const T *B, int64_t ldb, T beta, T *C,
                      int64_t ldc, const int32_t *xs, const int32_t *ys, T *carry, int32_t *carry_row,
                      bool carry_pass, int tile_bytes, const SweepAsk &ask, hipStream_t s)
{
    if (m <= 0 || ncols <= 0) return ASX_STATUS_SUCCESS;
    // Tiles of columns are blocks along a grid's y, of which there are at most 65535: more columns are walked in slabs of whole
    // tiles, one after the other in the same workspace.
    const int64_t slab = (int64_t)65535 * (tile_bytes / (int64_t)sizeof(T));
    if (ncols > slab) {
        for (int64_t c = 0; c < ncols; c += slab) {
            const int32_t wide = (int32_t)(ncols - c < slab ? ncols - c : slab);
            const int st = launch_spmm_merge<T>(chunked, rows, m, nnz, items, wide, alpha, row_ptr, col, val, B + c, ldb, beta, C + c,
                                                ldc, xs, ys, carry, carry_row, carry_pass, tile_bytes, ask, s);
            if (st) return st;
        }
        return ASX_STATUS_SUCCESS;
    }
    const int32_t nseg = spmm_segments(m, nnz, items);
    const SpmmTiling tiling = spmm_tiling(ncols, tile_bytes, sizeof(T));
    if (!carry_pass) carry = nullptr, carry_row = nullptr;  // no row is cut: nothing is left for the pass
    if (chunked) {
        launch_chunk<T>(tiling, rows, m, nnz, items, nseg, ncols, alpha, row_ptr, col, val, B, ldb, beta, C, ldc, xs, ys, carry, carry_row, s);
    } else {
        const auto launch = [&](auto seg_) {
            launch_merge_seg<T, decltype(seg_)::value>(tiling, m, nnz, items, nseg, ncols, alpha, row_ptr, col, val, B, ldb, beta, C, ldc,
                                                       xs, ys, carry, carry_row, ask, s);
        };
        if (items <= kSpmmSegmentSmall)
            launch(Int<kSpmmSegmentSmall>{});
        else if (items <= kSpmmSegmentMedium)
            launch(Int<kSpmmSegmentMedium>{});
        else if constexpr (sizeof(T) == 4)
            launch(Int<kSpmmSegmentLarge>{});
    }
    if (carry_pass)
        hipLaunchKernelGGL((k_spmm_merge_fixup<T>), dim3((unsigned)ceil_div64(ceil_div64(nseg, kFixupSegs), kBlock / kWave)),
                           dim3(kBlock), 0, s, m, nseg, ncols, alpha, carry, carry_row, C, ldc);
    return check_launch();
}

#define ASX_INST(T)                                                                                  \
    template int launch_spmm_row<T>(int32_t, int32_t, T, const int32_t *, const int32_t *, const T *, \
                                    const T *, int64_t, T, T *, int64_t, hipStream_t);               \
    template int launch_spmm_merge<T>(bool, int32_t, int32_t, int32_t, int32_t, int32_t, T, const int32_t *, const int32_t *, \
                                      const T *, const T *, int64_t, T, T *, int64_t, const int32_t *, \
                                      const int32_t *, T *, int32_t *, bool, int, const SweepAsk &, hipStream_t);
ASX_INST(float)
ASX_INST(double)
#undef ASX_INST

}  // namespace asx
