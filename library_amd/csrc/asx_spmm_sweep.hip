// CSR x dense SpMM for gfx950 where the columns of A lie all over B: C = alpha*A*B + beta*C, B and C row-major.
//
// The row-ordered kernels (asx_spmm.hip) fetch a row of B for every stored element, and where B is larger than an L2 nearly each
// fetch goes past it, at 56 to 59 G lines/s whatever the kernel does.  An XCD's registers, though, hold the rows of C that its
// share of A makes (32 compute units with 512 KB each), so here every wave keeps its rows of C in registers, and all waves go
// through the columns of A together, in windows: while a window lasts, its part of B stays in the XCD's L2 and serves the
// elements of all rows.  Nothing orders the waves but that they do the same work a window; those ahead wait for memory, those
// behind find their rows of B in the L2.
//
// Calls whose columns nobody has looked at ask the device (sweep_suits): the first wave of every workgroup looks at 64 rows spread over
// A, all workgroups come to the same answer, and where it is no they end; the merge kernel, launched behind them, finds the
// answer in the call's workspace and does what is left: everything, or the rows that are too long to be walked by one lane group.
//
// Uniform columns, 25 per row, 100 columns fp32 of 150001 rows: 255 us with the merge kernel, 14.7 M lines past the L2s, 4.8 M here; 124 us here
// where B is in the Infinity Cache, 141 where inputs change from call to call.  49 per row, 96 columns of 94796 rows 316 and 136, 100
// columns, where such rows are two sums, 289 and 158; 24 per row, 103 columns fp64 of 97486 337 and 215 (in the cache).
#include "asx_internal.hpp"

namespace asx {

namespace {

template <typename T>
struct Vec16 {  // 16 bytes of a row, aligned as an element is
    static constexpr int N = 16 / sizeof(T);
    typedef T type __attribute__((ext_vector_type(16 / sizeof(T)), aligned(sizeof(T))));
};

template <int I>
struct Const {
    static constexpr int value = I;
};
template <int I, int N, typename F>
__device__ __forceinline__ void static_for(const F &f)
{
    if constexpr (I < N) {
        f(Const<I>{});
        static_for<I + 1, N>(f);
    }
}

// what lane J of every group of 2^LOGL lanes holds, in all lanes of the group
template <int LOGL, int J>
__device__ __forceinline__ uint32_t group_lane(uint32_t v)
{
    if constexpr (LOGL == 6)
        return (uint32_t)__builtin_amdgcn_readlane((int)v, J);
    else
        return (uint32_t)__builtin_amdgcn_ds_swizzle((int)v, ((32 - (1 << LOGL)) & 31) | J << 5);
}
template <int LOGL, int J>
__device__ __forceinline__ float group_lane(float v)
{
    return __builtin_bit_cast(float, group_lane<LOGL, J>(__builtin_bit_cast(uint32_t, v)));
}
template <int LOGL, int J>
__device__ __forceinline__ double group_lane(double v)
{
    return __hiloint2double((int)group_lane<LOGL, J>((uint32_t)__double2hiint(v)), (int)group_lane<LOGL, J>((uint32_t)__double2loint(v)));
}

}  // namespace

// lanes j0 .. j0 + n - 1 of every group of l
constexpr uint64_t lanes_of_groups(int l, int j0, int n)
{
    uint64_t mask = 0;
    for (int g = 0; g < kWave; g += l) mask |= ((1ull << n) - 1) << (g + j0);
    return mask;
}
constexpr uint32_t kNoColumn = 0xffffffffu, kAllColumns = 0x80000000u;

// Whether A looks as if its columns lay all over B and ascended in a row, and its rows were of one length: by the first and last
// column and one between of 64 rows spread over A, one a lane, of which most have to say so (counted with ballots: every workgroup
// looks, and sums over the lanes took half a microsecond of the 4 to 5 that asking costs).
//   No row is longer than the sweep takes (some 4 of 64 power-law rows with exponents of up to 2.6 and a mean of 16 are), 48 have half of
//   the mean or more (power-law rows with an exponent of 2.2 some 30).
//   Columns ascend; 44 rows reach three quarters as far as uniform columns do on average, (len - 1) / (len + 1) of B (of uniform rows
//   of 4 51 do, of longer ones more); and in 44 a column is a tenth of B or more from one of the next row (uniform columns 52, matrices near a
//   diagonal, whose next row is a 64th of B away, none).
__device__ __forceinline__ bool sweep_suits(const SweepAsk &ask, int32_t m, int32_t nnz, int lane, const int32_t *__restrict__ row_ptr,
                                            const int32_t *__restrict__ col)
{
    const int64_t r = (int64_t)m * (2 * lane + 1) / (2 * kWave);
    const int32_t s = row_ptr[r], len = row_ptr[r + 1] - s;
    const int64_t last = (int64_t)nnz - 1, l = len > 0 ? len : 1;
    const int64_t k0 = s < last ? s : last, k1 = k0 + l - 1 < last ? k0 + l - 1 : last;
    const int64_t kx = k0 + ((int64_t)(lane * 0x9e3779b1u >> 8) * l >> 24);
    const int32_t c0 = col[k0], cx = col[kx < last ? kx : last], c1 = col[k1];
    const float n = (float)ask.n, apart = fabsf((float)cx - (float)__shfl(cx, (lane + 1) & (kWave - 1), kWave));
    const uint64_t far = __ballot(len > ask.longest), half = __ballot(2.0f * (float)len * (float)m >= (float)nnz);
    const uint64_t falls = __ballot(cx < c0 || c1 < cx);
    const uint64_t reach = __ballot(((float)c1 - (float)c0) * (float)(l + 1) >= 0.75f * n * (float)(l - 1)), across = __ballot(apart >= 0.1f * n);
    return far == 0 && falls == 0 && __popcll(half) >= 48 && __popcll(reach) >= 44 && __popcll(across) >= 44;
}
constexpr int sweep_batch(int slots) { return slots == 20 ? 5 : slots == 12 ? 6 : slots == 4 ? 4 : 8; }

// A group of L = 2^LOGL lanes, 16 bytes a lane, spans a tile of a row of B; the wave's NG groups have `rows` rows of C each, in S
// slots of registers (a slot is an array element by a constant: registers indexed at run time gave wrong sums where an indexed
// write is followed closely by an indexed read).  Lane j of a group knows where its slot j is in the row of A, which the wave has
// staged in LDS.  A step is a window: slots whose next element lies in it fetch a row of B, one element a slot and step, so
// that loads and sums need no more than a broadcast of slot j's column and value over the group; a slot that has several elements
// in a window is late for a step or two.  What bounds it: a step costs a slot ~10 instructions whether it has an element or not,
// and a load 16 cycles of a compute unit's L1 where all lanes take part, none where none does - slots without an element are
// masked out, not sent past a buffer's end (119 us against 157 for the first example above) -; and lines past the L2s for what
// waves are apart.  Batches of G slots, all loads of a batch ahead of its sums.
// LONG: rows of more than 32 elements are two or four sums of a stretch each (rows >> 8 says how many), S / 2 or S / 4 slots apart, so that
// most steps have nothing to do for the batches of one stretch or the other.  A variant of its own: the usual one's registers are
// given out otherwise as soon as it knows of stretches (260 columns fp32, 100001 rows of 10 180 -> 213 us).
//
// ASK: the call does not know its columns (above).  Rows longer than ask.longest are left to the merge kernel.
template <typename T, int LOGL, int S, bool ASK, bool LONG>
__global__ __launch_bounds__(kBlock, 4) void k_spmm_sweep(
    SweepAsk ask, int32_t m, int32_t nnz, int32_t rows, int32_t cap, uint32_t width, uint32_t last, int32_t ncols, T alpha, const int32_t *__restrict__ row_ptr,
    const int32_t *__restrict__ col, const T *__restrict__ val, const T *__restrict__ B, int64_t ldb, T beta, T *__restrict__ C, int64_t ldc)
{
    typedef typename Vec16<T>::type V;
    constexpr int VEC = Vec16<T>::N, L = 1 << LOGL, NG = kWave / L, G = sweep_batch(S);
    static_assert(S <= L && S % G == 0, "a lane knows where one row of its group is");
    extern __shared__ __align__(16) char s_all[];
    const int32_t chains = LONG ? rows >> 8 : 1;
    if (LONG) rows &= 255;
    const int lane = threadIdx.x & (kWave - 1);
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const uint32_t per_xcd = gridDim.x / kXcds;
    const int64_t wave = ((int64_t)(blockIdx.x % kXcds) * per_xcd + blockIdx.x / kXcds) * (kBlock / kWave) + w;
    const int64_t x0 = wave * rows * NG;
    if (!ASK && x0 >= m) return;
    const int32_t nrow = (int32_t)(x0 >= m ? 0 : m - x0 < rows * NG ? m - x0 : rows * NG);
    const int grp = lane >> LOGL, gl = lane & (L - 1);
    const int32_t t0 = (int32_t)((int64_t)blockIdx.y * ncols / gridDim.y), t1 = (int32_t)((int64_t)(blockIdx.y + 1) * ncols / gridDim.y);
    int32_t c = t0 + gl * VEC;
    const bool active = c < t1;
    c = c < t1 - VEC ? c : t1 - VEC;
    uint32_t *s_col = (uint32_t *)(s_all + (size_t)w * cap * (sizeof(T) + 4) + (size_t)cap * sizeof(T));
    T *s_val = (T *)(s_all + (size_t)w * cap * (sizeof(T) + 4));
    const char *Bc = (const char *)(B + c);
    const uint32_t pitch = (uint32_t)((uint64_t)ldb * sizeof(T));

    // the lane's row, or its part of one: element s up to e
    const int32_t apart = chains == 2 ? S / 2 : S / 4, part = LONG ? (gl >= apart) + (gl >= 2 * apart) + (gl >= 3 * apart) : 0;
    const int32_t mine = grp * rows + gl - (LONG ? part * apart : 0);
    bool has_row = (LONG ? gl - part * apart : gl) < rows && mine < nrow;
    if (LONG) has_row = has_row && part < chains;
    int32_t s = has_row ? row_ptr[x0 + mine] : 0, e = has_row ? row_ptr[x0 + mine + 1] : 0;
    if constexpr (ASK) {
        __shared__ int s_yes, s_long[kBlock / kWave];
        const bool too_long = e - s > ask.longest;
        const bool some = __ballot(too_long) != 0;
        if (lane == 0) s_long[w] = some;
        if (w == 0) {
            const bool yes = sweep_suits(ask, m, nnz, lane, row_ptr, col);
            if (lane == 0) s_yes = yes;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            int any = 0;
            for (int i = 0; i < kBlock / kWave; ++i) any |= s_long[i];
            ask.too_long[blockIdx.x] = (uint8_t)any;
            if (blockIdx.x == 0) *ask.answer = s_yes;
        }
        if (!s_yes || x0 >= m) return;
        if (too_long) has_row = false, s = e = 0;
    }
    const uint64_t kept = __ballot(LONG ? has_row && part == 0 : has_row);
    if constexpr (LONG) {
        if (e - s > spmm_dealt(4)) {  // several sums, of a stretch each
            const int32_t share = (e - s + chains - 1) / chains;
            s = s + part * share < e ? s + part * share : e;
            e = s + share < e ? s + share : e;
        } else if (part > 0) {
            s = e;
        }
    }
    const int32_t begin = __builtin_amdgcn_readfirstlane(row_ptr[x0]), end = __builtin_amdgcn_readfirstlane(row_ptr[x0 + nrow]);

    V acc[S];
#pragma unroll
    for (int j = 0; j < S; ++j) acc[j] = T(0);
    for (int32_t from = begin; from < end;) {  // once, unless rows are longer than usual
        const int32_t nel = end - from < cap ? end - from : cap;
        for (int i0 = 0; i0 < nel; i0 += 4 * kWave) {
            int32_t tc[4];
            T tv[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int i = i0 + j * kWave + lane;
                const int64_t k = (int64_t)from + (i < nel ? i : nel - 1);
                tc[j] = __builtin_nontemporal_load(col + k);
                tv[j] = __builtin_nontemporal_load(val + k);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int i = i0 + j * kWave + lane;
                if (i < nel) s_col[i] = (uint32_t)tc[j] & ~kAllColumns, s_val[i] = tv[j];  // 31 bits: every column comes up in a window
            }
        }
        // the staged data is private to this wave: order its LDS writes before its LDS reads
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        int32_t p = s < from ? 0 : s - from < nel ? s - from : nel;
        const int32_t pe = e < from ? 0 : e - from < nel ? e - from : nel;
        uint32_t next = p < pe ? s_col[p] : kNoColumn;
        T a_next = p < pe ? s_val[p] : T(0);
        uint32_t wend = width;
        bool more;
        do {
            const bool go = next < wend;
            wend = wend < last ? wend + width : kAllColumns;
            const uint32_t at = go ? next : kNoColumn;
            const T a = go ? a_next : T(0);
            p += go ? 1 : 0;
            if (go) next = kNoColumn;
            more = __ballot(p < pe) != 0;
            const uint64_t now = __ballot(go);
            if (now == 0) continue;
            if (go && p < pe) next = s_col[p], a_next = s_val[p];
            static_for<0, S / G>([&](auto g_) {
                constexpr int j0 = decltype(g_)::value * G;
                if ((now & lanes_of_groups(L, j0, G)) == 0) return;
                V b[G];
                uint32_t o[G];
                __builtin_amdgcn_sched_barrier(0);
                static_for<0, G>([&](auto u_) { o[decltype(u_)::value] = group_lane<LOGL, j0 + decltype(u_)::value>(at); });
                static_for<0, G>([&](auto u_) {
                    constexpr int u = decltype(u_)::value;
                    b[u] = T(0);
                    if (o[u] != kNoColumn) b[u] = *(const V *)(Bc + (uint64_t)o[u] * pitch);
                });
                __builtin_amdgcn_sched_barrier(0);
                static_for<0, G>([&](auto u_) {
                    constexpr int u = decltype(u_)::value;
                    V t = __builtin_elementwise_fma((V)group_lane<LOGL, j0 + u>(a), b[u], acc[j0 + u]);
                    static_for<0, VEC>([&](auto v_) {  // keeps the sum here: left alone, all of a step's move behind its last load
                        T x = t[decltype(v_)::value];
                        asm volatile("" : "+v"(x));
                        acc[j0 + u][decltype(v_)::value] = x;
                    });
                });
                __builtin_amdgcn_sched_barrier(0);
            });
        } while (more);
        from += nel;
        if (from < end) {
            __builtin_amdgcn_wave_barrier();
            if constexpr (ASK) {  // past rows that are left out
                int32_t at = e > from ? (s > from ? s : from) : end;
#pragma unroll
                for (int d = 1; d < kWave; d <<= 1) {
                    const int32_t other = __shfl_xor(at, d, kWave);
                    at = other < at ? other : at;
                }
                from = __builtin_amdgcn_readfirstlane(at);
            }
        }
    }
    if constexpr (LONG) {
        static_for<0, S / 2>([&](auto j_) { acc[decltype(j_)::value] += acc[decltype(j_)::value + S / 2]; });
        if (chains > 2) static_for<0, S / 4>([&](auto j_) { acc[decltype(j_)::value] += acc[decltype(j_)::value + S / 4]; });
    }
    static_for<0, S / G>([&](auto g_) {
        constexpr int j0 = decltype(g_)::value * G;
        V c_old[G];
        static_for<0, G>([&](auto u_) {
            constexpr int j = j0 + decltype(u_)::value;
            c_old[decltype(u_)::value] = T(0);
            if (beta != T(0) && (kept >> (grp * L + j) & 1))
                c_old[decltype(u_)::value] = *(const V *)(C + (x0 + grp * rows + j) * ldc + c);
        });
        static_for<0, G>([&](auto u_) {
            constexpr int j = j0 + decltype(u_)::value;
            const V y = beta == T(0) ? (V)(alpha * acc[j]) : __builtin_elementwise_fma((V)alpha, acc[j], (V)(beta * c_old[decltype(u_)::value]));
            if (active && (kept >> (grp * L + j) & 1)) *(V *)(C + (x0 + grp * rows + j) * ldc + c) = y;
        });
    });
}

template <typename T, bool ASK>
static int launch_sweep(const SpmmSweep &sw, const SweepAsk &ask, int32_t m, int32_t n, int32_t nnz, int32_t ncols, T alpha, const int32_t *row_ptr,
                        const int32_t *col, const T *val, const T *B, int64_t ldb, T beta, T *C, int64_t ldc, hipStream_t s)
{
    const dim3 grid((unsigned)spmm_sweep_blocks(sw, m), (unsigned)sw.tiles);
    const int32_t cap = ASK ? std::min(sw.cap, spmm_sweep_cap(sizeof(T)) - 2) : sw.cap;  // asking takes 20 bytes of LDS, 32 ahead of the aligned rest
    const size_t lds = (size_t)cap * (sizeof(T) + 4) * (kBlock / kWave);
    const uint32_t last = (uint32_t)n > sw.width ? (uint32_t)n - sw.width : 0;
#define ASX_SWEEP(LOGL, S)                                                                                                              \
    if (sw.log_lanes == LOGL && sw.slots == S) {                                                                                        \
        if constexpr (LOGL >= 4)                                                                                                        \
            if (sw.chains > 1) {                                                                                                        \
                hipLaunchKernelGGL((k_spmm_sweep<T, LOGL, S, ASK, true>), grid, dim3(kBlock), lds, s, ask, m, nnz, sw.rows | sw.chains << 8, cap, \
                                   sw.width, last, ncols, alpha, row_ptr, col, val, B, ldb, beta, C, ldc);                              \
                return check_launch();                                                                                                  \
            }                                                                                                                           \
        hipLaunchKernelGGL((k_spmm_sweep<T, LOGL, S, ASK, false>), grid, dim3(kBlock), lds, s, ask, m, nnz, sw.rows, cap, sw.width, last,      \
                           ncols, alpha, row_ptr, col, val, B, ldb, beta, C, ldc);                                                      \
        return check_launch();                                                                                                          \
    }
    ASX_SWEEP(3, 4)
    ASX_SWEEP(3, 8)
    ASX_SWEEP(4, 4)
    ASX_SWEEP(4, 8)
    ASX_SWEEP(4, 12)
    ASX_SWEEP(4, 16)
    ASX_SWEEP(5, 4)
    ASX_SWEEP(5, 8)
    ASX_SWEEP(5, 12)
    ASX_SWEEP(5, 16)
    ASX_SWEEP(5, 20)
    ASX_SWEEP(6, 4)
    ASX_SWEEP(6, 8)
    ASX_SWEEP(6, 12)
    ASX_SWEEP(6, 16)
    ASX_SWEEP(6, 20)
#undef ASX_SWEEP
    return ASX_STATUS_INTERNAL_ERROR;
}

template <typename T>
int launch_spmm_sweep(const SpmmSweep &sw, const SweepAsk *ask, int32_t m, int32_t n, int32_t nnz, int32_t ncols, T alpha, const int32_t *row_ptr,
                      const int32_t *col, const T *val, const T *B, int64_t ldb, T beta, T *C, int64_t ldc, hipStream_t s)
{
    if (ask) return launch_sweep<T, true>(sw, *ask, m, n, nnz, ncols, alpha, row_ptr, col, val, B, ldb, beta, C, ldc, s);
    return launch_sweep<T, false>(sw, SweepAsk{}, m, n, nnz, ncols, alpha, row_ptr, col, val, B, ldb, beta, C, ldc, s);
}

#define ASX_INST(T)                                                                                                                      \
    template int launch_spmm_sweep<T>(const SpmmSweep &, const SweepAsk *, int32_t, int32_t, int32_t, int32_t, T, const int32_t *,       \
                                      const int32_t *, const T *, const T *, int64_t, T, T *, int64_t, hipStream_t);
ASX_INST(float)
ASX_INST(double)
#undef ASX_INST

}  // namespace asx
