// Element-wise operators of the hot path: Diag multiply, row gather/scatter
// (Permutation, Partial) and scaled accumulation (Sum, Product scalars).
//
// Reference behaviour replaced:
//   Diag._forwardC / _backwardC + cmath._multiply   Diag.pyx:149-167, cmath.pyx:1294-1326
//   Permutation._forward / _backward                Permutation.pyx:121-125
//   Partial._forward / _backward (scatter/gather)   Partial.pyx:268-294
//   Sum._forwardC / _backwardC                      Sum.pyx:151-175
//   Product scalar factor                           Product.pyx:213-238
// Integer types use wrap-around (two's-complement) arithmetic like the
// reference's C loops.  All kernels work on n x k blocks of column-major data and
// stream HBM once.
#include <algorithm>
#include <type_traits>

#include "fm_common.hpp"

namespace fm {

template <typename S> struct ElemOps {
    using U = S;
    __device__ static S mul(S a, S b) { return a * b; }
    __device__ static S mulc(S a, S b) { return a * b; }  // real: conj(b) == b
    __device__ static S add(S a, S b) { return a + b; }
    __device__ static S conjv(S a) { return a; }
    __host__ static S from(const double *v) { return S(v[0]); }
};
template <typename I> struct IntOps {
    using U = typename std::make_unsigned<I>::type;
    __device__ static I mul(I a, I b) { return I(U(U(a) * U(b))); }
    __device__ static I mulc(I a, I b) { return mul(a, b); }
    __device__ static I add(I a, I b) { return I(U(U(a) + U(b))); }
    __device__ static I conjv(I a) { return a; }
    __host__ static I from(const double *v) { return I(int64_t(v[0])); }
};
template <> struct ElemOps<int8_t> : IntOps<int8_t> {};
template <> struct ElemOps<int16_t> : IntOps<int16_t> {};
template <> struct ElemOps<int32_t> : IntOps<int32_t> {};
template <> struct ElemOps<int64_t> : IntOps<int64_t> {};
template <typename T> struct ElemOps<cpx<T>> {
    __device__ static cpx<T> mul(cpx<T> a, cpx<T> b) { return cmul(a, b); }
    __device__ static cpx<T> mulc(cpx<T> a, cpx<T> b) { return cmulc(a, b); }
    __device__ static cpx<T> add(cpx<T> a, cpx<T> b) { return a + b; }
    __device__ static cpx<T> conjv(cpx<T> a) { return conj(a); }
    __host__ static cpx<T> from(const double *v) { return mk(T(v[0]), T(v[1])); }
};

// Row-wise kernels: the n k elements of a launch in order, E of them a thread, 256
// apart, so that a wave's accesses are contiguous, a thread's loads are all in flight
// together and no lane idles whatever n and k are.  The column of element t is
// floor(t / n), a multiplication by n's reciprocal.  Bound by HBM, and by the launch
// below some 8 MB.  Measured in us against a thread per row of eight columns, which
// leaves most lanes without a row below 64 rows and most columns empty below eight
// (and a gather by tiles of 1024 rows of one column), and against a flat loop with a
// 64-bit division per element:
//   Diag    float32     4 x 2^20    61 /  8.5 ->   6.5     2^24 x 1    211 /  34 ->  32
//           complex64  10^6 x 64   208 /  234 -> 194     2^20 x 16    62 /  44 ->  46
//           complex128  4 x 2^20    74 /   21 ->  20     2^18 x 32    50 /  39 ->  38
//   gather  float32     4 x 2^20   742 /  9.0 ->   7.2   10^6 x 64   404 / 917 -> 404
//           complex64   4 x 2^20   738 / 13.5 ->  12.4    2^18 x 32   48 /  73 ->  46
//           complex128  4 x 2^20   925 /   20 ->  20     2^18 x 32    96 / 108 ->  75
// Slower than that loop: Diag on 3 x 5 10^7 int8 190 (175) and int16 247 (205), a third
// of 2^20 x 16 float32 rows in order 20.7 (16.9).
constexpr int kElemThreads = 256;
struct Rows {
    uint32_t total, n, mul, shift;
    // column of element t < 2^31: for s = ceil(log2 n) and m = 2^32 (2^s / n - 1)
    // rounded up, floor((t + floor(t m / 2^32)) / 2^s) = floor(t / n) (Granlund and
    // Montgomery, "Division by invariant integers using multiplication")
    __device__ __forceinline__ uint32_t column(uint32_t t) const {
        return (__umulhi(t, mul) + t) >> shift;
    }
};

// f(row, column) of this thread's elements e, where there is one.
template <int E, typename F>
__device__ __forceinline__ void each_element(const Rows &r, int64_t block, F f) {
    const uint32_t t0 = uint32_t(block) * (kElemThreads * E) + threadIdx.x;
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const uint32_t t = t0 + e * kElemThreads, j = r.column(t);
        if (t < r.total) f(e, t - j * r.n, j);
    }
}

// Elements per thread: four of up to 8 bytes, from the size on where that leaves every
// CU four workgroups.
constexpr uint32_t kElemMany = 1u << 20;
template <typename S> constexpr int elem_each() { return sizeof(S) <= 8 ? 4 : 1; }

// Launches of a row-wise kernel on n x k elements, of at most 2^30 each (one as a
// rule): launch(elements per thread, rows, grid, first row, first column).
template <int E, typename F> static void launch_rows(int64_t n, int64_t k, F launch) {
    constexpr int64_t part = int64_t(1) << 30;
    const int64_t rows = std::min(n, part), cols = std::max<int64_t>(1, part / rows);
    for (int64_t j = 0; j < k; j += cols)
        for (int64_t i = 0; i < n; i += rows) {
            const uint64_t nn = std::min(n - i, rows), kk = std::min(k - j, cols);
            Rows r;
            r.total = uint32_t(nn * kk);
            r.n = uint32_t(nn);
            r.shift = 0;
            while ((uint64_t(1) << r.shift) < nn) ++r.shift;
            r.mul = uint32_t((((uint64_t(1) << r.shift) - nn) << 32) / nn + 1);
            if (r.total >= kElemMany)
                launch(std::integral_constant<int, E>(), r,
                       dim3(ceil_div(r.total, E * kElemThreads)), i, j);
            else
                launch(std::integral_constant<int, 1>(), r, dim3(ceil_div(r.total, kElemThreads)),
                       i, j);
        }
}

// y[i, j] = x[i, j] * d[i] (or conj(d[i])), column-major n x k
template <typename S, int E>
__global__ __launch_bounds__(kElemThreads) void diag_kernel(const Rows r, const S *__restrict__ d,
                                                            const S *__restrict__ x, int64_t ldx,
                                                            S *__restrict__ y, int64_t ldy,
                                                            int conj_d) {
    S v[E], w[E];
    each_element<E>(r, blockIdx.x, [&](int e, uint32_t i, uint32_t j) {
        v[e] = x[j * ldx + i];
        w[e] = d[i];
    });
    each_element<E>(r, blockIdx.x, [&](int e, uint32_t i, uint32_t j) {
        y[j * ldy + i] = conj_d ? ElemOps<S>::mulc(v[e], w[e]) : ElemOps<S>::mul(v[e], w[e]);
    });
}

// The kernels that only move elements take them as bytes of their size (a conditional
// copy of a complex128 object goes through LDS, 13 us a launch for it).
typedef uint32_t Bytes16 __attribute__((ext_vector_type(4)));
#define FM_DISPATCH_SIZE(dtype, FN, ...)                                                \
    switch (dtype) {                                                                  \
    case FM_INT8: return FN<uint8_t>(__VA_ARGS__);                                    \
    case FM_INT16: return FN<uint16_t>(__VA_ARGS__);                                  \
    case FM_INT32:                                                                    \
    case FM_FLOAT32: return FN<uint32_t>(__VA_ARGS__);                                \
    case FM_INT64:                                                                    \
    case FM_FLOAT64:                                                                  \
    case FM_COMPLEX64: return FN<uint64_t>(__VA_ARGS__);                              \
    case FM_COMPLEX128: return FN<Bytes16>(__VA_ARGS__);                              \
    default: set_error("Unsupported type: %d", dtype); return FM_ERR_TYPE;            \
    }

// y[i, j] = x[idx[i], j]; rows with idx[i] < 0 are zero (EXPAND).  The reads of
// one column hit its cache lines in any order, so neighbouring workgroups run on one
// XCD: a column's lines then come from HBM once, into one L2, not once per XCD (a
// third of 2^18 rows x 32 complex64 in any order: 20.5 us, 40 with columns spread over
// all XCDs).
template <typename S, bool EXPAND, int E>
__global__ __launch_bounds__(kElemThreads) void gather_kernel(const Rows r,
                                                              const int64_t *__restrict__ idx,
                                                              const S *__restrict__ x, int64_t ldx,
                                                              S *__restrict__ y, int64_t ldy) {
    const int64_t block = xcd_remap(blockIdx.x, gridDim.x);
    int64_t at[E];
    S v[E];
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = S(0);
    each_element<E>(r, block, [&](int e, uint32_t i, uint32_t) { at[e] = idx[i]; });
    each_element<E>(r, block, [&](int e, uint32_t, uint32_t j) {
        if (at[e] >= 0) v[e] = x[j * ldx + at[e]];
    });
    each_element<E>(r, block, [&](int e, uint32_t i, uint32_t j) {
        if (EXPAND || at[e] >= 0) y[j * ldy + i] = v[e];
    });
}

template <typename S, int E>
__global__ __launch_bounds__(kElemThreads) void zero_kernel(const Rows r, S *__restrict__ y,
                                                            int64_t ldy) {
    each_element<E>(r, blockIdx.x,
                    [&](int, uint32_t i, uint32_t j) { y[j * ldy + i] = S(0); });
}

template <typename S, int E>
__global__ __launch_bounds__(kElemThreads) void scatter_kernel(const Rows r,
                                                               const int64_t *__restrict__ idx,
                                                               const S *__restrict__ x, int64_t ldx,
                                                               S *__restrict__ y, int64_t ldy) {
    S v[E];
    int64_t at[E];
    each_element<E>(r, blockIdx.x, [&](int e, uint32_t i, uint32_t j) {
        at[e] = idx[i];
        v[e] = x[j * ldx + i];
    });
    each_element<E>(r, blockIdx.x,
                    [&](int e, uint32_t, uint32_t j) { y[j * ldy + at[e]] = v[e]; });
}

// A selection's inverse (fm_invert_index): the entries and the flag before, then the
// selected rows, the largest of equal indices.
template <typename I>
__global__ __launch_bounds__(kElemThreads) void invert_fill_kernel(I *__restrict__ inverse,
                                                                   int64_t n, I *twice) {
    const int64_t i = blockIdx.x * int64_t(kElemThreads) + threadIdx.x;
    if (i < n) inverse[i] = -1;
    if (i == 0) *twice = 0;
}
template <typename I>
__global__ __launch_bounds__(kElemThreads) void invert_kernel(const int64_t *__restrict__ idx,
                                                              int64_t first, int64_t m,
                                                              I *inverse, int64_t n, I *twice) {
    const int64_t i = first + blockIdx.x * int64_t(kElemThreads) + threadIdx.x;
    if (i >= m) return;
    const int64_t r = idx[i];
    if (r >= 0 && r < n && atomicMax(inverse + r, I(i)) >= 0) *twice = 1;
}

// y = alpha x + beta y (BETA: beta is not 0, a constant of the kernel, as the compiler
// got the choice wrong for int8: alpha x + beta y + 1 by v_dot4_u32_u8).
template <typename S, bool BETA, int E>
__global__ __launch_bounds__(kElemThreads) void axpby_kernel(const Rows r, S alpha, const S *x,
                                                             int64_t ldx, int conj_x, S beta,
                                                             S *y, int64_t ldy) {
    S v[E], w[E];
    each_element<E>(r, blockIdx.x, [&](int e, uint32_t i, uint32_t j) {
        v[e] = x[j * ldx + i];
        if (BETA) w[e] = y[j * ldy + i];
    });
    each_element<E>(r, blockIdx.x, [&](int e, uint32_t i, uint32_t j) {
        S t = conj_x ? ElemOps<S>::conjv(v[e]) : v[e];
        t = ElemOps<S>::mul(alpha, t);
        if (BETA) t = ElemOps<S>::add(t, ElemOps<S>::mul(beta, w[e]));
        y[j * ldy + i] = t;
    });
}

// dst[c][i] = src[i][c] for i < n, c < k: rows of k neighbouring elements to
// columns of n (a caller's row-major (n, k) array to the library's blocks).  A
// 256-thread workgroup moves a tile of 2^LOGC columns by 2^(LOGT - LOGC) rows
// through LDS: it reads the rows' k elements side by side (for k <= 2^LOGC the
// whole tile is one contiguous range) and writes runs of rows of each column.
// LDS columns are one element longer than the tile, so that both sides touch
// distinct banks.  Bound by HBM: one read and one write per element; complex64
// 2^18 x 32 (67 MB each way) 26 us, 5.2 TB/s, where torch's strided copy takes 63;
// float32 3072 x 1024 8 us against 17; 16-byte elements 2^18 x 32 46 us (107 as objects
// of cpx<double>, whose copies go through scratch memory).
template <typename S, int LOGT, int LOGC>
__global__ __launch_bounds__(256) void transpose_kernel(const S *__restrict__ src, int64_t lds_,
                                                        S *__restrict__ dst, int64_t ldd,
                                                        int64_t n, int64_t k) {
    constexpr int TC = 1 << LOGC, TR = 1 << (LOGT - LOGC), PER = (1 << LOGT) / 256;
    __shared__ S tile[TC * (TR + 1)];
    const int64_t i0 = blockIdx.x * int64_t(TR), c0 = blockIdx.y * int64_t(TC);
    S v[PER] = {};
#pragma unroll
    for (int e = 0; e < PER; ++e) {
        const int idx = threadIdx.x + e * 256, c = idx & (TC - 1), r = idx >> LOGC;
        if (i0 + r < n && c0 + c < k) v[e] = src[(i0 + r) * lds_ + c0 + c];
    }
#pragma unroll
    for (int e = 0; e < PER; ++e) {
        const int idx = threadIdx.x + e * 256, c = idx & (TC - 1), r = idx >> LOGC;
        tile[c * (TR + 1) + r] = v[e];
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < PER; ++e) {
        const int idx = threadIdx.x + e * 256, r = idx & (TR - 1), c = idx >> (LOGT - LOGC);
        if (i0 + r < n && c0 + c < k) dst[(c0 + c) * ldd + i0 + r] = tile[c * (TR + 1) + r];
    }
}

template <typename S, int LOGC>
static fm_status transpose_launch(int64_t n, int64_t k, const void *src, int64_t lds_, void *dst,
                                  int64_t ldd, hipStream_t s) {
    constexpr int LOGT = sizeof(S) == 16 ? 11 : 12;
    constexpr int TR = 1 << (LOGT - LOGC);
    constexpr int TC = 1 << LOGC;
    ProfToken tok;
    prof_begin(s, &tok);
    // (a launch for what one grid does not take: loops in the kernel would hold its
    // addresses in registers, 256 of them in place of 55)
    constexpr int64_t rows = (int64_t(1) << 22) * TR, cols = 65535 * int64_t(TC);
    for (int64_t i = 0; i < n; i += rows)
        for (int64_t c = 0; c < k; c += cols) {
            const int64_t nn = std::min(n - i, rows), kk = std::min(k - c, cols);
            hipLaunchKernelGGL((transpose_kernel<S, LOGT, LOGC>),
                               dim3(unsigned(ceil_div(nn, TR)), unsigned(ceil_div(kk, TC))),
                               dim3(256), 0, s, (const S *)src + i * lds_ + c, lds_,
                               (S *)dst + c * ldd + i, ldd, nn, kk);
        }
    FM_CHECK_LAUNCH();
    prof_elem(s, &tok, "transpose_kernel", sizeof(S), 2.0 * double(n) * double(k) * sizeof(S));
    return FM_SUCCESS;
}

// Tile width by the row length: at most 32 columns (runs of 128 rows), fewer
// where the rows are shorter, so that lanes do not idle past them.
template <typename S>
static fm_status transpose_t(int64_t n, int64_t k, const void *src, int64_t lds_, void *dst,
                             int64_t ldd, hipStream_t s) {
    if (k <= 2) return transpose_launch<S, 1>(n, k, src, lds_, dst, ldd, s);
    if (k <= 4) return transpose_launch<S, 2>(n, k, src, lds_, dst, ldd, s);
    if (k <= 8) return transpose_launch<S, 3>(n, k, src, lds_, dst, ldd, s);
    if (k <= 16) return transpose_launch<S, 4>(n, k, src, lds_, dst, ldd, s);
    return transpose_launch<S, 5>(n, k, src, lds_, dst, ldd, s);
}

#define FM_DISPATCH_ALL(dtype, FN, ...)                                                 \
    switch (dtype) {                                                                  \
    case FM_INT8: return FN<int8_t>(__VA_ARGS__);                                     \
    case FM_INT16: return FN<int16_t>(__VA_ARGS__);                                   \
    case FM_INT32: return FN<int32_t>(__VA_ARGS__);                                   \
    case FM_INT64: return FN<int64_t>(__VA_ARGS__);                                   \
    case FM_FLOAT32: return FN<float>(__VA_ARGS__);                                   \
    case FM_FLOAT64: return FN<double>(__VA_ARGS__);                                  \
    case FM_COMPLEX64: return FN<cpx<float>>(__VA_ARGS__);                            \
    case FM_COMPLEX128: return FN<cpx<double>>(__VA_ARGS__);                          \
    default: set_error("Unsupported type: %d", dtype); return FM_ERR_TYPE;            \
    }

template <typename S>
static fm_status diag_t(int conj_d, int64_t n, const void *d, const void *x, int64_t ldx,
                        void *y, int64_t ldy, int64_t k, hipStream_t s) {
    ProfToken tok;
    prof_begin(s, &tok);
    launch_rows<elem_each<S>()>(n, k, [&](auto e, const Rows &r, dim3 grid, int64_t i, int64_t j) {
        hipLaunchKernelGGL((diag_kernel<S, decltype(e)::value>), grid, dim3(kElemThreads), 0, s, r,
                           (const S *)d + i, (const S *)x + j * ldx + i, ldx,
                           (S *)y + j * ldy + i, ldy, conj_d);
    });
    FM_CHECK_LAUNCH();
    prof_elem(s, &tok, "diag_kernel", sizeof(S), (2.0 * double(n) * double(k) + double(n)) *
                                                     sizeof(S));
    return FM_SUCCESS;
}

template <typename S, bool EXPAND>
static fm_status gather_any(int64_t n_out, const int64_t *idx, const void *x, int64_t ldx, void *y,
                          int64_t ldy, int64_t k, hipStream_t s) {
    ProfToken tok;
    prof_begin(s, &tok);
    // (8-byte elements one by one: 8 x 2^20 rows in any order 22 us, four a thread 26)
    constexpr int E = sizeof(S) <= 4 ? 4 : 1;
    launch_rows<E>(n_out, k, [&](auto e, const Rows &r, dim3 grid, int64_t i, int64_t j) {
        hipLaunchKernelGGL((gather_kernel<S, EXPAND, decltype(e)::value>), grid,
                           dim3(kElemThreads), 0, s, r, idx + i, (const S *)x + j * ldx, ldx,
                           (S *)y + j * ldy + i, ldy);
    });
    FM_CHECK_LAUNCH();
    prof_elem(s, &tok, EXPAND ? "expand_kernel" : "gather_kernel", sizeof(S),
              2.0 * double(n_out) * double(k) * sizeof(S) + 8.0 * double(n_out));
    return FM_SUCCESS;
}

template <typename S>
static fm_status gather_t(int64_t n_out, const int64_t *idx, const void *x, int64_t ldx, void *y,
                          int64_t ldy, int64_t k, hipStream_t s) {
    return gather_any<S, false>(n_out, idx, x, ldx, y, ldy, k, s);
}
template <typename S>
static fm_status expand_t(int64_t n_out, const int64_t *idx, const void *x, int64_t ldx, void *y,
                          int64_t ldy, int64_t k, hipStream_t s) {
    return gather_any<S, true>(n_out, idx, x, ldx, y, ldy, k, s);
}

template <typename S>
static fm_status scatter_t(int64_t n_in, const int64_t *idx, const void *x, int64_t ldx, void *y,
                           int64_t ldy, int64_t n_out, int64_t k, hipStream_t s) {
    ProfToken tok;
    prof_begin(s, &tok);
    launch_rows<elem_each<S>()>(n_out, k, [&](auto e, const Rows &r, dim3 grid, int64_t i, int64_t j) {
        hipLaunchKernelGGL((zero_kernel<S, decltype(e)::value>), grid, dim3(kElemThreads), 0, s, r,
                           (S *)y + j * ldy + i, ldy);
    });
    if (n_in > 0)
        launch_rows<elem_each<S>()>(n_in, k, [&](auto e, const Rows &r, dim3 grid, int64_t i, int64_t j) {
            hipLaunchKernelGGL((scatter_kernel<S, decltype(e)::value>), grid, dim3(kElemThreads),
                               0, s, r, idx + i, (const S *)x + j * ldx + i, ldx,
                               (S *)y + j * ldy, ldy);
        });
    FM_CHECK_LAUNCH();
    // zero fill and scatter together: every output row written, every input
    // row and index read
    prof_elem(s, &tok, "scatter_rows", sizeof(S),
              (double(n_in) + double(n_out)) * double(k) * sizeof(S) + 8.0 * double(n_in));
    return FM_SUCCESS;
}

template <typename S, bool BETA>
static fm_status axpby_any(int64_t n, int64_t k, const double *alpha, const void *x, int64_t ldx,
                           int conj_x, const double *beta, void *y, int64_t ldy, hipStream_t s) {
    ProfToken tok;
    prof_begin(s, &tok);
    const S a = ElemOps<S>::from(alpha), b = ElemOps<S>::from(beta);
    launch_rows<elem_each<S>()>(n, k, [&](auto e, const Rows &r, dim3 grid, int64_t i, int64_t j) {
        hipLaunchKernelGGL((axpby_kernel<S, BETA, decltype(e)::value>), grid, dim3(kElemThreads),
                           0, s, r, a, (const S *)x + j * ldx + i, ldx, conj_x, b,
                           (S *)y + j * ldy + i, ldy);
    });
    FM_CHECK_LAUNCH();
    prof_elem(s, &tok, "axpby_kernel", sizeof(S),
              (2.0 + BETA) * double(n) * double(k) * sizeof(S));
    return FM_SUCCESS;
}

template <typename S>
static fm_status axpby_t(int64_t n, int64_t k, const double *alpha, const void *x, int64_t ldx,
                         int conj_x, const double *beta, void *y, int64_t ldy, hipStream_t s) {
    if (beta[0] != 0.0 || beta[1] != 0.0)
        return axpby_any<S, true>(n, k, alpha, x, ldx, conj_x, beta, y, ldy, s);
    return axpby_any<S, false>(n, k, alpha, x, ldx, conj_x, beta, y, ldy, s);
}

template <typename I>
static fm_status invert_t(int64_t m, const int64_t *idx, int64_t n, void *inverse, void *twice,
                          hipStream_t s) {
    constexpr int64_t part = int64_t(1) << 30;  // elements per launch
    auto grid = [](int64_t count) {
        return dim3(unsigned(ceil_div(count < part ? count : part, kElemThreads)));
    };
    ProfToken tok;
    prof_begin(s, &tok);
    for (int64_t i = 0; i < n; i += part)
        hipLaunchKernelGGL(invert_fill_kernel<I>, grid(n - i), dim3(kElemThreads), 0, s,
                           (I *)inverse + i, std::min(n - i, part), (I *)twice);
    for (int64_t i = 0; i < m; i += part)
        hipLaunchKernelGGL(invert_kernel<I>, grid(m - i), dim3(kElemThreads), 0, s, idx, i, m,
                           (I *)inverse, n, (I *)twice);
    FM_CHECK_LAUNCH();
    prof_elem(s, &tok, "invert_index", sizeof(I),
              8.0 * double(m) + sizeof(I) * (double(n) + double(m)));
    return FM_SUCCESS;
}

}  // namespace fm

using namespace fm;

extern "C" fm_status fm_diag_apply(int dtype, int conj_d, int64_t n, const void *d, const void *x,
                                   int64_t ldx, void *y, int64_t ldy, int64_t k, void *stream) {
    FM_REQUIRE(n >= 0 && k >= 0, FM_ERR_VALUE, "negative size");
    if (n == 0 || k == 0) return FM_SUCCESS;
    FM_REQUIRE(d && x && y, FM_ERR_VALUE, "NULL data pointer");
    FM_REQUIRE(ldx >= n && ldy >= n, FM_ERR_VALUE, "leading dimension below n");
    FM_DISPATCH_ALL(dtype, diag_t, conj_d, n, d, x, ldx, y, ldy, k, as_stream(stream));
}

extern "C" fm_status fm_transpose(int elem_bytes, int64_t n, int64_t k, const void *src,
                                  int64_t ld_src, void *dst, int64_t ld_dst, void *stream) {
    FM_REQUIRE(n >= 0 && k >= 0, FM_ERR_VALUE, "negative size");
    if (n == 0 || k == 0) return FM_SUCCESS;
    FM_REQUIRE(src && dst && src != dst, FM_ERR_VALUE, "bad data pointers");
    FM_REQUIRE(ld_src >= k && ld_dst >= n, FM_ERR_VALUE, "leading dimension too small");
    hipStream_t s = as_stream(stream);
    switch (elem_bytes) {
    case 1: return transpose_t<uint8_t>(n, k, src, ld_src, dst, ld_dst, s);
    case 2: return transpose_t<uint16_t>(n, k, src, ld_src, dst, ld_dst, s);
    case 4: return transpose_t<uint32_t>(n, k, src, ld_src, dst, ld_dst, s);
    case 8: return transpose_t<uint64_t>(n, k, src, ld_src, dst, ld_dst, s);
    case 16: return transpose_t<Bytes16>(n, k, src, ld_src, dst, ld_dst, s);
    default: break;
    }
    set_error("transpose: unsupported element size %d", elem_bytes);
    return FM_ERR_TYPE;
}

extern "C" fm_status fm_gather_rows(int dtype, int64_t n_out, const int64_t *idx, const void *x,
                                    int64_t ldx, void *y, int64_t ldy, int64_t k, void *stream) {
    FM_REQUIRE(n_out >= 0 && k >= 0, FM_ERR_VALUE, "negative size");
    if (n_out == 0 || k == 0) return FM_SUCCESS;
    FM_REQUIRE(idx && x && y, FM_ERR_VALUE, "NULL data pointer");
    FM_REQUIRE(ldy >= n_out, FM_ERR_VALUE, "leading dimension below n_out");
    FM_DISPATCH_SIZE(dtype, gather_t, n_out, idx, x, ldx, y, ldy, k, as_stream(stream));
}

extern "C" fm_status fm_expand_rows(int dtype, int64_t n_out, const int64_t *src, const void *x,
                                    int64_t ldx, void *y, int64_t ldy, int64_t k, void *stream) {
    FM_REQUIRE(n_out >= 0 && k >= 0, FM_ERR_VALUE, "negative size");
    if (n_out == 0 || k == 0) return FM_SUCCESS;
    FM_REQUIRE(src && x && y, FM_ERR_VALUE, "NULL data pointer");
    FM_REQUIRE(ldy >= n_out, FM_ERR_VALUE, "leading dimension below n_out");
    FM_DISPATCH_SIZE(dtype, expand_t, n_out, src, x, ldx, y, ldy, k, as_stream(stream));
}

extern "C" fm_status fm_invert_index(int elem_bytes, int64_t m, const int64_t *idx, int64_t n,
                                     void *inverse, void *twice, void *stream) {
    FM_REQUIRE(m >= 0 && n >= 1, FM_ERR_VALUE, "sizes out of range");
    FM_REQUIRE((idx || m == 0) && inverse && twice, FM_ERR_VALUE, "NULL data pointer");
    if (elem_bytes == 4) return invert_t<int32_t>(m, idx, n, inverse, twice, as_stream(stream));
    if (elem_bytes == 8) return invert_t<long long>(m, idx, n, inverse, twice, as_stream(stream));
    set_error("index inversion: unsupported element size %d", elem_bytes);
    return FM_ERR_TYPE;
}

extern "C" fm_status fm_scatter_rows(int dtype, int64_t n_in, const int64_t *idx, const void *x,
                                     int64_t ldx, void *y, int64_t ldy, int64_t n_out, int64_t k,
                                     void *stream) {
    FM_REQUIRE(n_in >= 0 && n_out >= 0 && k >= 0, FM_ERR_VALUE, "negative size");
    if (n_out == 0 || k == 0) return FM_SUCCESS;
    FM_REQUIRE(x && y && (idx || n_in == 0), FM_ERR_VALUE, "NULL data pointer");
    FM_REQUIRE(ldy >= n_out && ldx >= n_in, FM_ERR_VALUE, "leading dimension too small");
    FM_DISPATCH_SIZE(dtype, scatter_t, n_in, idx, x, ldx, y, ldy, n_out, k, as_stream(stream));
}

extern "C" fm_status fm_axpby(int dtype, int64_t n, int64_t k, const double *alpha, const void *x,
                              int64_t ldx, int conj_x, const double *beta, void *y, int64_t ldy,
                              void *stream) {
    FM_REQUIRE(n >= 0 && k >= 0, FM_ERR_VALUE, "negative size");
    if (n == 0 || k == 0) return FM_SUCCESS;
    FM_REQUIRE(alpha && beta && x && y, FM_ERR_VALUE, "NULL argument");
    FM_REQUIRE(ldx >= n && ldy >= n, FM_ERR_VALUE, "leading dimension below n");
    FM_DISPATCH_ALL(dtype, axpby_t, n, k, alpha, x, ldx, conj_x, beta, y, ldy, as_stream(stream));
}

namespace fm {
// Plain device copy in 16-byte vectors (grid-strided, four loads in flight
// per thread before their stores), the reference point for HBM bandwidth and
// for scaling the FETCH_SIZE / WRITE_SIZE counters.
__global__ __launch_bounds__(256) void copy16_kernel(const uint4 *__restrict__ src,
                                                      uint4 *__restrict__ dst, int64_t n) {
    constexpr int U = 4;
    const int64_t stride = int64_t(gridDim.x) * blockDim.x;
    int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x;
    for (; i + (U - 1) * stride < n; i += U * stride) {
        uint4 v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = src[i + u * stride];
#pragma unroll
        for (int u = 0; u < U; ++u) dst[i + u * stride] = v[u];
    }
    for (; i < n; i += stride) dst[i] = src[i];
}
}  // namespace fm

extern "C" fm_status fm_device_copy(void *dst, const void *src, int64_t bytes, void *stream) {
    FM_REQUIRE(bytes >= 0, FM_ERR_VALUE, "negative size");
    if (bytes == 0) return FM_SUCCESS;
    FM_REQUIRE(dst && src && (bytes % 16) == 0 && (uintptr_t(dst) % 16) == 0 &&
                   (uintptr_t(src) % 16) == 0,
               FM_ERR_VALUE, "copy needs 16-byte aligned pointers and a multiple of 16 bytes");
    const int64_t n = bytes / 16;
    int ncu = 256;
    int dev = 0;
    if (hipGetDevice(&dev) == hipSuccess)
        (void)hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
    int64_t grid = ceil_div(n, 256);
    if (grid > int64_t(ncu) * 8) grid = int64_t(ncu) * 8;
    ProfToken tok;
    prof_begin(as_stream(stream), &tok);
    hipLaunchKernelGGL(copy16_kernel, dim3(unsigned(grid)), dim3(256), 0, as_stream(stream),
                       (const uint4 *)src, (uint4 *)dst, n);
    FM_CHECK_LAUNCH();
    if (tok.active) prof_end(as_stream(stream), &tok, "copy16_kernel", 2.0 * double(bytes), 0.0);
    return FM_SUCCESS;
}
