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

// Launch shape of the row-wise kernels: a thread works on one row of a few
// columns, so that a row's index or diagonal entry is read once for them, their
// loads are all in flight together, and no element needs a division to find its
// row (a flat grid-stride loop over n k elements did: 64-bit, ~40 instructions).
constexpr int kElemCols = 8;
// Workgroups per grid dimension: a dimension of a launch has less than 2^32
// threads (and y at most 65535 workgroups); the kernels stride over the rest.
constexpr int64_t kElemGridX = int64_t(1) << 22;
static inline dim3 row_grid(int64_t n, int64_t k, unsigned *threads) {
    *threads = n >= 256 ? 256u : unsigned(ceil_div(n, 64) * 64);
    const int64_t gx = ceil_div(n, *threads), gy = ceil_div(k, kElemCols);
    return dim3(unsigned(std::min(gx, kElemGridX)), unsigned(std::min<int64_t>(gy, 65535)));
}

// f(row, first column, columns) for this thread's rows and column groups, with a
// full group's count as a constant.
template <typename F> __device__ __forceinline__ void each_group(int64_t n, int64_t k, F f) {
    for (int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; i < n;
         i += int64_t(gridDim.x) * blockDim.x)
        for (int64_t j = blockIdx.y * int64_t(kElemCols); j < k;
             j += int64_t(gridDim.y) * kElemCols) {
            if (j + kElemCols <= k) f(i, j, kElemCols);
            else f(i, j, int(k - j));
        }
}

// y[i, j] = x[i, j] * d[i] (or conj(d[i])), column-major n x k
template <typename S>
__global__ void diag_kernel(const S *__restrict__ d, const S *__restrict__ x, int64_t ldx,
                            S *__restrict__ y, int64_t ldy, int64_t n, int64_t k, int conj_d) {
    each_group(n, k, [&](int64_t i, int64_t j0, int cols) {
        const S di = d[i];
        S v[kElemCols];
#pragma unroll
        for (int c = 0; c < kElemCols; ++c)
            if (c < cols) v[c] = x[(j0 + c) * ldx + i];
#pragma unroll
        for (int c = 0; c < kElemCols; ++c)
            if (c < cols)
                y[(j0 + c) * ldy + i] =
                    conj_d ? ElemOps<S>::mulc(v[c], di) : ElemOps<S>::mul(v[c], di);
    });
}

// y[i, j] = x[idx[i], j]; rows with idx[i] < 0 are zero (EXPAND).  The reads of
// one column hit its cache lines in any order, so a column's tiles run together
// and on one XCD: its lines then come from HBM once, into one L2, not once per
// XCD (70001 of 2^18 rows x 32 complex64: 36 us with columns spread over all
// XCDs, 39 us with eight columns per thread).  A tile is 1024 rows of one column.
constexpr int kGatherRows = 4;
template <typename S, bool EXPAND>
__global__ __launch_bounds__(256) void gather_kernel(const int64_t *__restrict__ idx,
                                                     const S *__restrict__ x, int64_t ldx,
                                                     S *__restrict__ y, int64_t ldy, int64_t n_out,
                                                     int64_t row_tiles, int64_t tiles) {
    for (int64_t tile = xcd_remap(blockIdx.x, gridDim.x); tile < tiles; tile += gridDim.x) {
        // (tile indices below 2^32, all but a few, divide as such)
        const int64_t col = tile >> 32 ? tile / row_tiles : unsigned(tile) / unsigned(row_tiles);
        const int64_t i0 = (tile - col * row_tiles) * int64_t(256 * kGatherRows) + threadIdx.x;
        const S *xc = x + col * ldx;
        S *yc = y + col * ldy;
        int64_t r[kGatherRows];
#pragma unroll
        for (int e = 0; e < kGatherRows; ++e)
            r[e] = i0 + e * 256 < n_out ? idx[i0 + e * 256] : -1;
        S v[kGatherRows] = {};
#pragma unroll
        for (int e = 0; e < kGatherRows; ++e)
            if (r[e] >= 0) v[e] = xc[r[e]];
#pragma unroll
        for (int e = 0; e < kGatherRows; ++e)
            if (EXPAND ? i0 + e * 256 < n_out : r[e] >= 0) yc[i0 + e * 256] = v[e];
    }
}

template <typename S>
__global__ void zero_kernel(S *__restrict__ y, int64_t ldy, int64_t n, int64_t k) {
    each_group(n, k, [&](int64_t i, int64_t j0, int cols) {
#pragma unroll
        for (int c = 0; c < kElemCols; ++c)
            if (c < cols) y[(j0 + c) * ldy + i] = S{};
    });
}

template <typename S>
__global__ void scatter_kernel(const int64_t *__restrict__ idx, const S *__restrict__ x,
                               int64_t ldx, S *__restrict__ y, int64_t ldy, int64_t n_in,
                               int64_t k) {
    each_group(n_in, k, [&](int64_t i, int64_t j0, int cols) {
        const int64_t r = idx[i];
        S v[kElemCols];
#pragma unroll
        for (int c = 0; c < kElemCols; ++c)
            if (c < cols) v[c] = x[(j0 + c) * ldx + i];
#pragma unroll
        for (int c = 0; c < kElemCols; ++c)
            if (c < cols) y[(j0 + c) * ldy + r] = v[c];
    });
}

template <typename S>
__global__ void axpby_kernel(S alpha, const S *x, int64_t ldx, int conj_x, S beta, int use_beta,
                             S *y, int64_t ldy, int64_t n, int64_t k) {
    each_group(n, k, [&](int64_t i, int64_t j0, int cols) {
        S v[kElemCols], w[kElemCols];
#pragma unroll
        for (int c = 0; c < kElemCols; ++c)
            if (c < cols) {
                v[c] = x[(j0 + c) * ldx + i];
                if (use_beta) w[c] = y[(j0 + c) * ldy + i];
            }
#pragma unroll
        for (int c = 0; c < kElemCols; ++c)
            if (c < cols) {
                S t = v[c];
                if (conj_x) t = ElemOps<S>::conjv(t);
                t = ElemOps<S>::mul(alpha, t);
                if (use_beta) t = ElemOps<S>::add(t, ElemOps<S>::mul(beta, w[c]));
                y[(j0 + c) * ldy + i] = t;
            }
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
// float32 3072 x 1024 8 us against 17.
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
    constexpr int64_t rows = kElemGridX * TR, cols = 65535 * int64_t(TC);
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
    unsigned nt;
    const dim3 grid = row_grid(n, k, &nt);
    hipLaunchKernelGGL(diag_kernel<S>, grid, dim3(nt), 0, s, (const S *)d, (const S *)x,
                       ldx, (S *)y, ldy, n, k, conj_d);
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
    const int64_t row_tiles = ceil_div(n_out, 256 * kGatherRows), tiles = row_tiles * k;
    hipLaunchKernelGGL((gather_kernel<S, EXPAND>), dim3(unsigned(std::min(tiles, kElemGridX))),
                       dim3(256), 0, s, idx, (const S *)x, ldx, (S *)y, ldy, n_out, row_tiles,
                       tiles);
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
    unsigned nt;
    const dim3 zgrid = row_grid(n_out, k, &nt);
    hipLaunchKernelGGL(zero_kernel<S>, zgrid, dim3(nt), 0, s, (S *)y, ldy, n_out, k);
    if (n_in > 0) {
        const dim3 grid = row_grid(n_in, k, &nt);
        hipLaunchKernelGGL(scatter_kernel<S>, grid, dim3(nt), 0, s, idx, (const S *)x, ldx,
                           (S *)y, ldy, n_in, k);
    }
    FM_CHECK_LAUNCH();
    // zero fill and scatter together: every output row written, every input
    // row and index read
    prof_elem(s, &tok, "scatter_rows", sizeof(S),
              (double(n_in) + double(n_out)) * double(k) * sizeof(S) + 8.0 * double(n_in));
    return FM_SUCCESS;
}

template <typename S>
static fm_status axpby_t(int64_t n, int64_t k, const double *alpha, const void *x, int64_t ldx,
                         int conj_x, const double *beta, void *y, int64_t ldy, hipStream_t s) {
    const int use_beta = (beta[0] != 0.0 || beta[1] != 0.0) ? 1 : 0;
    ProfToken tok;
    prof_begin(s, &tok);
    unsigned nt;
    const dim3 grid = row_grid(n, k, &nt);
    hipLaunchKernelGGL(axpby_kernel<S>, grid, dim3(nt), 0, s, ElemOps<S>::from(alpha),
                       (const S *)x, ldx, conj_x, ElemOps<S>::from(beta), use_beta, (S *)y, ldy,
                       n, k);
    FM_CHECK_LAUNCH();
    prof_elem(s, &tok, "axpby_kernel", sizeof(S),
              (2.0 + use_beta) * double(n) * double(k) * sizeof(S));
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
    case 16: return transpose_t<cpx<double>>(n, k, src, ld_src, dst, ld_dst, s);
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
    FM_DISPATCH_ALL(dtype, gather_t, n_out, idx, x, ldx, y, ldy, k, as_stream(stream));
}

extern "C" fm_status fm_expand_rows(int dtype, int64_t n_out, const int64_t *src, const void *x,
                                    int64_t ldx, void *y, int64_t ldy, int64_t k, void *stream) {
    FM_REQUIRE(n_out >= 0 && k >= 0, FM_ERR_VALUE, "negative size");
    if (n_out == 0 || k == 0) return FM_SUCCESS;
    FM_REQUIRE(src && x && y, FM_ERR_VALUE, "NULL data pointer");
    FM_REQUIRE(ldy >= n_out, FM_ERR_VALUE, "leading dimension below n_out");
    FM_DISPATCH_ALL(dtype, expand_t, n_out, src, x, ldx, y, ldy, k, as_stream(stream));
}

extern "C" fm_status fm_scatter_rows(int dtype, int64_t n_in, const int64_t *idx, const void *x,
                                     int64_t ldx, void *y, int64_t ldy, int64_t n_out, int64_t k,
                                     void *stream) {
    FM_REQUIRE(n_in >= 0 && n_out >= 0 && k >= 0, FM_ERR_VALUE, "negative size");
    if (n_out == 0 || k == 0) return FM_SUCCESS;
    FM_REQUIRE(x && y && (idx || n_in == 0), FM_ERR_VALUE, "NULL data pointer");
    FM_REQUIRE(ldy >= n_out && ldx >= n_in, FM_ERR_VALUE, "leading dimension too small");
    FM_DISPATCH_ALL(dtype, scatter_t, n_in, idx, x, ldx, y, ldy, n_out, k, as_stream(stream));
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
