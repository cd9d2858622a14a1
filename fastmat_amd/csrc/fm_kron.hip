// The last two factors of a Kron product, a Circulant of N = 64 or 128 points
// and a dense M x M float32 matrix (M = 64, 96 or 128), applied to complex64
// data in one pass over HBM.
//
// Replaces two mode passes of Kron._forward / _backward (Kron.pyx:267-303:
// one factor per mode, each a full read and write of the data) for x viewed as
// (outer, n = N, m = M) with the dense axis contiguous: every N x M slab is
// read, transformed by both factors on the chip and written once.  The factors
// act on different axes, so their order does not matter; the adjoint of
// (Circulant x A) is the conjugate spectrum with A^T, which the caller passes
// as the matrix (A is real).
//
// A workgroup of 4 N / 64 waves computes 64 of a slab's M output columns and
// walks slabs persistently:
//   1. Z[n][i] = sum_j A[i][j] X[n][j] on FP32 MFMA (v_mfma_f32_16x16x4f32).  A
//      wave owns 16 columns i (its rows of A stay in registers for its life)
//      and 64 of the rows n, real and imaginary parts as separate blocks.  X
//      comes in chunks of 16 j through two LDS buffers; a chunk's loads are
//      issued two chunks ahead (the next slab's first ones before this slab's
//      transform).  Which row n an MFMA row stands for is free, and is chosen
//      so that the 16 rows in a lane's accumulators are n0 + r N / 16, r = 0
//      ... 15: the inputs of a radix-16 butterfly.
//   2. The circulant along n, from those registers: radix 16 and N / 16, the
//      spectrum, radix N / 16 and 16 back (Stockham stages as in
//      fm_fft_core.hpp) with two exchanges through LDS.  From the first
//      exchange on a wave's 64 lanes are 64 neighbouring columns i and share
//      the butterfly, so twiddles and spectrum are wave-uniform.
//   3. The last stage stores from registers, 512 contiguous bytes a wave.
// LDS holds the 64 columns once (68 KB for N = 128; the X buffers share it), so
// two workgroups run per CU and the MFMAs of one overlap the butterflies,
// exchanges and stores of the other.  The workgroups of a slab run side by side
// on one XCD, so the slab comes from HBM once.
//
// What bounds it: HBM 16 bytes and the MFMA pipes 4 M flop per complex element
// (52 and 55 us for 2^24 elements at M = 128).  Measured there: 102 us, against
// 189 us for the slab at a time through one workgroup per CU (transform, LDS,
// MFMA and staged store in turn), and 143 us with X loaded straight into MFMA
// registers by every wave (512 KB a workgroup through the L1).
#include <algorithm>

#include "fm_fft_plan.hpp"

namespace fm {

typedef float kp_f32x4 __attribute__((ext_vector_type(4)));
typedef float kp_f32x2u __attribute__((ext_vector_type(2), aligned(4)));
typedef float kp_f32x4u __attribute__((ext_vector_type(4), aligned(8)));

// Element i (wave-uniform) of a table in device memory, through scalar loads.
__device__ __forceinline__ cpx<float> kp_uniform(const cpx<float> *p, int i) {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef const float __attribute__((address_space(4))) CF;
    CF *q = (CF *)(const float *)p + 2 * i;
    return mk(float(q[0]), float(q[1]));
#else
    return p[i];
#endif
}

struct KronPairArgs {
    const cpx<float> *x;
    cpx<float> *y;
    const float *A;          // the dense factor as applied, M x M row-major
    const cpx<float> *D;     // spectrum, N entries
    const cpx<float> *tw;    // W_N^e
    int conj_d;
    int64_t outer;           // slabs
};

template <int LOGN, int M>
__global__ __launch_bounds__(4 << LOGN, 4) void kron_pair_kernel(const KronPairArgs k) {
    constexpr int N = 1 << LOGN, WN = N / 64, NT = 256 * WN;
    constexpr int LOGB = 6, E = 16;
    constexpr int SB = tile_row<float>(LOGN, LOGB);
    constexpr int NR0 = N / 16;                       // radix-16 butterflies
    constexpr int LOGR = LOGN - 4, R = 1 << LOGR;     // the other radix
    constexpr int NB = E / R;                         // its butterflies per thread
    constexpr int C = M / 16;                         // chunks of 16 j
    constexpr int IB = (M + 63) / 64;                 // workgroups per slab
    constexpr int XROW = 9;                           // 16-byte pieces per chunk row (8, padded)
    static_assert(NT == (4 << LOGN) && M % 16 == 0, "shape");
    extern __shared__ __align__(16) unsigned char smem_raw[];
    cpx<float> *lds = reinterpret_cast<cpx<float> *>(smem_raw);
    kp_f32x4 *xbuf = reinterpret_cast<kp_f32x4 *>(smem_raw);  // [2][N][XROW]
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, h = lane >> 4;
    const int wi = wave & 3, wn = wave >> 2;
    // workgroup g of the grid (a multiple of IB) keeps its columns: slabs g / IB,
    // g / IB + grid / IB, ...
    const int64_t g = xcd_remap(blockIdx.x, gridDim.x);
    const int i0 = int(g % IB) * 64;
    const int64_t stride = gridDim.x / IB;
    const bool cols = M % 64 == 0 || i0 + 16 * wi < M;  // the wave has columns

    // A[i][16 c + 8 t + 2 h + s] of column i = i0 + 16 wi + r at a[4 c + 2 t + s]
    float a[4 * C];
    {
        const uint32_t abase = uint32_t(cols ? i0 + 16 * wi + r : 0) * M + 2 * h;
#pragma unroll
        for (int t = 0; t < 2 * C; ++t) {
            const kp_f32x2u w = *reinterpret_cast<const kp_f32x2u *>(k.A + abase + 8 * t);
            a[2 * t] = w.x;
            a[2 * t + 1] = w.y;
        }
    }
    // This thread's two 16-byte pieces of a chunk: piece tid % 8 of rows
    // tid / 8 and tid / 8 + N / 2.  MFMA row m of block f of row group wn is
    // n = (m / 4 + 4 wn) + NR0 (4 f + m % 4), and stands at row 16 (4 wn + f) + m
    // of the buffer.
    uint32_t xoff[2];
    int xpos[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int n = (threadIdx.x >> 3) + q * (N / 2);
        const int n0 = n % NR0, rr = n / NR0;
        const int m = 4 * (n0 & 3) + (rr & 3);
        xpos[q] = (16 * (4 * (n0 >> 2) + (rr >> 2)) + m) * XROW + (threadIdx.x & 7);
        xoff[q] = uint32_t(n) * (8 * M) + 16 * (threadIdx.x & 7);
    }
    kp_f32x4u piece[2];
    auto load = [&](int64_t slab, int c) {
        const char *x = reinterpret_cast<const char *>(k.x + slab * (int64_t(N) * M));
#pragma unroll
        for (int q = 0; q < 2; ++q)
            piece[q] = *reinterpret_cast<const kp_f32x4u *>(x + xoff[q] + 128 * c);
    };
    auto put = [&](int c) {
#pragma unroll
        for (int q = 0; q < 2; ++q) xbuf[(c & 1) * (N * XROW) + xpos[q]] = piece[q];
    };

    int64_t slab = g / IB;
    if (slab < k.outer) load(slab, 0);
    for (; slab < k.outer; slab += stride) {
        kp_f32x4 re[4], im[4];
#pragma unroll
        for (int f = 0; f < 4; ++f) re[f] = im[f] = kp_f32x4{0.f, 0.f, 0.f, 0.f};
        put(0);
        load(slab, 1);
        __syncthreads();
#pragma unroll
        for (int c = 0; c < C; ++c) {
            // buffer c + 1 was last read in chunk c - 1, before a barrier
            if (c + 1 < C) put(c + 1);
            if (c + 2 < C) load(slab, c + 2);
            else if (c + 2 == C && slab + stride < k.outer) load(slab + stride, 0);
            if (cols) {
                const kp_f32x4 *xp = xbuf + (c & 1) * (N * XROW) + (64 * wn + r) * XROW + h;
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    kp_f32x4 w[4];
#pragma unroll
                    for (int f = 0; f < 4; ++f) w[f] = xp[16 * f * XROW + 4 * t];
#pragma unroll
                    for (int s = 0; s < 2; ++s)
#pragma unroll
                        for (int f = 0; f < 4; ++f) {
                            const float av = a[4 * c + 2 * t + s];
                            re[f] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[f][2 * s], av, re[f], 0,
                                                                         0, 0);
                            im[f] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[f][2 * s + 1], av,
                                                                         im[f], 0, 0, 0);
                        }
                }
            }
            __syncthreads();
        }
        cpx<float> v[E];
        if (cols) {
#pragma unroll
            for (int f = 0; f < 4; ++f)
#pragma unroll
                for (int u = 0; u < 4; ++u) v[4 * f + u] = mk(re[f][u], im[f][u]);
            // radix 16 of butterfly n0 = h + 4 wn, column 16 wi + r
            dftr<4, -1>(v);
            const int base = (16 * wi + r) * SB, n0 = h + 4 * wn;
#pragma unroll
            for (int q = 0; q < 16; ++q) lds[base + lpad(16 * n0 + q)] = v[q];
        }
        __syncthreads();

        // from here lane = column, butterflies i = wave + e NT / 64 (wave-uniform)
        const int row = lane * SB;
#pragma unroll
        for (int e = 0; e < NB; ++e) {
            const int i = wave + e * (NT / 64);       // < 16
            cpx<float> *w = v + e * R;
#pragma unroll
            for (int q = 0; q < R; ++q) w[q] = lds[row + lpad(i + 16 * q)];
#pragma unroll
            for (int q = 1; q < R; ++q) w[q] = cmul(w[q], kp_uniform(k.tw, i * q));
            dftr<LOGR, -1>(w);
#pragma unroll
            for (int q = 0; q < R; ++q) {
                const cpx<float> d = kp_uniform(k.D, i + 16 * q);
                w[q] = k.conj_d ? cmulc(w[q], d) : cmul(w[q], d);
            }
            dftr<LOGR, +1>(w);
        }
        __syncthreads();
#pragma unroll
        for (int e = 0; e < NB; ++e) {
            const int i = wave + e * (NT / 64);
#pragma unroll
            for (int q = 0; q < R; ++q) lds[row + lpad(R * i + q)] = v[e * R + q];
        }
        __syncthreads();
        const int i = wave;                           // < NR0 = R
#pragma unroll
        for (int q = 0; q < 16; ++q) v[q] = lds[row + lpad(i + NR0 * q)];
        __syncthreads();  // the LDS holds the next slab's chunks from here
#pragma unroll
        for (int q = 1; q < 16; ++q) v[q] = cmulc(v[q], kp_uniform(k.tw, i * q));
        dftr<4, +1>(v);
        if (M % 64 == 0 || i0 + lane < M) {
            // (scalar row address, the lane as the offset)
            cpx<float> *y = k.y + slab * (int64_t(N) * M) + i0 + i * M;
#pragma unroll
            for (int q = 0; q < 16; ++q, y += NR0 * M) stg_stream(y, uint32_t(lane), v[q]);
        }
    }
}

template <int LOGN, int M>
static fm_status kron_pair_launch(const KronPairArgs &k, int64_t outer, hipStream_t stream) {
    constexpr int N = 1 << LOGN;
    const size_t lds = tile_lds_bytes<float>(LOGN, 64);
    static bool attr = false;
    if (!attr) {
        (void)hipFuncSetAttribute((const void *)kron_pair_kernel<LOGN, M>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        attr = true;
    }
    constexpr int IB = (M + 63) / 64;
    // as many workgroups as run at once (two of 68 KB, or four of 34 KB, per CU)
    int dev = 0, ncu = 256;
    if (hipGetDevice(&dev) == hipSuccess)
        (void)hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
    const int64_t grid = std::min<int64_t>(outer, int64_t(ncu) * (LOGN == 6 ? 4 : 2) / IB) * IB;
    ProfToken tok;
    prof_begin(stream, &tok);
    hipLaunchKernelGGL((kron_pair_kernel<LOGN, M>), dim3(unsigned(grid)), dim3(4 << LOGN), lds,
                       stream, k);
    FM_CHECK_LAUNCH();
    if (tok.active) {
        const double bytes = 2.0 * double(outer) * N * M * 8.0 + double(M) * M * 4.0 + N * 8.0;
        prof_end(stream, &tok, "kron_pair_kernel", bytes,
                 4.0 * double(M) * M * double(N) * double(outer));
    }
    return FM_SUCCESS;
}

}  // namespace fm

using namespace fm;

extern "C" fm_status fm_kron_pair_apply(const fm_conv_plan *plan, int conj_circulant,
                                        const void *A, int64_t m, const void *x, void *y,
                                        int64_t outer, void *stream) {
    FM_REQUIRE(plan != nullptr && A != nullptr, FM_ERR_VALUE, "NULL plan or matrix");
    const int64_t n = plan->rows;
    FM_REQUIRE(plan->kind != 2 && plan->prec == FM_COMPLEX64 && plan->cols == n && plan->L == n &&
                   (n == 64 || n == 128) && (m == 64 || m == 96 || m == 128),
               FM_ERR_NOT_IMPLEMENTED,
               "the fused Kron pair needs a complex64 Circulant plan of 64 or 128 points and a "
               "matrix of 64, 96 or 128 rows");
    FM_REQUIRE(outer >= 0, FM_ERR_VALUE, "negative slab count");
    if (outer == 0) return FM_SUCCESS;
    FM_REQUIRE(x != nullptr && y != nullptr, FM_ERR_VALUE, "NULL data pointer");
    FM_REQUIRE(x != y, FM_ERR_VALUE, "the fused Kron pair does not run in place");
    KronPairArgs k;
    k.x = (const cpx<float> *)x;
    k.y = (cpx<float> *)y;
    k.A = (const float *)A;
    k.D = (const cpx<float> *)plan->D;
    k.tw = (const cpx<float> *)plan->geo.tw32;
    k.conj_d = conj_circulant ? 1 : 0;
    k.outer = outer;
    hipStream_t s = as_stream(stream);
    if (n == 64)
        return m == 64   ? kron_pair_launch<6, 64>(k, outer, s)
               : m == 96 ? kron_pair_launch<6, 96>(k, outer, s)
                         : kron_pair_launch<6, 128>(k, outer, s);
    return m == 64   ? kron_pair_launch<7, 64>(k, outer, s)
           : m == 96 ? kron_pair_launch<7, 96>(k, outer, s)
                     : kron_pair_launch<7, 128>(k, outer, s);
}

extern "C" fm_status fm_kron_conv_dense_apply(const fm_conv_plan *plan, int conj_circulant,
                                              const void *M, int64_t ldm, const void *x, void *y,
                                              int64_t outer, void *stream) {
    FM_REQUIRE(plan != nullptr && M != nullptr, FM_ERR_VALUE, "NULL plan or matrix");
    FM_REQUIRE(plan->kind != 2 && plan->prec == FM_COMPLEX64 && plan->rows == 128 &&
                   plan->cols == 128 && plan->L == 128,
               FM_ERR_NOT_IMPLEMENTED,
               "the fused Kron pair needs a complex64 128-point Circulant plan");
    FM_REQUIRE(ldm == 128, FM_ERR_VALUE, "the fused Kron pair needs a contiguous 128 x 128 matrix");
    FM_REQUIRE(outer >= 0, FM_ERR_VALUE, "negative slab count");
    FM_REQUIRE(outer == 0 || (uintptr_t(y) & 15) == 0, FM_ERR_VALUE,
               "output must be 16-byte aligned");
    return fm_kron_pair_apply(plan, conj_circulant, M, ldm, x, y, outer, stream);
}
