// Dense products on the matrix cores with operands loaded straight into the
// MFMA register layout (float32, float32 x complex64, float64, complex128).
//
//   Y[c][i] = sum_l A_eff[i][l] X[c][l],   A_eff = A or A^T (A^H)
//
// for A row-major (lda), X and Y columns contiguous (ldx, ldy): what
// ndarray.dot does for a dense Matrix (fastmat/Matrix.pyx:1831-1842,
// 1924-1935).
//
// Each wave64 owns a (16 FM) x (16 FN) piece of Y as FM x FN blocks of a
// 16x16x4 MFMA and keeps its operands in registers; there is no LDS staging
// and so no barrier in the K loop.  The fp32 and fp64 matrix instructions are
// slow enough (32 and 64 cycles) that the L1 serves the operands: a 64 x 64
// float wave tile needs 4 bytes per clock and SIMD.  One step covers K =
// 64 / sizeof(S) = 4 KS: lane (r, h) = (lane & 15, lane >> 4) holds KS = 16 /
// sizeof(S) consecutive l from l0 + KS h, one 16-byte load per row (a row's
// four lanes read 64 contiguous bytes), and the KS MFMAs of the step take l =
// l0 + KS h + s from lane h.  The next step's loads are issued before the
// current step's MFMAs.
//
// Rows of Y: fragment q, lane r stands for row 16 V (q / V) + V r + q mod V
// with V = min(KS, FM): a lane's V fragments are V neighbouring rows, so the
// transposed product (A_eff contiguous along i) loads 16 bytes along i for V
// fragments at once, and results are stored 16 bytes at a time.
//
// A workgroup is WM x WN waves over rows and columns and WK waves over K
// (steps dealt round robin, partial sums added through LDS in wave order, so
// results do not depend on timing): where M x NC has too few tiles for the
// chip, the K split supplies the waves.
//
// Out-of-range rows and columns read clamped addresses and are not stored;
// the last K step loads element by element with zeros beyond K, so no load
// leaves A or X.
//
// What bounds it: the matrix pipes (fp32 157, fp64 78.6 TFLOP/s).  Measured on
// one MI355X against the kernels it replaced (LDS tiles of 64 x 64 with K
// slabs of 16 in fp32, no matrix instructions in fp64): see the dispatch in
// fm_gemm.hip.
#pragma once

#include <type_traits>

#include "fm_common.hpp"

namespace fm {

template <typename S> struct DirectArgs {
    int64_t M, K, NC;  // rows of Y, length of the sum, columns of X (complex ones with XC)
    const S *A;
    int64_t lda;
    const S *X;
    int64_t ldx;
    S *Y;
    int64_t ldy;
    int conj_a;  // complex A: multiply by its conjugate
    int64_t tile0;  // the launch's first tile
};

typedef float dg_f4 __attribute__((ext_vector_type(4)));
typedef double dg_d4 __attribute__((ext_vector_type(4)));

// 16 bytes of elements at an element-aligned address
template <typename S> struct Vec16;
template <> struct Vec16<float> {
    typedef float T __attribute__((ext_vector_type(4), aligned(4)));
};
template <> struct Vec16<double> {
    typedef double T __attribute__((ext_vector_type(2), aligned(8)));
};

// One element / 16 bytes of elements, `off` elements (a lane's own) from a
// wave-uniform base.  A 32-bit offset makes it one load from scalar base plus
// vector offset.
template <typename Off, typename S>
__device__ __forceinline__ const S *direct_at(const S *base, Off off) {
    if constexpr (sizeof(Off) == 4)
        return reinterpret_cast<const S *>(reinterpret_cast<const char *>(base) +
                                           uint32_t(off * uint32_t(sizeof(S))));
    else return base + off;
}
template <typename Off, typename S>
__device__ __forceinline__ void load16(S *dst, const S *base, Off off) {
    if constexpr (sizeof(S) == 16) {
        *dst = *direct_at(base, off);
    } else {
        const auto v = *reinterpret_cast<const typename Vec16<S>::T *>(direct_at(base, off));
#pragma unroll
        for (int e = 0; e < 16 / int(sizeof(S)); ++e) dst[e] = v[e];
    }
}

// 16 bytes of elements to an element-aligned address
template <typename S> __device__ __forceinline__ void store16(S *dst, const S *src) {
    typename Vec16<S>::T v;
#pragma unroll
    for (int e = 0; e < 16 / int(sizeof(S)); ++e) v[e] = src[e];
    *reinterpret_cast<typename Vec16<S>::T *>(dst) = v;
}

// Accumulator of one 16 x 16 block and its update by one MFMA.  Element v of a
// lane is column (4 (lane >> 4) + v) for float, (4 v + (lane >> 4)) for double.
template <typename S> struct DirectAcc;
template <> struct DirectAcc<float> {
    dg_f4 d;
    static constexpr int R = 4;  // registers' worth of S per lane
    __device__ __forceinline__ void zero() { d = dg_f4{0.f, 0.f, 0.f, 0.f}; }
    __device__ __forceinline__ void mac(float x, float a) {
        d = __builtin_amdgcn_mfma_f32_16x16x4f32(x, a, d, 0, 0, 0);
    }
    __device__ __forceinline__ float get(int v) const { return d[v]; }
    __device__ static __forceinline__ int col(int lane, int v) { return 4 * (lane >> 4) + v; }
};
template <> struct DirectAcc<double> {
    dg_d4 d;
    __device__ __forceinline__ void zero() { d = dg_d4{0., 0., 0., 0.}; }
    __device__ __forceinline__ void mac(double x, double a) {
        d = __builtin_amdgcn_mfma_f64_16x16x4f64(x, a, d, 0, 0, 0);
    }
    __device__ __forceinline__ double get(int v) const { return d[v]; }
    __device__ static __forceinline__ int col(int lane, int v) { return 4 * v + (lane >> 4); }
};
template <> struct DirectAcc<cpx<double>> {
    dg_d4 re, im;
    __device__ __forceinline__ void zero() { re = im = dg_d4{0., 0., 0., 0.}; }
    __device__ __forceinline__ void mac(cpx<double> x, cpx<double> a) {
        re = __builtin_amdgcn_mfma_f64_16x16x4f64(x.x, a.x, re, 0, 0, 0);
        im = __builtin_amdgcn_mfma_f64_16x16x4f64(x.x, a.y, im, 0, 0, 0);
        re = __builtin_amdgcn_mfma_f64_16x16x4f64(x.y, -a.y, re, 0, 0, 0);
        im = __builtin_amdgcn_mfma_f64_16x16x4f64(x.y, a.x, im, 0, 0, 0);
    }
    __device__ __forceinline__ cpx<double> get(int v) const { return mk(re[v], im[v]); }
    __device__ static __forceinline__ int col(int lane, int v) { return 4 * v + (lane >> 4); }
};

template <typename S> __device__ __forceinline__ S direct_zero() {
    if constexpr (std::is_same<S, cpx<double>>::value) return mk(0.0, 0.0);
    else return S(0);
}

template <typename S, int FM_> struct DirectShape {
    static constexpr int KS = 16 / int(sizeof(S));   // MFMAs (of K = 4) per step
    static constexpr int BK = 4 * KS;                // K per step
    static constexpr int V = KS < FM_ ? KS : FM_;    // neighbouring rows per lane
};

// XC: real A, complex X and Y (S = float): fragments 2 b and 2 b + 1 are the
// real and imaginary parts of the same 16 columns.  AK: A_eff is contiguous
// along K (A itself), else along its rows (the transposed product).  Off: type
// of a lane's offset from its wave's base pointer.
template <typename S, typename Off, bool XC, bool AK, int FM, int FN, int WM, int WN, int WK>
__global__ __launch_bounds__(64 * WM * WN * WK, 2) void gemm_direct_kernel(
    const DirectArgs<S> g) {
    using Sh = DirectShape<S, FM>;
    constexpr int KS = Sh::KS, BK = Sh::BK, V = Sh::V;
    constexpr int TM = 16 * FM * WM;
    constexpr int CW = XC ? 8 * FN : 16 * FN;  // columns of X per wave
    constexpr int TN = CW * WN;
    constexpr int NB = XC ? FN / 2 : FN;       // column groups of 16
    static_assert(FM % V == 0 && (V == KS || V == 1) && (!XC || FN % 2 == 0), "fragment shape");
    extern __shared__ __align__(16) unsigned char direct_smem[];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, h = lane >> 4;
    const int wk = wave % WK, wn = (wave / WK) % WN, wm = wave / (WK * WN);
    const int64_t tiles_n = ceil_div(g.NC, TN);
    const int64_t tile = g.tile0 + xcd_remap(blockIdx.x, gridDim.x);
    const int64_t tm = tile / tiles_n, tn = tile - tm * tiles_n;
    const int64_t i0 = tm * TM + wm * (16 * FM), c0 = tn * TN + wn * CW;
    const int64_t steps = ceil_div(g.K, BK);

    // the wave's first row and column (clamped: a wave past the edge works on
    // the last ones and stores nothing), and the lanes' offsets from them,
    // clamped likewise
    const int64_t ib = i0 < g.M ? i0 : g.M - 1, cb = c0 < g.NC ? c0 : g.NC - 1;
    const Off ilast = Off(g.M - 1 - ib), clast = Off(g.NC - 1 - cb);
    const S *abase = g.A + (AK ? ib * g.lda : ib);
    const S *xbase = g.X + (XC ? 2 : 1) * cb * g.ldx;
    const Off lda = Off(g.lda);
    Off ao[AK ? FM : FM / V];
    if constexpr (AK) {
#pragma unroll
        for (int q = 0; q < FM; ++q) {
            const Off i = Off(16 * V * (q / V) + V * r + q % V);
            ao[q] = (i < ilast ? i : ilast) * lda + Off(KS * h);
        }
    } else {
#pragma unroll
        for (int u = 0; u < FM / V; ++u) {
            const Off i = Off(16 * V * u + V * r);
            ao[u] = Off(KS * h) * lda + (i < ilast ? i : ilast);
        }
    }
    Off xo[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        const Off c = Off(16 * b + r);
        xo[b] = Off(XC ? 2 : 1) * ((c < clast ? c : clast) * Off(g.ldx) + Off(KS * h));
    }

    DirectAcc<S> acc[FM][FN];
#pragma unroll
    for (int q = 0; q < FM; ++q)
#pragma unroll
        for (int b = 0; b < FN; ++b) acc[q][b].zero();

    // Operands of step st, for steps before the last: a transposed product's
    // vector may run up to V - 1 elements past row l's end, into row l + 1,
    // which exists there.
    auto load = [&](int64_t st, S a[FM][KS], S x[FN][KS]) {
        const int64_t l0 = st * BK;
        const S *xl = xbase + (XC ? 2 : 1) * l0;
        if constexpr (AK) {
#pragma unroll
            for (int q = 0; q < FM; ++q) load16(a[q], abase + l0, ao[q]);
        } else {
            const S *al = abase + l0 * g.lda;
#pragma unroll
            for (int s = 0; s < KS; ++s, al += g.lda)
#pragma unroll
                for (int u = 0; u < FM / V; ++u) {
                    if constexpr (V == KS) {
                        S t[KS];
                        load16(t, al, ao[u]);
#pragma unroll
                        for (int e = 0; e < V; ++e) a[u * V + e][s] = t[e];
                    } else {
                        a[u][s] = *direct_at(al, ao[u]);
                    }
                }
        }
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            if constexpr (XC) {
                S t[2 * KS];
                load16(t, xl, xo[b]);
                load16(t + KS, xl, xo[b] + Off(KS));
#pragma unroll
                for (int s = 0; s < KS; ++s) {
                    x[2 * b][s] = t[2 * s];
                    x[2 * b + 1][s] = t[2 * s + 1];
                }
            } else {
                load16(x[b], xl, xo[b]);
            }
        }
    };
    // Any step, element by element: zero beyond K, rows beyond the last clamped.
    auto load_tail = [&](int64_t st, S a[FM][KS], S x[FN][KS]) {
        const int64_t l0 = st * BK;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const bool ok = l0 + KS * h + s < g.K;
#pragma unroll
            for (int q = 0; q < FM; ++q) {
                S v = direct_zero<S>();
                if (ok) {
                    if constexpr (AK) {
                        v = *direct_at(abase + l0 + s, ao[q]);
                    } else {
                        const int64_t i = i0 + 16 * V * (q / V) + V * r + q % V;
                        v = *direct_at(abase + (l0 + s) * g.lda,
                                       ao[q / V] + Off(i < g.M ? q % V : 0));
                    }
                }
                a[q][s] = v;
            }
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                if constexpr (XC) {
                    const S *p = direct_at(xbase + 2 * (l0 + s), xo[b]);
                    x[2 * b][s] = ok ? p[0] : S(0);
                    x[2 * b + 1][s] = ok ? p[1] : S(0);
                } else {
                    x[b][s] = ok ? *direct_at(xbase + l0 + s, xo[b]) : direct_zero<S>();
                }
            }
        }
    };
    auto multiply = [&](S a[FM][KS], S x[FN][KS]) {
        if constexpr (std::is_same<S, cpx<double>>::value) {
            if (g.conj_a) {
#pragma unroll
                for (int q = 0; q < FM; ++q)
#pragma unroll
                    for (int s = 0; s < KS; ++s) a[q][s].y = -a[q][s].y;
            }
        }
#pragma unroll
        for (int s = 0; s < KS; ++s)
#pragma unroll
            for (int b = 0; b < FN; ++b)
#pragma unroll
                for (int q = 0; q < FM; ++q) acc[q][b].mac(x[b][s], a[q][s]);
    };

    // whole steps with the next one's loads in flight, then the wave's share
    // of the rest (the last step; every step of a transposed product whose rows
    // are shorter than a vector, which could pass row l + 1 too)
    const int64_t full = (AK || g.lda >= V) && steps > 0 ? steps - 1 : 0;
    S a0[FM][KS], x0[FN][KS];
    int64_t st = wk;
    if (st < full) {
        load(st, a0, x0);
#pragma unroll 1
        for (; st + WK < full; st += WK) {
            S a1[FM][KS], x1[FN][KS];
            load(st + WK, a1, x1);
            multiply(a0, x0);
#pragma unroll
            for (int s = 0; s < KS; ++s) {
#pragma unroll
                for (int q = 0; q < FM; ++q) a0[q][s] = a1[q][s];
#pragma unroll
                for (int b = 0; b < FN; ++b) x0[b][s] = x1[b][s];
            }
        }
        multiply(a0, x0);
        st += WK;
    }
#pragma unroll 1
    for (; st < steps; st += WK) {
        load_tail(st, a0, x0);
        multiply(a0, x0);
    }

    // Partial sums of the K split: unit (b, v) of a lane is FM elements; the
    // WK waves of a tile share its units, each adding all waves' parts in order.
    constexpr int UNITS = FN * 4;
    if constexpr (WK > 1) {
        S *red = reinterpret_cast<S *>(direct_smem) +
                 int64_t(wave / WK) * (int64_t(WK) * UNITS * FM * 64);
#pragma unroll
        for (int b = 0; b < FN; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v)
#pragma unroll
                for (int q = 0; q < FM; ++q)
                    red[((wk * UNITS + b * 4 + v) * FM + q) * 64 + lane] = acc[q][b].get(v);
        __syncthreads();
    }
    auto emit = [&](int b, int v, const S *re, const S *im) {
        // FM elements (XC: their real and imaginary parts) of column group b, register v
        const int64_t c = c0 + 16 * b + DirectAcc<S>::col(lane, v);
        if (c >= g.NC) return;
#pragma unroll
        for (int u = 0; u < FM / V; ++u) {
            const int64_t i = i0 + 16 * V * u + V * r;
            if constexpr (XC) {
                S *y = g.Y + 2 * (c * g.ldy + i);
                if constexpr (V > 1) {
                    if (i + V <= g.M) {
                        S t[2 * V];
#pragma unroll
                        for (int e = 0; e < V; ++e) {
                            t[2 * e] = re[u * V + e];
                            t[2 * e + 1] = im[u * V + e];
                        }
#pragma unroll
                        for (int e = 0; e < 2 * V; e += KS) store16(y + e, t + e);
                        continue;
                    }
                }
#pragma unroll
                for (int e = 0; e < V; ++e)
                    if (i + e < g.M) {
                        y[2 * e] = re[u * V + e];
                        y[2 * e + 1] = im[u * V + e];
                    }
            } else {
                S *y = g.Y + c * g.ldy + i;
                if constexpr (V > 1 && V == KS) {
                    if (i + V <= g.M) {
                        store16(y, re + u * V);
                        continue;
                    }
                }
#pragma unroll
                for (int e = 0; e < V; ++e)
                    if (i + e < g.M) y[e] = re[u * V + e];
            }
        }
    };
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            S re[FM], im[FM];
            const int b0 = XC ? 2 * b : b;
            if constexpr (WK > 1) {
                if ((b * 4 + v) % WK != wk) continue;
                const S *red = reinterpret_cast<const S *>(direct_smem) +
                               int64_t(wave / WK) * (int64_t(WK) * UNITS * FM * 64);
#pragma unroll
                for (int q = 0; q < FM; ++q) {
                    S t = direct_zero<S>(), t2 = direct_zero<S>();
                    for (int w = 0; w < WK; ++w) {
                        t = t + red[((w * UNITS + b0 * 4 + v) * FM + q) * 64 + lane];
                        if constexpr (XC)
                            t2 = t2 + red[((w * UNITS + (b0 + 1) * 4 + v) * FM + q) * 64 + lane];
                    }
                    re[q] = t;
                    im[q] = t2;
                }
            } else {
#pragma unroll
                for (int q = 0; q < FM; ++q) {
                    re[q] = acc[q][b0].get(v);
                    im[q] = XC ? acc[q][XC ? b0 + 1 : b0].get(v) : re[q];
                }
            }
            emit(b, v, re, im);
        }
}

}  // namespace fm
