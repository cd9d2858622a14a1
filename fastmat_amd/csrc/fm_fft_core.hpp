// FFT engine: the tile body used by every Fourier / Circulant / Toeplitz /
// Bluestein pass (per-operator kernels and the batched persistent kernels).
//
// Method (written from the published Stockham autosort formulation): a
// length-N transform (N = 2^LOGN, compile-time) is split into S stages of
// radix 2^bits(s) <= E, E = 4 to 32 elements per thread by the pass's shape (see
// PassShape).  Stage with radix R and sub-length p: butterfly i in [0, N/R) takes
// X[i + r N/R], multiplies input r by W_{pR}^{r k} (k = i mod p), runs an
// R-point DFT in registers and produces Y[(i - k) R + k + r p]; outputs come
// out in natural order.  Stage 0 loads its inputs straight from HBM, the last
// stage stores straight to HBM, and the S-1 exchanges in between go through a
// padded LDS tile (see tile_row).  1024 = 32 x 32 needs one exchange.
//
// Tile: B = threads * E / N consecutive sequences s = o*J + j of an (O x J)
// sequence space.  Element n of sequence
// (o, j) is read at  x[o*in_os + j*in_js + n*in_ns]  and written at
// y[o*out_os + j*out_js + n*out_ns]; this one addressing form covers
// contiguous columns, the strided and the transposed sides of the four-step
// passes, and Kron mode axes.  Global accesses map neighbouring lanes to
// neighbouring sequences where those are adjacent in memory (strided sides)
// and to neighbouring elements otherwise.  Work fused around the transform:
//     load:  zero-pad (global index n*in_gn + j*in_gj >= n_valid), conj,
//            pre-multiply by a chirp, then FFT(sign1)
//     conv:  multiply by the spectrum D[n*d_gn + j*d_gj] (or conj) in
//            registers, then FFT(-sign1) with the radices reversed so it
//            starts from the forward transform's registers
//     store: twiddle W_L^{+-j n} of an enclosing four-step, crop
//            (n*out_gn + j*out_gj >= m_valid), post-multiply, conj, scale.
#pragma once

#include <type_traits>

#include "fm_common.hpp"

namespace fm {

// ------------------------------------------------------------ small DFTs
template <int SIGN, typename T> __device__ __forceinline__ void dft2(cpx<T> *v) {
    cpx<T> a = v[0];
    v[0] = a + v[1];
    v[1] = a - v[1];
}

template <int SIGN, typename T> __device__ __forceinline__ void dft4(cpx<T> *v) {
    cpx<T> t0 = v[0] + v[2];
    cpx<T> t1 = v[0] - v[2];
    cpx<T> t2 = v[1] + v[3];
    cpx<T> t3 = mul_i<SIGN>(v[1] - v[3]);
    v[0] = t0 + t2;
    v[2] = t0 - t2;
    v[1] = t1 + t3;
    v[3] = t1 - t3;
}

template <int SIGN, typename T> __device__ __forceinline__ void dft8(cpx<T> *v) {
    cpx<T> e[4] = {v[0], v[2], v[4], v[6]};
    cpx<T> o[4] = {v[1], v[3], v[5], v[7]};
    dft4<SIGN>(e);
    dft4<SIGN>(o);
    const T h = T(0.70710678118654752440084436210485);
    cpx<T> a = o[1], c = o[3];
    if (SIGN < 0) {
        o[1] = mk(h * (a.x + a.y), h * (a.y - a.x));        // * h(1 - i)
        o[3] = mk(h * (c.y - c.x), -h * (c.x + c.y));       // * h(-1 - i)
    } else {
        o[1] = mk(h * (a.x - a.y), h * (a.x + a.y));        // * h(1 + i)
        o[3] = mk(-h * (c.x + c.y), h * (c.x - c.y));       // * h(-1 + i)
    }
    o[2] = mul_i<SIGN>(o[2]);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        v[q] = e[q] + o[q];
        v[q + 4] = e[q] - o[q];
    }
}

// W_32^k = exp(-2 pi i k / 32), k < 16 (cos, sin)
__device__ __forceinline__ constexpr double w32c(int k) {
    constexpr double c[16] = {1.0, 0.98078528040323043, 0.92387953251128674, 0.83146961230254524,
                              0.70710678118654757, 0.55557023301960229, 0.38268343236508984,
                              0.19509032201612833, 0.0, -0.19509032201612819, -0.38268343236508973,
                              -0.55557023301960196, -0.70710678118654746, -0.83146961230254535,
                              -0.92387953251128674, -0.98078528040323043};
    return c[k];
}
__device__ __forceinline__ constexpr double w32s(int k) {
    constexpr double s[16] = {0.0, 0.19509032201612825, 0.38268343236508978, 0.55557023301960218,
                              0.70710678118654746, 0.83146961230254524, 0.92387953251128674,
                              0.98078528040323043, 1.0, 0.98078528040323043, 0.92387953251128674,
                              0.83146961230254546, 0.70710678118654757, 0.55557023301960218,
                              0.38268343236508989, 0.19509032201612861};
    return s[k];
}

// x * W_R^k (forward, SIGN < 0) or x * conj(W_R^k) (inverse), k < R/2, R <= 32;
// k is a compile-time constant after unrolling, so the branches fold away.
template <int R, int SIGN, typename T>
__device__ __forceinline__ cpx<T> wmul(cpx<T> x, int k) {
    if (k == 0) return x;
    if (4 * k == R) return mul_i<SIGN>(x);
    const int q = k * (32 / R);
    const T c = T(w32c(q)), s = T(w32s(q));
    // forward W = c - i s ; inverse conj(W) = c + i s
    return SIGN < 0 ? mk(x.x * c + x.y * s, x.y * c - x.x * s)
                    : mk(x.x * c - x.y * s, x.y * c + x.x * s);
}

// In-register DFT of length 2^LOGR (LOGR <= 5), natural order in and out.
template <int LOGR, int SIGN, typename T> __device__ __forceinline__ void dftr(cpx<T> *v) {
    if constexpr (LOGR == 1) dft2<SIGN>(v);
    else if constexpr (LOGR == 2) dft4<SIGN>(v);
    else if constexpr (LOGR == 3) dft8<SIGN>(v);
    else if constexpr (LOGR >= 4) {
        constexpr int R = 1 << LOGR, H = R / 2;
        cpx<T> e[H], o[H];
#pragma unroll
        for (int i = 0; i < H; ++i) {
            e[i] = v[2 * i];
            o[i] = v[2 * i + 1];
        }
        dftr<LOGR - 1, SIGN>(e);
        dftr<LOGR - 1, SIGN>(o);
#pragma unroll
        for (int k = 0; k < H; ++k) {
            const cpx<T> t = wmul<R, SIGN>(o[k], k);
            v[k] = e[k] + t;
            v[k + H] = e[k] - t;
        }
    }
}

template <int SIGN, typename T>
__device__ __forceinline__ cpx<T> twiddle_mul(cpx<T> v, cpx<T> w) {
    // w is the forward twiddle exp(-2 pi i e / N); the inverse uses conj(w)
    return SIGN < 0 ? cmul(v, w) : cmulc(v, w);
}

// Stage plan of a length-2^LOGN transform for threads holding 2^LOGE
// elements: S stages with radices 2^bits(s) <= 2^LOGE, bits as even as
// possible, larger radices first.
template <int LOGN, int LOGE, bool REV = false> struct FftPlan {
    static constexpr int S = LOGN == 0 ? 0 : (LOGN + LOGE - 1) / LOGE;
    static constexpr int SD = S > 0 ? S : 1;  // (LOGN == 0 has no stages)
    static constexpr int fbits(int s) { return LOGN / SD + (s < LOGN % SD ? 1 : 0); }
    // REV runs the same radices last-to-first (any order is a valid Stockham
    // factorisation); a transform whose first radix equals the previous
    // transform's last radix can start from that transform's registers.
    static constexpr int bits(int s) { return REV ? fbits(S - 1 - s) : fbits(s); }
    static constexpr int logp(int s) {
        int t = 0;
        for (int q = 0; q < s; ++q) t += bits(q);
        return t;
    }
};

// Padded LDS index: one spare slot every 32 elements (16 of 16 bytes) keeps
// the strided exchanges of the stages free of most bank conflicts.
template <typename T = float> __host__ __device__ __forceinline__ constexpr int lpad(int n) {
    return n + (n >> (sizeof(T) == 4 ? 5 : 4));
}

// LDS elements between the sequences of a tile of 2^LOGB sequences of 2^LOGN.
// Accesses in the sequence-fastest mapping take 32 lanes (16 of 16 bytes) at a
// time, 2^LOGB sequences by 32 / 2^LOGB neighbouring elements (one slot apart
// after padding), so rows 32 / 2^LOGB slots apart (modulo 32) put them into
// distinct banks; with one spare slot the 1024-point strided tiles (8
// sequences) hit each bank four times.  With TwiddleChain below, measured in
// one step: the 1024-point column pass of 2^20 x 64 columns 353 -> 317 us (64 MB
// of columns: 38.2 -> 34.6), Fourier 2^20 x 64 forward and adjoint 1058 ->
// 1016 us, 50 FISTA iterations on 2^18 x 8 8256 -> 7748 us.
template <typename T> __host__ __device__ constexpr int tile_row(int logn, int logb) {
    const int span = sizeof(T) == 4 ? 32 : 16;
    const int spare = logb == 0 ? 0 : ((span >> logb) > 1 ? (span >> logb) : 1);
    return lpad<T>(1 << logn) + spare;
}

// LDS bytes of a tile of B (a power of two) sequences of 2^logn.
template <typename T> inline size_t tile_lds_bytes(int logn, int B) {
    return size_t(B) * tile_row<T>(logn, ilog2(B)) * sizeof(cpx<T>);
}

// ------------------------------------------------------------ tile kernel
template <typename T> struct TileArgs {
    int logN;          // transform length N = 2^logN
    int B;             // sequences per tile (power of two)
    int64_t O, J;      // sequence space, s = o*J + j
    int64_t ntiles;
    // input
    const cpx<T> *x;
    int64_t in_os, in_js, in_ns;
    int64_t in_gn, in_gj, n_valid;  // zero-pad predicate
    const cpx<T> *pre;              // optional chirp, indexed by global input index
    int conj_in;
    int seqfast_in;
    // transform
    int sign1;                      // -1 forward, +1 inverse
    const cpx<double> *tw;          // W_N^e table (FP64)
    // spectral multiply + second transform (conv mode)
    const cpx<T> *D;
    int64_t d_gn, d_gj;
    int conj_d;
    // enclosing four-step twiddle applied before the store: W_L^{tw_sign * j * n}
    const cpx<double> *twb_hi, *twb_lo;  // W_L^{a * 2^twb_shift}, W_L^{b} (FP64)
    int twb_shift;
    int twb_sign;
    // output
    cpx<T> *y;
    int64_t out_os, out_js, out_ns;
    int64_t out_gn, out_gj, m_valid;
    const cpx<T> *post;
    int conj_out;
    T out_scale;
    int seqfast_out;
    // batch engine: this pass writes the caller's output of its direction;
    // a redirected apply moves y by a byte shift and multiplies out_scale by
    // a device scalar for such passes only
    int redirect;
    // non-temporal (streaming) accesses (the batch engine's passes): bit 0
    // the output stores, bit 1 the input loads
    int stream_out;
    int logJ;                       // log2(J) when J is a power of two, else -1
    int64_t o_group;                // > 1: tiles walk groups of o_group o's (see tile_first_seq)
    // optional residual epilogue (target != NULL): the store writes
    // out_scale * (u - t) with t read from `target` at the output's position
    // (same layout as y), and the tile's sum of |u - t|^2 over the stored
    // elements goes to res_part[res_base + tile] (FP64) unless res_part is NULL
    const cpx<T> *target;
    double *res_part;
    int64_t res_base;
    // optional residual between the two transforms of a conv-mode pass, in
    // place of the spectrum (mid_t != NULL): element n of sequence (o, j)
    // of the first transform's output stands at index g = n*mid_gn + j*mid_gj
    // of column o; for g < mid_valid it becomes mid_scale * (u - t) with
    // t = mid_t[o*mid_os + g] (|u - t|^2 adds to the tile's residual sum
    // res_part[res_base + tile]), beyond mid_valid it becomes 0
    const cpx<T> *mid_t;
    int64_t mid_os, mid_gn, mid_gj, mid_valid;
    T mid_scale;
    // host only: this pass's share of its transform's algorithmic bytes (the
    // input and output blocks and the generator, split over the passes),
    // for the library's profiler; 0 = count the pass's own reads and writes
    double alg_bytes;
};

// Index arithmetic of a pass: int64_t in general, uint32_t when every
// element offset and logical index of the launch is below 2^32 / sizeof
// (32-bit offsets from a uniform base become saddr + voffset addressing).
template <bool I32> using IdxT = typename std::conditional<I32, uint32_t, int64_t>::type;

// Load / store element `idx` of a uniform base pointer, as global memory:
// every data pointer of the library is device memory, and kernels that read
// their pointers from descriptors in memory (the batch engine) would
// otherwise get flat loads and stores, which count against the LDS wait
// counter too and so serialise the tile's LDS exchanges behind its
// outstanding HBM traffic.
// (the host pass of the same source sees plain pointers)
#if defined(__HIP_DEVICE_COMPILE__)
#define FM_GLOBAL __attribute__((address_space(1)))
#else
#define FM_GLOBAL
#endif
template <typename Ix, typename V>
__device__ __forceinline__ V ldg(const V *base, Ix idx) {
    const FM_GLOBAL char *b = (const FM_GLOBAL char *)base;
    if constexpr (sizeof(Ix) == 4)
        return *(const FM_GLOBAL V *)(b + uint32_t(idx * uint32_t(sizeof(V))));
    else
        return ((const FM_GLOBAL V *)b)[idx];
}
template <typename Ix, typename V>
__device__ __forceinline__ void stg(V *base, Ix idx, V val) {
    FM_GLOBAL char *b = (FM_GLOBAL char *)base;
    if constexpr (sizeof(Ix) == 4)
        *(FM_GLOBAL V *)(b + uint32_t(idx * uint32_t(sizeof(V)))) = val;
    else
        ((FM_GLOBAL V *)b)[idx] = val;
}

// Non-temporal store of one complex element (see stg).
template <typename Ix, typename T>
__device__ __forceinline__ void stg_stream(cpx<T> *base, Ix idx, cpx<T> val) {
    typedef T v2 __attribute__((ext_vector_type(2)));
    FM_GLOBAL char *b = (FM_GLOBAL char *)base;
    FM_GLOBAL v2 *q;
    if constexpr (sizeof(Ix) == 4)
        q = (FM_GLOBAL v2 *)(b + uint32_t(idx * uint32_t(sizeof(cpx<T>))));
    else
        q = (FM_GLOBAL v2 *)(b + idx * int64_t(sizeof(cpx<T>)));
    v2 v = {val.x, val.y};
    __builtin_nontemporal_store(v, q);
}

// Non-temporal load of one complex element (see ldg).
template <typename Ix, typename T>
__device__ __forceinline__ cpx<T> ldg_stream(const cpx<T> *base, Ix idx) {
    typedef T v2 __attribute__((ext_vector_type(2)));
    const FM_GLOBAL char *b = (const FM_GLOBAL char *)base;
    const FM_GLOBAL v2 *q;
    if constexpr (sizeof(Ix) == 4)
        q = (const FM_GLOBAL v2 *)(b + uint32_t(idx * uint32_t(sizeof(cpx<T>))));
    else
        q = (const FM_GLOBAL v2 *)(b + idx * int64_t(sizeof(cpx<T>)));
    const v2 v = __builtin_nontemporal_load(q);
    return mk(v.x, v.y);
}

// Bound of a logical index in the launch's index type.
template <typename Ix> __device__ __forceinline__ Ix idx_bound(int64_t v) {
    if constexpr (sizeof(Ix) == 4) return v > int64_t(0xffffffffu) ? Ix(0xffffffffu) : Ix(v);
    else return v;
}

// Sequence (o, j) of tile-local sequence b.
template <typename Ix> struct SeqPos {
    Ix in_base, out_base, j;
    bool ok;
};

template <typename Ix, typename T>
__device__ __forceinline__ SeqPos<Ix> seq_pos(const TileArgs<T> &a, int64_t s) {
    SeqPos<Ix> p;
    p.ok = s < a.O * a.J;
    const Ix si = Ix(s);
    Ix o, j;
    if (a.logJ >= 0) {
        o = si >> a.logJ;
        j = si & ((Ix(1) << a.logJ) - 1);
    } else {
        o = si / Ix(a.J);
        j = si - o * Ix(a.J);
    }
    p.in_base = o * Ix(a.in_os) + j * Ix(a.in_js);
    p.out_base = o * Ix(a.out_os) + j * Ix(a.out_js);
    p.j = j;
    return p;
}

// Map butterfly g of a stage to (sequence b, butterfly index i): sequence-
// fastest for strided global sides (neighbouring sequences are adjacent in
// memory), butterfly-fastest otherwise.
template <int LOGB, int LOGNR>
__device__ __forceinline__ void bfly_pos(int g, bool seqfast, int &b, int &i) {
    if (seqfast) {
        b = g & ((1 << LOGB) - 1);
        i = g >> LOGB;
    } else {
        i = g & ((1 << LOGNR) - 1);
        b = g >> LOGNR;
    }
}

// base * step^r for r = 0, 1, ... R - 1 in order, in FP64: up to four
// interleaved recurrences by step^4, so that four products are in flight where
// a single recurrence would wait for each (a product depends on the one four
// back) and rounding errors pass through R / 4 products instead of R.
template <int R> struct TwiddleChain {
    static constexpr int C = R >= 8 ? 4 : (R >= 4 ? 2 : 1);
    cpx<double> w[C], s;
    // elements r = 0, 1, ...
    __device__ __forceinline__ void start(cpx<double> base, cpx<double> step) {
        start_powers(step);
        if constexpr (C > 1) {
#pragma unroll
            for (int c = 1; c < C; ++c) w[c] = cmul(base, w[c]);
        }
        w[0] = base;
    }
    // the powers step^r alone, elements r = 1, 2, ...
    __device__ __forceinline__ void start_powers(cpx<double> step) {
        if constexpr (C == 1) {
            s = step;
        } else {
            w[1] = step;
            const cpx<double> s2 = cmul(step, step);
            if constexpr (C == 2) {
                s = s2;
            } else {
                w[2] = s2;
                w[3] = cmul(step, s2);
                s = cmul(s2, s2);
            }
        }
        w[0] = s;
    }
    // element r, asked for in order
    __device__ __forceinline__ cpx<double> at(int r) {
        const cpx<double> t = w[r % C];
        if (r + C < R) w[r % C] = cmul(t, s);
        return t;
    }
};

// One radix-2^LOGR stage with sub-length 2^LOGP on registers v (E per thread,
// NB = E / R butterflies).  SRC: 0 = v already holds this stage's inputs,
// 1 = read them from LDS.  DST: 0 = write outputs to LDS, 1 = leave them in v.
template <typename T, int LOGN, int LOGR, int LOGP, int SIGN, int NT, int E, int LOGB, int SRC,
          int DST>
__device__ __forceinline__ void fft_stage2(cpx<T> *v, cpx<T> *lds,
                                           const cpx<double> *__restrict__ tw, bool sf) {
    // sf: mapping of the stage's butterflies (see bfly_pos): that of v when
    // SRC == 0, free when the inputs come from LDS.
    constexpr int R = 1 << LOGR, NB = E / R;
    constexpr int LOGNR = LOGN - LOGR, NR = 1 << LOGNR;
    constexpr int P = 1 << LOGP;
    constexpr int SB = tile_row<T>(LOGN, LOGB);
    if constexpr (SRC == 1) {
#pragma unroll
        for (int e = 0; e < NB; ++e) {
            int b, i;
            bfly_pos<LOGB, LOGNR>(threadIdx.x + e * NT, sf, b, i);
#pragma unroll
            for (int r = 0; r < R; ++r) v[e * R + r] = lds[b * SB + lpad<T>(i + r * NR)];
        }
    }
#pragma unroll
    for (int e = 0; e < NB; ++e) {
        int b, i;
        bfly_pos<LOGB, LOGNR>(threadIdx.x + e * NT, sf, b, i);
        if constexpr (LOGP > 0) {
            const int k = i & (P - 1);
            // W_{pR}^{r k} = W_N^{r k N / (p R)}: one FP64 lookup of
            // W_{pR}^k, its powers by FP64 products, rounded once to T
            const int step = k << (LOGN - LOGP - LOGR);
            TwiddleChain<R> w;
            w.start_powers(ldg(tw, uint32_t(step)));
#pragma unroll
            for (int r = 1; r < R; ++r) {
                const cpx<double> t = w.at(r);
                v[e * R + r] = twiddle_mul<SIGN>(v[e * R + r], mk(T(t.x), T(t.y)));
            }
        }
        dftr<LOGR, SIGN>(v + e * R);
    }
    if constexpr (DST == 0) {
        __syncthreads();  // every thread has read its inputs of this stage
#pragma unroll
        for (int e = 0; e < NB; ++e) {
            int b, i;
            bfly_pos<LOGB, LOGNR>(threadIdx.x + e * NT, sf, b, i);
            const int k = i & (P - 1);
            const int base = ((i - k) << LOGR) + k;
#pragma unroll
            for (int r = 0; r < R; ++r) lds[b * SB + lpad<T>(base + r * P)] = v[e * R + r];
        }
        __syncthreads();
    }
}

// All stages of one transform.  FIRST_SRC: 0 = v holds stage-0 inputs
// (loaded from global), 1 = they are in LDS in natural order.  LAST_DST:
// 0 = leave natural-order outputs in LDS, 1 = leave the last stage's outputs
// in v.  sf0: mapping of v's inputs; sf1: mapping of the last stage where it is
// not the first one too.  A strided side that follows takes sf1 = true: the last
// stage then reads its inputs from LDS in the mapping its outputs leave in, where
// outputs in the other mapping would go through LDS once more (Fourier 2^20 x 64
// forward and adjoint 2-3% faster, four-step passes of 16 MB 0.5-1 us), and
// operands between two transforms come in rows of neighbouring sequences (a column
// pass with a shrinkage in its middle 48.9 -> 21.8 us).
template <typename T, int LOGN, int LOGE, int SIGN, int NT, int LOGB, int FIRST_SRC, int LAST_DST,
          bool REV = false, int s = 0>
__device__ __forceinline__ void fft_all(cpx<T> *v, cpx<T> *lds,
                                        const cpx<double> *__restrict__ tw, bool sf0,
                                        bool sf1 = false) {
    using P = FftPlan<LOGN, LOGE, REV>;
    constexpr int E = 1 << LOGE;
    if constexpr (s < P::S) {
        constexpr int src = s == 0 ? FIRST_SRC : 1;
        constexpr int dst = (s == P::S - 1) ? (LAST_DST == 1 ? 1 : 0) : 0;
        const bool sf = s == 0 ? sf0 : (dst == 1 ? sf1 : false);
        fft_stage2<T, LOGN, P::bits(s), P::logp(s), SIGN, NT, E, LOGB, src, dst>(v, lds, tw, sf);
        fft_all<T, LOGN, LOGE, SIGN, NT, LOGB, FIRST_SRC, LAST_DST, REV, s + 1>(v, lds, tw, sf0,
                                                                                sf1);
    }
}

// Compile-time shape of one tile of a length-2^LOGN pass with NT threads.
template <typename T, int LOGN, int NT, int LE = -1> struct TileShape {
    // elements per thread: 2^LE, by default 32 (complex64) / 16 (complex128)
    static constexpr int LOGE = LE >= 0 ? LE : (sizeof(T) == 4 ? 5 : 4);
    static constexpr int E = 1 << LOGE;
    static constexpr int N = 1 << LOGN;
    using P = FftPlan<LOGN, LOGE>;
    static constexpr int LOGR0 = P::S > 0 ? P::bits(0) : 0;
    static constexpr int R0 = 1 << LOGR0;
    static constexpr int LOGNT = NT == 64 ? 6 : NT == 128 ? 7 : NT == 256 ? 8 : NT == 512 ? 9 : 10;
    // sequences per tile (NT * E / N, at least one)
    static constexpr int LOGB = LOGNT + LOGE - LOGN;
    static constexpr int B = 1 << LOGB;
    static_assert(LOGB >= 0, "tile must hold at least one sequence");
};

// First sequence of a tile.  Plain order: consecutive tiles step through the
// j-blocks of one o.  With o_group = G > 1 (G divides O, B divides J) the o's
// form groups of G and, inside a group, consecutive tiles step through the G
// o's of one j-block before the next j-block: tiles that share per-j data (a
// spectrum row, chirp or twiddle values) run close together and reuse it
// from cache, while each o still streams through neighbouring j-blocks.
template <typename T, int LOGB>
__device__ __forceinline__ int64_t tile_first_seq(const TileArgs<T> &a, int64_t tile) {
    if (a.o_group <= 1) return tile << LOGB;
    const int64_t G = a.o_group;
    const int64_t per = G * (a.J >> LOGB);  // tiles of one group
    const int64_t grp = tile / per, rem = tile - grp * per;
    const int64_t jb = rem / G, o = grp * G + (rem - jb * G);
    return o * a.J + (jb << LOGB);
}

// Where a pass's input elements come from: their own places (PlainLoad), or an
// object whose table(e) names the element of the column to read in place of
// element e, negative for a zero; a NULL table is the plain load.
struct PlainLoad {};

// Stage-0 inputs of one tile straight from global memory (zero outside the
// valid range); only loads, so a caller can issue them ahead of compute.
template <typename T, int LOGN, int NT, bool I32 = false, int LE = -1, typename LP = PlainLoad>
__device__ __forceinline__ void fft_tile_load(const TileArgs<T> &a, int64_t tile, cpx<T> *v,
                                              const LP &lp = LP()) {
    using S = TileShape<T, LOGN, NT, LE>;
    using Ix = IdxT<I32>;
    constexpr int NB = S::E / S::R0;
    constexpr int LOGNR = LOGN - S::LOGR0, NR = 1 << LOGNR;
    const int64_t s0 = tile_first_seq<T, S::LOGB>(a, tile);
    const Ix nv = idx_bound<Ix>(a.n_valid);
    const Ix in_gn = Ix(a.in_gn), in_gj = Ix(a.in_gj), in_ns = Ix(a.in_ns);
    // one loop per load kind (uniform), so that all the tile's loads issue
    // before the first use
    auto body = [&](auto load) {
#pragma unroll
        for (int e = 0; e < NB; ++e) {
            int b, i;
            bfly_pos<S::LOGB, LOGNR>(threadIdx.x + e * NT, a.seqfast_in, b, i);
            const SeqPos<Ix> sp = seq_pos<Ix>(a, s0 + b);
#pragma unroll
            for (int r = 0; r < S::R0; ++r) {
                const Ix n = Ix(i + r * NR);
                const Ix gidx = n * in_gn + sp.j * in_gj;
                const bool ok = sp.ok && gidx < nv;
                v[e * S::R0 + r] = ok ? load(Ix(sp.in_base + n * in_ns)) : mk(T(0), T(0));
            }
        }
    };
    if constexpr (!std::is_same<LP, PlainLoad>::value) {
        if (lp.in) {
            // the tile's table entries first, then its elements: the two are
            // dependent loads, so each kind issues as a whole
            int at[S::E];
            Ix base[NB];
#pragma unroll
            for (int e = 0; e < NB; ++e) {
                int b, i;
                bfly_pos<S::LOGB, LOGNR>(threadIdx.x + e * NT, a.seqfast_in, b, i);
                const SeqPos<Ix> sp = seq_pos<Ix>(a, s0 + b);
                base[e] = sp.in_base;
#pragma unroll
                for (int r = 0; r < S::R0; ++r) {
                    const Ix gidx = Ix(i + r * NR) * in_gn + sp.j * in_gj;
                    at[e * S::R0 + r] = sp.ok && gidx < nv ? ldg(lp.in, gidx) : -1;
                }
            }
#pragma unroll
            for (int e = 0; e < NB; ++e)
#pragma unroll
                for (int r = 0; r < S::R0; ++r) {
                    const int q = at[e * S::R0 + r];
                    v[e * S::R0 + r] = q >= 0 ? ldg(a.x, Ix(base[e] + Ix(q))) : mk(T(0), T(0));
                }
            return;
        }
    }
    if (a.stream_out & 2)
        body([&](Ix k) { return ldg_stream(a.x, k); });
    else
        body([&](Ix k) { return ldg(a.x, k); });
}

// The tile's sum of the threads' res2 (sums of |u - t|^2) into
// a.res_part[a.res_base + tile]: shuffle within each wave, one value per
// wave through LDS, summed in wave order by thread 0 (deterministic).  Every
// thread of the tile calls it; it waits for the tile's earlier LDS reads.
template <typename T, int NT>
__device__ __forceinline__ void tile_residual_sum(const TileArgs<T> &a, int64_t tile, double res2,
                                                  cpx<T> *lds) {
    double sum = res2;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) sum += __shfl_down(sum, off, 64);
    __syncthreads();  // the tile's LDS data is no longer read
    double *red = reinterpret_cast<double *>(lds);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = sum;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int q = 0; q < NT / 64; ++q) t += red[q];
        stg(a.res_part, int64_t(a.res_base + tile), t);
    }
    __syncthreads();  // red is read before the LDS is written again
}

// Epilogue of a pass's store: none (plain stores), or an object whose
// store<Ix, R>(idx, row, ok, u) takes over R elements u at offsets idx (those
// with ok set) of the output's layout, which are elements `row` of their columns;
// it is called for a few elements at a time so that it can load all of them
// before its first store.
struct PlainStore {};
constexpr int kEpilogueElems = 8;

// Store the last stage's outputs of one tile: v[e*RL + r] holds element
// i + r*N/RL (RL = 2^LOGRL, the radix of the stage that produced them) of
// sequence b in mapping cur_sf; re-stage through LDS when the store wants the
// other mapping, then apply the enclosing four-step twiddle / post-multiply /
// conj / scale and write, cropping at m_valid.
template <typename T, int LOGN, int NT, int LOGRL, bool I32 = false, int LE = -1,
          typename EP = PlainStore>
__device__ __forceinline__ void fft_tile_store(const TileArgs<T> &a, int64_t tile, cpx<T> *v,
                                               cpx<T> *lds, bool cur_sf, const EP &ep = EP()) {
    using S = TileShape<T, LOGN, NT, LE>;
    using Ix = IdxT<I32>;
    constexpr int E = S::E;
    constexpr int N = S::N;
    constexpr int RL = 1 << LOGRL;
    constexpr int LOGB = S::LOGB;
    constexpr int B = S::B;
    constexpr int SB = tile_row<T>(LOGN, LOGB);
    const int64_t s0 = tile_first_seq<T, LOGB>(a, tile);
    constexpr int NBL = E / RL;
    constexpr int LOGNRL = LOGN - LOGRL, NRL = 1 << LOGNRL;
    const bool want_sf = a.seqfast_out && B > 1;
    if (want_sf != cur_sf) {
        __syncthreads();
#pragma unroll
        for (int e = 0; e < NBL; ++e) {
            int b, i;
            bfly_pos<LOGB, LOGNRL>(threadIdx.x + e * NT, cur_sf, b, i);
#pragma unroll
            for (int r = 0; r < RL; ++r) lds[b * SB + lpad<T>(i + r * NRL)] = v[e * RL + r];
        }
        __syncthreads();
#pragma unroll
        for (int e = 0; e < NBL; ++e) {
            int b, i;
            bfly_pos<LOGB, LOGNRL>(threadIdx.x + e * NT, want_sf, b, i);
#pragma unroll
            for (int r = 0; r < RL; ++r) v[e * RL + r] = lds[b * SB + lpad<T>(i + r * NRL)];
        }
        cur_sf = want_sf;
    }
    const Ix lo_mask = (Ix(1) << a.twb_shift) - 1;
    const Ix mv = idx_bound<Ix>(a.m_valid);
    const Ix out_gn = Ix(a.out_gn), out_gj = Ix(a.out_gj), out_ns = Ix(a.out_ns);
    double res2 = 0.0;  // residual epilogue: sum of |u - t|^2 of this thread
#pragma unroll
    for (int e = 0; e < NBL; ++e) {
        int b, i;
        bfly_pos<LOGB, LOGNRL>(threadIdx.x + e * NT, cur_sf, b, i);
        const SeqPos<Ix> sp = seq_pos<Ix>(a, s0 + b);
        if (!sp.ok) continue;
        if (a.twb_hi) {
            // four-step twiddle W_L^{j n} for n = i + r NRL: the FP64 base
            // W_L^{j i} times FP64 powers of W_L^{j NRL} (two table lookups
            // each, j n < L), rounded once to T
            const Ix e0 = sp.j * Ix(i), e1 = sp.j * Ix(NRL);
            TwiddleChain<RL> w;
            w.start(cmul(ldg(a.twb_hi, Ix(e0 >> a.twb_shift)), ldg(a.twb_lo, Ix(e0 & lo_mask))),
                    cmul(ldg(a.twb_hi, Ix(e1 >> a.twb_shift)), ldg(a.twb_lo, Ix(e1 & lo_mask))));
#pragma unroll
            for (int r = 0; r < RL; ++r) {
                const cpx<double> t = w.at(r);
                v[e * RL + r] = cmul(v[e * RL + r], mk(T(t.x), T(a.twb_sign > 0 ? -t.y : t.y)));
            }
        }
        if (a.post) {
#pragma unroll
            for (int r = 0; r < RL; ++r) {
                const Ix gidx = Ix(i + r * NRL) * out_gn + sp.j * out_gj;
                if (gidx < mv) v[e * RL + r] = cmul(v[e * RL + r], ldg(a.post, gidx));
            }
        }
        if constexpr (!std::is_same<EP, PlainStore>::value) {
            constexpr int C = RL < kEpilogueElems ? RL : kEpilogueElems;
#pragma unroll
            for (int r0 = 0; r0 < RL; r0 += C) {
                Ix idx[C], row[C];
                bool ok[C];
#pragma unroll
                for (int r = 0; r < C; ++r) {
                    const Ix n = Ix(i + (r0 + r) * NRL);
                    row[r] = n * out_gn + sp.j * out_gj;
                    ok[r] = row[r] < mv;
                    idx[r] = sp.out_base + n * out_ns;
                }
                ep.template store<Ix, C>(idx, row, ok, v + e * RL + r0);
            }
            continue;
        }
#pragma unroll
        for (int r = 0; r < RL; ++r) {
            const Ix n = Ix(i + r * NRL);
            const Ix gidx = n * out_gn + sp.j * out_gj;
            if (gidx >= mv) continue;
            cpx<T> u = v[e * RL + r];
            if (a.conj_out) u = conj(u);
            if (a.target) {
                const cpx<T> d = u - ldg(a.target, Ix(sp.out_base + n * out_ns));
                if (a.res_part) res2 += double(d.x) * double(d.x) + double(d.y) * double(d.y);
                u = d;
            }
            if (a.stream_out & 1)
                stg_stream(a.y, Ix(sp.out_base + n * out_ns), scale(u, a.out_scale));
            else
                stg(a.y, Ix(sp.out_base + n * out_ns), scale(u, a.out_scale));
        }
    }
    if (a.target && a.res_part) tile_residual_sum<T, NT>(a, tile, res2, lds);
}

// Between the two transforms of a conv-mode pass: the spectrum or the residual
// (PlainMid), or an object whose apply<Ix, R>(idx, ok, u) replaces R elements u,
// which stand at offsets idx of the layout that mid_os, mid_gn, mid_gj describe
// (those with ok set: inside mid_valid).
struct PlainMid {};

// Everything after the stage-0 loads of one tile: conj / pre-multiply, the
// transform (conv: forward, spectrum, inverse), twiddle / post-multiply and
// the stores.  `lds` holds B * tile_row<T>(LOGN, LOGB) elements (tile_lds_bytes).
template <typename T, int LOGN, int NT, bool CONV, bool I32 = false, int LE = -1,
          typename EP = PlainStore, typename MP = PlainMid>
__device__ __forceinline__ void fft_tile_compute(const TileArgs<T> &a, int64_t tile, cpx<T> *v,
                                                 cpx<T> *lds, const EP &ep = EP(),
                                                 const MP &mp = MP()) {
    using S = TileShape<T, LOGN, NT, LE>;
    using Ix = IdxT<I32>;
    constexpr int LOGE = S::LOGE;
    constexpr int E = S::E;
    constexpr int N = S::N;
    using P = typename S::P;
    constexpr int LOGR0 = S::LOGR0;
    // radix of the stage that produces the stored outputs (the inverse of a
    // conv runs the radices reversed, so it ends with bits(0))
    constexpr int LOGRL = P::S > 0 ? (CONV ? P::bits(0) : P::bits(P::S - 1)) : 0;
    constexpr int R0 = 1 << LOGR0, RL = 1 << LOGRL;
    constexpr int LOGB = S::LOGB;
    constexpr int B = S::B;
    constexpr int SB = tile_row<T>(LOGN, LOGB);
    const int64_t s0 = tile_first_seq<T, LOGB>(a, tile);

    // ---- conj, pre-multiply (zero-padded positions hold zeros already)
    if (a.conj_in) {
#pragma unroll
        for (int q = 0; q < E; ++q) v[q] = conj(v[q]);
    }
    if (a.pre) {
        constexpr int NB = E / R0;
        constexpr int LOGNR = LOGN - LOGR0, NR = 1 << LOGNR;
#pragma unroll
        for (int e = 0; e < NB; ++e) {
            int b, i;
            bfly_pos<LOGB, LOGNR>(threadIdx.x + e * NT, a.seqfast_in, b, i);
            const SeqPos<Ix> sp = seq_pos<Ix>(a, s0 + b);
#pragma unroll
            for (int r = 0; r < R0; ++r) {
                const Ix n = Ix(i + r * NR);
                const Ix gidx = n * Ix(a.in_gn) + sp.j * Ix(a.in_gj);
                const bool ok = sp.ok && gidx < idx_bound<Ix>(a.n_valid);
                v[e * R0 + r] = cmul(v[e * R0 + r], ok ? ldg(a.pre, gidx) : mk(T(0), T(0)));
            }
        }
    }
    // mapping of the butterflies currently held in v (see bfly_pos), and the one
    // the store wants
    bool cur_sf = a.seqfast_in && B > 1;
    const bool out_sf = a.seqfast_out && B > 1;
    if constexpr (P::S == 0) {
        // N == 1: identity transform (conv: multiply by the single spectrum value)
        if constexpr (CONV) {
#pragma unroll
            for (int e = 0; e < E; ++e) {
                int b, i;
                bfly_pos<LOGB, 0>(threadIdx.x + e * NT, cur_sf, b, i);
                const SeqPos<Ix> sp = seq_pos<Ix>(a, s0 + b);
                if (sp.ok) {
                    const cpx<T> d = ldg(a.D, Ix(sp.j * Ix(a.d_gj)));
                    v[e] = a.conj_d ? cmulc(v[e], d) : cmul(v[e], d);
                }
            }
        }
    } else if constexpr (!CONV) {
        if (a.sign1 < 0) fft_all<T, LOGN, LOGE, -1, NT, LOGB, 0, 1>(v, lds, a.tw, cur_sf, out_sf);
        else fft_all<T, LOGN, LOGE, +1, NT, LOGB, 0, 1>(v, lds, a.tw, cur_sf, out_sf);
        if (P::S > 1) cur_sf = out_sf;
    } else {
        // forward transform ends in registers (last radix RL); multiply by the
        // spectrum there and run the inverse with the radices reversed, so its
        // first stage (radix RL, p = 1) consumes exactly those registers
        // (a residual or shrinkage in between reads and writes strided operands)
        const bool mid_sf =
            (!std::is_same<MP, PlainMid>::value || a.mid_t) && a.seqfast_in && B > 1;
        if (a.sign1 < 0) fft_all<T, LOGN, LOGE, -1, NT, LOGB, 0, 1>(v, lds, a.tw, cur_sf, mid_sf);
        else fft_all<T, LOGN, LOGE, +1, NT, LOGB, 0, 1>(v, lds, a.tw, cur_sf, mid_sf);
        if (P::S > 1) cur_sf = mid_sf;
        {
            constexpr int RF = 1 << P::bits(P::S - 1);
            constexpr int NBF = E / RF;
            constexpr int LOGNRF = LOGN - P::bits(P::S - 1), NRF = 1 << LOGNRF;
            if constexpr (!std::is_same<MP, PlainMid>::value) {
                const Ix mv = idx_bound<Ix>(a.mid_valid);
                constexpr int C = RF < kEpilogueElems ? RF : kEpilogueElems;
#pragma unroll
                for (int e = 0; e < NBF; ++e) {
                    int b, i;
                    bfly_pos<LOGB, LOGNRF>(threadIdx.x + e * NT, cur_sf, b, i);
                    const SeqPos<Ix> sp = seq_pos<Ix>(a, s0 + b);
                    const Ix si = Ix(s0 + b);
                    const Ix o = a.logJ >= 0 ? Ix(si >> a.logJ) : Ix(si / Ix(a.J));
#pragma unroll
                    for (int r0 = 0; r0 < RF; r0 += C) {
                        Ix idx[C];
                        bool ok[C];
#pragma unroll
                        for (int r = 0; r < C; ++r) {
                            const Ix g = Ix(i + (r0 + r) * NRF) * Ix(a.mid_gn) + sp.j * Ix(a.mid_gj);
                            ok[r] = sp.ok && g < mv;
                            idx[r] = o * Ix(a.mid_os) + g;
                        }
                        mp.template apply<Ix, C>(idx, ok, v + e * RF + r0);
                    }
                }
            } else if (a.mid_t) {
                // residual in place of the spectrum (see TileArgs::mid_t)
                const Ix mv = idx_bound<Ix>(a.mid_valid);
                double res2 = 0.0;
#pragma unroll
                for (int e = 0; e < NBF; ++e) {
                    int b, i;
                    bfly_pos<LOGB, LOGNRF>(threadIdx.x + e * NT, cur_sf, b, i);
                    const SeqPos<Ix> sp = seq_pos<Ix>(a, s0 + b);
                    if (!sp.ok) continue;
                    const Ix si = Ix(s0 + b);
                    const Ix o = a.logJ >= 0 ? Ix(si >> a.logJ) : Ix(si / Ix(a.J));
                    const Ix tb = o * Ix(a.mid_os);
#pragma unroll
                    for (int r = 0; r < RF; ++r) {
                        const Ix n = Ix(i + r * NRF);
                        const Ix g = n * Ix(a.mid_gn) + sp.j * Ix(a.mid_gj);
                        cpx<T> u = mk(T(0), T(0));
                        if (g < mv) {
                            const cpx<T> d = v[e * RF + r] - ldg(a.mid_t, Ix(tb + g));
                            if (a.res_part)
                                res2 += double(d.x) * double(d.x) + double(d.y) * double(d.y);
                            u = scale(d, a.mid_scale);
                        }
                        v[e * RF + r] = u;
                    }
                }
                if (a.res_part) tile_residual_sum<T, NT>(a, tile, res2, lds);
            } else {
#pragma unroll
                for (int e = 0; e < NBF; ++e) {
                    int b, i;
                    bfly_pos<LOGB, LOGNRF>(threadIdx.x + e * NT, cur_sf, b, i);
                    const SeqPos<Ix> sp = seq_pos<Ix>(a, s0 + b);
                    if (!sp.ok) continue;
#pragma unroll
                    for (int r = 0; r < RF; ++r) {
                        const Ix n = Ix(i + r * NRF);
                        const cpx<T> d = ldg(a.D, Ix(n * Ix(a.d_gn) + sp.j * Ix(a.d_gj)));
                        v[e * RF + r] =
                            a.conj_d ? cmulc(v[e * RF + r], d) : cmul(v[e * RF + r], d);
                    }
                }
            }
        }
        if (a.sign1 < 0)
            fft_all<T, LOGN, LOGE, +1, NT, LOGB, 0, 1, true>(v, lds, a.tw, cur_sf, out_sf);
        else
            fft_all<T, LOGN, LOGE, -1, NT, LOGB, 0, 1, true>(v, lds, a.tw, cur_sf, out_sf);
        if (P::S > 1) cur_sf = out_sf;
    }

    fft_tile_store<T, LOGN, NT, LOGRL, I32, LE, EP>(a, tile, v, lds, cur_sf, ep);
}

template <typename T, int LOGN, int NT, bool CONV, bool I32 = false, int LE = -1,
          typename EP = PlainStore, typename LP = PlainLoad, typename MP = PlainMid>
__device__ __forceinline__ void fft_pass_body(const TileArgs<T> &a, int64_t tile, cpx<T> *lds,
                                              const EP &ep = EP(), const LP &lp = LP(),
                                              const MP &mp = MP()) {
    cpx<T> v[TileShape<T, LOGN, NT, LE>::E];
    fft_tile_load<T, LOGN, NT, I32, LE, LP>(a, tile, v, lp);
    fft_tile_compute<T, LOGN, NT, CONV, I32, LE, EP, MP>(a, tile, v, lds, ep, mp);
}

template <typename T, int LOGN, int NT, bool CONV, bool I32, int LE = -1>
__global__ __launch_bounds__(NT) void fft_pass_kernel(const TileArgs<T> a) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    fft_pass_body<T, LOGN, NT, CONV, I32, LE>(a, xcd_remap(blockIdx.x, gridDim.x),
                                              reinterpret_cast<cpx<T> *>(smem_raw));
}

// Host-side launcher for one pass: plain or spectrum (defined in
// fm_fft_pass_*.hip).
template <typename T, bool CONV>
fm_status launch_kind(const TileArgs<T> &a, hipStream_t stream);
template <typename T>
inline fm_status launch_tile(const TileArgs<T> &a, bool conv, hipStream_t stream) {
    return conv ? launch_kind<T, true>(a, stream) : launch_kind<T, false>(a, stream);
}

// Largest tile (B*N elements) the engine supports for one precision.
template <typename T> constexpr int max_tile_elems() {
    return sizeof(T) == 4 ? 16384 : 8192;
}

// Launch shapes of a length-2^logn pass: elements per thread (2^le) and threads
// per tile.  Strided and transposed sides want several sequences per tile (a
// row segment of B elements, 8 of them 64 bytes of complex64); contiguous
// sequences do not, and run better as many small tiles, whose load, exchange
// and store phases overlap on a CU.  Where a launch has too few elements to give
// every CU a tile of the large shapes, fewer elements per thread (shorter
// chains of dependent butterflies and twiddle products) and smaller tiles cut
// its latency.
//   SHAPE_WIDE        strided or transposed sides
//   SHAPE_ROW         contiguous sides
//   SHAPE_SMALL_WIDE  the same for at most 2^19 elements,
//   SHAPE_SMALL_ROW   and for at most 2^20
// Measured (us, fft / spectrum pass; MI355X), shape = elements x threads:
//   contiguous complex64      one shape for all before   ROW            SMALL_ROW
//   1024 x 32768               32x256  111 / 142     16x128 102 / 120
//   2048 x 16384               16x512  113 / 152     16x128 104 / 127
//   4096 x 8192                16x512  109 / 149     16x256 102 / 128
//   256 x 131072               16x512  104 / 118     16x256  99 / 107
//   1024 x 16                  32x256  8.6 / 12.6                  8x128 4.5 / 6.5
//   256 x 1024                 16x512  6.2 / 8.8                   8x64  4.1 / 5.3
//   4096 x 4                   16x512  7.3 / 11.3                  8x512 5.3 / 8.2
//   four-step 2^18 complex64, 512-point columns / rows
//   32 columns                 32x256   32 / 40      8x512 28 (B = 8), 8x256 36
//   1 column                   32x256   11 / 14      8x256 5.5 / 6.3
//   contiguous complex128 1024 x 16  16x256 6.7 / 10.1   8x128 4.9 / 6.8
enum PassShape { SHAPE_WIDE = 0, SHAPE_ROW = 1, SHAPE_SMALL_WIDE = 2, SHAPE_SMALL_ROW = 3 };
constexpr int64_t kSmallWide = int64_t(1) << 19, kSmallRow = int64_t(1) << 20;

template <typename T> constexpr int pass_le(int logn, int shape) {
    const bool small = shape == SHAPE_SMALL_WIDE || shape == SHAPE_SMALL_ROW;
    if (sizeof(T) == 4) {
        if (logn == 0 || logn >= 14) return 5;
        if (logn <= 6) return shape == SHAPE_WIDE ? 4 : 3;
        if (logn <= 8) return small ? 3 : 4;
        if (logn == 9) return 3;
        if (logn == 10) return shape == SHAPE_WIDE ? 5 : (shape == SHAPE_SMALL_ROW ? 3 : 4);
        if (logn <= 12) return shape == SHAPE_SMALL_ROW ? 3 : 4;
        return 4;
    }
    if (logn == 0 || logn >= 12) return 4;
    if (logn <= 8 && shape == SHAPE_SMALL_ROW) return 2;
    if (logn <= 7) return 3;
    if (logn <= 9) return shape == SHAPE_WIDE ? 4 : 3;
    return shape == SHAPE_WIDE || shape == SHAPE_SMALL_WIDE ? 4 : 3;
}

template <typename T> constexpr int pass_nt(int logn, int shape) {
    const bool small = shape == SHAPE_SMALL_WIDE || shape == SHAPE_SMALL_ROW;
    const bool row = shape == SHAPE_ROW || shape == SHAPE_SMALL_ROW;
    if (sizeof(T) == 4) {
        if (logn == 0) return 256;
        if (logn <= 6) return small ? 64 : 256;
        if (logn == 7) return !small ? 256 : (row ? 64 : 128);
        if (logn == 8) return shape == SHAPE_SMALL_ROW ? 64 : 256;
        if (logn == 9) return shape == SHAPE_WIDE ? 512 : (shape == SHAPE_SMALL_ROW ? 128 : 256);
        if (logn == 10) return row ? 128 : 256;
        if (logn == 11) return !row ? 512 : (small ? 256 : 128);
        if (logn == 12) return shape == SHAPE_ROW ? 256 : 512;
        return 512;
    }
    if (logn == 0) return 256;
    if (logn <= 6) return small ? 64 : 256;
    if (logn == 7) return !small ? 256 : (row ? 64 : 128);
    if (logn == 8) return shape == SHAPE_SMALL_ROW ? 64 : 256;
    if (logn == 9) return !row ? 256 : (small ? 64 : 128);
    if (logn == 10) return row ? 128 : 256;
    return logn >= 13 ? 512 : 256;
}

template <typename T, int LOGN, int SHAPE> struct PassCfg {
    static constexpr int LE = pass_le<T>(LOGN, SHAPE);
    static constexpr int NT = pass_nt<T>(LOGN, SHAPE);
};

// Sequences per tile of a shape.
template <typename T> inline int pass_batch(int logn, int shape) {
    return (pass_nt<T>(logn, shape) << pass_le<T>(logn, shape)) >> logn;
}

}  // namespace fm
