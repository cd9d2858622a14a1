// ISTA / FISTA steps on a 1-D convolution operator, with the residual and the
// shrinkage inside the convolution's own passes.
//
// Replaces the operator applies and the numpy arithmetic of the steps
// (algorithms/ISTA.py:152-168, algorithms/FISTA.py:154-178):
//     step   = y - L A^H (A y - b)
//     x_new  = step * m / (m + alpha),   m = max(|step| - alpha, 0)
//     y_next = x_new + beta (x_new - x_old)          (FISTA only)
// The forward's last pass forms A y - b: for a four-step its column inverse is
// fused with the adjoint's column transform (inverse transform, residual, zero
// beyond the rows, forward transform), so neither A y nor the residual is
// written.  The adjoint's last pass holds A^H (A y - b) in registers and writes x
// and y_next (and step where asked); for a four-step it goes on with the next
// step's column transform of y_next, whose columns are the same tile.  Per step and
// column of n = L elements that is 13 blocks of reads and writes against 21 for
// applies, residual and shrinkage apart, in 4 kernels instead of 9, launched one
// after another from here (a replayed graph of one step took longer: its nodes
// start 2 us apart, and it has to be captured and instantiated first).  50 FISTA
// iterations on 2^18 x 8 complex64: 6.71 ms with nine kernels a step, 4.75 with a
// replayed graph of five, 3.56 with these four (2 x 16.2, 16.8 and 21.8 us, the last
// one 22.5 + 10.6 as two), bound by the latency of 16 MB passes.
#pragma once

#include "fm_fft_plan.hpp"

namespace fm {

template <typename T> struct ShrinkArgs {
    const cpx<T> *y;     // the point the gradient was taken at
    cpx<T> *x;           // iterate, updated
    cpx<T> *step;        // NULL: not written
    cpx<T> *y_next;      // momentum point (may be y), or NULL
    T L, alpha, beta;    // beta: momentum of this step
};

// The shrinkage of a pass's elements: the store of a pass that ends with the
// adjoint, or the middle of one that goes on with the next point's transform.
template <typename T> struct Shrink {
    const ShrinkArgs<T> &s;
    // g: A^H (A y - b) on entry, the next point (0 outside the columns) on return
    template <typename Ix, int R>
    __device__ __forceinline__ void apply(const Ix *idx, const bool *ok, cpx<T> *g) const {
        // y, x and y_next may be one buffer: every load before the first store
        cpx<T> y[R], xo[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            y[r] = xo[r] = mk(T(0), T(0));
            if (ok[r]) {
                y[r] = ldg(s.y, idx[r]);
                if (s.y_next) xo[r] = ldg(s.x, idx[r]);
            }
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if (!ok[r]) {
                g[r] = mk(T(0), T(0));
                continue;
            }
            const cpx<T> st = mk(y[r].x - s.L * g[r].x, y[r].y - s.L * g[r].y);
            const T m = fmax(T(hypot(st.x, st.y)) - s.alpha, T(0));
            const T f = m / (m + s.alpha);
            const cpx<T> xn = scale(st, f);
            if (s.step) stg(s.step, idx[r], st);
            g[r] = xn;
            if (s.y_next) {
                g[r] = xn + scale(xn - xo[r], s.beta);
                stg(s.y_next, idx[r], g[r]);
            }
            stg(s.x, idx[r], xn);
        }
    }
    template <typename Ix, int R>
    __device__ __forceinline__ void store(const Ix *idx, const Ix *, const bool *ok,
                                          cpx<T> *g) const {
        apply<Ix, R>(idx, ok, g);
    }
};

// Where the shrinkage stands in a pass: after a column inverse (four-step), after a
// one-pass convolution, or between a column inverse and a column transform.
enum ShrinkPass { SHRINK_COLUMN, SHRINK_CONV, SHRINK_NEXT };

template <typename T, int PASS>
fm_status launch_shrink(const TileArgs<T> &a, const ShrinkArgs<T> &s, hipStream_t stream);

// Lengths launch_shrink is compiled for.
template <typename T> inline bool shrink_length(int logn, bool conv) {
    return conv ? logn <= (sizeof(T) == 4 ? 13 : 12) : logn >= 6 && logn <= 11;
}

}  // namespace fm
