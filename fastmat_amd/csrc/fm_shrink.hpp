// One ISTA / FISTA step on a 1-D convolution operator, with the residual and the
// shrinkage inside the convolution's own passes.
//
// Replaces the operator applies and the numpy arithmetic of one step
// (algorithms/ISTA.py:152-168, algorithms/FISTA.py:154-178):
//     step   = y - L A^H (A y - b)
//     x_new  = step * m / (m + alpha),   m = max(|step| - alpha, 0)
//     y_next = x_new + beta (x_new - x_old)          (FISTA only)
// The forward's last pass forms A y - b: for a four-step its column inverse is
// fused with the adjoint's column transform (inverse transform, residual, zero
// beyond the rows, forward transform), so neither A y nor the residual is
// written.  The adjoint's last pass holds A^H (A y - b) in registers and writes x
// and y_next (and step where asked).  Per step and column of n = L elements that
// is 14 blocks of reads and writes against 21 for applies, residual and shrinkage
// apart, in 5 kernels instead of 9: 50 FISTA iterations on 2^18 x 8 complex64 take
// 4.78 ms against 6.71 ms, bound by the latency of the 16 MB passes (11-23 us each).
#pragma once

#include "fm_fft_plan.hpp"

namespace fm {

template <typename T> struct ShrinkArgs {
    const cpx<T> *y;     // the point the gradient was taken at
    cpx<T> *x;           // iterate, updated
    cpx<T> *step;        // NULL: not written
    cpx<T> *y_next;      // momentum point (may be y), or NULL
    T L, alpha;
    const double *beta_tab;  // momentum per step, or NULL (0)
    int64_t *counter;        // [0] step index, [1] workgroups done (0 between launches)
};

template <typename T> struct ShrinkStore {
    const ShrinkArgs<T> &s;
    T beta;
    template <typename Ix, int R>
    __device__ __forceinline__ void store(const Ix *idx, const Ix *, const bool *ok,
                                          const cpx<T> *g) const {
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
            if (!ok[r]) continue;
            const cpx<T> st = mk(y[r].x - s.L * g[r].x, y[r].y - s.L * g[r].y);
            const T m = fmax(T(hypot(st.x, st.y)) - s.alpha, T(0));
            const T f = m / (m + s.alpha);
            const cpx<T> xn = scale(st, f);
            if (s.step) stg(s.step, idx[r], st);
            if (s.y_next)
                stg(s.y_next, idx[r], xn + scale(xn - xo[r], beta));
            stg(s.x, idx[r], xn);
        }
    }
};

// The adjoint's last pass with the shrinkage as its store.  The last workgroup to
// finish moves the step counter on: by then every workgroup has read it.
template <typename T, int LOGN, bool CONV, int LE, int NT>
__global__ __launch_bounds__(NT) void fft_pass_shrink_kernel(const TileArgs<T> a,
                                                             const ShrinkArgs<T> s) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const ShrinkStore<T> ep{s, s.beta_tab ? T(s.beta_tab[s.counter[0]]) : T(0)};
    fft_pass_body<T, LOGN, NT, CONV, true, LE, ShrinkStore<T>>(
        a, xcd_remap(blockIdx.x, gridDim.x), reinterpret_cast<cpx<T> *>(smem_raw), ep);
    if (s.beta_tab) {
        // every thread's stores used beta, so the workgroup has read the counter
        // by now; a relaxed count is enough (an agent-scope fence here would
        // write the L2 back once per workgroup: 36 us a launch instead of 23)
        __syncthreads();
        if (threadIdx.x == 0) {
            const unsigned long long done =
                __hip_atomic_fetch_add(reinterpret_cast<unsigned long long *>(s.counter + 1), 1ull,
                                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (done == gridDim.x - 1) {
                s.counter[1] = 0;
                s.counter[0] += 1;
            }
        }
    }
}

// Launch of that pass: column pass (CONV = false) or one-pass convolution.
template <typename T, bool CONV>
fm_status launch_shrink(const TileArgs<T> &a, const ShrinkArgs<T> &s, hipStream_t stream);

// Lengths launch_shrink is compiled for.
template <typename T> inline bool shrink_length(int logn, bool conv) {
    return conv ? logn <= (sizeof(T) == 4 ? 13 : 12) : logn >= 6 && logn <= 11;
}

}  // namespace fm
