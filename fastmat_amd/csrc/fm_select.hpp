// Fourier transforms of selected elements: the first pass reads its column through
// an index table and the last one stores through one.
//
// Replaces the zero-padded copy and the row gather around a Fourier matrix
// (Partial.pyx:268-294).  The tables name, per element of the full column, its
// place in the selected one or -1, so what is not selected is neither read nor
// written: a transform of 2^18 x 32 complex64 with 70001 selected elements moves
// 85 MB less on its selected side than expansion or gather beside it.  The passes
// stay bound by their strided side; a table is 4 bytes an element and one for all
// columns, and the tiles of a column run on one XCD, so the table and the selected
// column (560 KB) are in its L2 while their elements come and go in random order.
// Measured on that transform, rows in random order: a selecting pass 31 us, the plain
// pass and the separate gather (24 us) or expansion (26 us) together 54; forward and
// adjoint behind a diagonal 208 -> 161 us.  2048 x 16, two launches in place of four:
// 78 -> 33 us with the host work that went.
#pragma once

#include "fm_fft_plan.hpp"

namespace fm {

template <typename T> struct SelectArgs {
    const int *in;   // NULL: elements in place
    const int *out;  // NULL: elements in place
    cpx<T> *y;       // the pass's output and its last conjugation and scale
    int conj_out;
    T out_scale;

    template <typename Ix, int R>
    __device__ __forceinline__ void store(const Ix *idx, const Ix *row, const bool *ok,
                                          const cpx<T> *v) const {
        int at[R];
#pragma unroll
        for (int r = 0; r < R; ++r) at[r] = !ok[r] ? -1 : out ? ldg(out, row[r]) : 0;
#pragma unroll
        for (int r = 0; r < R; ++r)
            if (at[r] >= 0)
                stg(y, Ix(idx[r] + Ix(at[r])),
                    scale(conj_out ? conj(v[r]) : v[r], out_scale));
    }
};

// One plain pass with its input and / or output through the tables of s.
template <typename T>
fm_status launch_select(const TileArgs<T> &a, const SelectArgs<T> &s, hipStream_t stream);

// Lengths launch_select is compiled for: contiguous passes of one-pass transforms,
// strided passes of four-step ones.
inline bool select_length(int logn, bool wide) { return wide ? logn >= 6 && logn <= 11 : logn <= 13; }

// run_pipeline with the first pass's input and the last pass's output selected.
template <typename T>
inline fm_status run_selected(const Geometry &g, PipeIO io, const int *in, const int *out,
                              hipStream_t stream, const Lanes *lanes) {
    const bool one = g.passes == 1;
    FM_REQUIRE(!(one && io.D), FM_ERR_NOT_IMPLEMENTED,
               "selected elements of a one-pass chirp transform");
    FM_REQUIRE(one || (select_length(g.logN1, true) && select_length(g.logN2, true)),
               FM_ERR_NOT_IMPLEMENTED, "selected elements of a transform of length 2^%d", g.logL);
    const int64_t cc = chunk_columns(g, io.k, sizeof(cpx<T>), lanes);
    const int64_t L = int64_t(1) << g.logL;
    const int64_t ld = io.ldx > io.ldy ? io.ldx : io.ldy;
    // (the padding covers the index sums of a last partial tile)
    FM_REQUIRE((double(cc) + 1) * double(ld > L ? ld : L) + 512 <
                   double((uint64_t(1) << 32) / sizeof(cpx<T>)),
               FM_ERR_NOT_IMPLEMENTED, "selected elements beyond 32-bit offsets");
    return run_pipeline_with<T>(
        g, io, stream, lanes, [&](const PassSpec<T> &p, int i, int n, hipStream_t s) {
            SelectArgs<T> sel;
            sel.in = i == 0 ? in : nullptr;
            sel.out = i == n - 1 ? out : nullptr;
            if (!sel.in && !sel.out) return launch_tile<T>(p.a, p.conv, s);
            TileArgs<T> a = p.a;
            // selected sides: an offset is the column's start plus the table's entry
            if (sel.in) a.in_js = a.in_ns = 0;
            if (sel.out) a.out_js = a.out_ns = 0;
            sel.y = a.y;
            sel.conj_out = a.conj_out;
            sel.out_scale = a.out_scale;
            return launch_select<T>(a, sel, s);
        });
}

}  // namespace fm
