// Kernels and launch of the passes over selected elements (see fm_select.hpp),
// compiled per precision in fm_select_f32.hip and fm_select_f64.hip.
#pragma once

#include "fm_select.hpp"

namespace fm {

template <typename T, int LOGN, int LE, int NT>
__global__ __launch_bounds__(NT) void fft_pass_select_kernel(const TileArgs<T> a,
                                                             const SelectArgs<T> s) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    fft_pass_body<T, LOGN, NT, false, true, LE, SelectArgs<T>, SelectArgs<T>>(
        a, xcd_remap(blockIdx.x, gridDim.x), reinterpret_cast<cpx<T> *>(smem_raw), s, s);
}

template <typename T, int LOGN, int SHAPE>
static fm_status select_shape(TileArgs<T> a, const SelectArgs<T> &s, hipStream_t stream) {
    // (1024 complex64 points with 16 elements per thread: the tables' entries
    // come on top of the butterflies' registers)
    constexpr bool half = sizeof(T) == 4 && LOGN == 10 && SHAPE == SHAPE_WIDE;
    constexpr int LE = half ? 4 : PassCfg<T, LOGN, SHAPE>::LE;
    constexpr int NT = half ? 512 : PassCfg<T, LOGN, SHAPE>::NT;
    fm_status st = normalize_pass(a, TileShape<T, LOGN, NT, LE>::B);
    if (st) return st;
    const size_t lds = tile_lds_bytes<T>(LOGN, a.B);
    static bool attr_set = false;
    if (!attr_set) {
        (void)hipFuncSetAttribute((const void *)fft_pass_select_kernel<T, LOGN, LE, NT>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        attr_set = true;
    }
    FM_REQUIRE(a.ntiles > 0 && a.ntiles < (int64_t(1) << 31), FM_ERR_VALUE,
               "tile count %lld out of range", (long long)a.ntiles);
    ProfToken tok;
    prof_begin(stream, &tok);
    hipLaunchKernelGGL((fft_pass_select_kernel<T, LOGN, LE, NT>), dim3(unsigned(a.ntiles)),
                       dim3(NT), lds, stream, a, s);
    FM_CHECK_LAUNCH();
    if (tok.active) {
        const double own = 2.0 * double(a.O) * double(a.J) * (int64_t(1) << LOGN) * sizeof(cpx<T>);
        prof_end(stream, &tok, "fft_pass_select_kernel", a.alg_bytes > 0 ? a.alg_bytes : own,
                 5.0 * LOGN * double(a.O) * double(a.J) * (int64_t(1) << LOGN), own);
    }
    return FM_SUCCESS;
}

template <typename T, int LOGN>
static fm_status select_length_launch(const TileArgs<T> &a, const SelectArgs<T> &s,
                                      hipStream_t stream) {
    const int shape = pick_shape(a, true);
    if constexpr (LOGN >= 6 && LOGN <= 11) {
        if (shape == SHAPE_WIDE) return select_shape<T, LOGN, SHAPE_WIDE>(a, s, stream);
        if (shape == SHAPE_SMALL_WIDE) return select_shape<T, LOGN, SHAPE_SMALL_WIDE>(a, s, stream);
    }
    FM_REQUIRE(shape == SHAPE_ROW || shape == SHAPE_SMALL_ROW, FM_ERR_NOT_IMPLEMENTED,
               "strided pass of length 2^%d over selected elements", LOGN);
    if (shape == SHAPE_SMALL_ROW) return select_shape<T, LOGN, SHAPE_SMALL_ROW>(a, s, stream);
    return select_shape<T, LOGN, SHAPE_ROW>(a, s, stream);
}

template <typename T>
fm_status launch_select(const TileArgs<T> &a, const SelectArgs<T> &s, hipStream_t stream) {
#define FM_CASE(L) \
    case L: return select_length_launch<T, L>(a, s, stream);
    switch (a.logN) {
        FM_CASE(0) FM_CASE(1) FM_CASE(2) FM_CASE(3) FM_CASE(4) FM_CASE(5) FM_CASE(6) FM_CASE(7)
        FM_CASE(8) FM_CASE(9) FM_CASE(10) FM_CASE(11) FM_CASE(12)
    case 13:
        if constexpr (sizeof(T) == 4) return select_length_launch<T, 13>(a, s, stream);
        break;
    default: break;
    }
#undef FM_CASE
    set_error("unsupported pass length 2^%d over selected elements", a.logN);
    return FM_ERR_VALUE;
}

}  // namespace fm
