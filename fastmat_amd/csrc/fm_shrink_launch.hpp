// Kernels and launch of the shrinkage pass (see fm_shrink.hpp), compiled per
// precision in fm_shrink_f32.hip and fm_shrink_f64.hip.
#pragma once

#include "fm_shrink.hpp"

namespace fm {

template <typename T, int LOGN, int PASS, int LE, int NT>
__global__ __launch_bounds__(NT) void fft_pass_shrink_kernel(const TileArgs<T> a,
                                                             const ShrinkArgs<T> s) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int64_t tile = xcd_remap(blockIdx.x, gridDim.x);
    cpx<T> *lds = reinterpret_cast<cpx<T> *>(smem_raw);
    const Shrink<T> sh{s};
    if constexpr (PASS == SHRINK_NEXT)
        fft_pass_body<T, LOGN, NT, true, true, LE, PlainStore, PlainLoad, Shrink<T>>(
            a, tile, lds, PlainStore(), PlainLoad(), sh);
    else
        fft_pass_body<T, LOGN, NT, PASS == SHRINK_CONV, true, LE, Shrink<T>>(a, tile, lds, sh);
}

template <typename T, int LOGN, int PASS, int LE, int NT>
static fm_status shrink_shape(TileArgs<T> a, const ShrinkArgs<T> &s, hipStream_t stream) {
    fm_status st = normalize_pass(a, TileShape<T, LOGN, NT, LE>::B);
    if (st) return st;
    const size_t lds = tile_lds_bytes<T>(LOGN, a.B);
    static bool attr_set = false;
    if (!attr_set) {
        (void)hipFuncSetAttribute((const void *)fft_pass_shrink_kernel<T, LOGN, PASS, LE, NT>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        attr_set = true;
    }
    FM_REQUIRE(a.ntiles > 0 && a.ntiles < (int64_t(1) << 31), FM_ERR_VALUE,
               "tile count %lld out of range", (long long)a.ntiles);
    ProfToken tok;
    prof_begin(stream, &tok);
    hipLaunchKernelGGL((fft_pass_shrink_kernel<T, LOGN, PASS, LE, NT>), dim3(unsigned(a.ntiles)),
                       dim3(NT), lds, stream, a, s);
    FM_CHECK_LAUNCH();
    if (tok.active) {
        // the pass's input, y (and the old x), x (and step, the momentum point)
        const double span = double(a.J) * (int64_t(1) << LOGN);
        const int64_t valid = PASS == SHRINK_NEXT ? a.mid_valid : a.m_valid;
        const double out = double(a.O) * (double(valid) < span ? double(valid) : span);
        const double in = double(a.O) * (double(a.n_valid) < span ? double(a.n_valid) : span);
        const double next = PASS == SHRINK_NEXT ? span * double(a.O) : 0.0;
        const double own =
            sizeof(cpx<T>) *
            (in + next + out * (2.0 + (s.y_next ? 2.0 : 0.0) + (s.step ? 1.0 : 0.0)));
        prof_end(stream, &tok, "fft_pass_shrink_kernel", own, 0.0);
    }
    return FM_SUCCESS;
}

template <typename T, int LOGN, int PASS>
static fm_status shrink_length_launch(const TileArgs<T> &a, const ShrinkArgs<T> &s,
                                      hipStream_t stream) {
    const int shape = pick_shape(a, true);
    if constexpr (PASS == SHRINK_CONV) {
        if (shape == SHAPE_SMALL_ROW)
            return shrink_shape<T, LOGN, PASS, PassCfg<T, LOGN, SHAPE_SMALL_ROW>::LE,
                                PassCfg<T, LOGN, SHAPE_SMALL_ROW>::NT>(a, s, stream);
        return shrink_shape<T, LOGN, PASS, PassCfg<T, LOGN, SHAPE_ROW>::LE,
                            PassCfg<T, LOGN, SHAPE_ROW>::NT>(a, s, stream);
    } else {
        if (shape == SHAPE_SMALL_WIDE)
            return shrink_shape<T, LOGN, PASS, PassCfg<T, LOGN, SHAPE_SMALL_WIDE>::LE,
                                PassCfg<T, LOGN, SHAPE_SMALL_WIDE>::NT>(a, s, stream);
        // (1024 complex64 points with 16 elements per thread: the epilogue's
        // operands come on top of the butterflies' registers)
        constexpr bool half = sizeof(T) == 4 && LOGN == 10;
        return shrink_shape<T, LOGN, PASS, half ? 4 : PassCfg<T, LOGN, SHAPE_WIDE>::LE,
                            half ? 512 : PassCfg<T, LOGN, SHAPE_WIDE>::NT>(a, s, stream);
    }
}

template <typename T, int PASS>
fm_status launch_shrink(const TileArgs<T> &a, const ShrinkArgs<T> &s, hipStream_t stream) {
#define FM_CASE(L) \
    case L: return shrink_length_launch<T, L, PASS>(a, s, stream);
    if constexpr (PASS == SHRINK_CONV) {
        switch (a.logN) {
            FM_CASE(0) FM_CASE(1) FM_CASE(2) FM_CASE(3) FM_CASE(4) FM_CASE(5) FM_CASE(6)
            FM_CASE(7) FM_CASE(8) FM_CASE(9) FM_CASE(10) FM_CASE(11) FM_CASE(12)
        case 13:
            if constexpr (sizeof(T) == 4) return shrink_length_launch<T, 13, PASS>(a, s, stream);
            break;
        default: break;
        }
    } else {
        switch (a.logN) {
            FM_CASE(6) FM_CASE(7) FM_CASE(8) FM_CASE(9) FM_CASE(10) FM_CASE(11)
        default: break;
        }
    }
#undef FM_CASE
    set_error("unsupported shrinkage pass length 2^%d", a.logN);
    return FM_ERR_VALUE;
}

}  // namespace fm
