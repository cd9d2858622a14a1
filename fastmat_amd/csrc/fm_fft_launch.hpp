// Launch of one pass kernel (single-operator paths): tile shape, index width and
// the kernel of its length.  The kernels are compiled per precision and kind in
// fm_fft_pass_*.hip, one source each so that they build side by side.
#pragma once

#include "fm_fft_plan.hpp"

namespace fm {

template <typename T, int LOGN, bool CONV, int LE, int NT, bool I32>
static fm_status launch_shape(TileArgs<T> a, hipStream_t stream) {
    constexpr int N = 1 << LOGN;
    fm_status st = normalize_pass(a, TileShape<T, LOGN, NT, LE>::B);
    if (st) return st;
    const size_t lds = tile_lds_bytes<T>(LOGN, a.B);
    static bool attr_set = false;
    if (!attr_set) {
        (void)hipFuncSetAttribute((const void *)fft_pass_kernel<T, LOGN, NT, CONV, I32, LE>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        attr_set = true;
    }
    FM_REQUIRE(lds <= 160 * 1024, FM_ERR_VALUE, "tile of %d x %d needs %zu bytes of LDS", a.B, N,
               lds);
    FM_REQUIRE(a.ntiles > 0 && a.ntiles < (int64_t(1) << 31), FM_ERR_VALUE,
               "tile count %lld out of range", (long long)a.ntiles);
    ProfToken tok;
    prof_begin(stream, &tok);
    hipLaunchKernelGGL((fft_pass_kernel<T, LOGN, NT, CONV, I32, LE>), dim3(unsigned(a.ntiles)),
                       dim3(NT), lds, stream, a);
    FM_CHECK_LAUNCH();
    if (tok.active) {
        const double span = double(a.J) * N;
        const double esz = double(sizeof(cpx<T>));
        const double in = double(a.O) * (double(a.n_valid) < span ? double(a.n_valid) : span);
        const double out = double(a.O) * (double(a.m_valid) < span ? double(a.m_valid) : span);
        const double spec = CONV ? (a.d_gj ? span : double(N)) : 0.0;
        char name[96];
        snprintf(name, sizeof(name), "fft_pass_kernel<%s,%d,%d,%s>",
                 sizeof(T) == 4 ? "float" : "double", LOGN, NT, CONV ? "conv" : "fft");
        const double nseq = double(a.O) * double(a.J);
        const double flops = nseq * 5.0 * N * LOGN * (CONV ? 2.0 : 1.0);
        const double own = (in + out + spec) * esz;
        prof_end(stream, &tok, name, a.alg_bytes > 0 ? a.alg_bytes : own, flops, own);
    }
    return FM_SUCCESS;
}

template <typename T, int LOGN, bool CONV>
static fm_status launch_length(const TileArgs<T> &a, hipStream_t stream) {
#define FM_SHAPE(S, I32) \
    launch_shape<T, LOGN, CONV, PassCfg<T, LOGN, S>::LE, PassCfg<T, LOGN, S>::NT, I32>(a, stream)
    // offsets beyond 32 bits are rare (4 GiB tensors): one shape, right for any sides
    if (!fits_idx32(a, int64_t(1) << LOGN)) return FM_SHAPE(SHAPE_WIDE, false);
    // 1024-point complex64 passes that also multiply by a chirp (Bluestein
    // pass A / C): with the chirp loads they gain more from the extra waves of
    // 16 elements per thread than they lose to the extra stage
    if constexpr (sizeof(T) == 4 && LOGN == 10) {
        if ((a.seqfast_in || a.seqfast_out) && (a.pre || a.post))
            return launch_shape<T, LOGN, CONV, 4, 512, true>(a, stream);
    }
    switch (pick_shape(a, true)) {
    case SHAPE_ROW: return FM_SHAPE(SHAPE_ROW, true);
    case SHAPE_SMALL_WIDE: return FM_SHAPE(SHAPE_SMALL_WIDE, true);
    case SHAPE_SMALL_ROW: return FM_SHAPE(SHAPE_SMALL_ROW, true);
    default: return FM_SHAPE(SHAPE_WIDE, true);
    }
#undef FM_SHAPE
}

// Plain (CONV = false) and spectrum (CONV = true) passes of every length.
template <typename T, bool CONV>
fm_status launch_kind(const TileArgs<T> &a, hipStream_t stream) {
#define FM_PASS_CASE(L) \
    case L: return launch_length<T, L, CONV>(a, stream);
    switch (a.logN) {
        FM_PASS_CASE(0) FM_PASS_CASE(1) FM_PASS_CASE(2) FM_PASS_CASE(3) FM_PASS_CASE(4)
        FM_PASS_CASE(5) FM_PASS_CASE(6) FM_PASS_CASE(7) FM_PASS_CASE(8) FM_PASS_CASE(9)
        FM_PASS_CASE(10) FM_PASS_CASE(11) FM_PASS_CASE(12) FM_PASS_CASE(13)
    case 14:
        if constexpr (sizeof(T) == 4) return launch_length<T, 14, CONV>(a, stream);
        break;
    default:
        break;
    }
#undef FM_PASS_CASE
    set_error("unsupported sub-transform length 2^%d", a.logN);
    return FM_ERR_VALUE;
}

}  // namespace fm
