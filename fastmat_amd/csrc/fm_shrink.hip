// C entry points of the fused shrinkage step (see fm_shrink.hpp).
#include "fm_shrink.hpp"

using namespace fm;

namespace fm {

// Whether every pass of the step has a kernel: the step's last pass is compiled
// for these lengths and with 32-bit offsets.
static bool shrink_supported(const fm_conv_plan *p, int64_t k) {
    if (p->kind == 2) return false;
    const double lim = 4294967296.0 / double(esize(p->prec));
    if (double(p->L) * double(k) + 512.0 >= lim) return false;
    const bool one = p->geo.passes == 1;
    const int logn = one ? p->geo.logL : p->geo.logN1;
    return p->prec == FM_COMPLEX64 ? shrink_length<float>(logn, one)
                                   : shrink_length<double>(logn, one);
}

template <typename T>
static fm_status shrink_step(const fm_conv_plan *p, const ShrinkArgs<T> &s, const cpx<T> *b,
                             int64_t k, cpx<T> *work, hipStream_t stream) {
    PassList<T> fw, ad;
    PipeIO io;
    memset(&io, 0, sizeof(io));
    io.k = k;
    io.D = p->D;
    // forward of y; a four-step works in place in `work`, a one-pass
    // convolution writes its residual there
    io.x = s.y; io.ldx = p->cols; io.n_in = p->cols;
    io.y = work; io.ldy = p->rows; io.m_out = p->rows;
    io.work = work;
    fm_status st = build_pipeline<T>(p->geo, io, &fw);
    if (st) return st;
    io.x = work; io.ldx = p->rows; io.n_in = p->rows;
    io.y = s.x; io.ldy = p->cols; io.m_out = p->cols;
    io.conj_d = 1;
    st = build_pipeline<T>(p->geo, io, &ad);
    if (st) return st;
    if (p->geo.passes == 1) {
        TileArgs<T> &a = fw[0].a;
        a.target = b;
        st = launch_tile<T>(a, true, stream);
        if (!st) st = launch_shrink<T, true>(ad[0].a, s, stream);
        return st;
    }
    // the forward's column inverse, the residual and the adjoint's column
    // transform in one pass, in place
    TileArgs<T> f = fw[2].a;
    const TileArgs<T> &pa = ad[0].a;
    f.mid_t = b;
    f.mid_os = p->rows;
    f.mid_gn = f.out_gn;
    f.mid_gj = f.out_gj;
    f.mid_valid = p->rows;
    f.mid_scale = T(1);
    f.y = pa.y;
    f.out_os = pa.out_os; f.out_js = pa.out_js; f.out_ns = pa.out_ns;
    f.out_gn = pa.out_gn; f.out_gj = pa.out_gj; f.m_valid = pa.m_valid;
    f.seqfast_out = pa.seqfast_out;
    f.twb_hi = pa.twb_hi; f.twb_lo = pa.twb_lo;
    f.twb_shift = pa.twb_shift; f.twb_sign = pa.twb_sign;
    st = launch_tile<T>(fw[0].a, false, stream);
    if (!st) st = launch_tile<T>(fw[1].a, true, stream);
    if (!st) st = launch_tile<T>(f, true, stream);
    if (!st) st = launch_tile<T>(ad[1].a, true, stream);
    if (!st) st = launch_shrink<T, false>(ad[2].a, s, stream);
    return st;
}

template <typename T>
static fm_status shrink_call(const fm_conv_plan *p, const void *y, const void *b, int64_t k,
                             double L, double alpha, void *x, void *step, void *y_next,
                             const double *beta_tab, int64_t *counter, void *work,
                             hipStream_t stream) {
    ShrinkArgs<T> s;
    s.y = (const cpx<T> *)y;
    s.x = (cpx<T> *)x;
    s.step = (cpx<T> *)step;
    s.y_next = (cpx<T> *)y_next;
    s.L = T(L);
    s.alpha = T(alpha);
    s.beta_tab = beta_tab;
    s.counter = counter;
    return shrink_step<T>(p, s, (const cpx<T> *)b, k, (cpx<T> *)work, stream);
}

}  // namespace fm

extern "C" fm_status fm_conv_shrink_workspace_size(const fm_conv_plan *p, int64_t k,
                                                   int64_t *bytes) {
    FM_REQUIRE(p != nullptr && bytes != nullptr, FM_ERR_VALUE, "NULL argument");
    FM_REQUIRE(k >= 1, FM_ERR_VALUE, "the shrinkage step needs at least one column");
    FM_REQUIRE(shrink_supported(p, k), FM_ERR_NOT_IMPLEMENTED,
               "no fused shrinkage step for this convolution plan and column count");
    *bytes = int64_t(esize(p->prec)) * k * (p->geo.passes == 1 ? p->rows : p->L);
    return FM_SUCCESS;
}

extern "C" fm_status fm_conv_shrink_step(const fm_conv_plan *p, const void *y, const void *b,
                                         int64_t k, double L, double alpha, void *x, void *step,
                                         void *y_next, const double *beta_tab, int64_t *counter,
                                         void *workspace, int64_t workspace_bytes, void *stream) {
    int64_t need = 0;
    fm_status st = fm_conv_shrink_workspace_size(p, k, &need);
    if (st) return st;
    FM_REQUIRE(y && b && x && workspace, FM_ERR_VALUE, "NULL data pointer");
    FM_REQUIRE((beta_tab == nullptr) == (counter == nullptr), FM_ERR_VALUE,
               "momentum table and step counter come together");
    FM_REQUIRE(workspace_bytes >= need, FM_ERR_VALUE,
               "workspace of %lld bytes is smaller than the %lld required",
               (long long)workspace_bytes, (long long)need);
    if (p->prec == FM_COMPLEX64)
        return shrink_call<float>(p, y, b, k, L, alpha, x, step, y_next, beta_tab, counter,
                                  workspace, as_stream(stream));
    return shrink_call<double>(p, y, b, k, L, alpha, x, step, y_next, beta_tab, counter, workspace,
                               as_stream(stream));
}
