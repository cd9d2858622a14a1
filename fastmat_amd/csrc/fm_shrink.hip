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

// The passes of a step: what the four-step runs in order, or the two of a one-pass
// convolution (whose residual goes through `work`).
template <typename T> struct StepPasses {
    bool one;
    TileArgs<T> first;     // column transform of y, or the forward with its residual
    TileArgs<T> rows;      // forward's spectrum pass
    TileArgs<T> residual;  // column inverse, residual, column transform
    TileArgs<T> rows_adj;  // adjoint's spectrum pass
    TileArgs<T> last;      // column inverse (or adjoint) that ends in the shrinkage
    TileArgs<T> next;      // ... and goes on with the next point's column transform
};

// a, a column inverse, goes on with the column transform `to` after its middle, in
// place in the workspace.
template <typename T>
static TileArgs<T> join_columns(TileArgs<T> a, const TileArgs<T> &to, int64_t valid) {
    a.mid_os = valid;
    a.mid_gn = a.out_gn;
    a.mid_gj = a.out_gj;
    a.mid_valid = valid;
    a.y = to.y;
    a.out_os = to.out_os; a.out_js = to.out_js; a.out_ns = to.out_ns;
    a.out_gn = to.out_gn; a.out_gj = to.out_gj; a.m_valid = to.m_valid;
    a.seqfast_out = to.seqfast_out;
    a.twb_hi = to.twb_hi; a.twb_lo = to.twb_lo;
    a.twb_shift = to.twb_shift; a.twb_sign = to.twb_sign;
    return a;
}

template <typename T>
static fm_status step_passes(const fm_conv_plan *p, const cpx<T> *y, const cpx<T> *b, int64_t k,
                             cpx<T> *x, cpx<T> *work, StepPasses<T> *out) {
    PassList<T> fw, ad;
    PipeIO io;
    memset(&io, 0, sizeof(io));
    io.k = k;
    io.D = p->D;
    io.x = y; io.ldx = p->cols; io.n_in = p->cols;
    io.y = work; io.ldy = p->rows; io.m_out = p->rows;
    io.work = work;
    fm_status st = build_pipeline<T>(p->geo, io, &fw);
    if (st) return st;
    io.x = work; io.ldx = p->rows; io.n_in = p->rows;
    io.y = x; io.ldy = p->cols; io.m_out = p->cols;
    io.conj_d = 1;
    st = build_pipeline<T>(p->geo, io, &ad);
    if (st) return st;
    out->one = p->geo.passes == 1;
    out->first = fw[0].a;
    if (out->one) {
        out->first.target = b;
        out->last = ad[0].a;
        return FM_SUCCESS;
    }
    out->rows = fw[1].a;
    out->residual = join_columns<T>(fw[2].a, ad[0].a, p->rows);
    out->residual.mid_t = b;
    out->residual.mid_scale = T(1);
    out->rows_adj = ad[1].a;
    out->last = ad[2].a;
    out->next = join_columns<T>(ad[2].a, fw[0].a, p->cols);
    return FM_SUCCESS;
}

template <typename T>
static fm_status shrink_run(const fm_conv_plan *p, const void *y, const void *b, int64_t k,
                            double L, double alpha, void *x, void *step, void *y_next,
                            const double *betas, int64_t steps, int flags, void *work,
                            hipStream_t stream) {
    StepPasses<T> q;
    fm_status st = step_passes<T>(p, (const cpx<T> *)y, (const cpx<T> *)b, k, (cpx<T> *)x,
                                  (cpx<T> *)work, &q);
    ShrinkArgs<T> s;
    s.y = (const cpx<T> *)y;
    s.x = (cpx<T> *)x;
    s.y_next = (cpx<T> *)y_next;
    s.L = T(L);
    s.alpha = T(alpha);
    for (int64_t i = 0; !st && i < steps; ++i) {
        const bool last = i == steps - 1;
        s.step = last ? (cpx<T> *)step : nullptr;
        s.beta = betas ? T(betas[i]) : T(0);
        if (q.one) {
            st = launch_tile<T>(q.first, true, stream);
            if (!st) st = launch_shrink<T, SHRINK_CONV>(q.last, s, stream);
            continue;
        }
        if (i == 0 && !(flags & 1)) st = launch_tile<T>(q.first, false, stream);
        if (!st) st = launch_tile<T>(q.rows, true, stream);
        if (!st) st = launch_tile<T>(q.residual, true, stream);
        if (!st) st = launch_tile<T>(q.rows_adj, true, stream);
        if (st) break;
        st = last && !(flags & 2) ? launch_shrink<T, SHRINK_COLUMN>(q.last, s, stream)
                                  : launch_shrink<T, SHRINK_NEXT>(q.next, s, stream);
    }
    return st;
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

extern "C" fm_status fm_conv_shrink_run(const fm_conv_plan *p, const void *y, const void *b,
                                        int64_t k, double L, double alpha, void *x, void *step,
                                        void *y_next, const double *betas, int64_t steps,
                                        int flags, void *workspace, int64_t workspace_bytes,
                                        void *stream) {
    int64_t need = 0;
    fm_status st = fm_conv_shrink_workspace_size(p, k, &need);
    if (st) return st;
    FM_REQUIRE(y && b && x && workspace, FM_ERR_VALUE, "NULL data pointer");
    FM_REQUIRE(steps >= 1, FM_ERR_VALUE, "at least one step expected");
    FM_REQUIRE(alpha > 0.0, FM_ERR_VALUE, "shrinkage threshold must be positive");
    FM_REQUIRE(steps == 1 || y == (y_next ? y_next : x), FM_ERR_VALUE,
               "several steps need the next point in place of the point");
    FM_REQUIRE(workspace_bytes >= need, FM_ERR_VALUE,
               "workspace of %lld bytes is smaller than the %lld required",
               (long long)workspace_bytes, (long long)need);
    if (p->prec == FM_COMPLEX64)
        return shrink_run<float>(p, y, b, k, L, alpha, x, step, y_next, betas, steps, flags,
                                 workspace, as_stream(stream));
    return shrink_run<double>(p, y, b, k, L, alpha, x, step, y_next, betas, steps, flags, workspace,
                              as_stream(stream));
}
