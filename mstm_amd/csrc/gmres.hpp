// gmres.hpp -- the small quantities of restarted GMRES for one system: what a
// step does to them (one thread of gm_final_kernel, krylov.hip) and when a
// cycle opens.  Plain host and device code, so that it can be driven without
// a GPU.
#pragma once
#include "common.hpp"

#define GM_M 120  // longest cycle
struct GmSys {
    double bb, eps, err, scale;  // |b|^2, stop test |g|^2 / bb < eps, its last value; 1 / norm of the next vector
    int active, done;            // iterating; stopped for good (eps, niter, or a step that is not finite)
    int k, it0, niter, m;        // steps of this cycle, steps before it, step limits
    double cs[GM_M];
    cplx<double> sn[GM_M], g[GM_M + 1], h[2][GM_M + 1];
    cplx<double> R[GM_M * (GM_M + 1) / 2];  // columns of the triangular factor
};
struct GmStart {
    double bb, eps, beta;  // beta = |v_0| as given, 0: not in this cycle
    int it0, niter, m;
};

MSTM_HD bool gm_finite(double v) { return fabs(v) <= 1.7976931348623157e308; }  // false for NaN

// Does a (further) cycle start from a residual with |r|^2 = rr, after it
// steps?  Not from one that is not finite: no step could be taken from it, so
// the cycles would never end.
MSTM_HD bool gm_opens(double rr, double bb, double eps, int it, int niter)
{
    return rr > 0.0 && gm_finite(rr) && rr / bb >= eps && it < niter;
}

MSTM_HD void gm_begin(GmSys &S, const GmStart &st)
{
    S.bb = st.bb;
    S.eps = st.eps;
    S.err = st.beta * st.beta / st.bb;
    S.active = st.beta > 0.0;
    S.done = 0;
    S.k = 0;
    S.it0 = st.it0;
    S.niter = st.niter;
    S.m = st.m;
    S.scale = 1.0 / st.beta;
    S.g[0] = cmk(st.beta, 0.0);
}

// Step nv: col = the projections of column j = nv - 1, ww = |w|^2 after them,
// cs, sn = the rotations of the columns before.  A column that is not finite (a
// product that overflowed in FP32, say) is not taken: the system stops for good
// with the steps before it and their error.
MSTM_HD void gm_column(GmSys &S, const cplx<double> *col, const double *cs, const cplx<double> *sn, int nv, double ww)
{
    typedef cplx<double> Z;
    const int j = nv - 1;
    const double hn = sqrt(ww > 0.0 ? ww : 0.0);
    Z *R = S.R + (j * (j + 1)) / 2;
    Z cur = col[0];
    for (int r = 0; r < j; r++) {  // earlier rotations on column j
        const Z b = col[r + 1];
        R[r] = cadd(cscale(cur, cs[r]), cmul(sn[r], b));
        cur = csub(cscale(b, cs[r]), cmul(cconj(sn[r]), cur));
    }
    const double ca = sqrt(cur.re * cur.re + cur.im * cur.im), nu = sqrt(ca * ca + hn * hn);
    double c = 0.0;
    Z s = cmk(1.0, 0.0);
    if (ca != 0.0) {
        c = ca / nu;
        s = cscale(cur, hn / (ca * nu));
    }
    const Z d = cadd(cscale(cur, c), cscale(s, hn));
    const Z gj = S.g[j], gn = cmul(cmk(-s.re, s.im), gj);
    const double err = (gn.re * gn.re + gn.im * gn.im) / S.bb;
    // what is not finite in col has reached cur, c and d through the rotations
    if (!(gm_finite(ww) && gm_finite(d.re) && gm_finite(d.im) && gm_finite(err))) {
        S.active = 0;
        S.done = 1;
        return;
    }
    R[j] = d;
    S.cs[j] = c;
    S.sn[j] = s;
    S.g[j + 1] = gn;
    S.g[j] = cscale(gj, c);
    S.k = nv;
    S.scale = 1.0 / hn;
    S.err = err;
    S.done = S.err < S.eps || S.it0 + nv >= S.niter;
    if (S.done || hn == 0.0 || nu == 0.0 || nv == S.m) S.active = 0;
}

// g / d of the back substitution, 0 for a singular factor
MSTM_HD cplx<double> gm_pivot(cplx<double> g, cplx<double> d)
{
    const cplx<double> y = cdiv(g, d);
    return gm_finite(y.re) && gm_finite(y.im) ? y : cmk(0.0, 0.0);
}
