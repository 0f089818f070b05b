// GMRES of one dense system on the host with the package's own step and cycle
// decisions (gmres.hpp): the cycles, products and corrections follow the
// device driver, a product from number `bad` on returns `poison`.
#include <cmath>
#include <vector>

#include "../../mstm_amd/csrc/gmres.hpp"

typedef cplx<double> Z;

// A row-major n x n.  out: {steps, err, cycles}; returns 0, or 1 if max_cycles
// did not close the system
extern "C" int gmres_host(int n, const Z *A, const Z *b, double eps, int niter, int m, int bad, double poison,
                          int max_cycles, Z *x, double *out)
{
    static GmSys S;
    int products = 0;
    auto mul = [&](const Z *v, Z *w) {
        for (int i = 0; i < n; i++) {
            w[i] = cmk(0.0, 0.0);
            for (int j = 0; j < n; j++) cfma(w[i], A[i * n + j], v[j]);
        }
        if (products++ >= bad) w[n / 2].re = poison;
    };
    auto dot = [&](const Z *a, const Z *c) {
        Z s = cmk(0.0, 0.0);
        for (int i = 0; i < n; i++) cfma(s, cconj(a[i]), c[i]);
        return s;
    };
    for (int i = 0; i < n; i++) x[i] = cmk(0.0, 0.0);
    const double bb = dot(b, b).re;
    double rr = bb, err = 1.0;
    int it = 0, cycle = 0;
    std::vector<Z> V((size_t)(m + 1) * n), r(b, b + n);
    bool open = gm_opens(bb, bb, 0.0, 0, 1);
    for (; open; cycle++) {
        if (cycle == max_cycles) return 1;
        if (cycle > 0) {
            std::vector<Z> w(n);
            mul(x, w.data());
            for (int i = 0; i < n; i++) r[i] = csub(b[i], w[i]);
            rr = dot(r.data(), r.data()).re;
            if (gm_finite(rr)) err = rr / bb;
            open = gm_opens(rr, bb, eps, it, niter);
            if (!open) break;
        }
        gm_begin(S, GmStart{bb, eps, std::sqrt(rr), it, niter, m});
        for (int i = 0; i < n; i++) V[i] = cscale(r[i], S.scale);
        for (int nv = 1; S.active; nv++) {
            Z *w = &V[(size_t)nv * n];
            mul(&V[(size_t)(nv - 1) * n], w);
            std::vector<Z> col(nv, cmk(0.0, 0.0));
            for (int pass = 0; pass < 2; pass++) {
                std::vector<Z> h(nv);
                for (int q = 0; q < nv; q++) h[q] = dot(&V[(size_t)q * n], w);
                for (int q = 0; q < nv; q++) {
                    for (int i = 0; i < n; i++) cfma(w[i], cscale(h[q], -1.0), V[(size_t)q * n + i]);
                    col[q] = cadd(col[q], h[q]);
                }
            }
            gm_column(S, col.data(), S.cs, S.sn, nv, dot(w, w).re);
            if (S.active)
                for (int i = 0; i < n; i++) w[i] = cscale(w[i], S.scale);
        }
        it += S.k;
        err = S.err;
        if (S.done) open = false;
        std::vector<Z> y(S.g, S.g + S.k);
        for (int q = S.k - 1; q >= 0; q--) {
            for (int t = q + 1; t < S.k; t++) y[q] = csub(y[q], cmul(S.R[t * (t + 1) / 2 + q], y[t]));
            y[q] = gm_pivot(y[q], S.R[q * (q + 1) / 2 + q]);
        }
        for (int q = 0; q < S.k; q++)
            for (int i = 0; i < n; i++) cfma(x[i], y[q], V[(size_t)q * n + i]);
    }
    out[0] = it;
    out[1] = err;
    out[2] = cycle;
    return 0;
}
