// observe.hip -- post-solve observables of a single-origin run on MI355X.
//
// Replaces, for a cluster without plane boundaries (single_origin_expansion,
// the reference default):
//   merge_to_common_origin     mstm-scatprops-26.f90:447-559
//       every sphere's solution is carried to the common origin by a regular
//       (vswf_type = 1) rotate-axial-rotate translation and summed, then
//       written in the E/M form of the reference;
//   the angle loop of scattering_matrix_calculation
//                              mstm-input-37.f90:3015-3118
//       over scatteringmatrix  mstm-scatprops-26.f90:1498-1573
//       (taufunc mstm-modules-33.f90:1324-1344, amplitude_to_scattering_matrix
//       mstm-scatprops-26.f90:1410-1436);
//   the w = 0, 1 moments of s00(1,1,w) of fosmexpansion
//                              mstm-scatprops-26.f90:1820-1951,
//       which give the asymmetry parameter g = s00(1,1,1) / (3 s00(1,1,0)).
// All arithmetic is FP64.  Thread j of a 256-thread workgroup owns the
// azimuthal index k = j - OBS_KOFF, so common-origin orders up to 127 are
// supported (the reference caps them at max_t_matrix_order = 100).
#include <cmath>

#include "common.hpp"
#include "kernels.hpp"
#include "specfun.hpp"

#define OBS_THREADS 256
#define OBS_KOFF 127
#define OBS_RB (2 * OBS_KOFF + 3)  // Wigner row buffer: index k + OBS_KOFF + 1
#define OBS_NB (MSTM_MAX_L * (MSTM_MAX_L + 2))
#define OBS_NCH (2 * (2 * MSTM_MAX_L + 1))  // axial chains: (m, mode)

// the reference's pi: a real(4) literal widened to real(8) (mstm-modules-33.f90:18)
#define OBS_PI_R4 3.1415927410125732

namespace {

// e^{i k phi} from e^{i phi} by repeated multiplication (as ephicoef)
__device__ cplx<double> epow(cplx<double> e1, int k)
{
    cplx<double> r = cmk(1.0, 0.0);
    cplx<double> b = k < 0 ? cconj(e1) : e1;
    for (int q = 0; q < iab(k); q++) r = cmul(r, b);
    return r;
}

// m = 0 row of the Wigner d recurrence of rotcoef (mstm-modules-33.f90:
// 1098-1175) for the thread's column k: advances (d0, d1) from degree n-1
// to n.  sben/bc/sgn are the shared edge terms, updated by the caller.
__device__ void wigner_m0(int n, int k, double ct, double edge, double &d0, double &d1)
{
    if (iab(k) > n) return;
    if (iab(k) == n) {
        d0 = (k >= 0) ? edge : ((n & 1) ? -edge : edge);
        d1 = 0.0;
        return;
    }
    double dkt = d1;
    d1 = d0;
    d0 = (ct * (double)(2 * n - 1) * d1 - sqrt((double)(n - k - 1)) * sqrt((double)(n + k - 1)) * dkt) /
         (sqrt((double)(n + k)) * sqrt((double)(n - k)));
}

// row m from row m-1 (same degree n) at column k; rp indexed k + OBS_KOFF + 1
__device__ double wigner_up(const double *rp, int n, int m, int k, double cbe2, double sbe2, double sbe)
{
    const double fmn = 1.0 / sqrt((double)(n - m + 1)) / sqrt((double)(n + m));
    double km1 = (k - 1 >= -n) ? rp[k - 1 + OBS_KOFF + 1] : 0.0;
    double kp1 = (k + 1 <= n) ? rp[k + 1 + OBS_KOFF + 1] : 0.0;
    return (sqrt((double)(n + k)) * sqrt((double)(n - k + 1)) * cbe2 * km1 -
            sqrt((double)(n - k)) * sqrt((double)(n + k + 1)) * sbe2 * kp1 - (double)k * sbe * rp[k + OBS_KOFF + 1]) *
           fmn;
}

}  // namespace

// ===========================================================================
// merge_to_common_origin.  Workgroup g takes spheres g, g+G, ... and adds
// their translated expansions (both columns, both L/R modes) into its own
// partial block part[g][4][T(T+2)] (complex), in a fixed order, so the sum
// is deterministic.  For sphere i with order L and target order
// Ti = min(T, torder_i), along r = r0 - r_i:
//   xp(n,k) = e^{ik phi} a(k,n)                           (n <= L)
//   y_m(n)  = sum_k d^n_{m,k}(beta) xp(n,k)                (forward rotation)
//   z_m(t)  = sum_s A_m(t,s) y_m(s)                        (axial, t <= Ti)
//   W(t,k)  = e^{-ik phi} sum_m d^t_{m,k}(beta) z_m(t)     (back rotation)
// The axial coefficients A_m(t,s) of axialtrancoefrecurrence
// (mstm-modules-33.f90:1566-1676, regular type) are generated upward in t
// by one thread per (m, mode) chain, seeded by vector-coupling sums of
// j_w(r); the Wigner rows of degree t are generated by the k threads in the
// same t loop, so no table larger than a few rows is ever stored.
// ===========================================================================
struct MergeArgs {
    const double *amnp;  // complex FP64, column c at amnp + 2*ldc*c
    int64_t ldc;
    const int *order, *offset, *torder;
    const double *pos;
    int nsph, T, LS;  // LS: order bound of the vccm table
    double r0x, r0y, r0z, rimed;
    const double *vccm;
    double *part;
};

__global__ __launch_bounds__(OBS_THREADS) void merge_kernel(MergeArgs a)
{
    const int g = blockIdx.x, G = gridDim.x, j = threadIdx.x, k = j - OBS_KOFF;
    const int T = a.T, b0 = T * (T + 2);
    cplx<double> *P = reinterpret_cast<cplx<double> *>(a.part) + ((int64_t)blockIdx.y * G + g) * 4 * b0;
    for (int e = j; e < 4 * b0; e += OBS_THREADS) P[e] = cmk(0.0, 0.0);

    __shared__ double jw[128 + MSTM_MAX_L + 2];
    __shared__ cplx<double> xp[4][OBS_NB];
    __shared__ cplx<double> ys[4][OBS_NB];
    __shared__ double rowF[(2 * MSTM_MAX_L + 1) * (2 * MSTM_MAX_L + 1)];
    __shared__ double rb[2][OBS_RB];
    __shared__ cplx<double> zt[2 * MSTM_MAX_L + 1][4];
    __shared__ cplx<double> act[OBS_NCH][3][MSTM_MAX_L + 1];
    __syncthreads();

    const cplx<double> *A = reinterpret_cast<const cplx<double> *>(a.amnp) + (int64_t)blockIdx.y * 2 * a.ldc;
    for (int i = g; i < a.nsph; i += G) {
        const int L = a.order[i], bl = L * (L + 2);
        const int Ti = imn(T, a.torder[i]);
        const double rx = a.r0x - a.pos[3 * i], ry = a.r0y - a.pos[3 * i + 1], rz = a.r0z - a.pos[3 * i + 2];
        const double r = sqrt(rx * rx + ry * ry + rz * rz);
        const cplx<double> *src = A + a.offset[i];
        if (r < 1e-12) {  // zero translation of regular waves: truncated copy (mtransfer)
            for (int t = imx(1, iab(k)); t <= imn(L, Ti); t++)
                for (int c = 0; c < 4; c++) {
                    cplx<double> v = src[(c >> 1) * a.ldc + (c & 1) * bl + amn(k, t, L)];
                    cplx<double> &o = P[c * b0 + amn(k, t, T)];
                    o = cadd(o, v);
                }
            continue;
        }
        const double ct = rz / r, rho = sqrt(rx * rx + ry * ry);
        cplx<double> e1 = cmk(1.0, 0.0);
        if (!(rx == 0.0 && ry == 0.0)) e1 = cmk(rx / rho, ry / rho);
        const double sbe = (fabs(ct) >= 1.0) ? 0.0 : sqrt(fabs((1.0 + ct) * (1.0 - ct)));
        const double cbe2 = 0.5 * (1.0 + ct), sbe2 = 0.5 * (1.0 - ct);
        if (j == 0) sph_bessel_j(Ti + L, r * a.rimed, jw);
        for (int e = j; e < 4 * bl; e += OBS_THREADS) {
            const int c = e / bl, q = e - c * bl;
            int n = (int)sqrt((double)(q + 1));
            while (n * (n + 2) < q + 1) n++;
            while ((n - 1) * (n + 1) >= q + 1) n--;
            const int kk = q + 1 - n * (n + 1);
            xp[c][q] = cmul(epow(e1, kk), src[(c >> 1) * a.ldc + (c & 1) * bl + amn(kk, n, L)]);
        }
        __syncthreads();

        // ---- forward rotation, degrees n <= L ----------------------------
        double d0 = (k == 0) ? 1.0 : 0.0, d1 = 0.0, sben = 1.0, bc = 1.0;
        int sgn = 1;
        for (int n = 1; n <= L; n++) {
            sgn = -sgn;
            sben = sben * sbe / 2.0;
            if (sben < 1e-30) sben = 0.0;
            bc = bc * sqrt((double)(2 * n) * (double)(2 * n - 1)) / (double)n;
            wigner_m0(n, k, ct, sgn * sben * bc, d0, d1);
            const int w2 = 2 * n + 1;
            if (iab(k) <= n) {
                rb[0][k + OBS_KOFF + 1] = d0;
                rowF[n * w2 + (k + n)] = d0;
            }
            __syncthreads();
            int cur = 0;
            for (int m = 1; m <= n; m++) {
                if (iab(k) <= n) {
                    double v = wigner_up(rb[cur], n, m, k, cbe2, sbe2, sbe);
                    rb[1 - cur][k + OBS_KOFF + 1] = v;
                    rowF[(m + n) * w2 + (k + n)] = v;
                    rowF[(-m + n) * w2 + (-k + n)] = v * (((m + k) & 1) ? -1.0 : 1.0);
                }
                __syncthreads();
                cur ^= 1;
            }
            for (int e = j; e < 4 * w2; e += OBS_THREADS) {
                const int c = e / w2, m = e - c * w2 - n;
                cplx<double> s = cmk(0.0, 0.0);
                for (int kk = -n; kk <= n; kk++) crfma(s, rowF[(m + n) * w2 + (kk + n)], xp[c][nk(n, kk)]);
                ys[c][nk(n, m)] = s;
            }
            __syncthreads();
        }

        // ---- axial chains + back rotation, degrees t <= Ti ----------------
        const int nch = 2 * (2 * L + 1);
        const int cm = (j >> 1) - L, cp = j & 1, cm1 = imx(1, iab(cm));
        d0 = (k == 0) ? 1.0 : 0.0;
        d1 = 0.0;
        sben = 1.0;
        bc = 1.0;
        sgn = 1;
        const cplx<double> ephk = epow(e1, -k);
        for (int t = 1; t <= Ti; t++) {
            if (j < nch) {
                cplx<double> z0 = cmk(0.0, 0.0), z1 = cmk(0.0, 0.0);
                if (t >= cm1) {
                    cplx<double> *Rt = act[j][t % 3], *Rn = act[j][(t + 2) % 3], *Rm = act[j][(t + 1) % 3];
                    auto seed = [&](int n, int l) -> cplx<double> {
                        const int wmin = iab(n - l), wmax = n + l;
                        const double *vc = a.vccm + (((int64_t)n * (a.LS + 1) + l) * (2 * a.LS + 1) + (cm + a.LS)) *
                                                        (2 * a.LS + 1) - wmin;
                        double se = 0.0, so = 0.0;
                        for (int w = wmin; w <= wmax; w += 2) se = fma(vc[w], jw[w], se);
                        for (int w = wmin + 1; w <= wmax - 1; w += 2) so = fma(vc[w], jw[w], so);
                        return cmk(se, cp == 0 ? so : -so);
                    };
                    if (t == cm1) {
                        for (int l = cm1; l <= L; l++) Rt[l] = seed(t, l);
                    } else {
                        // row t from rows t-1 (Rn) and t-2 (Rm); column l = L from its seed
                        const int n = t - 1;
                        const double sp = (cp == 0) ? 1.0 : -1.0;
                        for (int l = cm1; l <= L - 1; l++) {
                            cplx<double> v = cscale(Rn[l + 1], -ax_fnp1(cm, l));
                            const double f = sp * (ax_fn(cm, l) - ax_fn(cm, n));
                            v = cadd(v, cmk(-f * Rn[l].im, f * Rn[l].re));
                            if (l >= cm1 + 1) v = cadd(v, cscale(Rn[l - 1], ax_fnm1(cm, l)));
                            if (n > cm1) v = cadd(v, cscale(Rm[l], ax_fnm1(cm, n)));
                            Rt[l] = cscale(v, 1.0 / ax_fnp1(cm, n));
                        }
                        Rt[L] = seed(t, L);
                    }
                    for (int s = cm1; s <= L; s++) {
                        cfma(z0, Rt[s], ys[cp][nk(s, cm)]);
                        cfma(z1, Rt[s], ys[2 + cp][nk(s, cm)]);
                    }
                }
                zt[cm + L][cp] = z0;
                zt[cm + L][2 + cp] = z1;
            }
            sgn = -sgn;
            sben = sben * sbe / 2.0;
            if (sben < 1e-30) sben = 0.0;
            bc = bc * sqrt((double)(2 * t) * (double)(2 * t - 1)) / (double)t;
            wigner_m0(t, k, ct, sgn * sben * bc, d0, d1);
            if (iab(k) <= t) rb[0][k + OBS_KOFF + 1] = d0;
            __syncthreads();
            cplx<double> W[4] = {cmk(0.0, 0.0), cmk(0.0, 0.0), cmk(0.0, 0.0), cmk(0.0, 0.0)};
            const int kmx = imn(t, L);
            int cur = 0;
            for (int m = 0; m <= kmx; m++) {
                if (iab(k) <= t) {
                    const double dm = rb[cur][k + OBS_KOFF + 1];
                    for (int c = 0; c < 4; c++) crfma(W[c], dm, zt[m + L][c]);
                    if (m > 0) {
                        const double dn = rb[cur][-k + OBS_KOFF + 1] * (((m + k) & 1) ? -1.0 : 1.0);
                        for (int c = 0; c < 4; c++) crfma(W[c], dn, zt[-m + L][c]);
                    }
                    if (m < kmx) rb[1 - cur][k + OBS_KOFF + 1] = wigner_up(rb[cur], t, m + 1, k, cbe2, sbe2, sbe);
                }
                __syncthreads();
                cur ^= 1;
            }
            if (iab(k) <= t) {
                const int ad = amn(k, t, T);
                for (int c = 0; c < 4; c++) {
                    cplx<double> &o = P[c * b0 + ad];
                    o = cadd(o, cmul(ephk, W[c]));
                }
            }
        }
        __syncthreads();
    }
}

// a0[col][0][e] = sum_g (W_L + W_R), a0[col][1][e] = sum_g (W_L - W_R).
// KS lanes share an output: lane j adds the partials g = j, j + KS, ...,
// then a fixed butterfly over the lanes (deterministic), so that the G
// partials of an output are loaded many at a time.
template <int KS>
__global__ __launch_bounds__(256) void merge_reduce_kernel(const double *part, int G, int T, double *a0)
{
    const int b0 = T * (T + 2);
    const int e = (int)(((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / KS), j = threadIdx.x % KS;
    const bool live = e < 2 * b0;
    const int col = live ? e / b0 : 0, q = live ? e - col * b0 : 0;
    const cplx<double> *P = reinterpret_cast<const cplx<double> *>(part) + (int64_t)blockIdx.y * G * 4 * b0;
    cplx<double> s0 = cmk(0.0, 0.0), s1 = cmk(0.0, 0.0);
    if (live) {
#pragma unroll 4
        for (int g = j; g < G; g += KS) {
            s0 = cadd(s0, P[(int64_t)g * 4 * b0 + (2 * col) * b0 + q]);
            s1 = cadd(s1, P[(int64_t)g * 4 * b0 + (2 * col + 1) * b0 + q]);
        }
    }
#pragma unroll
    for (int w = 1; w < KS; w <<= 1) {
        s0.re += __shfl_xor(s0.re, w, KS);
        s0.im += __shfl_xor(s0.im, w, KS);
        s1.re += __shfl_xor(s1.re, w, KS);
        s1.im += __shfl_xor(s1.im, w, KS);
    }
    if (!live || j) return;
    cplx<double> *O = reinterpret_cast<cplx<double> *>(a0) + ((int64_t)blockIdx.y * 2 + col) * 2 * b0;
    O[q] = cadd(s0, s1);
    O[b0 + q] = csub(s0, s1);
}

hipError_t launch_merge(const double *amnp, int64_t ldc, const int *order, const int *offset, const int *torder,
                        const double *pos, int nsph, int T, int LS, const double *r0, double rimed, const double *vccm,
                        double *part, int G, double *a0, hipStream_t st, int npair)
{
    if (npair < 1 || npair > 65535 || T < 1 || T > OBS_KOFF || LS < 1 || LS > MSTM_MAX_L || G < 1) return hipErrorInvalidValue;
    MergeArgs a{amnp, ldc, order, offset, torder, pos, nsph, T, LS, r0[0], r0[1], r0[2], rimed, vccm, part};
    hipLaunchKernelGGL(merge_kernel, dim3(G, npair), dim3(OBS_THREADS), 0, st, a);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const int64_t n = 2 * T * (T + 2);
    if (G >= 64)
        hipLaunchKernelGGL(merge_reduce_kernel<16>, dim3((unsigned)((n * 16 + 255) / 256), npair), dim3(256), 0, st,
                           part, G, T, a0);
    else
        hipLaunchKernelGGL(merge_reduce_kernel<4>, dim3((unsigned)((n * 4 + 255) / 256), npair), dim3(256), 0, st,
                           part, G, T, a0);
    return hipGetLastError();
}

// ===========================================================================
// distribute_from_common_origin (mstm-scatprops-26.f90:561-669), vswf_type 1,
// for the unit excitations of tmatrix_solution (mstm-solver-8.f90:162-182):
// every column of common-origin degree l at once.  Column (k0, q) holds the
// origin expansion a(k0, l) = (1/2, -(-1)^q / 2) in the two L/R modes
// (the TE/TM unit vector of the T-matrix basis); it is carried to sphere i
// along d = r_i - r0, from order l to the sphere's order L:
//   W_p(t,k) = e^{-ik phi} sum_m d^t_{m,k} A^p_m(t <- l) d^l_{m,k0} e^{ik0 phi}
// for t <= L, |m| <= min(t, l).  The axial coefficients are the explicit
// vector-coupling sums A^p_m(t <- l) = sum_w c(t,l,m,w) j_w(|d|), even w - |t-l|
// real, odd imaginary with the sign of the mode (the seeds of
// axialtrancoefrecurrence, mstm-modules-33.f90:1566-1676).  The degree-l
// Wigner rows and the rows of every degree t <= L come from the recurrences
// of rotcoef in one degree loop, one thread per column k.  Column kq =
// 2(k0+l) + q-1 is written at out + 2*ldc*kq (complex, solver packing).
// One 256-thread workgroup per sphere (spheres g, g+G, ...); every output
// element is written once.
// ===========================================================================
struct DistArgs {
    const int *order, *offset;
    const double *pos;
    int nsph, l, LS;  // LS: order bound of the vccd table
    double r0x, r0y, r0z, rimed;
    const double *vccd;  // [l'][t][m + LS][w - |t - l'|], l' source, t target
    double *out;
    int64_t ldc;
};

#define DIST_ROWB ((MSTM_MAX_L) * (2 * MSTM_MAX_L - 1) * (2 * MSTM_MAX_L + 1) / 3 + (2 * MSTM_MAX_L + 1) * (2 * MSTM_MAX_L + 1))

__device__ inline int rowb_off(int t) { return t * (2 * t - 1) * (2 * t + 1) / 3; }  // sum_{t'<t} (2t'+1)^2

__global__ __launch_bounds__(OBS_THREADS) void distribute_kernel(DistArgs a)
{
    const int g = blockIdx.x, G = gridDim.x, j = threadIdx.x, k = j - OBS_KOFF;
    const int l = a.l, ncol = 2 * (2 * l + 1);
    __shared__ double jw[128 + MSTM_MAX_L + 2];
    __shared__ double rowL[MSTM_MAX_L + 1][2 * OBS_KOFF + 1];  // d^l_{m,k0}, m >= 0
    __shared__ double rowB[DIST_ROWB];                          // d^t_{m,k}, t <= L
    __shared__ double rb[2][OBS_RB];
    __shared__ cplx<double> az[2][2 * MSTM_MAX_L + 1][MSTM_MAX_L + 1];
    __shared__ cplx<double> ph[2 * OBS_KOFF + 1];  // e^{i k phi}
    cplx<double> *O = reinterpret_cast<cplx<double> *>(a.out);

    for (int i = g; i < a.nsph; i += G) {
        const int L = a.order[i], bl = L * (L + 2), mm = imn(l, L);
        const double dx = a.pos[3 * i] - a.r0x, dy = a.pos[3 * i + 1] - a.r0y, dz = a.pos[3 * i + 2] - a.r0z;
        const double r = sqrt(dx * dx + dy * dy + dz * dz);
        cplx<double> *dst = O + a.offset[i];
        const int nel = (2 * l + 1) * 2 * bl;
        if (r < 1e-12) {  // zero translation of regular waves: truncated copy (mtransfer)
            for (int e = j; e < nel; e += OBS_THREADS) {
                const int k0i = e / (2 * bl), rem = e - k0i * 2 * bl, p = rem / bl, w = rem - p * bl;
                int t = (int)sqrt((double)(w + 1));
                while (t * (t + 2) < w + 1) t++;
                while ((t - 1) * (t + 1) >= w + 1) t--;
                const int kk = w + 1 - t * (t + 1), k0 = k0i - l;
                const double v = (t == l && kk == k0) ? 0.5 : 0.0;
                const int ad = p * bl + amn(kk, t, L);
                dst[(int64_t)(2 * k0i) * a.ldc + ad] = cmk(v, 0.0);
                dst[(int64_t)(2 * k0i + 1) * a.ldc + ad] = cmk(p == 0 ? v : -v, 0.0);
            }
            continue;
        }
        const double ct = dz / r, rho = sqrt(dx * dx + dy * dy);
        cplx<double> e1 = cmk(1.0, 0.0);
        if (!(dx == 0.0 && dy == 0.0)) e1 = cmk(dx / rho, dy / rho);
        const double sbe = (fabs(ct) >= 1.0) ? 0.0 : sqrt(fabs((1.0 + ct) * (1.0 - ct)));
        const double cbe2 = 0.5 * (1.0 + ct), sbe2 = 0.5 * (1.0 - ct);
        const int nph = imx(l, L);
        if (iab(k) <= nph) ph[k + OBS_KOFF] = epow(e1, k);
        if (j == 0) sph_bessel_j(l + L, r * a.rimed, jw);
        __syncthreads();

        // ---- axial coefficients A^p_m(t <- l), t = m1..L ------------------
        for (int e = j; e < 2 * (2 * mm + 1) * L; e += OBS_THREADS) {
            const int p = e / ((2 * mm + 1) * L), rem = e - p * (2 * mm + 1) * L, mi = rem / L, t = rem - mi * L + 1;
            const int m = mi - mm;
            if (t < imx(1, iab(m))) continue;
            const int wmin = iab(t - l), wmax = t + l;
            const double *vc = a.vccd + (((int64_t)l * (a.LS + 1) + t) * (2 * a.LS + 1) + (m + a.LS)) *
                                            (2 * a.LS + 1) - wmin;
            double se = 0.0, so = 0.0;
            for (int w = wmin; w <= wmax; w += 2) se = fma(vc[w], jw[w], se);
            for (int w = wmin + 1; w <= wmax - 1; w += 2) so = fma(vc[w], jw[w], so);
            az[p][m + MSTM_MAX_L][t] = cmk(se, p == 0 ? so : -so);
        }

        // ---- Wigner rows: degree l (m <= min(l, L)) and every degree t <= L
        double d0 = (k == 0) ? 1.0 : 0.0, d1 = 0.0, sben = 1.0, bc = 1.0;
        int sgn = 1;
        for (int n = 1; n <= nph; n++) {
            sgn = -sgn;
            sben = sben * sbe / 2.0;
            if (sben < 1e-30) sben = 0.0;
            bc = bc * sqrt((double)(2 * n) * (double)(2 * n - 1)) / (double)n;
            wigner_m0(n, k, ct, sgn * sben * bc, d0, d1);
            const bool needB = n <= L, needL = n == l;
            if (!needB && !needL) continue;
            const int w2 = 2 * n + 1, ob = rowb_off(n);
            if (iab(k) <= n) {
                rb[0][k + OBS_KOFF + 1] = d0;
                if (needB) rowB[ob + n * w2 + (k + n)] = d0;
                if (needL) rowL[0][k + OBS_KOFF] = d0;
            }
            __syncthreads();
            const int mtop = needB ? n : mm;
            int cur = 0;
            for (int m = 1; m <= mtop; m++) {
                if (iab(k) <= n) {
                    const double v = wigner_up(rb[cur], n, m, k, cbe2, sbe2, sbe);
                    rb[1 - cur][k + OBS_KOFF + 1] = v;
                    if (needB) {
                        rowB[ob + (m + n) * w2 + (k + n)] = v;
                        rowB[ob + (-m + n) * w2 + (-k + n)] = v * (((m + k) & 1) ? -1.0 : 1.0);
                    }
                    if (needL && m <= mm) rowL[m][k + OBS_KOFF] = v;
                }
                __syncthreads();
                cur ^= 1;
            }
        }
        __syncthreads();

        // ---- columns: back rotation of the translated unit harmonic -------
        for (int e = j; e < nel; e += OBS_THREADS) {
            const int k0i = e / (2 * bl), rem = e - k0i * 2 * bl, p = rem / bl, w = rem - p * bl;
            int t = (int)sqrt((double)(w + 1));
            while (t * (t + 2) < w + 1) t++;
            while ((t - 1) * (t + 1) >= w + 1) t--;
            const int kk = w + 1 - t * (t + 1), k0 = k0i - l, mt = imn(t, l), w2 = 2 * t + 1, ob = rowb_off(t);
            cplx<double> acc = cmk(0.0, 0.0);
            for (int m = -mt; m <= mt; m++) {
                // d^l_{m,k0}; negative m from d^l_{-m,-k0} (-1)^{m+k0}
                const double dl = (m >= 0) ? rowL[m][k0 + OBS_KOFF]
                                           : rowL[-m][-k0 + OBS_KOFF] * (((m + k0) & 1) ? -1.0 : 1.0);
                crfma(acc, rowB[ob + (m + t) * w2 + (kk + t)] * dl, az[p][m + MSTM_MAX_L][t]);
            }
            const cplx<double> v = cmul(cmul(ph[-kk + OBS_KOFF], ph[k0 + OBS_KOFF]), acc);
            const int ad = p * bl + amn(kk, t, L);
            dst[(int64_t)(2 * k0i) * a.ldc + ad] = cscale(v, 0.5);
            dst[(int64_t)(2 * k0i + 1) * a.ldc + ad] = cscale(v, p == 0 ? 0.5 : -0.5);
        }
        __syncthreads();
    }
}

hipError_t launch_distribute(int l, const int *order, const int *offset, const double *pos, int nsph, int LS,
                             const double *r0, double rimed, const double *vccd, double *out, int64_t ldc, int G,
                             hipStream_t st)
{
    if (l < 1 || l > OBS_KOFF || LS < 1 || LS > MSTM_MAX_L || G < 1) return hipErrorInvalidValue;
    DistArgs a{order, offset, pos, nsph, l, LS, r0[0], r0[1], r0[2], rimed, vccd, out, ldc};
    hipLaunchKernelGGL(distribute_kernel, dim3(G), dim3(OBS_THREADS), 0, st, a);
    return hipGetLastError();
}

// ===========================================================================
// scatteringmatrix at one (cos theta, phi) per workgroup, rotate_plane = F,
// normalize_s11 = F.  Thread j owns the azimuthal index c = j - OBS_KOFF;
// the d^n_{+-1,c} rows of taufunc come from the same recurrences as above.
// sm[16*ia + ...] holds the Fortran sm(4,4) (column-major) of angle ia.
// ===========================================================================
__global__ __launch_bounds__(OBS_THREADS) void scatmat_kernel(const double *a0, int T, const double *ctv,
                                                              const double *phiv, double rimed, double *sm)
{
    const int ia = blockIdx.x, j = threadIdx.x, c = j - OBS_KOFF;
    const int b0 = T * (T + 2);
    const double ct = ctv[ia], ph = phiv[ia];
    const double sbe = (fabs(ct) >= 1.0) ? 0.0 : sqrt(fabs((1.0 + ct) * (1.0 - ct)));
    const double cbe2 = 0.5 * (1.0 + ct), sbe2 = 0.5 * (1.0 - ct);
    __shared__ double r0b[OBS_RB], r1b[OBS_RB];
    __shared__ cplx<double> red[4][OBS_THREADS];
    const cplx<double> *A = reinterpret_cast<const cplx<double> *>(a0);
    const cplx<double> eph = epow(cmk(cos(ph), sin(ph)), c);
    cplx<double> acc[4] = {cmk(0.0, 0.0), cmk(0.0, 0.0), cmk(0.0, 0.0), cmk(0.0, 0.0)};
    double d0 = (c == 0) ? 1.0 : 0.0, d1 = 0.0, sben = 1.0, bc = 1.0;
    int sgn = 1;
    cplx<double> cin = cmk(1.0, 0.0);
    for (int n = 1; n <= T; n++) {
        cin = cmk(cin.im, -cin.re);  // (-i)^n
        sgn = -sgn;
        sben = sben * sbe / 2.0;
        if (sben < 1e-30) sben = 0.0;
        bc = bc * sqrt((double)(2 * n) * (double)(2 * n - 1)) / (double)n;
        wigner_m0(n, c, ct, sgn * sben * bc, d0, d1);
        const bool on = iab(c) <= n;
        if (on) r0b[c + OBS_KOFF + 1] = d0;
        __syncthreads();
        double dp1 = 0.0;
        if (on) {
            dp1 = wigner_up(r0b, n, 1, c, cbe2, sbe2, sbe);
            r1b[c + OBS_KOFF + 1] = dp1;
        }
        __syncthreads();
        if (on) {
            // d^n_{-1,c} = (-1)^{1+c} d^n_{1,-c}
            const double dm1 = r1b[-c + OBS_KOFF + 1] * ((c & 1) ? 1.0 : -1.0);
            const double fnm = sqrt((double)(2 * n + 1) / 2.0) / 4.0;
            const double tau[2] = {-fnm * (-dm1 + dp1), -fnm * (dm1 + dp1)};
            const int ad = amn(c, n, T);
            for (int p = 0; p < 2; p++) {
                const cplx<double> va = A[p * b0 + ad];
                const cplx<double> vb = cscale(A[2 * b0 + p * b0 + ad], -1.0);
                const cplx<double> ca = cmul(cin, eph);
                const cplx<double> ci_ca = cmk(-ca.im, ca.re);
                cfma(acc[0], cscale(ca, tau[1 - p]), vb);
                cfma(acc[1], cscale(ci_ca, tau[p]), va);
                cfma(acc[2], cscale(ci_ca, tau[p]), vb);
                cfma(acc[3], cscale(ca, tau[1 - p]), va);
            }
        }
        __syncthreads();
    }
    for (int q = 0; q < 4; q++) red[q][j] = acc[q];
    __syncthreads();
    for (int s = OBS_THREADS / 2; s > 0; s >>= 1) {
        if (j < s)
            for (int q = 0; q < 4; q++) red[q][j] = cadd(red[q][j], red[q][j + s]);
        __syncthreads();
    }
    if (j == 0) {
        const double f = 4.0 / sqrt(2.0 * (1.0 / OBS_PI_R4));
        cplx<double> sa[4];
        for (int q = 0; q < 4; q++) sa[q] = cscale(red[q][0], f);
        auto sp = [&](int x, int y) { return cmul(sa[x - 1], cconj(sa[y - 1])); };
        double o[16];
#define SMO(x, y) o[((x) - 1) + 4 * ((y) - 1)]
        SMO(1, 1) = sp(1, 1).re + sp(2, 2).re + sp(3, 3).re + sp(4, 4).re;
        SMO(1, 2) = -sp(1, 1).re + sp(2, 2).re - sp(3, 3).re + sp(4, 4).re;
        SMO(2, 1) = -sp(1, 1).re + sp(2, 2).re + sp(3, 3).re - sp(4, 4).re;
        SMO(2, 2) = sp(1, 1).re + sp(2, 2).re - sp(3, 3).re - sp(4, 4).re;
        SMO(3, 3) = 2.0 * (sp(1, 2).re + sp(3, 4).re);
        SMO(3, 4) = 2.0 * (sp(2, 1).im + sp(4, 3).im);
        SMO(4, 3) = 2.0 * (sp(1, 2).im - sp(3, 4).im);
        SMO(4, 4) = 2.0 * (sp(1, 2).re - sp(3, 4).re);
        SMO(1, 3) = 2.0 * (sp(2, 3).re + sp(1, 4).re);
        SMO(3, 1) = 2.0 * (sp(2, 4).re + sp(1, 3).re);
        SMO(1, 4) = -2.0 * (sp(2, 3).im - sp(1, 4).im);
        SMO(4, 1) = -2.0 * (sp(4, 2).im + sp(1, 3).im);
        SMO(2, 3) = -2.0 * (sp(2, 3).re - sp(1, 4).re);
        SMO(3, 2) = -2.0 * (sp(2, 4).re - sp(1, 3).re);
        SMO(2, 4) = -2.0 * (sp(2, 3).im + sp(1, 4).im);
        SMO(4, 2) = -2.0 * (sp(4, 2).im - sp(1, 3).im);
#undef SMO
        for (int q = 0; q < 16; q++) sm[16 * (int64_t)ia + q] = o[q] / (4.0 * OBS_PI_R4) / rimed;
    }
}

hipError_t launch_scatmat(const double *a0, int T, int nang, const double *ct, const double *phi, double rimed,
                          double *sm, hipStream_t st)
{
    if (T < 1 || T > OBS_KOFF || nang < 1) return hipErrorInvalidValue;
    hipLaunchKernelGGL(scatmat_kernel, dim3(nang), dim3(OBS_THREADS), 0, st, a0, T, ct, phi, rimed, sm);
    return hipGetLastError();
}

// ===========================================================================
// s00(1,1,w), w = 0, 1, of fosmexpansion: one thread per (n, m) of the
// common-origin expansion sums over l = n-1..n+1 and the E/M indices
// (p, q); only the terms whose Clebsch-Gordan coefficients reach w <= 1
// are nonzero.  cgm[((n*3 + l-n+1)*(2T+1) + m+T)*2 + w] = C(n,-m;l,m|w,0),
// cg1[(n*3 + l-n+1)*2 + w] = C(n,-1;l,1|w,0).  Block partials out[2*block].
// ===========================================================================
__global__ __launch_bounds__(256) void s00_moments_kernel(const double *a0, int T, const double *cgm,
                                                          const double *cg1, double *out)
{
    const int b0 = T * (T + 2);
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    double s[2] = {0.0, 0.0};
    if (e < b0) {
        int n = (int)sqrt((double)(e + 1));
        while (n * (n + 2) < e + 1) n++;
        while ((n - 1) * (n + 1) >= e + 1) n--;
        const int m = e + 1 - n * (n + 1);
        const cplx<double> *A = reinterpret_cast<const cplx<double> *>(a0);
        const double m1m = (iab(m) & 1) ? -1.0 : 1.0;
        for (int l = imx(1, n - 1); l <= imn(T, n + 1); l++) {
            if (iab(m) > l) continue;
            const int li = l - n + 1;
            // fnl = sqrt((2n+1)(2l+1)) i^(l-n)
            const double fm = sqrt((double)((2 * n + 1) * (2 * l + 1)));
            const int ph = ((l - n) % 4 + 4) % 4;
            const cplx<double> fnl = ph == 0 ? cmk(fm, 0.0) : ph == 1 ? cmk(0.0, fm) : ph == 2 ? cmk(-fm, 0.0) : cmk(0.0, -fm);
            for (int p = 0; p < 2; p++)
                for (int q = 0; q < 2; q++) {
                    const cplx<double> a1n = A[p * b0 + amn(m, n, T)], a1l = A[q * b0 + amn(m, l, T)];
                    const cplx<double> a2n = A[2 * b0 + p * b0 + amn(m, n, T)], a2l = A[2 * b0 + q * b0 + amn(m, l, T)];
                    const cplx<double> a1122 = cadd(cmul(a1n, cconj(a1l)), cmul(a2n, cconj(a2l)));
                    const cplx<double> fa = cmul(fnl, a1122);
                    for (int w = iab(n - l); w <= 1; w++) {
                        if (((n + l + w + p + q) & 1) != 0) continue;
                        const double cw = cg1[(n * 3 + li) * 2 + w] * cgm[((n * 3 + li) * (2 * T + 1) + m + T) * 2 + w];
                        s[w] += -(m1m * fa.re * cw) / 2.0;
                    }
                }
        }
    }
    __shared__ double red[2][256];
    red[0][threadIdx.x] = s[0];
    red[1][threadIdx.x] = s[1];
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) {
            red[0][threadIdx.x] += red[0][threadIdx.x + h];
            red[1][threadIdx.x] += red[1][threadIdx.x + h];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        out[2 * blockIdx.x] = red[0][0];
        out[2 * blockIdx.x + 1] = red[1][0];
    }
}

int s00_moment_blocks(int T) { return (T * (T + 2) + 255) / 256; }

hipError_t launch_s00_moments(const double *a0, int T, const double *cgm, const double *cg1, double *out,
                              hipStream_t st)
{
    if (T < 1 || T > OBS_KOFF) return hipErrorInvalidValue;
    hipLaunchKernelGGL(s00_moments_kernel, dim3(s00_moment_blocks(T)), dim3(256), 0, st, a0, T, cgm, cg1, out);
    return hipGetLastError();
}

// ===========================================================================
// fosmexpansion (mstm-scatprops-26.f90:1820-1951): the eight nonzero
// sequences over w of s00, s02, sp22 and sm22 (before the sign patch and the
// 1/(2 m_medium) scale, which the host applies).  One 256-thread workgroup
// per (n, block of FOSM_LB degrees l); thread w owns w = 0..2T.
// Vector-coupling coefficients C(n,m;l,k|w,m+k) for all w come from the
// recurrences of vcfunc / vcfuncuprec (mstm-modules-33.f90:950-1056),
// one coefficient array per thread, in LDS; bc is the bcof table of init
// (mstm-modules-33.f90:46-50), leading dimension ldb.
// part[(block*8 + e)*W + w], e: s00(1,1), s00(4,4), s02(2,1), s02(1,2),
// s02(3,4), s02(4,3), sm22(2,2), sp22(2,2).
// ===========================================================================
#define FOSM_LB 4
#define FOSM_CH 16

__device__ static void vc_up(int m, int n, int k, int l, int wmax, double *v, const double *bc, int ldb,
                             const double *fnr)
{
#define BC(a, b) bc[(a) * ldb + (b)]
    int mk = iab(m + k);
    const int nl = iab(n - l);
    int w;
    double vc1;
    if (nl >= mk) {
        w = nl;
        int m1, l1, k1;
        if (n >= l) {
            m1 = m;
            l1 = l;
            k1 = k;
        } else {
            m1 = k;
            k1 = m;
            l1 = n;
        }
        vc1 = (double)(((k1 + l1) & 1) ? -1 : 1) * BC(l1 + k1, w - m1 - k1) * BC(l1 - k1, w + m1 + k1) / BC(l1 + l1, w + w + 1);
    } else {
        w = mk;
        if (m + k >= 0)
            vc1 = (double)(((n + m) & 1) ? -1 : 1) * BC(n - l + w, l - k) * BC(l - n + w, n - m) / BC(w + w + 1, n + l - w);
        else
            vc1 = (double)(((l + k) & 1) ? -1 : 1) * BC(n - l + w, l + k) * BC(l - n + w, n + m) / BC(w + w + 1, n + l - w);
    }
    const int w1 = w;
    v[w] = vc1;
    w = w1 + 1;
    mk = m + k;
    const int w2 = imn(wmax, n + l);
    if (w2 > w1) {
        const double t1 = (double)(2 * w) * fnr[w + w + 1] * fnr[w + w - 1] /
                          (fnr[w + mk] * fnr[w - mk] * fnr[n - l + w] * fnr[l - n + w] * fnr[n + l - w + 1] * fnr[n + l + w + 1]);
        const double t2 = w1 == 0 ? 0.5 * (double)(m - k)
                                  : (double)((m - k) * w * (w - 1) - mk * n * (n + 1) + mk * l * (l + 1)) / (double)(2 * w * (w - 1));
        v[w] = t1 * t2 * v[w1];
    }
    for (w = w1 + 2; w <= w2; w++) {
        const double t1 = (double)(2 * w) * fnr[w + w + 1] * fnr[w + w - 1] /
                          (fnr[w + mk] * fnr[w - mk] * fnr[n - l + w] * fnr[l - n + w] * fnr[n + l - w + 1] * fnr[n + l + w + 1]);
        const double t2 = (double)((m - k) * w * (w - 1) - mk * n * (n + 1) + mk * l * (l + 1)) / (double)(2 * w * (w - 1));
        const double t3 = fnr[w - mk - 1] * fnr[w + mk - 1] * fnr[l - n + w - 1] * fnr[n - l + w - 1] * fnr[n + l - w + 2] *
                          fnr[n + l + w] / ((double)(2 * (w - 1)) * fnr[2 * w - 3] * fnr[2 * w - 1]);
        v[w] = t1 * (t2 * v[w - 1] - t3 * v[w - 2]);
    }
#undef BC
}

// C(n,m;l,k|w,m+k), w = 0..n+l, into v (zero where the coefficient is)
__device__ static void vc_all(int m, int n, int k, int l, double *v, const double *bc, int ldb, const double *fnr)
{
#define BC(a, b) bc[(a) * ldb + (b)]
    for (int w = 0; w <= n + l; w++) v[w] = 0.0;
    const int wmax = n + l, wmin = imx(iab(n - l), iab(m + k));
    v[wmax] = BC(n + m, l + k) * BC(n - m, l - k) / BC(n + n, l + l);
    if (wmin == wmax) return;
    v[wmax - 1] = v[wmax] * (double)(l * m - k * n) * fnr[2 * (l + n) - 1] / fnr[l] / fnr[n] / fnr[n + l + m + k] /
                  fnr[n + l - m - k];
    if (wmin == wmax - 1) return;
    const int mk = m + k;
    double vcmax = fabs(v[wmax]) + fabs(v[wmax - 1]);
    // downward first; once the coefficients shrink, upward from wmin
    int w;
    for (w = wmax; w >= wmin + 2; w--) {
        const double t1 = (double)(2 * w) * fnr[w + w + 1] * fnr[w + w - 1] /
                          (fnr[w + mk] * fnr[w - mk] * fnr[n - l + w] * fnr[l - n + w] * fnr[n + l - w + 1] * fnr[n + l + w + 1]);
        const double t2 = (double)((m - k) * w * (w - 1) - mk * n * (n + 1) + mk * l * (l + 1)) / (double)(2 * w * (w - 1));
        const double t3 = fnr[w - mk - 1] * fnr[w + mk - 1] * fnr[l - n + w - 1] * fnr[n - l + w - 1] * fnr[n + l - w + 2] *
                          fnr[n + l + w] / ((double)(2 * (w - 1)) * fnr[2 * w - 3] * fnr[2 * w - 1]);
        v[w - 2] = (t2 * v[w - 1] - v[w] / t1) / t3;
        if ((wmax - w) % 2 == 1) {
            const double vctest = fabs(v[w - 2]) + fabs(v[w - 1]);
            vcmax = fmax(vcmax, vctest);
            if (vctest / vcmax < 0.01) break;
        }
    }
    if (w - 2 > wmin) vc_up(m, n, k, l, w - 3, v, bc, ldb, fnr);
#undef BC
}

__global__ __launch_bounds__(256) void fosm_kernel(const double *__restrict__ a0, int T, const double *__restrict__ bc,
                                                   int ldb, int ch, double *__restrict__ part)
{
    extern __shared__ double lds[];
    const int W = 2 * T + 1, nlb = (T + FOSM_LB - 1) / FOSM_LB;
    const int n = blockIdx.x / nlb + 1, l0 = (blockIdx.x % nlb) * FOSM_LB + 1, l1 = imn(T, l0 + FOSM_LB - 1);
    const int nfnr = 4 * T + 4;
    double *fnr = lds;                   // sqrt(i), i < nfnr
    double *vl = fnr + nfnr;             // C(n,-1;l,1|w,0), C(n,-1;l,-1|w,-2)
    double *vm = vl + 2 * W;             // [j][kind][w] of a chunk of ch values of m
    for (int i = threadIdx.x; i < nfnr; i += blockDim.x) fnr[i] = sqrt((double)i);
    const int w = threadIdx.x;
    const cplx<double> *A = reinterpret_cast<const cplx<double> *>(a0);
    const int b0 = T * (T + 2);
    // a1(m,n,p) = A[p b0 + amn(m,n,T)], a2(m,n,p) = A[(2 + p) b0 + amn(m,n,T)]; zero for |m| > n
    auto amp = [&](int t, int m, int nn, int p) -> cplx<double> {
        if (iab(m) > nn) return cmk(0.0, 0.0);
        return A[(2 * t + p) * b0 + amn(m, nn, T)];
    };
    double acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    const cplx<double> ci = cmk(0.0, 1.0);
    for (int l = l0; l <= l1; l++) {
        __syncthreads();
        if (threadIdx.x == 0) vc_all(-1, n, 1, l, vl, bc, ldb, fnr);
        if (threadIdx.x == 1) vc_all(-1, n, -1, l, vl + W, bc, ldb, fnr);
        const int wmin = iab(n - l), wmax = n + l;
        const double fm = sqrt((double)((n + n + 1) * (l + l + 1)));
        const int ph = ((l - n) % 4 + 4) % 4;  // fnl = fm i^(l-n)
        const cplx<double> fnl = ph == 0 ? cmk(fm, 0.0) : ph == 1 ? cmk(0.0, fm) : ph == 2 ? cmk(-fm, 0.0) : cmk(0.0, -fm);
        const int mhi = imn(n, l + 2);
        for (int mc = -mhi; mc <= mhi; mc += ch) {
            __syncthreads();
            if (threadIdx.x >= 2 && threadIdx.x < 2 + 3 * ch) {
                const int t = threadIdx.x - 2, j = t / 3, kind = t % 3, m = mc + j;
                double *v = vm + (j * 3 + kind) * W;
                if (m <= mhi) {
                    const int k = kind == 0 ? m : (kind == 1 ? m - 2 : m + 2);
                    if (iab(k) <= l) vc_all(-m, n, k, l, v, bc, ldb, fnr);
                    else
                        for (int q = 0; q <= n + l; q++) v[q] = 0.0;
                }
            }
            __syncthreads();
            if (w < wmin || w > wmax) continue;
            const double m1w = (w & 1) ? -1.0 : 1.0;
            const double cp1 = vl[w], cm1 = vl[W + w];
            for (int j = 0; j < ch && mc + j <= mhi; j++) {
                const int m = mc + j;
                const double cmm = vm[(j * 3) * W + w], cm2 = vm[(j * 3 + 1) * W + w], cp2 = vm[(j * 3 + 2) * W + w];
                const double m1m = (iab(m) & 1) ? -1.0 : 1.0;
                for (int p = 0; p < 2; p++)
                    for (int q = 0; q < 2; q++) {
                        // Fortran p, q = p + 1, q + 1
                        const double m1mq = ((iab(m) + q + 1) & 1) ? -1.0 : 1.0;
                        const double m1mnpl = ((iab(m) + n + p + 1 + l) & 1) ? -1.0 : 1.0;
                        const cplx<double> a1n = amp(0, m, n, p), a2n = amp(1, m, n, p);
                        const cplx<double> a1l = amp(0, m, l, q), a2l = amp(1, m, l, q);
                        const cplx<double> a1122 = cadd(cmul(a1n, cconj(a1l)), cmul(a2n, cconj(a2l)));
                        const cplx<double> a2112 = csub(cmul(a2n, cconj(a1l)), cmul(a1n, cconj(a2l)));
                        const cplx<double> a1pn = cadd(a1n, cmul(ci, a2n)), a1mn = csub(a1n, cmul(ci, a2n));
                        const cplx<double> lm2 = csub(amp(0, m - 2, l, q), cmul(ci, amp(1, m - 2, l, q)));
                        const cplx<double> lp2 = cadd(amp(0, m + 2, l, q), cmul(ci, amp(1, m + 2, l, q)));
                        const cplx<double> a1p2 = cmul(a1pn, cconj(lm2)), a1m2 = cmul(a1mn, cconj(lp2));
                        const cplx<double> f1122 = cmul(fnl, a1122), f2112 = cmul(fnl, a2112);
                        const cplx<double> fp2 = cmul(fnl, a1p2), fm2 = cmul(fnl, a1m2);
                        const bool even = ((n + l + w + p + q) & 1) == 0;
                        if (even) {
                            acc[0] += -(m1m * f1122.re * cp1 * cmm) / 2.0;
                        } else {
                            // (i/2 m1m fnl a2112 cp1 cmm): real part
                            acc[1] += -0.5 * m1m * f2112.im * cp1 * cmm;
                        }
                        if (w < 2) continue;
                        if (even) {
                            acc[2] += -(m1mq * f1122.re * cm1 * cmm) / 2.0;
                            acc[3] += -(m1m * fp2.re * cp1 * cm2) / 4.0;
                            acc[3] += -(m1m * fm2.re * cp1 * cp2) / 4.0;
                        } else {
                            // imag(-i/2 m1mq a2112 fnl cm1 cmm) = -1/2 m1mq re(fnl a2112) cm1 cmm
                            acc[4] += -0.5 * m1mq * f2112.re * cm1 * cmm;
                            acc[5] += m1m * fp2.im * cp1 * cm2 / 4.0;
                            acc[5] -= m1m * fm2.im * cp1 * cp2 / 4.0;
                        }
                        acc[6] += -(m1mnpl * m1w * fp2.re * cm1 * cm2) / 8.0;
                        acc[7] += -(m1mq * fp2.re * cm1 * cm2) / 8.0;
                        acc[6] += -(m1mq * fm2.re * cm1 * cp2) / 8.0;
                        acc[7] += -(m1mnpl * m1w * fm2.re * cm1 * cp2) / 8.0;
                    }
            }
        }
    }
    if (w < W)
        for (int e = 0; e < 8; e++) part[((int64_t)blockIdx.x * 8 + e) * W + w] = acc[e];
}

// sum of the per-block sequences in block order: one workgroup per (e, w)
__global__ __launch_bounds__(256) void fosm_reduce_kernel(const double *__restrict__ part, int nblocks, int W,
                                                          double *__restrict__ out)
{
    __shared__ double red[256];
    const int ew = blockIdx.x;  // e * W + w
    double s = 0.0;
    for (int b = threadIdx.x; b < nblocks; b += 256) s += part[(int64_t)b * 8 * W + ew];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[ew] = red[0];
}

int fosm_blocks(int T) { return T * ((T + FOSM_LB - 1) / FOSM_LB); }

hipError_t launch_fosm(const double *a0, int T, const double *bc, int ldb, double *part, double *out, hipStream_t st)
{
    if (T < 1 || T > OBS_KOFF) return hipErrorInvalidValue;
    const int W = 2 * T + 1, nb = fosm_blocks(T);
    // m values per chunk: as many as 64 KB of LDS holds, at most FOSM_CH
    const int ch = imn(FOSM_CH, (8192 - (4 * T + 4) - 2 * W) / (3 * W));
    const size_t lds = sizeof(double) * ((size_t)(4 * T + 4) + 2 * W + (size_t)3 * ch * W);
    hipLaunchKernelGGL(fosm_kernel, dim3(nb), dim3(256), lds, st, a0, T, bc, ldb, ch, part);
    hipLaunchKernelGGL(fosm_reduce_kernel, dim3(8 * W), dim3(256), 0, st, part, nb, W, out);
    return hipGetLastError();
}
