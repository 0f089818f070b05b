// direct.hip -- around the direct tiles (tile32.hip, tile64.hip) and the FFT
// operator: input preparation with the con_tran/Mie pre-op of
// sphereinteraction (mstm-scatprops-26.f90:88-97) and the sum of the partial
// results with its post-op (:158-168).
#include "common.hpp"
#include "kernels.hpp"
#include "tile.hpp"

// ---------------------------------------------------------------------------
// Input preparation (sphereinteraction :88-97): for a con_tran column
// x = S T^T conj(a) (S = m-flip with (-1)^m, T^T the transposed 2x2 Mie
// matrix when mie_mult); otherwise x = a.  The kernels behind work on a
// uniform-order copy (order Lp = max order, npad spheres); coefficients of
// degree n > order(i) and padding spheres are zero, which is exact because
// a translation table of order Lp contains those of lower orders.
// flags[r] (host array, r < nrhs <= 4) bit0 = con_tran, bit1 = mie_mult.
// an: Mie matrices, 4 complex per degree, at (sphere*Lp + n-1)*4.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void decode_mn(int e, int L, int &m, int &n)
{
    int row = e % (L + 2), colm = e / (L + 2) + 1;
    if (row <= colm) {
        m = row;
        n = colm;
    } else {
        m = -colm;
        n = row - 1;
    }
}
__device__ __forceinline__ int flag_of(int4 f, int r) { return r == 0 ? f.x : (r == 1 ? f.y : (r == 2 ? f.z : f.w)); }

// both modes of coefficient (m, n) of a sphere (order L >= n, its vector at
// a, its Mie matrix of degree n at t4) after the pre-op
__device__ __forceinline__ void pre_op(const cplx<double> *__restrict__ a, int m, int n, int L, int f,
                                       const cplx<double> *__restrict__ t4, cplx<double> (&v)[2])
{
    const int NB = L * (L + 2);
    if (!(f & 1)) {
        v[0] = a[amn(m, n, L)];
        v[1] = a[amn(m, n, L) + NB];
        return;
    }
    // flipped value at (m,n) is (-1)^m (T^T conj a)(-m,n)
    cplx<double> v0 = cconj(a[amn(-m, n, L)]), v1 = cconj(a[amn(-m, n, L) + NB]);
    if (f & 2) {  // t4[p + 2q] = T(p,q)
        const cplx<double> w0 = cadd(cmul(t4[0], v0), cmul(t4[1], v1));
        const cplx<double> w1 = cadd(cmul(t4[2], v0), cmul(t4[3], v1));
        v0 = w0;
        v1 = w1;
    }
    const double sg = (m & 1) ? -1.0 : 1.0;
    v[0] = cscale(v0, sg);
    v[1] = cscale(v1, sg);
}
// both modes of coefficient (m, n) of the result, written to the sphere's
// vector o: normal column out = T h (mie_mult) or h; con_tran out = conj(S h),
// h then being the sum at (-m, n)
__device__ __forceinline__ void post_op(cplx<double> *__restrict__ o, int m, int n, int L, int f,
                                        const cplx<double> *__restrict__ t4, cplx<double> h0, cplx<double> h1)
{
    const int NB = L * (L + 2), eo = amn(m, n, L);
    if (f & 1) {
        const double sg = (m & 1) ? -1.0 : 1.0;
        o[eo] = cmk(sg * h0.re, -sg * h0.im);
        o[eo + NB] = cmk(sg * h1.re, -sg * h1.im);
    } else if (f & 2) {
        o[eo] = cadd(cmul(t4[0], h0), cmul(t4[2], h1));
        o[eo + NB] = cadd(cmul(t4[1], h0), cmul(t4[3], h1));
    } else {
        o[eo] = h0;
        o[eo + NB] = h1;
    }
}

static int4 flags4(const int *flags, int nrhs)
{
    return make_int4(flags[0], nrhs > 1 ? flags[1] : 0, nrhs > 2 ? flags[2] : 0, nrhs > 3 ? flags[3] : 0);
}

// FFT operator: xin[r][sphere][mode][packed (m,n)], r < 2.  One thread per
// (r, sphere, e).
template <typename T>
__global__ void prep_kernel(const cplx<double> *__restrict__ ain, int ldain, cplx<T> *__restrict__ xin, int nrhs,
                            int4 flags, int nsph, int npad, int Lp, const int *__restrict__ order,
                            const int *__restrict__ offset, const cplx<double> *__restrict__ an,
                            const int *__restrict__ gate)
{
    if (gate && !*gate) return;
    const int NBP = Lp * (Lp + 2);
    int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= (int64_t)2 * npad * NBP) return;
    int e = (int)(q % NBP);
    int64_t t = q / NBP;
    int sph = (int)(t % npad);
    int r = (int)(t / npad);
    cplx<T> *o = xin + ((int64_t)(r * npad + sph) * 2) * NBP;
    int m, n;
    decode_mn(e, Lp, m, n);
    cplx<double> v[2] = {cmk(0.0, 0.0), cmk(0.0, 0.0)};
    if (r < nrhs && sph < nsph && n <= order[sph])
        pre_op(ain + (int64_t)r * ldain + offset[sph], m, n, order[sph], flag_of(flags, r),
               an + ((int64_t)sph * Lp + (n - 1)) * 4, v);
    o[e] = cmk((T)v[0].re, (T)v[0].im);
    o[e + NBP] = cmk((T)v[1].re, (T)v[1].im);
}

template <typename T>
hipError_t launch_prep(const double *ain, int ldain, T *xin, int nrhs, const int *flags, int nsph, int npad, int Lp,
                       const int *order, const int *offset, const double *an, hipStream_t st, const int *gate)
{
    if (nrhs < 1 || nrhs > 2) return hipErrorInvalidValue;
    const int64_t n = (int64_t)2 * npad * Lp * (Lp + 2);
    const int bs = 256;
    hipLaunchKernelGGL(prep_kernel<T>, dim3((unsigned)((n + bs - 1) / bs)), dim3(bs), 0, st,
                       reinterpret_cast<const cplx<double> *>(ain), ldain / 2, reinterpret_cast<cplx<T> *>(xin), nrhs,
                       flags4(flags, nrhs), nsph, npad, Lp, order, offset,
                       reinterpret_cast<const cplx<double> *>(an), gate);
    return hipGetLastError();
}
template hipError_t launch_prep<float>(const double *, int, float *, int, const int *, int, int, int, const int *,
                                       const int *, const double *, hipStream_t, const int *);
template hipError_t launch_prep<double>(const double *, int, double *, int, const int *, int, int, int, const int *,
                                        const int *, const double *, hipStream_t, const int *);

// Direct tiles: quad layout (tile.hpp).  Position, in T, of complex value idx
// of (column r, mode p) of a sphere.
template <typename T> __device__ __forceinline__ int64_t quad_pos(int64_t r, int sph, int p, int idx, int npad, int L)
{
    const int NB = L * (L + 2), UC = cvec_unit(L, sizeof(T));
    return ((r >> 1) * npad + sph) * (8 * NB) + 2 * (((idx / UC) * 4 + 2 * (int)(r & 1) + p) * UC + idx % UC);
}

// One thread per (column r < nr, sphere, degree n, k = 0..n): the values a_k,
// b_k of both modes.
template <typename T>
__global__ void prep_quad_kernel(const cplx<double> *__restrict__ ain, int ldain, T *__restrict__ xin, int nrhs,
                                 int4 flags, int nr, int nsph, int npad, int Lp, const int *__restrict__ order,
                                 const int *__restrict__ offset, const cplx<double> *__restrict__ an,
                                 const int *__restrict__ gate)
{
    if (gate && !gate[blockIdx.y]) return;
    const int NK = Lp * (Lp + 3) / 2;
    ain += (int64_t)blockIdx.y * nrhs * ldain;
    xin += (int64_t)blockIdx.y * nr * npad * 4 * Lp * (Lp + 2);
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= (int64_t)nr * npad * NK) return;
    const int e = (int)(q % NK);
    const int64_t t = q / NK;
    const int sph = (int)(t % npad), r = (int)(t / npad);
    int n = 1, k = e;  // e = (n-1)(n+2)/2 + k
    while (k > n) k -= ++n;
    cplx<double> vp[2] = {cmk(0.0, 0.0), cmk(0.0, 0.0)}, vm[2] = {vp[0], vp[0]};
    if (r < nrhs && sph < nsph && n <= order[sph]) {
        const cplx<double> *a = ain + (int64_t)r * ldain + offset[sph];
        const cplx<double> *t4 = an + ((int64_t)sph * Lp + (n - 1)) * 4;
        const int f = flag_of(flags, r), L = order[sph];
        pre_op(a, k, n, L, f, t4, vp);
        if (k) pre_op(a, -k, n, L, f, t4, vm);
    }
    const double sk = (k & 1) ? -1.0 : 1.0;
#pragma unroll
    for (int p = 0; p < 2; p++) {
        const cplx<double> fl = cscale(vm[p], sk), a = cadd(vp[p], fl), b = csub(vp[p], fl);
        T *o = xin + quad_pos<T>(r, sph, p, cvec(n, k, 0, Lp), npad, Lp);
        o[0] = (T)a.re;
        o[1] = (T)a.im;
        if (k) {
            o = xin + quad_pos<T>(r, sph, p, cvec(n, k, 1, Lp), npad, Lp);
            o[0] = (T)b.re;
            o[1] = (T)b.im;
        }
    }
}

template <typename T>
hipError_t launch_prep_quad(const double *ain, int ldain, T *xin, int nrhs, const int *flags, int nsph, int npad,
                            int Lp, const int *order, const int *offset, const double *an, int nq, hipStream_t st,
                            const int *gate)
{
    if (nrhs < 1 || nrhs > 4 || nq < 1 || nq > 65535) return hipErrorInvalidValue;
    const int nr = nrhs > 2 ? 4 : 2, bs = 256;
    const int64_t n = (int64_t)nr * npad * (Lp * (Lp + 3) / 2);
    hipLaunchKernelGGL(prep_quad_kernel<T>, dim3((unsigned)((n + bs - 1) / bs), nq), dim3(bs), 0, st,
                       reinterpret_cast<const cplx<double> *>(ain), ldain / 2, xin, nrhs, flags4(flags, nrhs), nr,
                       nsph, npad, Lp, order, offset, reinterpret_cast<const cplx<double> *>(an), gate);
    return hipGetLastError();
}
template hipError_t launch_prep_quad<float>(const double *, int, float *, int, const int *, int, int, int, const int *,
                                            const int *, const double *, int, hipStream_t, const int *);
template hipError_t launch_prep_quad<double>(const double *, int, double *, int, const int *, int, int, int,
                                             const int *, const int *, const double *, int, hipStream_t,
                                             const int *);

// ---------------------------------------------------------------------------
// Post-op (sphereinteraction :158-168).  FFT operator: the result of one
// product, in prep_kernel's layout, to the reference (unpadded) layout.
// ---------------------------------------------------------------------------
template <typename T>
__global__ void post_kernel(const cplx<T> *__restrict__ res, cplx<double> *__restrict__ aout, int ldaout, int nrhs,
                            int4 flags, int nsph, int npad, int Lp, const int *__restrict__ order,
                            const int *__restrict__ offset, const cplx<double> *__restrict__ an,
                            const int *__restrict__ gate)
{
    if (gate && !*gate) return;
    const int NBP = Lp * (Lp + 2);
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= (int64_t)nrhs * nsph * NBP) return;
    const int e = (int)(q % NBP);
    const int64_t t = q / NBP;
    const int sph = (int)(t % nsph), r = (int)(t / nsph);
    int m, n;
    decode_mn(e, Lp, m, n);
    if (n > order[sph]) return;
    const int f = flag_of(flags, r);
    const cplx<T> *p = res + ((int64_t)r * npad + sph) * 2 * NBP + ((f & 1) ? amn(-m, n, Lp) : e);
    post_op(aout + (int64_t)r * ldaout + offset[sph], m, n, order[sph], f, an + ((int64_t)sph * Lp + (n - 1)) * 4,
            cmk((double)p[0].re, (double)p[0].im), cmk((double)p[NBP].re, (double)p[NBP].im));
}

template <typename T>
hipError_t launch_post(const T *res, double *aout, int ldaout, int nrhs, const int *flags, int nsph, int npad, int Lp,
                       const int *order, const int *offset, const double *an, hipStream_t st, const int *gate)
{
    if (nrhs < 1 || nrhs > 2) return hipErrorInvalidValue;
    const int64_t n = (int64_t)nrhs * nsph * Lp * (Lp + 2);
    const int bs = 256;
    hipLaunchKernelGGL(post_kernel<T>, dim3((unsigned)((n + bs - 1) / bs)), dim3(bs), 0, st,
                       reinterpret_cast<const cplx<T> *>(res), reinterpret_cast<cplx<double> *>(aout), ldaout / 2,
                       nrhs, flags4(flags, nrhs), nsph, npad, Lp, order, offset,
                       reinterpret_cast<const cplx<double> *>(an), gate);
    return hipGetLastError();
}
template hipError_t launch_post<float>(const float *, double *, int, int, const int *, int, int, int, const int *,
                                       const int *, const double *, hipStream_t, const int *);
template hipError_t launch_post<double>(const double *, double *, int, int, const int *, int, int, int, const int *,
                                        const int *, const double *, hipStream_t, const int *);

// Direct tiles: the sum over the partials (quad layout) in FP64, then the
// post-op.  A workgroup owns SP spheres of one column pair: U units (16 bytes;
// 8 for odd FP32 orders) per sphere, KS threads per unit, each summing every
// KS-th partial (fixed order), then the sums meet in LDS and a thread per
// (column, sphere, n, k) writes the coefficients (+-k, n) of both modes.  The
// partials' reads are whole cache lines, each read once: bound by HBM with
// many spheres (5000 of order 4, two FP32 columns: 0.18 ms against 0.25 ms for
// one thread per coefficient, whose lanes read 8 bytes each), by the latency
// of a chain of loads with few, where KS shortens the chain.
template <typename T, int VC>
__global__ __launch_bounds__(1024) void reduce_quad_kernel(const T *__restrict__ part, int nparts,
                                                          cplx<double> *__restrict__ aout, int ldaout, int nrhs,
                                                          int4 flags, int nr, int nsph, int npad, int Lp, int SP,
                                                          int KS, const int *__restrict__ order,
                                                          const int *__restrict__ offset,
                                                          const cplx<double> *__restrict__ an,
                                                          const int *__restrict__ gate)
{
    if (gate && !gate[blockIdx.z]) return;  // uniform over the workgroup
    extern __shared__ double red[];  // [KS][SP][8 NB]
    typedef T vec __attribute__((ext_vector_type(VC)));
    const int NB = Lp * (Lp + 2), NK = Lp * (Lp + 3) / 2, U = 8 * NB / VC;
    const int sph0 = blockIdx.x * SP, rp = blockIdx.y;
    const int64_t stride = (int64_t)(nr / 2) * npad * U;  // one partial
    aout += (int64_t)blockIdx.z * nrhs * ldaout;
    const vec *p0 = reinterpret_cast<const vec *>(part) + blockIdx.z * nparts * stride +
                    ((int64_t)rp * npad + sph0) * U;
    const int nsp = imn(SP, npad - sph0);
    for (int e = threadIdx.x; e < KS * nsp * U; e += blockDim.x) {
        const int un = e % (nsp * U), j = e / (nsp * U);
        double s[VC];
#pragma unroll
        for (int q = 0; q < VC; q++) s[q] = 0.0;
        const vec *p = p0 + un;
#pragma unroll 8
        for (int b = j; b < nparts; b += KS) {
            const vec v = __builtin_nontemporal_load(p + (int64_t)b * stride);
#pragma unroll
            for (int q = 0; q < VC; q++) s[q] += (double)v[q];
        }
#pragma unroll
        for (int q = 0; q < VC; q++) red[(int64_t)j * SP * 8 * NB + un * VC + q] = s[q];
    }
    __syncthreads();
    for (int e = threadIdx.x; e < 2 * nsp * NK; e += blockDim.x) {
        const int kn = e % NK, i = (e / NK) % nsp, r = 2 * rp + e / (NK * nsp), sph = sph0 + i;
        int n = 1, k = kn;
        while (k > n) k -= ++n;
        if (r >= nrhs || sph >= nsph || n > order[sph]) continue;
        cplx<double> a[2], b[2];
        for (int p = 0; p < 2; p++) {
            const int64_t pa = quad_pos<T>(r & 1, i, p, cvec(n, k, 0, Lp), 0, Lp);
            const int64_t pb = quad_pos<T>(r & 1, i, p, cvec(n, k, k ? 1 : 0, Lp), 0, Lp);
            a[p] = b[p] = cmk(0.0, 0.0);
            for (int j = 0; j < KS; j++) {
                const double *d = red + (int64_t)j * SP * 8 * NB;
                a[p] = cadd(a[p], cmk(d[pa], d[pa + 1]));
                b[p] = cadd(b[p], cmk(d[pb], d[pb + 1]));
            }
        }
        const int f = flag_of(flags, r), L = order[sph];
        const cplx<double> *t4 = an + ((int64_t)sph * Lp + (n - 1)) * 4;
        cplx<double> *o = aout + (int64_t)r * ldaout + offset[sph];
        if (k == 0) {
            post_op(o, 0, n, L, f, t4, a[0], a[1]);
            continue;
        }
        // x_k = (a + b)/2, x_-k = (-1)^k (a - b)/2, the tiles giving a/2, b/2
        const double sk = (k & 1) ? -1.0 : 1.0;
        const cplx<double> hp[2] = {cadd(a[0], b[0]), cadd(a[1], b[1])};
        const cplx<double> hm[2] = {cscale(csub(a[0], b[0]), sk), cscale(csub(a[1], b[1]), sk)};
        const bool fl = f & 1;
        post_op(o, k, n, L, f, t4, fl ? hm[0] : hp[0], fl ? hm[1] : hp[1]);
        post_op(o, -k, n, L, f, t4, fl ? hp[0] : hm[0], fl ? hp[1] : hm[1]);
    }
}

template <typename T>
hipError_t launch_reduce_quad(const T *partial, int nparts, double *aout, int ldaout, int nrhs, const int *flags,
                              int nsph, int npad, int Lp, const int *order, const int *offset, const double *an,
                              int nq, hipStream_t st, const int *gate)
{
    if (nrhs < 1 || nrhs > 4 || nq < 1 || nq > 65535) return hipErrorInvalidValue;
    const int nr = nrhs > 2 ? 4 : 2, NB = Lp * (Lp + 2);
    const int VC = 2 * cvec_unit(Lp, sizeof(T)), U = 8 * NB / VC;
    // about one unit per thread of 256; fewer than two workgroups per CU: one
    // sphere and 1024 threads each, and chains of about four loads
    int SP = imx(1, 256 / U), threads = 256;
    if ((int64_t)nsph * (nr / 2) * nq / SP < 512) {
        SP = 1;
        threads = 1024;
    }
    const int KS = imx(1, imn(threads / (SP * U), (nparts + 3) / 4));
    const dim3 g((nsph + SP - 1) / SP, nr / 2, nq);
    const size_t lds = sizeof(double) * (size_t)KS * SP * 8 * NB;
#define RQ(V)                                                                                                          \
    hipLaunchKernelGGL((reduce_quad_kernel<T, V>), g, dim3(threads), lds, st, partial, nparts,                         \
                       reinterpret_cast<cplx<double> *>(aout), ldaout / 2, nrhs, flags4(flags, nrhs), nr, nsph, npad,  \
                       Lp, SP, KS, order, offset, reinterpret_cast<const cplx<double> *>(an), gate)
    if (VC == 2) RQ(2);
    else RQ((sizeof(T) == 8 ? 2 : 4));
#undef RQ
    return hipGetLastError();
}
template hipError_t launch_reduce_quad<float>(const float *, int, double *, int, int, const int *, int, int, int,
                                              const int *, const int *, const double *, int, hipStream_t,
                                              const int *);
template hipError_t launch_reduce_quad<double>(const double *, int, double *, int, int, const int *, int, int, int,
                                               const int *, const int *, const double *, int, hipStream_t, const int *);
