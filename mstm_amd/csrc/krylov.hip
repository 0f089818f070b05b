// krylov.hip -- FP64 vector kernels of the complex biconjugate-gradient
// iteration (cbicg, mstm-solver-8.f90:654-949) and of the mixed-precision
// refinement.  Inner products are written as per-block partial sums that the
// host adds in a fixed order (deterministic results).
#include "common.hpp"
#include "kernels.hpp"

#define KB 256  // threads per block
#define KGRID 512

__device__ __forceinline__ void block_sum3(cplx<double> *v, int nv)
{
    __shared__ cplx<double> sh[3][KB];
    for (int q = 0; q < nv; q++) sh[q][threadIdx.x] = v[q];
    __syncthreads();
    for (int s = KB / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s)
            for (int q = 0; q < nv; q++) sh[q][threadIdx.x] = cadd(sh[q][threadIdx.x], sh[q][threadIdx.x + s]);
        __syncthreads();
    }
    for (int q = 0; q < nv; q++) v[q] = sh[q][0];
}

// partial[b] = sum (conj_a ? conj(a) : a) * b over the block's grid-stride share
__global__ void zdot_kernel(const cplx<double> *__restrict__ a, const cplx<double> *__restrict__ b, int n, int conj_a,
                            cplx<double> *__restrict__ partials)
{
    cplx<double> s = cmk(0.0, 0.0);
    for (int i = blockIdx.x * KB + threadIdx.x; i < n; i += gridDim.x * KB) {
        cplx<double> x = a[i];
        if (conj_a) x = cconj(x);
        cfma(s, x, b[i]);
    }
    block_sum3(&s, 1);
    if (threadIdx.x == 0) partials[blockIdx.x] = s;
}

hipError_t launch_zdot(const double *a, const double *b, int n, int conj_a, double *partials, double *, hipStream_t st)
{
    hipLaunchKernelGGL(zdot_kernel, dim3(KGRID), dim3(KB), 0, st, reinterpret_cast<const cplx<double> *>(a),
                       reinterpret_cast<const cplx<double> *>(b), n, conj_a, reinterpret_cast<cplx<double> *>(partials));
    return hipGetLastError();
}

// y = a*x + b*y (complex scalars a, b)
__global__ void zaxpby_kernel(cplx<double> a, const cplx<double> *__restrict__ x, cplx<double> b,
                              cplx<double> *__restrict__ y, int n)
{
    for (int i = blockIdx.x * KB + threadIdx.x; i < n; i += gridDim.x * KB) {
        cplx<double> v = cmul(b, y[i]);
        cfma(v, a, x[i]);
        y[i] = v;
    }
}

int krylov_grid() { return KGRID; }
// blocks of the BiCG kernels: those of the full grid that have rows (the others'
// partial sums would be zeros)
static int bicg_grid(int n) { return imn(KGRID, (n + KB - 1) / KB); }

// ---------------------------------------------------------------------------
// Device-resident BiCG scalars (see BicgScal in kernels.hpp).  The vector
// kernels of a system whose state is inactive return at once, so the host
// may launch one iteration for both systems and learn only afterwards which
// of them stopped.
// An iteration's two reductions need no launch of their own: every workgroup
// of the vector step that follows adds the partial sums (at most 512, in one
// order) and works out the new scalars for itself; its first workgroup writes
// them to the other of two state arrays, so none reads what another writes.
// 20 spheres of order 5: 43 us per iteration with a 4.4 us launch after each
// reduction, now 34 us.
// ---------------------------------------------------------------------------
// the sums of nv values per block over nb blocks, in all threads
__device__ __forceinline__ void sum_blocks(const cplx<double> *__restrict__ p, int nv, int nb, cplx<double> *v)
{
    __shared__ cplx<double> red[2][KB];
    for (int q = 0; q < nv; q++) {
        cplx<double> s = cmk(0.0, 0.0);
        for (int b = threadIdx.x; b < nb; b += KB) s = cadd(s, p[(int64_t)nv * b + q]);
        red[q][threadIdx.x] = s;
    }
    __syncthreads();
    for (int h = KB / 2; h > 0; h >>= 1) {
        if (threadIdx.x < h)
            for (int q = 0; q < nv; q++) red[q][threadIdx.x] = cadd(red[q][threadIdx.x], red[q][threadIdx.x + h]);
        __syncthreads();
    }
    for (int q = 0; q < nv; q++) v[q] = red[q][0];
    __syncthreads();
}

// a new iteration: den = v0 = <w, A p>
__device__ __forceinline__ void bicg_alpha(BicgScal &S, cplx<double> v0)
{
    S.cur++;
    if (v0.re == 0.0 && v0.im == 0.0) {  // breakdown: the Fortran loop exits here
        S.active = 0;
        S.it = S.cur;
        S.brk = 1;
        S.cak = cmk(0.0, 0.0);
    } else {
        S.cak = cdiv(S.csk, v0);
    }
}
// its end: v0 = <q, r>, v1 = <r, r>
__device__ __forceinline__ void bicg_beta(BicgScal &S, cplx<double> v0, cplx<double> v1)
{
    S.err = v1.re / S.enorm;
    if (S.err < S.eps || (S.csk.re == 0.0 && S.csk.im == 0.0)) {
        S.active = 0;
        S.it = S.cur;
        S.cbk = cmk(0.0, 0.0);
    } else {
        S.cbk = cdiv(v0, S.csk);
        S.csk = v0;
    }
}

// start-up, one workgroup per pair of systems: step 0, enorm = |b|^2; step 1,
// csk = r.r
__global__ __launch_bounds__(KB) void bicg_scal_kernel(int step, const cplx<double> *__restrict__ partials,
                                                       int64_t region, BicgScal *__restrict__ sc, int ns,
                                                       int nb, int *__restrict__ gate)
{
    const int sa = 2 * blockIdx.x, se = imn(ns, sa + 2);
    int any = 0;
    for (int s = sa; s < se; s++) {
        BicgScal &S = sc[s];
        const bool skip = step >= 1 && !S.active;  // uniform: read by all threads
        cplx<double> v0 = cmk(0.0, 0.0);
        if (!skip) sum_blocks(partials + region * s, 1, nb, &v0);
        if (threadIdx.x == 0) {
            const cplx<double> zero = cmk(0.0, 0.0);
            if (step == 0) {
                S.enorm = v0.re;
                S.active = v0.re != 0.0;
                S.it = 0;
                S.brk = 0;
                S.cur = 0;
                S.err = 0.0;
                S.cak = S.cbk = zero;
            } else if (skip) {
                S.cak = S.cbk = zero;
            } else {
                S.csk = v0;
                if (v0.re == 0.0 && v0.im == 0.0) S.active = 0;  // it stays 0
            }
            any |= S.active != 0;
        }
    }
    if (gate && threadIdx.x == 0) gate[blockIdx.x] = any;
}

// The vector steps of ns systems in one launch: system s = blockIdx.y has
// its vectors at the base pointers plus s times a stride (complex elements:
// sv for x, r, q; sp for p, w, Ap, A^H w), its scalars at sc[s] and its
// partial sums at partials + s * region; a stopped system returns at once.
// |b|^2
__global__ void bicg_norm_kernel(const cplx<double> *__restrict__ b, int64_t sv, int n, cplx<double> *__restrict__ partials,
                                 int64_t region)
{
    b += blockIdx.y * sv;
    cplx<double> s = cmk(0.0, 0.0);
    for (int i = blockIdx.x * KB + threadIdx.x; i < n; i += gridDim.x * KB) cfma(s, cconj(b[i]), b[i]);
    block_sum3(&s, 1);
    if (threadIdx.x == 0) partials[blockIdx.y * region + blockIdx.x] = s;
}

// cr = pnp - anp + cr ; cq = cw = conj(cr) ; cp = cr ; partial sum cr*cr
// (bilinear, :828-834)
__global__ void bicg_init_kernel(cplx<double> *__restrict__ cr, cplx<double> *__restrict__ cq,
                                 cplx<double> *__restrict__ cw, cplx<double> *__restrict__ cp,
                                 const cplx<double> *__restrict__ pnp, const cplx<double> *__restrict__ anp, int64_t sv,
                                 int64_t sp, int n, cplx<double> *__restrict__ partials, int64_t region)
{
    const int64_t v = blockIdx.y * sv, p = blockIdx.y * sp;
    cplx<double> s = cmk(0.0, 0.0);
    for (int i = blockIdx.x * KB + threadIdx.x; i < n; i += gridDim.x * KB) {
        cplx<double> r = cadd(csub(pnp[v + i], anp[v + i]), cr[v + i]);
        cr[v + i] = r;
        cq[v + i] = cconj(r);
        cw[p + i] = cconj(r);
        cp[p + i] = r;
        cfma(s, r, r);
    }
    block_sum3(&s, 1);
    if (threadIdx.x == 0) partials[blockIdx.y * region + blockIdx.x] = s;
}

// cap = cp - cap ; caw = cw - caw ; partial <cw, cap>   (:897-903)
__global__ void bicg_a_dev_kernel(cplx<double> *__restrict__ cap, cplx<double> *__restrict__ caw,
                                  const cplx<double> *__restrict__ cp, const cplx<double> *__restrict__ cw, int64_t sp,
                                  int n, cplx<double> *__restrict__ partials, int64_t region,
                                  const BicgScal *__restrict__ sc)
{
    const int64_t y = blockIdx.y;
    if (!sc[y].active) return;
    cap += y * sp;
    caw += y * sp;
    cp += y * sp;
    cw += y * sp;
    partials += y * region;
    cplx<double> s = cmk(0.0, 0.0);
    for (int i = blockIdx.x * KB + threadIdx.x; i < n; i += gridDim.x * KB) {
        cplx<double> a = csub(cp[i], cap[i]);
        cap[i] = a;
        caw[i] = csub(cw[i], caw[i]);
        cfma(s, cconj(cw[i]), a);
    }
    block_sum3(&s, 1);
    if (threadIdx.x == 0) partials[blockIdx.x] = s;
}

// anp += cak cp ; cr -= cak cap ; cq -= conj(cak) caw ;
// partials <cq, cr>, <cr, cr>   (:912-920)
__global__ void bicg_b_dev_kernel(cplx<double> *__restrict__ anp, cplx<double> *__restrict__ cr,
                                  cplx<double> *__restrict__ cq, const cplx<double> *__restrict__ cp,
                                  const cplx<double> *__restrict__ cap, const cplx<double> *__restrict__ caw,
                                  int64_t sv, int64_t sp, const BicgScal *__restrict__ sc,
                                  BicgScal *__restrict__ sn, int n, const cplx<double> *__restrict__ den,
                                  cplx<double> *__restrict__ partials, int64_t region)
{
    const int64_t y = blockIdx.y;
    BicgScal S = sc[y];
    const bool first = blockIdx.x == 0 && threadIdx.x == 0;
    if (S.active) {
        cplx<double> v0;
        sum_blocks(den + y * region, 1, gridDim.x, &v0);
        bicg_alpha(S, v0);
    } else {
        S.cak = S.cbk = cmk(0.0, 0.0);
    }
    if (first) sn[y] = S;
    if (!S.active) return;
    anp += y * sv;
    cr += y * sv;
    cq += y * sv;
    cp += y * sp;
    cap += y * sp;
    caw += y * sp;
    partials += y * region;
    const cplx<double> cak = S.cak, cakc = cconj(cak);
    cplx<double> s[2] = {cmk(0.0, 0.0), cmk(0.0, 0.0)};
    for (int i = blockIdx.x * KB + threadIdx.x; i < n; i += gridDim.x * KB) {
        cplx<double> a = anp[i];
        cfma(a, cak, cp[i]);
        anp[i] = a;
        cplx<double> r = cr[i];
        cfma(r, cscale(cak, -1.0), cap[i]);
        cr[i] = r;
        cplx<double> q = cq[i];
        cfma(q, cscale(cakc, -1.0), caw[i]);
        cq[i] = q;
        cfma(s[0], cconj(q), r);
        cfma(s[1], cconj(r), r);
    }
    block_sum3(s, 2);
    if (threadIdx.x == 0) {
        partials[2 * blockIdx.x] = s[0];
        partials[2 * blockIdx.x + 1] = s[1];
    }
}

// cp = cr + cbk cp ; cw = cq + conj(cbk) cw   (:928-929)
__global__ void bicg_c_dev_kernel(cplx<double> *__restrict__ cp, cplx<double> *__restrict__ cw,
                                  const cplx<double> *__restrict__ cr, const cplx<double> *__restrict__ cq, int64_t sv,
                                  int64_t sp, const BicgScal *__restrict__ sc, BicgScal *__restrict__ sn, int n,
                                  const cplx<double> *__restrict__ partials, int64_t region, int *__restrict__ gate)
{
    const int64_t y = blockIdx.y;
    auto next = [&](int64_t s) {
        BicgScal S = sc[s];
        if (S.active) {
            cplx<double> v[2];
            sum_blocks(partials + s * region, 2, gridDim.x, v);
            bicg_beta(S, v[0], v[1]);
        } else {
            S.cak = S.cbk = cmk(0.0, 0.0);
        }
        return S;
    };
    const BicgScal S = next(y);
    if (blockIdx.x == 0) {
        if (threadIdx.x == 0) sn[y] = S;
        if (gate && y % 2 == 0) {  // the pair's gate: the other system's state too
            const bool any = S.active || (y + 1 < gridDim.y && next(y + 1).active);
            if (threadIdx.x == 0) gate[y / 2] = any;
        }
    }
    if (!S.active) return;
    cp += y * sp;
    cw += y * sp;
    cr += y * sv;
    cq += y * sv;
    const cplx<double> cbk = S.cbk, cbkc = cconj(cbk);
    for (int i = blockIdx.x * KB + threadIdx.x; i < n; i += gridDim.x * KB) {
        cplx<double> p = cr[i];
        cfma(p, cbk, cp[i]);
        cp[i] = p;
        cplx<double> w = cq[i];
        cfma(w, cbkc, cw[i]);
        cw[i] = w;
    }
}

hipError_t launch_bicg_scal(int step, const double *partials, int64_t region, BicgScal *sc, int ns, int n,
                            hipStream_t st, int *gate)
{
    if (ns < 1 || step < 0 || step > 1) return hipErrorInvalidValue;
    hipLaunchKernelGGL(bicg_scal_kernel, dim3((ns + 1) / 2), dim3(KB), 0, st, step,
                       reinterpret_cast<const cplx<double> *>(partials), region, sc, ns, bicg_grid(n), gate);
    return hipGetLastError();
}
hipError_t launch_bicg_norm(const double *b, int64_t sv, int n, double *partials, int64_t region, int ns,
                            hipStream_t st)
{
    typedef cplx<double> Z;
    hipLaunchKernelGGL(bicg_norm_kernel, dim3(bicg_grid(n), ns), dim3(KB), 0, st, (const Z *)b, sv / 2, n,
                       (Z *)partials, region);
    return hipGetLastError();
}
hipError_t launch_bicg_init(double *cr, double *cq, double *cw, double *cp, const double *pnp, const double *anp,
                            int64_t sv, int64_t sp, int n, double *partials, int64_t region, int ns, hipStream_t st)
{
    typedef cplx<double> Z;
    hipLaunchKernelGGL(bicg_init_kernel, dim3(bicg_grid(n), ns), dim3(KB), 0, st, (Z *)cr, (Z *)cq, (Z *)cw, (Z *)cp,
                       (const Z *)pnp, (const Z *)anp, sv / 2, sp / 2, n, (Z *)partials, region);
    return hipGetLastError();
}
hipError_t launch_bicg_a_dev(double *cap, double *caw, const double *cp, const double *cw, int64_t sp, int n,
                             double *partials, int64_t region, const BicgScal *sc, int ns, hipStream_t st)
{
    typedef cplx<double> Z;
    hipLaunchKernelGGL(bicg_a_dev_kernel, dim3(bicg_grid(n), ns), dim3(KB), 0, st, (Z *)cap, (Z *)caw, (const Z *)cp,
                       (const Z *)cw, sp / 2, n, (Z *)partials, region, sc);
    return hipGetLastError();
}
hipError_t launch_bicg_b_dev(double *anp, double *cr, double *cq, const double *cp, const double *cap,
                             const double *caw, int64_t sv, int64_t sp, const BicgScal *sc, BicgScal *sn, int n,
                             const double *den, double *partials, int64_t region, int ns, hipStream_t st)
{
    typedef cplx<double> Z;
    hipLaunchKernelGGL(bicg_b_dev_kernel, dim3(bicg_grid(n), ns), dim3(KB), 0, st, (Z *)anp, (Z *)cr, (Z *)cq, (const Z *)cp,
                       (const Z *)cap, (const Z *)caw, sv / 2, sp / 2, sc, sn, n, (const Z *)den, (Z *)partials, region);
    return hipGetLastError();
}
hipError_t launch_bicg_c_dev(double *cp, double *cw, const double *cr, const double *cq, int64_t sv, int64_t sp,
                             const BicgScal *sc, BicgScal *sn, int n, const double *partials, int64_t region, int ns,
                             hipStream_t st, int *gate)
{
    typedef cplx<double> Z;
    hipLaunchKernelGGL(bicg_c_dev_kernel, dim3(bicg_grid(n), ns), dim3(KB), 0, st, (Z *)cp, (Z *)cw, (const Z *)cr,
                       (const Z *)cq, sv / 2, sp / 2, sc, sn, n, (const Z *)partials, region, gate);
    return hipGetLastError();
}
hipError_t launch_zaxpby(double ar, double ai, const double *x, double br, double bi, double *y, int n, hipStream_t st)
{
    typedef cplx<double> Z;
    hipLaunchKernelGGL(zaxpby_kernel, dim3(KGRID), dim3(KB), 0, st, cmk(ar, ai), (const Z *)x, cmk(br, bi), (Z *)y, n);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// One Arnoldi step of GMRES for one or two systems, without the host: the
// kernels of a step take both systems in one launch (blockIdx.z), and the
// projections, the Givens rotations and the stop test stay on the device
// (GmSys).  After the product p = T H v_j:
//   dots   w = v_j - p, written to v_{j+1}; <v_i, w>, i <= j
//   reduce h_i;   axpy  w -= sum_i h_i v_i
//   dots, reduce, axpy once more (with the block sums of |w|^2)
//   final  |w|, the column of H, its rotations, g, the stop test
//   scale  v_{j+1} = w / |w|
// Bound by reading the basis, twice per projection.  Four waves of a workgroup
// take four basis vectors each of a chunk of 256 rows, a lane the rows of four
// threads of a 256-wide reduction tree, so a sum needs no barrier and a step
// has thousands of waves: 38 us on average over a cycle of 120 steps for the two
// systems of a 1000-sphere cylinder, axpy 30 us, reduce + final + scale 30 us per
// step (one workgroup per chunk and system going through the vectors with a tree
// for each: 142 us the dots of both, and the host decided each step).  Sums run in
// the order of that tree over the 512 chunks, whatever the launch, so an
// Arnoldi vector's bits depend on the vectors before it only.
// ---------------------------------------------------------------------------
#define GM_SPAN (KGRID * KB)  // rows i, i + GM_SPAN, ... belong to one thread of the tree
static_assert(KB == 256, "gm kernels: 256-row chunks, four rows per lane");

// the tree over a chunk's 256 threads, lane t holding threads t, t+64, t+128, t+192
__device__ __forceinline__ cplx<double> tree256(const cplx<double> (&s)[4])
{
    cplx<double> v = cadd(cadd(s[0], s[2]), cadd(s[1], s[3]));
#pragma unroll
    for (int d = 32; d; d >>= 1) v = cadd(v, cmk(__shfl_xor(v.re, d), __shfl_xor(v.im, d)));
    return v;  // lane 0
}

__global__ __launch_bounds__(KB) void gm_dots_kernel(cplx<double> *__restrict__ V, int64_t stride, int64_t vs, int nv,
                                                     const cplx<double> *__restrict__ P, int64_t ps, int n,
                                                     const GmSys *__restrict__ sys, int pass,
                                                     cplx<double> *__restrict__ part, int64_t region)
{
    if (!sys[blockIdx.z].active) return;
    V += blockIdx.z * vs;
    P += blockIdx.z * ps;
    part += blockIdx.z * region;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int v0 = (blockIdx.y * 4 + wave) * 4;
    if (v0 >= nv) return;
    const cplx<double> *vj = V + (int64_t)(nv - 1) * stride;
    cplx<double> *wn = V + (int64_t)nv * stride;
    const bool first = v0 == 0 && !pass;
    cplx<double> s[4][4];
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
        for (int r = 0; r < 4; r++) s[q][r] = cmk(0.0, 0.0);
    for (int k0 = blockIdx.x * KB; k0 < n; k0 += GM_SPAN) {
        cplx<double> w[4], v[4][4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int i = k0 + lane + 64 * r;
            w[r] = cmk(0.0, 0.0);
            if (i < n) w[r] = pass ? wn[i] : csub(vj[i], P[i]);
#pragma unroll
            for (int q = 0; q < 4; q++) {
                v[q][r] = cmk(0.0, 0.0);
                if (v0 + q < nv && i < n) v[q][r] = V[(int64_t)(v0 + q) * stride + i];
            }
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int i = k0 + lane + 64 * r;
            if (first && i < n) wn[i] = w[r];
#pragma unroll
            for (int q = 0; q < 4; q++)
                if (i < n) cfma(s[q][r], cconj(v[q][r]), w[r]);
        }
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const cplx<double> t = tree256(s[q]);
        if (lane == 0 && v0 + q < nv) part[(int64_t)(v0 + q) * gridDim.x + blockIdx.x] = t;
    }
}

// h_i = sum over the chunks, one wave per i (chunks beyond the last are zero)
__global__ __launch_bounds__(KB) void gm_reduce_kernel(int nv, int nch, GmSys *__restrict__ sys, int pass,
                                                       const cplx<double> *__restrict__ part, int64_t region)
{
    GmSys &S = sys[blockIdx.z];
    const int j = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (!S.active || j >= nv) return;
    part += blockIdx.z * region + (int64_t)j * nch;
    cplx<double> s[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int b = lane + 64 * r;
        s[r] = b < nch ? part[b] : cmk(0.0, 0.0);
        if (b + KB < nch) s[r] = cadd(s[r], part[b + KB]);
    }
    const cplx<double> t = tree256(s);
    if (lane == 0) S.h[pass][j] = t;
}

// w -= sum_i h_i v_i; second pass: block sums of |w|^2
__global__ __launch_bounds__(KB) void gm_axpy_kernel(cplx<double> *__restrict__ V, int64_t stride, int64_t vs, int nv,
                                                     int n, const GmSys *__restrict__ sys, int pass,
                                                     cplx<double> *__restrict__ part, int64_t region)
{
    const GmSys &S = sys[blockIdx.z];
    if (!S.active) return;
    __shared__ cplx<double> hs[GM_M + 2], sh[KB];
    V += blockIdx.z * vs;
    for (int j = threadIdx.x; j < nv; j += KB) hs[j] = cscale(S.h[pass][j], -1.0);
    __syncthreads();
    cplx<double> s = cmk(0.0, 0.0);
    for (int i = blockIdx.x * KB + threadIdx.x; i < n; i += GM_SPAN) {
        cplx<double> a = V[(int64_t)nv * stride + i];
#pragma unroll 8
        for (int j = 0; j < nv; j++) cfma(a, hs[j], V[(int64_t)j * stride + i]);
        V[(int64_t)nv * stride + i] = a;
        cfma(s, cconj(a), a);
    }
    if (!pass) return;
    sh[threadIdx.x] = s;
    __syncthreads();
    if (threadIdx.x >= 64) return;
    cplx<double> f[4];
#pragma unroll
    for (int r = 0; r < 4; r++) f[r] = sh[threadIdx.x + 64 * r];
    s = tree256(f);
    if (threadIdx.x == 0) part[blockIdx.z * region + blockIdx.x] = s;
}

__global__ __launch_bounds__(KB) void gm_scale_kernel(cplx<double> *__restrict__ v, int64_t vs, int n,
                                                      const GmSys *__restrict__ sys)
{
    if (!sys[blockIdx.z].active) return;
    const double f = sys[blockIdx.z].scale;
    const int i = blockIdx.x * KB + threadIdx.x;
    if (i < n) v[blockIdx.z * vs + i] = cscale(v[blockIdx.z * vs + i], f);
}

// |w|, column j of H through the earlier rotations and its own, g, and
// the stop test (one workgroup per system); gate = any system active
__global__ __launch_bounds__(KB) void gm_final_kernel(int nv, int nb, GmSys *__restrict__ sys, int ns,
                                                      const cplx<double> *__restrict__ part, int64_t region,
                                                      int *__restrict__ gate, GmStat *__restrict__ stat)
{
    typedef cplx<double> Z;
    __shared__ Z col[GM_M + 1], sn[GM_M];
    __shared__ double cs[GM_M], sq[KGRID];
    int any = 0;
    for (int q = 0; q < ns; q++) {
        GmSys &S = sys[q];
        if (!S.active) continue;  // uniform
        const int j = nv - 1;
        for (int b = threadIdx.x; b < nb; b += KB) sq[b] = part[q * region + b].re;
        for (int i = threadIdx.x; i < nv; i += KB) {
            col[i] = cadd(S.h[0][i], S.h[1][i]);
            if (i < j) {
                sn[i] = S.sn[i];
                cs[i] = S.cs[i];
            }
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            double ww = 0.0;
            for (int b = 0; b < nb; b++) ww += sq[b];
            gm_column(S, col, cs, sn, nv, ww);
        }
        __syncthreads();
        any |= S.active;
    }
    if (threadIdx.x == 0) {
        *gate = any;
        for (int q = 0; q < ns; q++) stat[q] = {sys[q].err, sys[q].active, sys[q].done, sys[q].k};
        __threadfence_system();  // stat is pinned host memory
    }
}

// R y = g, back substitution (one workgroup per system), y in h[0]
__global__ __launch_bounds__(128) void gm_solve_kernel(GmSys *__restrict__ sys)
{
    typedef cplx<double> Z;
    GmSys &S = sys[blockIdx.x];
    const int k = S.k, t = threadIdx.x;
    __shared__ Z piv;
    Z g = t < k ? S.g[t] : cmk(0.0, 0.0);
    for (int r = k - 1; r >= 0; r--) {
        const Z *R = S.R + (r * (r + 1)) / 2;
        if (t == r) {
            piv = gm_pivot(g, R[r]);
            S.h[0][r] = piv;
        }
        __syncthreads();
        if (t < r) g = csub(g, cmul(R[t], piv));
        __syncthreads();
    }
}

// x += sum_{i < k} y_i v_i
__global__ __launch_bounds__(KB) void gm_update_kernel(const cplx<double> *__restrict__ U, int64_t stride, int64_t vs,
                                                       cplx<double> *__restrict__ x, int64_t xs, int n,
                                                       const GmSys *__restrict__ sys)
{
    const GmSys &S = sys[blockIdx.z];
    const int k = S.k;
    __shared__ cplx<double> hs[GM_M + 2];
    U += blockIdx.z * vs;
    x += blockIdx.z * xs;
    for (int j = threadIdx.x; j < k; j += KB) hs[j] = S.h[0][j];
    __syncthreads();
    const int i = blockIdx.x * KB + threadIdx.x;
    if (i >= n) return;
    cplx<double> a = x[i];
#pragma unroll 8
    for (int j = 0; j < k; j++) cfma(a, hs[j], U[(int64_t)j * stride + i]);
    x[i] = a;
}

// start of a cycle (beta = 0: not a system of it)
__global__ void gm_begin_kernel(GmSys *__restrict__ sys, int ns, GmStart a, GmStart b, int *__restrict__ gate)
{
    const int q = threadIdx.x;
    if (q == 0) *gate = 1;
    if (q >= ns) return;
    gm_begin(sys[q], q ? b : a);
}

static int gm_chunks(int n) { return imn(KGRID, (n + KB - 1) / KB); }
size_t gm_partials(int n) { return (size_t)2 * (GM_M + 1) * gm_chunks(n); }

hipError_t launch_gm_begin(GmSys *sys, int ns, const GmStart *st, double *V, int64_t vs, int n, int *gate,
                           hipStream_t str)
{
    if (ns < 1 || ns > 2) return hipErrorInvalidValue;
    hipLaunchKernelGGL(gm_begin_kernel, dim3(1), dim3(64), 0, str, sys, ns, st[0], st[ns - 1], gate);
    hipLaunchKernelGGL(gm_scale_kernel, dim3((n + KB - 1) / KB, 1, ns), dim3(KB), 0, str, (cplx<double> *)V, vs / 2, n,
                       sys);
    return hipGetLastError();
}

hipError_t launch_gm_step(GmSys *sys, int ns, double *V, int64_t stride, int64_t vs, int nv, const double *p,
                          int64_t ps, int n, double *partials, int *gate, GmStat *stat, hipStream_t str)
{
    typedef cplx<double> Z;
    if (ns < 1 || ns > 2 || nv < 1 || nv > GM_M) return hipErrorInvalidValue;
    const int nch = gm_chunks(n);
    const int64_t region = (int64_t)gm_partials(n) / 2;
    Z *v = (Z *)V, *part = (Z *)partials;
    for (int pass = 0; pass < 2; pass++) {
        hipLaunchKernelGGL(gm_dots_kernel, dim3(nch, (nv + 15) / 16, ns), dim3(KB), 0, str, v, stride / 2, vs / 2, nv,
                           (const Z *)p, ps / 2, n, sys, pass, part, region);
        hipLaunchKernelGGL(gm_reduce_kernel, dim3((nv + 3) / 4, 1, ns), dim3(KB), 0, str, nv, nch, sys, pass, part,
                           region);
        hipLaunchKernelGGL(gm_axpy_kernel, dim3(nch, 1, ns), dim3(KB), 0, str, v, stride / 2, vs / 2, nv, n, sys, pass,
                           part, region);
    }
    hipLaunchKernelGGL(gm_final_kernel, dim3(1), dim3(KB), 0, str, nv, nch, sys, ns, part, region, gate, stat);
    hipLaunchKernelGGL(gm_scale_kernel, dim3((n + KB - 1) / KB, 1, ns), dim3(KB), 0, str, v + nv * (stride / 2), vs / 2,
                       n, sys);
    return hipGetLastError();
}

hipError_t launch_gm_update(GmSys *sys, int ns, const double *U, int64_t stride, int64_t vs, double *x, int64_t xs,
                            int n, hipStream_t str)
{
    typedef cplx<double> Z;
    hipLaunchKernelGGL(gm_solve_kernel, dim3(ns), dim3(128), 0, str, sys);
    hipLaunchKernelGGL(gm_update_kernel, dim3((n + KB - 1) / KB, 1, ns), dim3(KB), 0, str, (const Z *)U, stride / 2,
                       vs / 2, (Z *)x, xs / 2, n, sys);
    return hipGetLastError();
}
