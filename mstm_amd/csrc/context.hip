// context.hip -- C-ABI entry points (include/mstm_hip.h) and the host-side
// orchestration of the device kernels: sphere state, operator set-up, the
// BiCG driver of cbicg (mstm-solver-8.f90:654-949), the mixed-precision
// refinement around it, and fixedorsoln (mstm-solver-8.f90:350-569).
#include <chrono>
#include <complex>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/mstm_hip.h"
#include "common.hpp"
#include "kernels.hpp"
#include "specfun.hpp"
#include "fft.hpp"
#include "learned.hpp"

// largest number of workgroups sharing one direct tile's 16 steps
#ifndef MSTM_TGROUPS_MAX
#define MSTM_TGROUPS_MAX MSTM_SLOTS
#endif

namespace {

struct DirectOp {
    bool ready = false;
    void *tab = nullptr;
    void *xin = nullptr;
    void *part = nullptr;
    size_t tab_bytes = 0;
};

struct Stats {
    double tables_ms[2] = {0, 0};
    double tile_ms[2] = {0, 0};  // two-column launches
    long tile_launches[2] = {0, 0};
    double tile4_ms[2] = {0, 0};  // four-column launches (both polarizations)
    long tile4_launches[2] = {0, 0};
    double matvec_ms = 0;
    long matvecs[2] = {0, 0};
    double solve_ms = 0;
    long iters_fp64 = 0, iters_fp32 = 0, refinements = 0;
    double table_bytes[2] = {0, 0};
    double fft_setup_ms = 0, fft_conv_ms = 0;
    long fft_launches = 0;
    long lig_solves = 0, lig_fallbacks = 0, fgmres_steps = 0;
    double lig_ms = 0, lig_err0 = 0, lig_errb = 0;
};

// learned initial guess: network parameters and per-sphere work buffers
struct LearnedNet {
    bool ready = false;
    MlpShape s{};
    int Lnet = 0;
    float *params = nullptr;
    size_t np = 0;
    int cap = 0;
    float *feat = nullptr, *depth = nullptr, *out = nullptr;
    std::vector<float *> H;
};

// Krylov work-vector slots (complex FP64, neqns each).  Blocks that one
// product reads or writes are contiguous.
enum {
    KV_PW = 0,    // 0-3   product inputs  [p_0, w_0, p_1, w_1] of the two BiCG systems
    KV_CAPS = 4,  // 4-7   product outputs [A p_0, A^H w_0, A p_1, A^H w_1]
    KV_RB = 8,    // 8-9   BiCG residuals r_0, r_1
    KV_QB = 10,   // 10-11 BiCG shadow residuals q_0, q_1
    KV_X = 12,    // 12-13 solutions (both polarizations)
    KV_Y = 14,    // 14-15 refinement products
    KV_R = 16,    // 16-17 refinement residuals
    KV_D = 18,    // 18-19 refinement corrections
    KV_B = 20,    // 20-21 right-hand sides b = T f
    KV_PM = 22,   // 22-23 incident field f (pmnp)
    KV_ST = 24,   // 24-27 host staging
    KV_N = 28
};

}  // namespace

// a block of BiCG systems takes at most this much work space
#define BICG_BLOCK_BYTES ((size_t)512 << 20)

struct mstm_hip_ctx {
    int device = 0;
    hipStream_t st = nullptr;
    std::string err;
    int nsph = 0, npad = 0, Lmax = 0, neqns = 0;
    double rimed = 1.0;
    std::vector<int> order, offset;
    std::vector<double> pos, radius, ri;
    double *d_pos = nullptr, *d_radius = nullptr, *d_mre = nullptr, *d_mim = nullptr;
    int *d_order = nullptr, *d_offset = nullptr, *d_mieoff = nullptr;
    double *d_an = nullptr;  // complex, (npad*Lmax*4), sphere-uniform stride 4*Lmax
    int *d_excited = nullptr;  // excited_spheres mask of the last fixedorsoln (nsph)
    double *d_qeff = nullptr;  // per-sphere efficiencies of fixedorsoln (9 nsph)
    int2 *d_tiles = nullptr;
    int ntiles = 0, nblocks = 0;
    int tgroups = 1;  // workgroups per direct tile (its 16 steps split among them)
    double *d_vcc = nullptr;
    int vcc_LM = 0;
    DirectOp dop[2];
    FftOp *fft = nullptr;
    LearnedNet lig;
    double *d_fg = nullptr;  // FGMRES basis V (m+1) and Z (m), complex FP64
    size_t fg_bytes = 0;
    double *d_gm = nullptr;  // GMRES basis of the inner solver, two systems interleaved
    size_t gm_bytes = 0;
    GmSys *d_gsys = nullptr;  // small quantities of two GMRES systems
    GmStat *h_gstat = nullptr;  // pinned: their state after the last two steps
    hipEvent_t gm_ev[2] = {nullptr, nullptr};
    double *d_gp = nullptr;  // block sums of the GMRES projections
    size_t gp_bytes = 0;
    int inner = 1;           // inner solver of the mixed refinement: 0 BiCG, 1 GMRES
    int max_ref = 6;         // FP64 refinement cycles of the mixed solvers
    // Krylov work vectors (complex FP64, neqns each)
    double *d_kv = nullptr;
    size_t kv_n = 0;
    double *d_partials = nullptr;
    std::vector<double> h_partials;
    BicgScal *d_bscal = nullptr;  // device-resident BiCG scalars of two systems, twice
    BicgScal *h_bscal = nullptr;  // their pinned host copy
    bool graphs = true;           // replay lazily read BiCG iterations from HIP graphs
    int *d_gate = nullptr;        // 1 while any of those systems is active
    const int *gate = nullptr;    // set while a lazily read BiCG loop issues products
    // HIP graphs of K lazily read BiCG iterations, one per pattern of active
    // systems (both, the first, the second), with the buffers they were
    // captured on and the products one replay makes
    struct BicgGraph {
        hipGraphExec_t exec = nullptr;
        std::vector<intptr_t> key;
        int matvecs = 0;
    } bgraph[3];
    // event pool for tile-kernel timing
    std::vector<hipEvent_t> ev;
    std::vector<int> ev_prec;
    size_t ev_used = 0;
    bool timing = true;
    Stats stats;
    // post-solve observables of a single-origin expansion
    struct {
        bool x_valid = false;  // KV_X holds the last fixedorsoln solution
        int T = 0;             // common-origin order of the last translation_orders call
        double r0[3] = {0, 0, 0};
        std::vector<int> torder;
        int *d_torder = nullptr;
        double *d_vccm = nullptr;
        int vccm_T = 0, vccm_LS = 0;
        double *d_part = nullptr;
        size_t part_bytes = 0;
        double *d_a0 = nullptr;  // merged E/M coefficients, 2 columns x 2 x T(T+2) complex
        size_t a0_bytes = 0;
        int a0_T = 0;
        double *d_in = nullptr;  // caller-supplied common-origin coefficients
        size_t in_bytes = 0;
        double *d_ang = nullptr, *d_sm = nullptr;
        size_t ang_cap = 0;
        double *d_cg = nullptr, *d_mom = nullptr;
        int cg_T = 0;
        double *d_bc = nullptr, *d_fpart = nullptr;  // fosmexpansion: bcof table, block sums
        int bc_T = 0;
        double orders_ms = 0, merge_ms = 0, scatmat_ms = 0, moments_ms = 0, fosm_ms = 0;
        // T-matrix solution: distribute table and the unit-excitation columns
        double *d_vccd = nullptr;
        int vccd_T = 0, vccd_LS = 0;
        double *d_dist = nullptr, *d_dq = nullptr;
        size_t dist_bytes = 0, dq_bytes = 0;
        unsigned char *d_blk = nullptr;  // work space of a block of column pairs (BicgBlock)
        size_t blk_bytes = 0;
        double tmatrix_ms = 0;
        int tm_solves = 0;
        double *h_pin = nullptr;  // pinned host copies of each column pair's efficiencies and merge
        size_t pin_bytes = 0;
    } obs;
    // dense interaction matrix A = I - T H and its LU factors (direct solution)
    struct {
        double *A = nullptr, *LU = nullptr, *vv = nullptr, *work = nullptr;
        int *piv = nullptr, *err = nullptr;
        void *scr = nullptr;
        int n = 0;
        int polls = 1 << 21;  // looks of a panel's workgroups for each other, about a second
        bool ready = false;
        double build_ms = 0, factor_ms = 0, solve_ms = 0;
    } lu;
};

static int fail(mstm_hip_ctx *c, int code, const char *fmt, ...)
{
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    if (c) c->err = buf;
    return code;
}
#define HIPCHK(call)                                                                                                   \
    do {                                                                                                               \
        hipError_t e_ = (call);                                                                                        \
        if (e_ != hipSuccess) return fail(c, MSTM_HIP_EHIP, "%s failed: %s", #call, hipGetErrorString(e_));            \
    } while (0)

template <typename P> static hipError_t dalloc(P **p, size_t bytes)
{
    *p = nullptr;
    if (bytes == 0) return hipSuccess;
    return hipMalloc((void **)p, bytes);
}
template <typename P> static void dfree(P *&p)
{
    if (p) hipFree((void *)p);
    p = nullptr;
}

// ---------------------------------------------------------------- scratch
// Device scratch of mstm_hip_sphereinteraction_noalloc: one file-scope array
// per GPU, held until the process ends.  Host code never passes `scratch`
// itself to a kernel (in host code the name is only a stand-in for the
// symbol): each device's address comes from hipGetSymbolAddress, taken once
// per device with that device current (mstm_hip_create), and kernels get
// that address.
#define MSTM_SCRATCH_BYTES (32u << 20)
static __device__ __align__(256) unsigned char scratch[MSTM_SCRATCH_BYTES];
#define MSTM_MAX_DEVICES 64
static std::mutex g_scratch_mu;
static void *g_scratch_ptr[MSTM_MAX_DEVICES];
static hipError_t g_scratch_rc[MSTM_MAX_DEVICES];
static bool g_scratch_done[MSTM_MAX_DEVICES];

// address of this device's scratch array; the device must be current
static hipError_t scratch_bind(int device)
{
    if (device < 0 || device >= MSTM_MAX_DEVICES) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_done[device]) {
        void *p = nullptr;
        g_scratch_rc[device] = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        g_scratch_ptr[device] = g_scratch_rc[device] == hipSuccess ? p : nullptr;
        g_scratch_done[device] = true;
    }
    return g_scratch_rc[device];
}

// ---------------------------------------------------------------- constants
// vector-coupling products vcc(n, l, m, w) of axialtrancoefinit
// (mstm-modules-33.f90:1680-1710): -sqrt((2n+1)(2l+1)) (-1)^m
// C(n,-m;l,m|w,0) C(n,-1;l,1|w,0) (Re+Im)(i^(n-l+w)); Clebsch-Gordan
// coefficients from Racah's sum in long double.
static long double lfac(int n)
{
    static std::vector<long double> f;
    if (f.empty()) {
        f.resize(400);
        f[0] = 1.0L;
        for (int k = 1; k < 400; k++) f[k] = f[k - 1] * (long double)k;
    }
    return f[n];
}
static long double clebsch(int j1, int m1, int j2, int m2, int J)
{
    int M = m1 + m2;
    if (std::abs(m1) > j1 || std::abs(m2) > j2 || std::abs(M) > J || J < std::abs(j1 - j2) || J > j1 + j2) return 0;
    long double pre = (2.0L * J + 1.0L) * lfac(J + j1 - j2) * lfac(J - j1 + j2) * lfac(j1 + j2 - J) / lfac(j1 + j2 + J + 1);
    pre *= lfac(J + M) * lfac(J - M) * lfac(j1 - m1) * lfac(j1 + m1) * lfac(j2 - m2) * lfac(j2 + m2);
    int kmin = std::max(0, std::max(j2 - J - m1, j1 - J + m2)), kmax = std::min(j1 + j2 - J, std::min(j1 - m1, j2 + m2));
    long double s = 0;
    for (int k = kmin; k <= kmax; k++)
        s += ((k & 1) ? -1.0L : 1.0L) / (lfac(k) * lfac(j1 + j2 - J - k) * lfac(j1 - m1 - k) * lfac(j2 + m2 - k) *
                                          lfac(J - j2 + m1 + k) * lfac(J - j1 - m2 + k));
    return sqrtl(pre) * s;
}
void vcc_table(int LM, std::vector<double> &h)
{
    size_t n = (size_t)(LM + 1) * (LM + 1) * (2 * LM + 1) * (2 * LM + 1);
    h.assign(n, 0.0);
    for (int nn = 1; nn <= LM; nn++)
        for (int l = 1; l <= LM; l++) {
            long double c1 = sqrtl((long double)(2 * nn + 1)) * sqrtl((long double)(2 * l + 1));
            for (int m = -std::min(nn, l); m <= std::min(nn, l); m++)
                for (int w = std::abs(nn - l); w <= nn + l; w++) {
                    long double c2 = -c1 * ((std::abs(m) & 1) ? -1.0L : 1.0L);
                    int k4 = (nn - l + w) & 3;
                    long double sg = (k4 == 0 || k4 == 1) ? 1.0L : -1.0L;
                    h[vcc_index(nn, l, m, w, LM)] =
                        (double)(c2 * clebsch(nn, -m, l, m, w) * clebsch(nn, -1, l, 1, w) * sg);
                }
        }
}

static int ensure_vcc(mstm_hip_ctx *c, int LM)
{
    if (c->d_vcc && c->vcc_LM >= LM) return 0;
    dfree(c->d_vcc);
    std::vector<double> h;
    vcc_table(LM, h);
    const size_t n = h.size();
    HIPCHK(dalloc(&c->d_vcc, n * sizeof(double)));
    HIPCHK(hipMemcpy(c->d_vcc, h.data(), n * sizeof(double), hipMemcpyHostToDevice));
    c->vcc_LM = LM;
    return 0;
}

static void release_direct(mstm_hip_ctx *c, int p)
{
    dfree(c->dop[p].tab);
    dfree(c->dop[p].xin);
    dfree(c->dop[p].part);
    c->dop[p].ready = false;
}

static void release_lig_buffers(mstm_hip_ctx *c)
{
    dfree(c->lig.feat);
    dfree(c->lig.depth);
    dfree(c->lig.out);
    for (auto &q : c->lig.H) dfree(q);
    c->lig.H.clear();
    c->lig.cap = 0;
}

static void release_lu(mstm_hip_ctx *c)
{
    dfree(c->lu.A);
    dfree(c->lu.LU);
    dfree(c->lu.vv);
    dfree(c->lu.work);
    dfree(c->lu.piv);
    dfree(c->lu.err);
    dfree(c->lu.scr);
    c->lu.n = 0;
    c->lu.ready = false;
}

static void release_spheres(mstm_hip_ctx *c)
{
    release_lu(c);
    release_lig_buffers(c);
    release_direct(c, 0);
    release_direct(c, 1);
    if (c->fft) {
        fft_destroy(c->fft);
        c->fft = nullptr;
    }
    dfree(c->d_pos);
    dfree(c->d_radius);
    dfree(c->d_mre);
    dfree(c->d_mim);
    dfree(c->d_order);
    dfree(c->d_offset);
    dfree(c->d_mieoff);
    dfree(c->d_an);
    dfree(c->d_excited);
    dfree(c->d_qeff);
    dfree(c->d_tiles);
    dfree(c->d_kv);
    dfree(c->d_fg);
    c->fg_bytes = 0;
    dfree(c->d_gm);
    c->gm_bytes = 0;
    c->kv_n = 0;
    c->nsph = 0;
    c->obs.x_valid = false;
    c->obs.T = 0;
    c->obs.a0_T = 0;
    c->obs.torder.clear();
    dfree(c->obs.d_torder);
    dfree(c->obs.d_blk);
    c->obs.blk_bytes = 0;
}

static void release_observables(mstm_hip_ctx *c)
{
    dfree(c->obs.d_torder);
    dfree(c->obs.d_vccm);
    dfree(c->obs.d_part);
    dfree(c->obs.d_a0);
    dfree(c->obs.d_in);
    dfree(c->obs.d_ang);
    dfree(c->obs.d_sm);
    dfree(c->obs.d_cg);
    dfree(c->obs.d_mom);
    dfree(c->obs.d_bc);
    dfree(c->obs.d_fpart);
    c->obs.bc_T = 0;
    dfree(c->obs.d_vccd);
    dfree(c->obs.d_dist);
    dfree(c->obs.d_dq);
    if (c->obs.h_pin) hipHostFree(c->obs.h_pin);
    c->obs.h_pin = nullptr;
    c->obs.pin_bytes = 0;
    c->obs.vccm_T = c->obs.vccm_LS = c->obs.cg_T = c->obs.vccd_T = c->obs.vccd_LS = 0;
    c->obs.part_bytes = c->obs.a0_bytes = c->obs.in_bytes = c->obs.ang_cap = 0;
    c->obs.dist_bytes = c->obs.dq_bytes = 0;
}

// ------------------------------------------------------------------ C ABI
extern "C" {

int mstm_hip_create(mstm_hip_ctx **ctx, int device)
{
    if (!ctx) return MSTM_HIP_EARG;
    *ctx = nullptr;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= device || device < 0) return MSTM_HIP_EHIP;
    mstm_hip_ctx *c = new mstm_hip_ctx();
    c->device = device;
    HIPCHK(hipSetDevice(device));
    // the allocation-free entry point's scratch on this device; a failure is
    // kept and reported by that entry point, other calls do not need it
    (void)scratch_bind(device);
    HIPCHK(hipStreamCreateWithFlags(&c->st, hipStreamNonBlocking));
    HIPCHK(dalloc(&c->d_partials, sizeof(double) * 16 * krylov_grid()));  // 8 regions of one value per block
    c->h_partials.resize(16 * krylov_grid());
    HIPCHK(dalloc(&c->d_bscal, sizeof(BicgScal) * 4));
    HIPCHK(dalloc(&c->d_gate, sizeof(int)));
    HIPCHK(hipHostMalloc((void **)&c->h_bscal, sizeof(BicgScal) * 2, hipHostMallocDefault));
    *ctx = c;
    return 0;
}

int mstm_hip_destroy(mstm_hip_ctx *c)
{
    if (!c) return 0;
    hipSetDevice(c->device);
    hipStreamSynchronize(c->st);
    release_spheres(c);
    release_observables(c);
    dfree(c->lig.params);
    dfree(c->d_gsys);
    dfree(c->d_gp);
    for (auto &e : c->gm_ev)
        if (e) hipEventDestroy(e);
    if (c->h_gstat) hipHostFree(c->h_gstat);
    dfree(c->d_vcc);
    dfree(c->d_partials);
    dfree(c->d_bscal);
    dfree(c->d_gate);
    for (auto &g : c->bgraph)
        if (g.exec) hipGraphExecDestroy(g.exec);
    if (c->h_bscal) hipHostFree(c->h_bscal);
    for (auto &e : c->ev) hipEventDestroy(e);
    hipStreamDestroy(c->st);
    delete c;
    return 0;
}

const char *mstm_hip_last_error(const mstm_hip_ctx *c) { return c ? c->err.c_str() : "null context"; }

static int finish_sphere_layout(mstm_hip_ctx *c)
{
    int n = c->nsph;
    c->offset.assign(n + 1, 0);
    c->Lmax = 0;
    for (int i = 0; i < n; i++) {
        c->offset[i + 1] = c->offset[i] + 2 * c->order[i] * (c->order[i] + 2);
        c->Lmax = std::max(c->Lmax, c->order[i]);
    }
    c->neqns = c->offset[n];
    if (c->Lmax > 8) return fail(c, MSTM_HIP_EUNSUP, "sphere order %d > 8 not compiled", c->Lmax);
    std::vector<int> mieoff(n);
    for (int i = 0; i < n; i++) mieoff[i] = 4 * c->Lmax * i;
    dfree(c->d_offset);
    dfree(c->d_mieoff);
    HIPCHK(dalloc(&c->d_offset, sizeof(int) * (n + 1)));
    HIPCHK(dalloc(&c->d_mieoff, sizeof(int) * n));
    HIPCHK(hipMemcpy(c->d_order, c->order.data(), sizeof(int) * n, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(c->d_offset, c->offset.data(), sizeof(int) * (n + 1), hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(c->d_mieoff, mieoff.data(), sizeof(int) * n, hipMemcpyHostToDevice));
    // direct-operator tiling over blocks of MSTM_SLOTS spheres
    c->npad = (n + MSTM_SLOTS - 1) / MSTM_SLOTS * MSTM_SLOTS;
    c->nblocks = c->npad / MSTM_SLOTS;
    std::vector<int2> tiles;
    for (int bi = 0; bi < c->nblocks; bi++)
        for (int bj = bi; bj < c->nblocks; bj++) tiles.push_back(make_int2(bi, bj));
    c->ntiles = (int)tiles.size();
    // few tiles (small clusters): split each tile's 16 steps over up to 16
    // workgroups, doubling while the launch stays within 512 workgroups (two
    // per CU of 256): more groups leave each with a few steps that cannot
    // pay for staging its sources, and more partial sums to add; each group
    // keeps its own partial sums (partial buffer at most 256 MiB at FP64,
    // four columns)
    c->tgroups = 1;
    {
        const size_t nbp = (size_t)c->Lmax * (c->Lmax + 2);
        auto part_bytes = [&](int G) { return sizeof(double) * 2 * (size_t)c->nblocks * G * 4 * 2 * c->npad * nbp; };
        while (c->tgroups < MSTM_TGROUPS_MAX && (int64_t)c->ntiles * c->tgroups * 2 <= 512 &&
               part_bytes(2 * c->tgroups) <= ((size_t)256 << 20))
            c->tgroups *= 2;
    }
    dfree(c->d_tiles);
    HIPCHK(dalloc(&c->d_tiles, sizeof(int2) * tiles.size()));
    HIPCHK(hipMemcpy(c->d_tiles, tiles.data(), sizeof(int2) * tiles.size(), hipMemcpyHostToDevice));
    // Krylov work space (slot plan KV_*)
    c->kv_n = (size_t)c->neqns;
    dfree(c->d_kv);
    HIPCHK(dalloc(&c->d_kv, sizeof(double) * 2 * c->kv_n * KV_N));
    return 0;
}

int mstm_hip_set_spheres(mstm_hip_ctx *c, int n, const double *pos, const double *radius, const double *ri,
                         double ri_medium, double mie_eps)
{
    if (!c || n <= 0 || !pos || !radius || !ri) return fail(c, MSTM_HIP_EARG, "set_spheres: bad arguments");
    HIPCHK(hipSetDevice(c->device));
    release_spheres(c);
    c->nsph = n;
    c->rimed = ri_medium;
    c->pos.assign(pos, pos + 3 * n);
    c->radius.assign(radius, radius + n);
    c->ri.assign(ri, ri + 2 * n);
    std::vector<double> mre(n), mim(n);
    for (int i = 0; i < n; i++) {
        mre[i] = ri[2 * i];
        mim[i] = ri[2 * i + 1];
    }
    HIPCHK(dalloc(&c->d_pos, sizeof(double) * 3 * n));
    HIPCHK(dalloc(&c->d_radius, sizeof(double) * n));
    HIPCHK(dalloc(&c->d_mre, sizeof(double) * n));
    HIPCHK(dalloc(&c->d_mim, sizeof(double) * n));
    HIPCHK(dalloc(&c->d_order, sizeof(int) * n));
    HIPCHK(dalloc(&c->d_excited, sizeof(int) * n));
    HIPCHK(dalloc(&c->d_qeff, sizeof(double) * 9 * n));
    HIPCHK(hipMemcpy(c->d_pos, pos, sizeof(double) * 3 * n, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(c->d_radius, radius, sizeof(double) * n, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(c->d_mre, mre.data(), sizeof(double) * n, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(c->d_mim, mim.data(), sizeof(double) * n, hipMemcpyHostToDevice));
    // pass 1: orders
    HIPCHK(launch_mie(c->d_radius, c->d_mre, c->d_mim, ri_medium, n, mie_eps, c->d_order, nullptr, 0, c->st));
    c->order.resize(n);
    HIPCHK(hipMemcpyAsync(c->order.data(), c->d_order, sizeof(int) * n, hipMemcpyDeviceToHost, c->st));
    HIPCHK(hipStreamSynchronize(c->st));
    int rc = finish_sphere_layout(c);
    if (rc) return rc;
    // pass 2: Mie matrices at the selected orders, stride 4*Lmax per sphere
    HIPCHK(dalloc(&c->d_an, sizeof(double) * 2 * 4 * (size_t)c->Lmax * c->npad));
    HIPCHK(hipMemsetAsync(c->d_an, 0, sizeof(double) * 2 * 4 * (size_t)c->Lmax * c->npad, c->st));
    HIPCHK(launch_mie(c->d_radius, c->d_mre, c->d_mim, ri_medium, n, mie_eps, c->d_order, c->d_an, 4 * c->Lmax, c->st));
    HIPCHK(hipStreamSynchronize(c->st));
    return 0;
}

int mstm_hip_set_mie(mstm_hip_ctx *c, const int *order, const double *an_mie)
{
    if (!c || !c->nsph || !order || !an_mie) return fail(c, MSTM_HIP_ESTATE, "set_mie: no spheres");
    int n = c->nsph;
    // everything built from the old orders or Mie matrices goes: operator
    // tables, the FFT grid, the LU factors and the held solution
    release_lu(c);
    release_direct(c, 0);
    release_direct(c, 1);
    if (c->fft) {
        fft_destroy(c->fft);
        c->fft = nullptr;
    }
    c->obs.x_valid = false;
    c->order.assign(order, order + n);
    int rc = finish_sphere_layout(c);
    if (rc) return rc;
    std::vector<double> h((size_t)2 * 4 * c->Lmax * c->npad, 0.0);
    size_t src = 0;
    for (int i = 0; i < n; i++)
        for (int q = 0; q < 4 * c->order[i]; q++, src++) {
            h[2 * ((size_t)i * 4 * c->Lmax + q)] = an_mie[2 * src];
            h[2 * ((size_t)i * 4 * c->Lmax + q) + 1] = an_mie[2 * src + 1];
        }
    dfree(c->d_an);
    HIPCHK(dalloc(&c->d_an, sizeof(double) * h.size()));
    HIPCHK(hipMemcpy(c->d_an, h.data(), sizeof(double) * h.size(), hipMemcpyHostToDevice));
    return 0;
}

int mstm_hip_get_orders(const mstm_hip_ctx *c, int *order, int *offset)
{
    if (!c || !c->nsph) return MSTM_HIP_ESTATE;
    if (order) memcpy(order, c->order.data(), sizeof(int) * c->nsph);
    if (offset) memcpy(offset, c->offset.data(), sizeof(int) * (c->nsph + 1));
    return 0;
}

int mstm_hip_number_eqns(const mstm_hip_ctx *c) { return c ? c->neqns : 0; }

int mstm_hip_get_mie(const mstm_hip_ctx *cc, double *an_mie)
{
    mstm_hip_ctx *c = const_cast<mstm_hip_ctx *>(cc);
    if (!c || !c->nsph || !an_mie) return MSTM_HIP_ESTATE;
    std::vector<double> h((size_t)2 * 4 * c->Lmax * c->npad);
    HIPCHK(hipMemcpy(h.data(), c->d_an, sizeof(double) * h.size(), hipMemcpyDeviceToHost));
    size_t dst = 0;
    for (int i = 0; i < c->nsph; i++)
        for (int q = 0; q < 4 * c->order[i]; q++, dst++) {
            an_mie[2 * dst] = h[2 * ((size_t)i * 4 * c->Lmax + q)];
            an_mie[2 * dst + 1] = h[2 * ((size_t)i * 4 * c->Lmax + q) + 1];
        }
    return 0;
}

// the tables, padded input and partial sums of one precision's operator
static int direct_alloc(mstm_hip_ctx *c, int prec)
{
    release_direct(c, prec);
    DirectOp &d = c->dop[prec];
    const int L = c->Lmax;
    const size_t esz = prec == MSTM_HIP_FP64 ? sizeof(double) : sizeof(float);
    size_t slot = (size_t)direct_slot_len(L, (int)esz);
    d.tab_bytes = (size_t)c->ntiles * MSTM_SLOTS * MSTM_SLOTS * slot * esz;
    size_t nbp = (size_t)L * (L + 2);
    HIPCHK(dalloc(&d.tab, d.tab_bytes));
    HIPCHK(dalloc(&d.xin, esz * 2 * 4 * 2 * (size_t)c->npad * nbp));
    HIPCHK(dalloc(&d.part, esz * 2 * (size_t)c->nblocks * c->tgroups * 4 * 2 * c->npad * nbp));
    return 0;
}

int mstm_hip_setup_direct(mstm_hip_ctx *c, int prec)
{
    if (!c || !c->nsph) return fail(c, MSTM_HIP_ESTATE, "setup_direct: no spheres");
    if (prec != MSTM_HIP_FP64 && prec != MSTM_HIP_FP32 && prec != MSTM_HIP_FP64_FP32)
        return fail(c, MSTM_HIP_EARG, "setup_direct: precision");
    HIPCHK(hipSetDevice(c->device));
    const int L = c->Lmax;
    if (prec == MSTM_HIP_FP64_FP32 && !direct_tables_both_ok(L)) {
        int rc = mstm_hip_setup_direct(c, MSTM_HIP_FP64);
        return rc ? rc : mstm_hip_setup_direct(c, MSTM_HIP_FP32);
    }
    int rc = ensure_vcc(c, L);
    if (rc) return rc;
    const int p0 = prec == MSTM_HIP_FP32 ? MSTM_HIP_FP32 : MSTM_HIP_FP64;
    const int p1 = prec == MSTM_HIP_FP64 ? MSTM_HIP_FP64 : MSTM_HIP_FP32;
    for (int p = p0; p <= p1; p++)
        if ((rc = direct_alloc(c, p))) return rc;
    auto t0 = std::chrono::steady_clock::now();
    if (prec == MSTM_HIP_FP64_FP32)
        HIPCHK(launch_direct_tables_both((double *)c->dop[0].tab, (float *)c->dop[1].tab, c->d_tiles, c->ntiles, L,
                                         c->nsph, c->d_pos, c->rimed, c->d_vcc, c->vcc_LM, c->st));
    else if (prec == MSTM_HIP_FP64)
        HIPCHK(launch_direct_tables<double>((double *)c->dop[0].tab, c->d_tiles, c->ntiles, L, c->nsph, c->d_pos,
                                            c->rimed, c->d_vcc, c->vcc_LM, c->st));
    else
        HIPCHK(launch_direct_tables<float>((float *)c->dop[1].tab, c->d_tiles, c->ntiles, L, c->nsph, c->d_pos,
                                           c->rimed, c->d_vcc, c->vcc_LM, c->st));
    HIPCHK(hipStreamSynchronize(c->st));
    const double ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    for (int p = p0; p <= p1; p++) {
        // one pass for both: its time is booked to the FP64 tables
        c->stats.tables_ms[p] = p == p0 ? ms : 0.0;
        c->stats.table_bytes[p] = (double)c->dop[p].tab_bytes;
        c->dop[p].ready = true;
    }
    return 0;
}

int mstm_hip_node_selection(mstm_hip_ctx *c, double *fva, const double *target_min, const double *target_max,
                            int d_specified, double *d_cell, int local_host, int node_order, int neighbor_node_model,
                            int *cell_dim, int *node_order_out)
{
    if (!c || !c->nsph) return fail(c, MSTM_HIP_ESTATE, "node_selection: no spheres");
    if (!fva || !cell_dim || !d_cell || !node_order_out) return fail(c, MSTM_HIP_EARG, "node_selection: null argument");
    if (local_host != 0)
        return fail(c, MSTM_HIP_EUNSUP, "node_selection: local_host %d (spheres inside a host sphere) is not on the "
                                        "GPU path", local_host);
    if (neighbor_node_model < 0 || neighbor_node_model > 3)
        return fail(c, MSTM_HIP_EARG, "node_selection: neighbor_node_model %d", neighbor_node_model);
    HIPCHK(hipSetDevice(c->device));
    if (c->fft) {
        fft_destroy(c->fft);
        c->fft = nullptr;
    }
    FftGeometry g{c->nsph,          c->Lmax,    c->neqns,   c->pos.data(), c->radius.data(), c->order.data(),
                  c->offset.data(), c->rimed,   c->d_pos,   c->d_order,    c->d_offset,      c->d_an,
                  c->d_vcc,         c->vcc_LM};
    int err = 0;
    const char *why = "node_selection failed";
    FftOp *f = fft_create(g, fva, target_min, target_max, d_specified, node_order, neighbor_node_model, cell_dim,
                          d_cell, node_order_out, &err, &why);
    if (!f) return fail(c, err ? err : MSTM_HIP_EHIP, "%s", why);
    c->fft = f;
    return 0;
}

int mstm_hip_fft_grid(const mstm_hip_ctx *c, double *cell_boundary, int *sphere_node, int *number_neighbor_nodes)
{
    if (!c || !c->fft) return MSTM_HIP_ESTATE;
    fft_grid(c->fft, cell_boundary, sphere_node, number_neighbor_nodes, nullptr);
    return 0;
}

int mstm_hip_setup_fft(mstm_hip_ctx *c, int prec)
{
    if (!c || !c->fft) return fail(c, MSTM_HIP_ESTATE, "setup_fft: call mstm_hip_node_selection first");
    HIPCHK(hipSetDevice(c->device));
    int rc = ensure_vcc(c, std::max(c->Lmax, fft_required_vcc(c->fft)));
    if (rc) return rc;
    FftGeometry g{c->nsph,          c->Lmax,    c->neqns,   c->pos.data(), c->radius.data(), c->order.data(),
                  c->offset.data(), c->rimed,   c->d_pos,   c->d_order,    c->d_offset,      c->d_an,
                  c->d_vcc,         c->vcc_LM};
    fft_bind(c->fft, g);
    rc = fft_setup(c->fft, prec, c->st);
    if (rc) return fail(c, rc, "setup_fft: %s", fft_last_error(c->fft));
    return 0;
}

}  // extern "C"

// --------------------------------------------------------------- operators
static hipEvent_t next_event(mstm_hip_ctx *c)
{
    if (c->ev_used >= c->ev.size()) {
        hipEvent_t e;
        hipEventCreate(&e);
        c->ev.push_back(e);
    }
    return c->ev[c->ev_used++];
}

// Device-side sphereinteraction on the direct operator: ain/aout are
// (neqns, nrhs) complex FP64 device arrays, nrhs <= 4; 3-4 columns run as
// one four-column tile launch.
// xin/part: the padded input and the partial sums (the context's, or the
// allocation-free entry point's scratch).
static int direct_matvec_buf(mstm_hip_ctx *c, int nrhs, const double *ain, double *aout, const int *flags, int prec,
                             void *xin, void *part, int G)
{
    DirectOp &d = c->dop[prec];
    if (nrhs < 1 || nrhs > 4) return fail(c, MSTM_HIP_EARG, "direct product: %d columns", nrhs);
    const int L = c->Lmax, nr = nrhs > 2 ? 4 : 2;
    // four-column products that run two workgroups per tile (step group):
    // fewer step groups keep the launch within the same 512 workgroups
    if (nr == 4 && tile_cols4(L, prec == MSTM_HIP_FP64 ? 8 : 4) == 2)
        while (G > 1 && (int64_t)c->ntiles * G * 2 > 512) G /= 2;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    if (c->timing) {
        e0 = next_event(c);
        e1 = next_event(c);
    }
    const int *gate = c->gate;
    if (prec == MSTM_HIP_FP64) {
        HIPCHK(launch_prep_quad<double>(ain, 2 * c->neqns, (double *)xin, nrhs, flags, c->nsph, c->npad, L, c->d_order,
                                   c->d_offset, c->d_an, 1, c->st, gate));
        if (e0) hipEventRecord(e0, c->st);
        HIPCHK(launch_direct_tiles<double>((const double *)d.tab, c->d_tiles, c->ntiles, L, (const double *)xin,
                                           (double *)part, c->npad, nr, G, 1, c->st, gate));
        if (e1) hipEventRecord(e1, c->st);
        HIPCHK(launch_reduce_quad<double>((const double *)part, c->nblocks * G, aout, 2 * c->neqns, nrhs, flags, c->nsph,
                                          c->npad, L, c->d_order, c->d_offset, c->d_an, 1, c->st, gate));
    } else {
        HIPCHK(launch_prep_quad<float>(ain, 2 * c->neqns, (float *)xin, nrhs, flags, c->nsph, c->npad, L, c->d_order,
                                  c->d_offset, c->d_an, 1, c->st, gate));
        if (e0) hipEventRecord(e0, c->st);
        HIPCHK(launch_direct_tiles<float>((const float *)d.tab, c->d_tiles, c->ntiles, L, (const float *)xin,
                                          (float *)part, c->npad, nr, G, 1, c->st, gate));
        if (e1) hipEventRecord(e1, c->st);
        HIPCHK(launch_reduce_quad<float>((const float *)part, c->nblocks * G, aout, 2 * c->neqns, nrhs, flags, c->nsph,
                                         c->npad, L, c->d_order, c->d_offset, c->d_an, 1, c->st, gate));
    }
    if (e0) c->ev_prec.push_back(prec + 2 * (nr == 4));
    c->stats.matvecs[prec]++;
    return 0;
}

static int direct_matvec(mstm_hip_ctx *c, int nrhs, const double *ain, double *aout, const int *flags, int prec)
{
    DirectOp &d = c->dop[prec];
    if (!d.ready) {
        int rc = mstm_hip_setup_direct(c, prec);
        if (rc) return rc;
    }
    return direct_matvec_buf(c, nrhs, ain, aout, flags, prec, d.xin, d.part, c->tgroups);
}

static int matvec(mstm_hip_ctx *c, int nrhs, const double *ain, double *aout, const int *flags, int prec, int use_fft)
{
    if (use_fft) {
        if (!c->fft) return fail(c, MSTM_HIP_ESTATE, "FFT operator not set up (call node_selection + setup_fft)");
        if (!fft_ready(c->fft, prec)) {  // first product at this precision: set up as mstm_hip_setup_fft does
            int rc = mstm_hip_setup_fft(c, prec);
            if (rc) return rc;
        }
        const size_t V = 2 * (size_t)c->neqns;
        for (int r0 = 0; r0 < nrhs; r0 += 2) {  // the node-grid operator takes two columns per call
            const int nr = std::min(2, nrhs - r0);
            int rc = fft_matvec(c->fft, nr, ain + V * r0, aout + V * r0, flags + r0, prec, c->st, c->gate);
            if (rc) return fail(c, rc, "fft matvec: %s", fft_last_error(c->fft));
            c->stats.matvecs[prec]++;
        }
        return 0;
    }
    return direct_matvec(c, nrhs, ain, aout, flags, prec);
}

// take the last product out of the counts (it was enqueued ahead and its
// gate was closed)
static void drop_product(mstm_hip_ctx *c, int prec, int use_fft)
{
    c->stats.matvecs[prec]--;
    if (use_fft) fft_drop_product(c->fft);
    else if (!c->ev_prec.empty() && c->ev_used >= 2) {
        c->ev_used -= 2;
        c->ev_prec.pop_back();
    }
}

static void collect_events(mstm_hip_ctx *c)
{
    hipStreamSynchronize(c->st);
    for (size_t q = 0; q + 1 < c->ev_used && q / 2 < c->ev_prec.size(); q += 2) {
        float ms = 0;
        hipEventElapsedTime(&ms, c->ev[q], c->ev[q + 1]);
        const int p = c->ev_prec[q / 2] & 1;
        if (c->ev_prec[q / 2] & 2) {
            c->stats.tile4_ms[p] += ms;
            c->stats.tile4_launches[p]++;
        } else {
            c->stats.tile_ms[p] += ms;
            c->stats.tile_launches[p]++;
        }
    }
    c->ev_used = 0;
    c->ev_prec.clear();
}

// Krylov partial sums: each kernel launch writes one complex value per
// block of its grid (krylov_grid()) into a region of d_partials; regions are
// fetched together and added on the host in a fixed order (deterministic).
static int fetch_partials(mstm_hip_ctx *c, int ncomplex)
{
    HIPCHK(hipMemcpyAsync(c->h_partials.data(), c->d_partials, sizeof(double) * 2 * ncomplex, hipMemcpyDeviceToHost,
                          c->st));
    HIPCHK(hipStreamSynchronize(c->st));
    return 0;
}
// sum of nvals interleaved values of the region starting at complex offset off
static void reduce_region(const mstm_hip_ctx *c, int off, int nvals, double *out)
{
    const int g = krylov_grid();
    for (int v = 0; v < nvals; v++) {
        double re = 0, im = 0;
        for (int b = 0; b < g; b++) {
            re += c->h_partials[2 * (off + nvals * b + v)];
            im += c->h_partials[2 * (off + nvals * b + v) + 1];
        }
        out[2 * v] = re;
        out[2 * v + 1] = im;
    }
}
static int sum_partials(mstm_hip_ctx *c, int nvals, double *out)
{
    int rc = fetch_partials(c, nvals * krylov_grid());
    if (rc) return rc;
    reduce_region(c, 0, nvals, out);
    return 0;
}
static inline double *pregion(mstm_hip_ctx *c, int s) { return c->d_partials + (size_t)4 * krylov_grid() * s; }
static inline int pregion_off(int s) { return 2 * krylov_grid() * s; }


// K iterations of a lazily read BiCG loop (small clusters, direct
// operator) as one replay of a HIP graph captured from step(): the launches
// of an iteration are identical every time (iteration numbers, scalars and
// the stop test live on the device; flags and pointers are fixed), so a
// graph captured once per pattern of active systems and set of buffers
// replaces 6 K launches by one.  Tile timing events are left out of the
// graph; the product count is kept.
template <typename F>
static int bicg_graph_steps(mstm_hip_ctx *c, int ns, int prec, const bool act[2], const double *x0, int K, F &&step)
{
    const DirectOp &d = c->dop[prec];
    const std::vector<intptr_t> key = {ns, prec, act[0], act[1], K, (intptr_t)x0, (intptr_t)c->d_kv, (intptr_t)c->kv_n,
                                       c->neqns, (intptr_t)d.tab, (intptr_t)d.xin, (intptr_t)d.part, c->tgroups,
                                       c->ntiles, c->nblocks, c->Lmax, c->nsph, c->npad, (intptr_t)c->d_tiles,
                                       (intptr_t)c->d_order, (intptr_t)c->d_offset, (intptr_t)c->d_an,
                                       (intptr_t)c->d_partials, (intptr_t)c->d_bscal, (intptr_t)c->gate};
    mstm_hip_ctx::BicgGraph &g = c->bgraph[act[0] && act[1] ? 0 : (act[0] ? 1 : 2)];
    if (!g.exec || g.key != key) {
        if (g.exec) (void)hipGraphExecDestroy(g.exec);
        g.exec = nullptr;
        g.key.clear();
        const bool timing = c->timing;
        c->timing = false;
        const long mv0 = c->stats.matvecs[prec];
        hipGraph_t gr = nullptr;
        int rc = 0;
        bool graph_ok = false;  // capture and instantiation both worked
        hipError_t e = hipStreamBeginCapture(c->st, hipStreamCaptureModeThreadLocal);
        if (e == hipSuccess) {
            for (int q = 0; q < K && !rc; q++) rc = step();
            const hipError_t e2 = hipStreamEndCapture(c->st, &gr);
            if (!rc && e2 == hipSuccess) {
                graph_ok = hipGraphInstantiate(&g.exec, gr, nullptr, nullptr, 0) == hipSuccess;
                if (!graph_ok) g.exec = nullptr;
            }
        }
        c->timing = timing;
        g.matvecs = (int)(c->stats.matvecs[prec] - mv0);
        c->stats.matvecs[prec] = mv0;
        if (gr) (void)hipGraphDestroy(gr);
        if (rc) return rc;  // a launch of the step itself failed
        if (!graph_ok) {
            // the stream could not be captured here (another capture, a tool
            // that intercepts graphs): this context issues the same launches
            // one by one from now on
            (void)hipGetLastError();
            c->graphs = false;
            for (int q = 0; q < K; q++)
                if ((rc = step())) return rc;
            return 0;
        }
        g.key = key;
    }
    HIPCHK(hipGraphLaunch(g.exec, c->st));
    c->stats.matvecs[prec] += g.matvecs;
    return 0;
}

// cbicg (mstm-solver-8.f90:654-949) for ns = 1 or 2 independent systems
// A x_s = b_s at once (the two polarizations of fixedorsoln).  b and x are
// blocks of ns contiguous vectors; every system keeps the reference's own
// recurrences and scalars, so each one runs exactly the iterations it would
// run alone, while both share every table stream of the product (one
// four-column launch while both are active).  it[s]: iterations as the
// Fortran do-variable (niter+1 if the loop ran out); err[s]: last |r|^2/|b|^2.
static int bicg2_dev(mstm_hip_ctx *c, int ns, int niter, const double *eps, const double *b, double *x, int prec,
                     int use_fft, int *it, double *err)
{
    const int n = c->neqns;
    const size_t V = 2 * c->kv_n;
    double *kv = c->d_kv;
    double *P[2], *W[2], *AP[2], *AW[2], *Rr[2], *Q[2];
    const double *B[2];
    double *X[2];
    BicgScal *S = c->d_bscal, *hS = c->h_bscal;
    const int64_t region = 2 * (int64_t)krylov_grid();  // complex values per partial region
    for (int s = 0; s < ns; s++) {
        P[s] = kv + V * (KV_PW + 2 * s);
        W[s] = P[s] + V;
        AP[s] = kv + V * (KV_CAPS + 2 * s);
        AW[s] = AP[s] + V;
        Rr[s] = kv + V * (KV_RB + s);
        Q[s] = kv + V * (KV_QB + s);
        B[s] = b + V * s;
        X[s] = x + V * s;
        it[s] = 0;
        err[s] = 0.0;
        hS[s] = BicgScal{};
        hS[s].eps = eps[s];
    }
    // the scalars live on the device; the host reads them every K iterations
    auto sync_state = [&]() -> int {
        HIPCHK(hipMemcpyAsync(hS, S, sizeof(BicgScal) * ns, hipMemcpyDeviceToHost, c->st));
        HIPCHK(hipStreamSynchronize(c->st));
        return 0;
    };
    // host reads of the scalars every K iterations: a stopped system's
    // kernels return at once on the device, so the iterates and counts are
    // the same for any K.  Products of small clusters cost less than the
    // read: there the loop does not wait for the start-up state either, and
    // its products carry the device gate (1 while a system is active), so
    // the up to K - 1 products enqueued after the last system stops return at
    // once.
    const bool lazy = !use_fft && c->nsph <= 500;
    const int K = lazy ? 4 : 1;
    int *gate = lazy ? c->d_gate : nullptr;
    struct GateScope {  // products outside this loop are never gated
        mstm_hip_ctx *c;
        ~GateScope() { c->gate = nullptr; }
    } gate_scope{c};
    c->gate = gate;
    HIPCHK(hipMemcpyAsync(S, hS, sizeof(BicgScal) * ns, hipMemcpyHostToDevice, c->st));
    // |b|^2
    HIPCHK(launch_bicg_norm(B[0], (int64_t)V, n, c->d_partials, region, ns, c->st));
    HIPCHK(launch_bicg_scal(0, c->d_partials, region, S, ns, n, c->st, gate));
    int rc = 0;
    bool act[2] = {true, ns == 2};
    if (!lazy) {
        rc = sync_state();
        if (rc) return rc;
        act[0] = hS[0].active != 0;
        act[1] = ns == 2 && hS[1].active != 0;
        if (!act[0] && !act[1]) return 0;
    }
    // r = b - A x (:827-834), one product for the active systems' x (lazy:
    // both, a system with b = 0 having been stopped on the device)
    {
        int f[2] = {2, 2};
        if (act[0] && act[1]) rc = matvec(c, 2, X[0], Rr[0], f, prec, use_fft);
        else
            for (int s = 0; s < ns && !rc; s++)
                if (act[s]) rc = matvec(c, 1, X[s], Rr[s], f, prec, use_fft);
        if (rc) return rc;
    }
    {
        const int s0 = act[0] ? 0 : 1, nact = act[0] && act[1] ? 2 : 1;
        HIPCHK(launch_bicg_init(Rr[s0], Q[s0], W[s0], P[s0], B[s0], X[s0], (int64_t)V, 2 * (int64_t)V, n,
                                pregion(c, s0), region, nact, c->st));
    }
    HIPCHK(launch_bicg_scal(1, c->d_partials, region, S, ns, n, c->st, gate));
    if (!lazy) {
        rc = sync_state();
        if (rc) return rc;
        act[0] = hS[0].active != 0;
        act[1] = ns == 2 && hS[1].active != 0;
    }
    // one iteration (:836-948) of the active systems: the product of p and
    // w, then both systems' vector steps in one launch each (the kernels of
    // a system the device has stopped return at once)
    auto step = [&]() -> int {
        int f4[4] = {2, 3, 2, 3};
        int rc_;
        if (act[0] && act[1]) rc_ = matvec(c, 4, P[0], AP[0], f4, prec, use_fft);
        else rc_ = matvec(c, 2, act[0] ? P[0] : P[1], act[0] ? AP[0] : AP[1], f4, prec, use_fft);
        if (rc_) return rc_;
        double *den = pregion(c, 2);  // partial sums of step a, those of step b in regions 0 and 1
        HIPCHK(launch_bicg_a_dev(AP[0], AW[0], P[0], W[0], 2 * (int64_t)V, n, den, region, S, ns, c->st));
        HIPCHK(launch_bicg_b_dev(X[0], Rr[0], Q[0], P[0], AP[0], AW[0], (int64_t)V, 2 * (int64_t)V, S, S + 2, n, den,
                                 pregion(c, 0), region, ns, c->st));
        HIPCHK(launch_bicg_c_dev(P[0], W[0], Rr[0], Q[0], (int64_t)V, 2 * (int64_t)V, S + 2, S, n, pregion(c, 0), region,
                                 ns, c->st, gate));
        return 0;
    };
    int iter = 1, synced = 0;
    while (iter <= niter) {
        if (!act[0] && !act[1]) break;
        const int nst = std::min(K, niter - iter + 1);
        if (lazy && nst == K && c->graphs) rc = bicg_graph_steps(c, ns, prec, act, X[0], K, step);
        else
            for (int q = 0; q < nst && !rc; q++) rc = step();
        if (rc) return rc;
        iter += nst;
        const int last = iter - 1;
        rc = sync_state();
        if (rc) return rc;
        for (int s = 0; s < ns; s++) {
            if (!act[s]) continue;
            // steps since the last read; a step that failed the breakdown test
            // does not count, as in the host loop
            const int done = hS[s].active ? last - synced : hS[s].it - synced - hS[s].brk;
            if (prec == MSTM_HIP_FP64) c->stats.iters_fp64 += done;
            else c->stats.iters_fp32 += done;
            act[s] = hS[s].active != 0;
        }
        synced = last;
    }
    if (lazy && niter < 1) {  // no iteration ran: the start-up state decides
        rc = sync_state();
        if (rc) return rc;
        for (int s = 0; s < ns; s++) act[s] = hS[s].active != 0;
    }
    for (int s = 0; s < ns; s++) {
        it[s] = act[s] ? iter : hS[s].it;  // ran out: niter + 1
        err[s] = hS[s].err;
    }
    return 0;
}

// ---------------------------------------------------------------------------
// cbicg for a block of np column pairs (2 np systems, FP64, direct operator):
// the T-matrix's columns of one degree share their operator, and a pair alone
// leaves most of the chip idle on a small cluster (200 spheres of order 4: 67 us
// per iteration, 31 of them the tiles; in blocks of up to 33 pairs 23 us per pair
// and iteration, 19 of them the tiles, which then run at the rate of a full
// chip: 335 -> 94 ms for the T-matrix of order 16).  Every system keeps its own recurrences, scalars, stop and count;
// the kernels of a step take all systems, and a pair whose two systems have
// stopped closes its gate.
// ---------------------------------------------------------------------------
struct BicgBlock {
    int np = 0, G = 1;  // pairs, workgroups per tile of the product
    double *x, *b, *pw, *cap, *r, *q, *partials, *den, *xin, *part;
    BicgScal *sc;
    int *gate;
};

// the parts of a work space at base (null: sizes only); returns its bytes
static size_t bicg_block_layout(const mstm_hip_ctx *c, unsigned char *base, BicgBlock &k)
{
    size_t o = 0;
    const size_t V = sizeof(double) * 2 * c->kv_n, np = (size_t)k.np;
    const size_t col = sizeof(double) * 2 * 4 * 2 * (size_t)c->npad * c->Lmax * (c->Lmax + 2);  // four product columns
    auto put = [&](auto *&p, size_t bytes) {
        p = reinterpret_cast<std::remove_reference_t<decltype(p)>>(base + o);
        o += (bytes + 255) / 256 * 256;
    };
    put(k.x, 2 * V * np);
    put(k.b, 2 * V * np);
    put(k.pw, 4 * V * np);
    put(k.cap, 4 * V * np);
    put(k.r, 2 * V * np);
    put(k.q, 2 * V * np);
    put(k.partials, sizeof(double) * 4 * (size_t)krylov_grid() * 2 * np);
    put(k.den, sizeof(double) * 4 * (size_t)krylov_grid() * 2 * np);
    put(k.xin, col * np);
    put(k.part, col * np * c->nblocks * k.G);
    put(k.sc, sizeof(BicgScal) * 4 * np);
    put(k.gate, sizeof(int) * np);
    return o;
}

// the block for np of the columns of one degree: as many pairs as the work
// space may hold, split evenly, and workgroups per tile while the tiles of all
// pairs are fewer than 2048.  Work space of 96 / 256 / 512 / 1024 MB, T-matrix:
// 200 spheres 114 / 97 / 94 / 94 ms, 500 spheres 510 / 337 / 302 / 292 ms, 900
// spheres 1492 (pairs alone) / 1492 / 1306 / 1291 ms.
static BicgBlock bicg_block_plan(const mstm_hip_ctx *c, int np)
{
    const size_t limit = (size_t)BICG_BLOCK_BYTES;
    BicgBlock k;
    k.np = np;
    while (k.np > 1 && bicg_block_layout(c, nullptr, k) > limit) {
        const int parts = (np + k.np - 1) / k.np + 1;
        k.np = std::min(k.np - 1, (np + parts - 1) / parts);
    }
    k.G = c->tgroups;
    while (k.G > 1 && ((int64_t)c->ntiles * k.G * k.np > 2048 || bicg_block_layout(c, nullptr, k) > limit)) k.G /= 2;
    return k;
}

// b in k.b; x in k.x = b at the start, the solutions at the end; hS: 2 np scalars
static int bicg_block(mstm_hip_ctx *c, const BicgBlock &k, int niter, double eps, BicgScal *hS, int *it, double *err)
{
    const int n = c->neqns, np = k.np, ns = 2 * np, L = c->Lmax, K = 4;
    const int64_t V = 2 * (int64_t)c->kv_n, region = 2 * (int64_t)krylov_grid();
    const DirectOp &d = c->dop[MSTM_HIP_FP64];
    // tile times as bicg2_dev has them: not for small clusters (200 spheres: the
    // events cost 1.2 of 97 ms)
    const bool timed = c->timing && c->nsph > 500;
    auto product = [&](int ncol, const double *in, double *out, const int *f, const int *gate) -> int {
        HIPCHK(launch_prep_quad<double>(in, (int)V, k.xin, ncol, f, c->nsph, c->npad, L, c->d_order, c->d_offset,
                                        c->d_an, np, c->st, gate));
        hipEvent_t e0 = nullptr, e1 = nullptr;
        if (timed) {
            e0 = next_event(c);
            e1 = next_event(c);
            hipEventRecord(e0, c->st);
        }
        HIPCHK(launch_direct_tiles<double>((const double *)d.tab, c->d_tiles, c->ntiles, L, k.xin, k.part, c->npad,
                                           ncol, k.G, np, c->st, gate));
        if (e1) {
            hipEventRecord(e1, c->st);
            c->ev_prec.push_back(MSTM_HIP_FP64 + 2 * (ncol == 4));
        }
        HIPCHK(launch_reduce_quad<double>(k.part, c->nblocks * k.G, out, (int)V, ncol, f, c->nsph, c->npad, L,
                                          c->d_order, c->d_offset, c->d_an, np, c->st, gate));
        return 0;
    };
    for (int s = 0; s < ns; s++) {
        hS[s] = BicgScal{};
        hS[s].eps = eps;
    }
    HIPCHK(hipMemcpyAsync(k.sc, hS, sizeof(BicgScal) * ns, hipMemcpyHostToDevice, c->st));
    HIPCHK(launch_bicg_norm(k.b, V, n, k.partials, region, ns, c->st));
    HIPCHK(launch_bicg_scal(0, k.partials, region, k.sc, ns, n, c->st, k.gate));
    const int f2[2] = {2, 2}, f4[4] = {2, 3, 2, 3};
    if (int rc = product(2, k.x, k.r, f2, k.gate)) return rc;
    HIPCHK(launch_bicg_init(k.r, k.q, k.pw + V, k.pw, k.b, k.x, V, 2 * V, n, k.partials, region, ns, c->st));
    HIPCHK(launch_bicg_scal(1, k.partials, region, k.sc, ns, n, c->st, k.gate));
    bool any = true;
    for (int iter = 0; iter < niter && any;) {
        const int nst = std::min(K, niter - iter);
        for (int q = 0; q < nst; q++) {
            if (int rc = product(4, k.pw, k.cap, f4, k.gate)) return rc;
            HIPCHK(launch_bicg_a_dev(k.cap, k.cap + V, k.pw, k.pw + V, 2 * V, n, k.den, region, k.sc, ns, c->st));
            HIPCHK(launch_bicg_b_dev(k.x, k.r, k.q, k.pw, k.cap, k.cap + V, V, 2 * V, k.sc, k.sc + ns, n, k.den,
                                     k.partials, region, ns, c->st));
            HIPCHK(launch_bicg_c_dev(k.pw, k.pw + V, k.r, k.q, V, 2 * V, k.sc + ns, k.sc, n, k.partials, region, ns,
                                     c->st, k.gate));
        }
        iter += nst;
        HIPCHK(hipMemcpyAsync(hS, k.sc, sizeof(BicgScal) * ns, hipMemcpyDeviceToHost, c->st));
        HIPCHK(hipStreamSynchronize(c->st));
        any = false;
        for (int s = 0; s < ns; s++) any |= hS[s].active != 0;
    }
    for (int s = 0; s < ns; s++) {
        it[s] = hS[s].active ? niter + 1 : hS[s].it;  // ran out: niter + 1
        err[s] = hS[s].err;
        c->stats.iters_fp64 += hS[s].active ? niter : hS[s].it - hS[s].brk;
    }
    for (int s = 0; s < ns; s += 2)  // a pair's products: the start, and one per iteration of either system
        if (hS[s].enorm != 0.0 || hS[s + 1].enorm != 0.0)
            c->stats.matvecs[MSTM_HIP_FP64] += 1 + std::max(hS[s].cur, hS[s + 1].cur);
    return 0;
}

// Order-of-scattering solution, cbicg with niter < 0 (mstm-solver-8.f90:
// 785-825), for ns = 1 or 2 systems at once: starting from x_s, the series
//   c_1 = T H x_s,  c_{k+1} = T H c_k,  x_s += c_k
// stops when |c_k|^2/|b_s|^2 < eps[s] (err[s] = that ratio, it[s] = k) or
// after nord terms (it[s] = nord + 1 and err[s] = 0, as the Fortran loop
// leaves them).  Each term of the active systems is one FP64 product.
static int oos2_dev(mstm_hip_ctx *c, int ns, int nord, const double *eps, const double *b, double *x, int use_fft,
                    int *it, double *err)
{
    const int n = c->neqns;
    const size_t V = 2 * c->kv_n;
    double *buf[2] = {c->d_kv + V * KV_PW, c->d_kv + V * KV_CAPS};  // two blocks of ns terms, alternating
    double enorm[2] = {0, 0};
    bool act[2] = {false, false};
    for (int s = 0; s < ns; s++) {
        it[s] = 0;
        err[s] = 0.0;
        HIPCHK(launch_zdot(b + V * s, b + V * s, n, 1, pregion(c, s), nullptr, c->st));
    }
    int rc = fetch_partials(c, 2 * krylov_grid() * ns);
    if (rc) return rc;
    for (int s = 0; s < ns; s++) {
        double v[2];
        reduce_region(c, pregion_off(s), 1, v);
        enorm[s] = v[0];
        act[s] = v[0] != 0.0;  // cbicg returns at once for pnp = 0
    }
    HIPCHK(hipMemcpyAsync(buf[0], x, sizeof(double) * V * ns, hipMemcpyDeviceToDevice, c->st));
    int f2[2] = {2, 2};
    int cur = 0, k;
    for (k = 1; k <= nord; k++) {
        if (!act[0] && !(ns == 2 && act[1])) break;
        double *in = buf[cur], *out = buf[cur ^ 1];
        if (ns == 2 && act[0] && act[1]) rc = matvec(c, 2, in, out, f2, MSTM_HIP_FP64, use_fft);
        else
            for (int s = 0; s < ns && !rc; s++)
                if (act[s]) rc = matvec(c, 1, in + V * s, out + V * s, f2, MSTM_HIP_FP64, use_fft);
        if (rc) return rc;
        for (int s = 0; s < ns; s++) {
            if (!act[s]) continue;
            HIPCHK(launch_zaxpby(1.0, 0.0, out + V * s, 1.0, 0.0, x + V * s, n, c->st));
            HIPCHK(launch_zdot(out + V * s, out + V * s, n, 1, pregion(c, s), nullptr, c->st));
        }
        rc = fetch_partials(c, 2 * krylov_grid() * ns);
        if (rc) return rc;
        for (int s = 0; s < ns; s++) {
            if (!act[s]) continue;
            double v[2];
            reduce_region(c, pregion_off(s), 1, v);
            c->stats.iters_fp64++;
            if (v[0] / enorm[s] < eps[s]) {
                err[s] = v[0] / enorm[s];
                it[s] = k;
                act[s] = false;
            }
        }
        cur ^= 1;
    }
    for (int s = 0; s < ns; s++)
        if (act[s]) it[s] = k;  // ran out: nord + 1
    return 0;
}

// GMRES(m) (Saad & Schultz, SIAM J. Sci. Stat. Comput. 7, 856 (1986)) for
// ns = 1 or 2 systems A d_s = b_s at once, from d_s = 0.  Arnoldi vectors
// are FP64 and orthogonalised by classical Gram-Schmidt applied twice; the
// products run at precision prec, one column per system (both systems in one
// launch) -- half the columns of a BiCG step.  A system stops when its residual
// estimate |g_{j+1}|^2/|b|^2 < eps[s], or for good at a step or a residual that
// is not finite, with the correction of the steps before and err[s] >= eps[s];
// it restarts every m steps from the residual b - A d.  it[s]: Arnoldi steps.
// Projections, rotations and the stop test stay on the device (launch_gm_step);
// the host enqueues one step ahead of the state it has read, and a step of
// systems that have all stopped returns at once (gate).
static int scaled_copy(mstm_hip_ctx *c, double *dst, const double *src, double sr, double si);
static int gmres2_dev(mstm_hip_ctx *c, int ns, int niter, const double *eps, const double *b, double *x, int prec,
                      int use_fft, int *it, double *err)
{
    const int n = c->neqns;
    const size_t V = 2 * c->kv_n;
    const size_t need = sizeof(double) * V * 2 * (GM_M + 1), npart = sizeof(double) * 2 * gm_partials(n);
    if (c->gm_bytes < need) {
        dfree(c->d_gm);
        c->gm_bytes = 0;
        HIPCHK(dalloc(&c->d_gm, need));
        c->gm_bytes = need;
    }
    if (c->gp_bytes < npart) {
        dfree(c->d_gp);
        c->gp_bytes = 0;
        HIPCHK(dalloc(&c->d_gp, npart));
        c->gp_bytes = npart;
    }
    if (!c->d_gsys) HIPCHK(dalloc(&c->d_gsys, sizeof(GmSys) * 2));
    if (!c->h_gstat) HIPCHK(hipHostMalloc((void **)&c->h_gstat, sizeof(GmStat) * 4, hipHostMallocDefault));
    for (auto &e : c->gm_ev)
        if (!e) HIPCHK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    auto basis = [&](int j, int sys) { return c->d_gm + V * (2 * (size_t)j + sys); };
    double *W = c->d_kv + V * KV_CAPS;  // products
    double *T = c->d_kv + V * KV_ST;    // temporaries t_s at T + s V
    double bb[2] = {0, 0};
    bool open[2] = {false, false};
    for (int q = 0; q < ns; q++) {
        it[q] = 0;
        err[q] = 0.0;
        HIPCHK(hipMemsetAsync(x + V * q, 0, sizeof(double) * V, c->st));
        HIPCHK(launch_zdot(b + V * q, b + V * q, n, 1, pregion(c, q), nullptr, c->st));
    }
    int rc = fetch_partials(c, 2 * krylov_grid() * ns);
    if (rc) return rc;
    for (int q = 0; q < ns; q++) {
        double v[2];
        reduce_region(c, pregion_off(q), 1, v);
        bb[q] = v[0];
        open[q] = gm_opens(bb[q], bb[q], 0.0, 0, 1);
        err[q] = bb[q] == 0.0 ? 0.0 : 1.0;
    }
    int f2[2] = {2, 2};
    for (int cycle = 0; open[0] || (ns == 2 && open[1]); cycle++) {
        double beta[2] = {0, 0};
        if (cycle == 0) {
            for (int q = 0; q < ns; q++)
                if (open[q]) {
                    beta[q] = std::sqrt(bb[q]);
                    HIPCHK(hipMemcpyAsync(basis(0, q), b + V * q, sizeof(double) * V, hipMemcpyDeviceToDevice, c->st));
                }
        } else {
            // r = b - A x = b - x + T H x
            if (ns == 2 && open[0] && open[1]) rc = matvec(c, 2, x, W, f2, prec, use_fft);
            else
                for (int q = 0; q < ns && !rc; q++)
                    if (open[q]) rc = matvec(c, 1, x + V * q, W + V * q, f2, prec, use_fft);
            if (rc) return rc;
            for (int q = 0; q < ns; q++) {
                if (!open[q]) continue;
                double *t = T + V * q;
                HIPCHK(hipMemcpyAsync(t, b + V * q, sizeof(double) * V, hipMemcpyDeviceToDevice, c->st));
                HIPCHK(launch_zaxpby(-1.0, 0.0, x + V * q, 1.0, 0.0, t, n, c->st));
                HIPCHK(launch_zaxpby(1.0, 0.0, W + V * q, 1.0, 0.0, t, n, c->st));
                HIPCHK(launch_zdot(t, t, n, 1, pregion(c, q), nullptr, c->st));
            }
            rc = fetch_partials(c, 2 * krylov_grid() * ns);
            if (rc) return rc;
            for (int q = 0; q < ns; q++) {
                if (!open[q]) continue;
                double v[2];
                reduce_region(c, pregion_off(q), 1, v);
                if (gm_finite(v[0])) err[q] = v[0] / bb[q];
                if (!gm_opens(v[0], bb[q], eps[q], it[q], niter)) {
                    open[q] = false;
                    continue;
                }
                beta[q] = std::sqrt(v[0]);
                HIPCHK(hipMemcpyAsync(basis(0, q), T + V * q, sizeof(double) * V, hipMemcpyDeviceToDevice, c->st));
            }
            if (!open[0] && !(ns == 2 && open[1])) break;
        }
        // the systems of this cycle: both, or the one that is open
        const int q0 = open[0] ? 0 : 1, nq = (open[0] ? 1 : 0) + (ns == 2 && open[1] ? 1 : 0);
        GmStart st[2];
        for (int q = 0; q < nq; q++) st[q] = {bb[q0 + q], eps[q0 + q], beta[q0 + q], it[q0 + q], niter, GM_M};
        HIPCHK(launch_gm_begin(c->d_gsys, nq, st, basis(0, q0), (int64_t)V, n, c->d_gate, c->st));
        struct GateScope {  // products outside this loop are never gated
            mstm_hip_ctx *c;
            ~GateScope() { c->gate = nullptr; }
        } gate_scope{c};
        c->gate = c->d_gate;
        // enqueue step j, then read the state after step j - 1
        auto stat = [&](int j) { return c->h_gstat + 2 * (j & 1); };
        auto enqueue = [&](int j) -> int {
            int r = matvec(c, nq, basis(j, q0), W, f2, prec, use_fft);
            if (r) return r;
            HIPCHK(launch_gm_step(c->d_gsys, nq, basis(0, q0), (int64_t)(2 * V), (int64_t)V, j + 1, W, (int64_t)V, n,
                                  c->d_gp, c->d_gate, stat(j), c->st));
            HIPCHK(hipEventRecord(c->gm_ev[j & 1], c->st));
            return 0;
        };
        rc = enqueue(0);
        if (rc) return rc;
        int last = 0;  // steps enqueued - 1
        for (int j = 0;; j++) {
            if (j + 1 < GM_M) {
                rc = enqueue(j + 1);
                if (rc) return rc;
                last = j + 1;
            }
            HIPCHK(hipEventSynchronize(c->gm_ev[j & 1]));
            bool any = false;
            for (int q = 0; q < nq; q++) any = any || stat(j)[q].active;
            if (!any) {
                if (last > j) drop_product(c, prec, use_fft);  // the step enqueued ahead did nothing
                for (int q = 0; q < nq; q++) {
                    const GmStat *s = stat(j) + q;
                    it[q0 + q] += s->k;
                    err[q0 + q] = s->err;
                    if (s->done) open[q0 + q] = false;
                    if (prec == MSTM_HIP_FP64) c->stats.iters_fp64 += s->k;
                    else c->stats.iters_fp32 += s->k;
                }
                break;
            }
        }
        HIPCHK(launch_gm_update(c->d_gsys, nq, basis(0, q0), (int64_t)(2 * V), (int64_t)V, x + V * q0, (int64_t)V, n,
                                c->st));
    }
    return 0;
}

// Mixed precision for ns = 1 or 2 systems: x_s <- x_s + d_s with A d_s = r_s
// solved by FP32 BiCG, r_s = b_s - A x_s evaluated with the FP64 operator;
// a system stops on the reference criterion |r|^2/|b|^2 < eps measured in
// FP64.  r_in (optional): the residual block of the starting x.  When
// r_in_exact is false it came from an FP32 product: it only steers the first
// inner solve, and a system it shows below eps gets no inner solve but one
// more pass whose FP64 residual decides.  iters[s] counts inner FP32
// iterations.
static int refine2_dev(mstm_hip_ctx *c, int ns, int niter, double eps, const double *b, double *x, int use_fft,
                       int *iters, double *errmax, const double *r_in = nullptr, bool r_in_exact = true)
{
    const int n = c->neqns;
    const size_t V = 2 * c->kv_n;
    double *Y = c->d_kv + V * KV_Y, *R = c->d_kv + V * KV_R, *D = c->d_kv + V * KV_D;
    double bb[2] = {0, 0};
    bool open[2] = {false, false};
    for (int s = 0; s < ns; s++) HIPCHK(launch_zdot(b + V * s, b + V * s, n, 1, pregion(c, s), nullptr, c->st));
    int rc = fetch_partials(c, 2 * krylov_grid() * ns);
    if (rc) return rc;
    for (int s = 0; s < ns; s++) {
        double v[2];
        reduce_region(c, pregion_off(s), 1, v);
        bb[s] = v[0];
        open[s] = bb[s] != 0.0;
        iters[s] = 0;
        errmax[s] = 0.0;
    }
    int f2[2] = {2, 2};
    // a system closes on an FP64 residual only: below eps, after max_ref
    // inner solves, or with its iteration budget spent.  An inexact starting
    // residual never closes one (pass 0 then only decides on an inner solve).
    const bool inexact = r_in && !r_in_exact;
    int nsolve[2] = {0, 0};
    for (int ref = 0;; ref++) {
        if (!open[0] && !(ns == 2 && open[1])) break;
        if (ref == 0 && r_in) {
            for (int s = 0; s < ns; s++)
                if (open[s] && r_in + V * s != R + V * s)
                    HIPCHK(hipMemcpyAsync(R + V * s, r_in + V * s, sizeof(double) * V, hipMemcpyDeviceToDevice, c->st));
        } else {
            if (ns == 2 && open[0] && open[1]) rc = matvec(c, 2, x, Y, f2, MSTM_HIP_FP64, use_fft);  // y = T H x
            else
                for (int s = 0; s < ns && !rc; s++)
                    if (open[s]) rc = matvec(c, 1, x + V * s, Y + V * s, f2, MSTM_HIP_FP64, use_fft);
            if (rc) return rc;
            for (int s = 0; s < ns; s++) {
                if (!open[s]) continue;  // r = b - x + y
                HIPCHK(hipMemcpyAsync(R + V * s, b + V * s, sizeof(double) * V, hipMemcpyDeviceToDevice, c->st));
                HIPCHK(launch_zaxpby(-1.0, 0.0, x + V * s, 1.0, 0.0, R + V * s, n, c->st));
                HIPCHK(launch_zaxpby(1.0, 0.0, Y + V * s, 1.0, 0.0, R + V * s, n, c->st));
            }
        }
        for (int s = 0; s < ns; s++)
            if (open[s]) HIPCHK(launch_zdot(R + V * s, R + V * s, n, 1, pregion(c, s), nullptr, c->st));
        rc = fetch_partials(c, 2 * krylov_grid() * ns);
        if (rc) return rc;
        double rr[2] = {0, 0}, eps_in[2] = {1, 1};
        int nin = 0, sidx[2];
        for (int s = 0; s < ns; s++) {
            if (!open[s]) continue;
            double v[2];
            reduce_region(c, pregion_off(s), 1, v);
            rr[s] = v[0];
            errmax[s] = rr[s] / bb[s];
            const bool done = errmax[s] < eps || nsolve[s] >= c->max_ref || iters[s] >= niter;
            if (done && ref == 0 && inexact) continue;  // no inner solve; the FP64 residual of pass 1 decides
            if (done) {
                open[s] = false;
                continue;
            }
            nsolve[s]++;
            // inner FP32 solve of A d = r from d = r, to half the outer
            // target: the FP32 operator's relative error (~2e-7) is far below
            // the 1e-3 relative residual asked for, so one refinement step
            // normally ends.  (0.9 of the target saves two GMRES steps at 5000
            // spheres but doubles the Q_ext error against FP64, to 8.7e-6.)
            eps_in[nin] = std::max(0.5 * eps * bb[s] / rr[s], 1e-12);
            sidx[nin++] = s;
            HIPCHK(hipMemcpyAsync(D + V * s, R + V * s, sizeof(double) * V, hipMemcpyDeviceToDevice, c->st));
        }
        if (!nin) continue;
        c->stats.refinements++;
        int it_in[2] = {0, 0};
        double e_in[2] = {0, 0};
        const int budget = std::max(1, niter - std::max(iters[sidx[0]], nin > 1 ? iters[sidx[1]] : 0));
        if (c->inner == 1)
            rc = gmres2_dev(c, nin, budget, eps_in, R + V * sidx[0], D + V * sidx[0], MSTM_HIP_FP32, use_fft, it_in,
                            e_in);
        else
            rc = bicg2_dev(c, nin, budget, eps_in, R + V * sidx[0], D + V * sidx[0], MSTM_HIP_FP32, use_fft, it_in,
                           e_in);
        if (rc) return rc;
        for (int q = 0; q < nin; q++) {
            const int s = sidx[q];
            iters[s] += std::min(it_in[q], std::max(0, niter - iters[s]));
            HIPCHK(launch_zaxpby(1.0, 0.0, D + V * s, 1.0, 0.0, x + V * s, n, c->st));
        }
    }
    return 0;
}

// features + network forward for the current spheres (learned.hpp model)
static int lig_predict(mstm_hip_ctx *c)
{
    LearnedNet &g = c->lig;
    const int n = c->nsph;
    if (g.cap < n) {
        release_lig_buffers(c);
        HIPCHK(dalloc(&g.feat, sizeof(float) * (size_t)n * LIG_NFEAT));
        HIPCHK(dalloc(&g.depth, sizeof(float) * (size_t)n));
        HIPCHK(dalloc(&g.out, sizeof(float) * (size_t)n * g.s.nout));
        g.H.assign(g.s.nlayers, nullptr);
        for (auto &q : g.H) HIPCHK(dalloc(&q, sizeof(float) * (size_t)n * g.s.hidden));
        g.cap = n;
    }
    HIPCHK(launch_lig_features(n, c->d_pos, c->d_radius, c->d_mre, c->d_mim, c->rimed, g.feat, g.depth, c->st));
    HIPCHK(mlp_forward(g.s, g.params, g.feat, n, g.H.data(), nullptr, g.out, c->st));
    return 0;
}

// Starting vectors of the learned solver for both polarizations: the
// network's prediction xl_p is checked against the zero start (residual b,
// |r|^2/|b|^2 = 1) with one two-column FP32 product; the better one goes to
// x_p and its residual to r_p.  That residual is an FP32 product: the
// refinement uses it to steer its first inner solve and accepts an answer
// only on an FP64 residual.  used[p]: prediction kept.
static int lig_start2(mstm_hip_ctx *c, const double *b, double *x, double *r, int use_fft, bool *used)
{
    const int n = c->neqns;
    const size_t V = 2 * c->kv_n;
    double *in = c->d_kv + V * KV_PW, *y = c->d_kv + V * KV_CAPS;  // [xl_0, xl_1] -> products
    for (int p = 0; p < 2; p++)
        HIPCHK(launch_lig_combine(c->nsph, p, c->d_order, c->d_offset, c->d_pos, c->rimed, c->lig.out, c->lig.Lnet,
                                  c->lig.depth, c->lig.params + c->lig.np - 2, b + V * p, in + V * p, c->st));
    int f2[2] = {2, 2};
    int rc = matvec(c, 2, in, y, f2, MSTM_HIP_FP32, use_fft);
    if (rc) return rc;
    for (int p = 0; p < 2; p++) {
        double *rp = r + V * p;
        HIPCHK(hipMemcpyAsync(rp, b + V * p, sizeof(double) * V, hipMemcpyDeviceToDevice, c->st));
        HIPCHK(launch_zaxpby(-1.0, 0.0, in + V * p, 1.0, 0.0, rp, n, c->st));
        HIPCHK(launch_zaxpby(1.0, 0.0, y + V * p, 1.0, 0.0, rp, n, c->st));
        HIPCHK(launch_zdot(rp, rp, n, 1, c->d_partials + (size_t)2 * krylov_grid() * p, nullptr, c->st));
        HIPCHK(launch_zdot(b + V * p, b + V * p, n, 1, c->d_partials + (size_t)2 * krylov_grid() * (2 + p), nullptr,
                           c->st));
    }
    rc = fetch_partials(c, 4 * krylov_grid());
    if (rc) return rc;
    for (int p = 0; p < 2; p++) {
        double el[2], eb[2];
        reduce_region(c, krylov_grid() * p, 1, el);
        reduce_region(c, krylov_grid() * (2 + p), 1, eb);
        const double bn = eb[0] > 0.0 ? eb[0] : 1.0;
        c->stats.lig_err0 = el[0] / bn;  // the second polarization's values remain, as maxerr does
        c->stats.lig_errb = 1.0;         // the zero start
        used[p] = el[0] < eb[0];
        if (used[p]) {
            HIPCHK(hipMemcpyAsync(x + V * p, in + V * p, sizeof(double) * V, hipMemcpyDeviceToDevice, c->st));
        } else {
            HIPCHK(hipMemsetAsync(x + V * p, 0, sizeof(double) * V, c->st));
            HIPCHK(hipMemcpyAsync(r + V * p, b + V * p, sizeof(double) * V, hipMemcpyDeviceToDevice, c->st));
        }
    }
    return 0;
}

// dst = s * src (dst cleared first: the update kernel reads it)
static int scaled_copy(mstm_hip_ctx *c, double *dst, const double *src, double sr, double si)
{
    HIPCHK(hipMemsetAsync(dst, 0, sizeof(double) * 2 * c->neqns, c->st));
    HIPCHK(launch_zaxpby(sr, si, src, 0.0, 0.0, dst, c->neqns, c->st));
    return 0;
}

static int zdot_host(mstm_hip_ctx *c, const double *a, const double *b, std::complex<double> &out)
{
    double v[2];
    HIPCHK(launch_zdot(a, b, c->neqns, 1, c->d_partials, nullptr, c->st));
    int rc = sum_partials(c, 1, v);
    out = std::complex<double>(v[0], v[1]);
    return rc;
}


// Flexible GMRES(m) (Saad, SIAM J. Sci. Comput. 14, 461 (1993)) in FP64 on
// A = I - T H from x = 0, right-preconditioned with a different map for every
// Arnoldi vector v_j: for the first vector of the first cycle (v_1 = b/|b|, a
// plane-wave right-hand side) the learned network's prediction when lig is
// set; for every other one an FP32 BiCG solve of A z = v_j to the relative
// accuracy the outer residual still needs.  Each cycle starts from the FP64
// residual b - A x, so an answer is accepted only on the reference criterion
// |r|^2/|b|^2 < eps.  iters counts the inner FP32 BiCG iterations.
static int fgmres_dev(mstm_hip_ctx *c, int niter, double eps, const double *b, double *x, int use_fft, bool lig,
                      int pol, int *iters, double *errmax)
{
    typedef std::complex<double> zc;
    const int m = 8, max_cycles = 8;
    const int n = c->neqns;
    const size_t V = 2 * c->kv_n;
    const size_t need = sizeof(double) * V * (2 * m + 1);
    if (c->fg_bytes < need) {
        dfree(c->d_fg);
        HIPCHK(dalloc(&c->d_fg, need));
        c->fg_bytes = need;
    }
    auto Vv = [&](int i) { return c->d_fg + V * i; };
    auto Zv = [&](int i) { return c->d_fg + V * (m + 1 + i); };
    double *w = c->d_kv + V * KV_D, *y = c->d_kv + V * KV_Y, *r = c->d_kv + V * KV_R;
    zc bbz;
    int rc = zdot_host(c, b, b, bbz);
    if (rc) return rc;
    const double bb = bbz.real();
    *iters = 0;
    *errmax = 0.0;
    HIPCHK(hipMemsetAsync(x, 0, sizeof(double) * V, c->st));
    if (bb == 0.0) return 0;
    int f1[2] = {2, 0};
    for (int cycle = 0; cycle <= max_cycles; cycle++) {
        double beta;
        if (cycle == 0) {
            HIPCHK(hipMemcpyAsync(r, b, sizeof(double) * V, hipMemcpyDeviceToDevice, c->st));
            beta = std::sqrt(bb);
        } else {
            rc = matvec(c, 1, x, y, f1, MSTM_HIP_FP64, use_fft);  // y = T H x
            if (rc) return rc;
            HIPCHK(hipMemcpyAsync(r, b, sizeof(double) * V, hipMemcpyDeviceToDevice, c->st));
            HIPCHK(launch_zaxpby(-1.0, 0.0, x, 1.0, 0.0, r, n, c->st));
            HIPCHK(launch_zaxpby(1.0, 0.0, y, 1.0, 0.0, r, n, c->st));
            zc rr;
            rc = zdot_host(c, r, r, rr);
            if (rc) return rc;
            beta = std::sqrt(std::max(rr.real(), 0.0));
        }
        *errmax = beta * beta / bb;
        if (*errmax < eps || *iters >= niter || cycle == max_cycles) break;
        rc = scaled_copy(c, Vv(0), r, 1.0 / beta, 0.0);
        if (rc) return rc;
        std::vector<zc> H((size_t)(m + 1) * m, zc(0.0)), g(m + 1, zc(0.0)), sn(m, zc(0.0));
        std::vector<double> cs(m, 0.0);
        auto h = [&](int i, int j) -> zc & { return H[(size_t)i * m + j]; };
        g[0] = beta;
        int k = 0;  // steps taken in this cycle
        for (int j = 0; j < m; j++) {
            const double rho = std::norm(g[j]);
            if (cycle == 0 && j == 0 && lig) {
                // learned prediction of A^{-1} b, scaled like v_1 = b/|b|
                HIPCHK(launch_lig_combine(c->nsph, pol, c->d_order, c->d_offset, c->d_pos, c->rimed, c->lig.out,
                                          c->lig.Lnet, c->lig.depth, c->lig.params + c->lig.np - 2, b, y, c->st));
                rc = scaled_copy(c, Zv(0), y, 1.0 / beta, 0.0);
                if (rc) return rc;
            } else {
                HIPCHK(hipMemcpyAsync(Zv(j), Vv(j), sizeof(double) * V, hipMemcpyDeviceToDevice, c->st));
                const double eps_in = std::max(0.5 * eps * bb / rho, 1e-12);
                int it = 0;
                double ein = 0.0;
                rc = bicg2_dev(c, 1, std::max(1, niter - *iters), &eps_in, Vv(j), Zv(j), MSTM_HIP_FP32, use_fft, &it,
                               &ein);
                if (rc) return rc;
                *iters += std::min(it, std::max(1, niter - *iters));
            }
            // w = A z_j in FP64
            rc = matvec(c, 1, Zv(j), y, f1, MSTM_HIP_FP64, use_fft);
            if (rc) return rc;
            HIPCHK(hipMemcpyAsync(w, Zv(j), sizeof(double) * V, hipMemcpyDeviceToDevice, c->st));
            HIPCHK(launch_zaxpby(-1.0, 0.0, y, 1.0, 0.0, w, n, c->st));
            for (int i = 0; i <= j; i++) {  // modified Gram-Schmidt
                rc = zdot_host(c, Vv(i), w, h(i, j));
                if (rc) return rc;
                HIPCHK(launch_zaxpby(-h(i, j).real(), -h(i, j).imag(), Vv(i), 1.0, 0.0, w, n, c->st));
            }
            zc ww;
            rc = zdot_host(c, w, w, ww);
            if (rc) return rc;
            const double hn = std::sqrt(std::max(ww.real(), 0.0));
            h(j + 1, j) = hn;
            c->stats.fgmres_steps++;
            k = j + 1;
            if (hn > 0.0) {
                rc = scaled_copy(c, Vv(j + 1), w, 1.0 / hn, 0.0);
                if (rc) return rc;
            }
            for (int i = 0; i < j; i++) {  // earlier rotations on column j
                const zc a = h(i, j), bq = h(i + 1, j);
                h(i, j) = cs[i] * a + sn[i] * bq;
                h(i + 1, j) = -std::conj(sn[i]) * a + cs[i] * bq;
            }
            const zc a = h(j, j), bq = h(j + 1, j);
            const double nu = std::sqrt(std::norm(a) + std::norm(bq));
            if (nu == 0.0) break;
            if (std::abs(a) == 0.0) {
                cs[j] = 0.0;
                sn[j] = 1.0;
            } else {
                cs[j] = std::abs(a) / nu;
                sn[j] = (a / std::abs(a)) * std::conj(bq) / nu;
            }
            h(j, j) = cs[j] * a + sn[j] * bq;
            h(j + 1, j) = 0.0;
            g[j + 1] = -std::conj(sn[j]) * g[j];
            g[j] = cs[j] * g[j];
            if (std::norm(g[j + 1]) / bb < eps || hn == 0.0 || *iters >= niter) break;
        }
        // x += Z y with R y = g
        std::vector<zc> yv(k);
        for (int i = k - 1; i >= 0; i--) {
            zc s = g[i];
            for (int q = i + 1; q < k; q++) s -= h(i, q) * yv[q];
            yv[i] = s / h(i, i);
        }
        for (int i = 0; i < k; i++) HIPCHK(launch_zaxpby(yv[i].real(), yv[i].imag(), Zv(i), 1.0, 0.0, x, n, c->st));
    }
    return 0;
}

extern "C" {

// ---- dense LU (direct_solver, mstm-solver-8.f90:571-642) ----------------
static const int LU_MAX_N = 16384;  // two n x n complex FP64 matrices: 8.6 GB at the limit

// A = I - T H column by column (the FP64 operator on unit vectors, four
// columns per product), then its LU factors with the reference's scaled
// pivot rule
static int lu_setup(mstm_hip_ctx *c)
{
    const int n = c->neqns;
    if (n > LU_MAX_N) return fail(c, MSTM_HIP_EUNSUP, "direct solver: %d equations > %d", n, LU_MAX_N);
    if (c->lu.n != n) {
        release_lu(c);
        const size_t mat = sizeof(double) * 2 * (size_t)n * n;
        HIPCHK(dalloc(&c->lu.A, mat));
        HIPCHK(dalloc(&c->lu.LU, mat));
        HIPCHK(dalloc(&c->lu.vv, sizeof(double) * n));
        HIPCHK(dalloc(&c->lu.work, sizeof(double) * 2 * (size_t)n * 8));
        HIPCHK(dalloc(&c->lu.piv, sizeof(int) * n));
        HIPCHK(dalloc(&c->lu.err, sizeof(int)));
        HIPCHK(dalloc(&c->lu.scr, lu_factor_scratch_bytes()));
        c->lu.n = n;
    }
    c->lu.ready = false;
    auto t0 = std::chrono::steady_clock::now();
    bool uniform = true;
    for (int i = 0; i < c->nsph; i++) uniform = uniform && c->order[i] == c->Lmax;
    int rc = 0;
    if (uniform) {
        // spheres of one order: every off-diagonal block of A straight from its
        // pair table (FP64, full layout), in chunks of pairs
        if (int r2 = ensure_vcc(c, c->Lmax)) return r2;
        const int L = c->Lmax, CH = 4096, se = slot_len(L, L, 2);
        double *tab = nullptr, *d_rt = nullptr;
        int2 *d_pr = nullptr;
        HIPCHK(hipMemsetAsync(c->lu.A, 0, sizeof(double) * 2 * (size_t)n * n, c->st));
        HIPCHK(launch_lu_identity(c->lu.A, n, c->st));
        hipError_t e = dalloc(&tab, sizeof(double) * (size_t)CH * se);
        if (e == hipSuccess) e = dalloc(&d_rt, sizeof(double) * 3 * CH);
        if (e == hipSuccess) e = dalloc(&d_pr, sizeof(int2) * CH);
        std::vector<double> rt(3 * CH);
        std::vector<int2> pr(CH);
        int np = 0;
        auto flush = [&]() {
            if (e != hipSuccess || np == 0) return;
            e = hipMemcpyAsync(d_rt, rt.data(), sizeof(double) * 3 * np, hipMemcpyHostToDevice, c->st);
            if (e == hipSuccess) e = hipMemcpyAsync(d_pr, pr.data(), sizeof(int2) * np, hipMemcpyHostToDevice, c->st);
            if (e == hipSuccess) e = launch_list_tables<double>(tab, d_rt, np, L, L, 3, c->rimed, c->d_vcc, c->vcc_LM, c->st);
            if (e == hipSuccess) e = launch_lu_expand(tab, se, d_pr, np, L, n, c->d_an, c->lu.A, c->st);
            if (e == hipSuccess) e = hipStreamSynchronize(c->st);  // rt/pr are refilled next
            np = 0;
        };
        for (int i = 0; i < c->nsph && e == hipSuccess; i++)
            for (int j = i + 1; j < c->nsph && e == hipSuccess; j++) {
                pr[np] = make_int2(i, j);
                for (int a = 0; a < 3; a++) rt[3 * np + a] = c->pos[3 * i + a] - c->pos[3 * j + a];
                if (++np == CH) flush();
            }
        flush();
        dfree(tab);
        dfree(d_rt);
        dfree(d_pr);
        if (e != hipSuccess) return fail(c, MSTM_HIP_EHIP, "direct solver build: %s", hipGetErrorString(e));
    } else {
        // mixed orders: the columns e_j - T H e_j from the FP64 operator, four at a time
        const int flags[4] = {2, 2, 2, 2};  // mie_mult, no con_tran
        double *ue = c->lu.work, *th = c->lu.work + 2 * (size_t)n * 4;
        const bool timing = c->timing;  // the build's products stay out of the tile timings
        c->timing = false;
        for (int j0 = 0; j0 < n && !rc; j0 += 4) {
            const int nc = std::min(4, n - j0);
            hipError_t e = launch_lu_unit(ue, n, n, j0, nc, c->st);
            if (e == hipSuccess) rc = direct_matvec(c, nc, ue, th, flags, MSTM_HIP_FP64);
            if (e == hipSuccess && !rc) e = launch_lu_store(c->lu.A, n, j0, nc, th, n, c->st);
            if (e != hipSuccess) rc = fail(c, MSTM_HIP_EHIP, "direct solver: %s", hipGetErrorString(e));
        }
        c->timing = timing;
    }
    if (rc) return rc;
    HIPCHK(hipStreamSynchronize(c->st));
    auto t1 = std::chrono::steady_clock::now();
    c->lu.build_ms = std::chrono::duration<double, std::milli>(t1 - t0).count();
    // where the workgroups of a panel did not meet (their CUs were held by other
    // work), the factorization is done again without an exchange between them
    int err = 0;
    for (int capacity = lu_panel_capacity(c->device);; capacity = 0) {
        HIPCHK(hipMemcpyAsync(c->lu.LU, c->lu.A, sizeof(double) * 2 * (size_t)n * n, hipMemcpyDeviceToDevice, c->st));
        HIPCHK(hipMemsetAsync(c->lu.err, 0, sizeof(int), c->st));
        HIPCHK(launch_lu_factor(c->lu.LU, n, c->lu.vv, c->lu.piv, c->lu.err, c->lu.scr, capacity, c->lu.polls, c->st));
        HIPCHK(hipMemcpyAsync(&err, c->lu.err, sizeof(int), hipMemcpyDeviceToHost, c->st));
        HIPCHK(hipStreamSynchronize(c->st));
        if (!(err & 2) || !capacity) break;
    }
    c->lu.factor_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t1).count();
    if (err) return fail(c, MSTM_HIP_EARG, "direct solver: lu decomposition failed (a zero row)");
    c->lu.ready = true;
    return 0;
}

// x <- LU^{-1} P x for nrhs device vectors 2*neqns doubles apart
static int lu_solve_dev(mstm_hip_ctx *c, double *x, int nrhs)
{
    auto t0 = std::chrono::steady_clock::now();
    HIPCHK(launch_lu_solve(c->lu.LU, c->lu.n, c->lu.piv, x, c->lu.n, nrhs, c->st));
    HIPCHK(hipStreamSynchronize(c->st));
    c->lu.solve_ms += std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    return 0;
}

int mstm_hip_direct_solver(mstm_hip_ctx *c, const double *pnp, double *anp, int initialize, int niter,
                           double *solution_error)
{
    if (!c || !c->nsph) return fail(c, MSTM_HIP_ESTATE, "direct_solver: no spheres");
    if (!pnp || !anp || niter < 0) return fail(c, MSTM_HIP_EARG, "direct_solver: bad arguments");
    HIPCHK(hipSetDevice(c->device));
    c->obs.x_valid = false;
    if (initialize || !c->lu.ready)
        if (int rc = lu_setup(c)) return rc;
    const int n = c->neqns;
    double *p = c->lu.work, *x = c->lu.work + 2 * (size_t)n, *r = c->lu.work + 4 * (size_t)n;
    HIPCHK(hipMemcpyAsync(p, pnp, sizeof(double) * 2 * n, hipMemcpyHostToDevice, c->st));
    HIPCHK(hipMemcpyAsync(x, p, sizeof(double) * 2 * n, hipMemcpyDeviceToDevice, c->st));
    if (int rc = lu_solve_dev(c, x, 1)) return rc;
    // niter refinement steps r = A x - p, x <- x - LU^{-1} r (:627-633)
    double serr = 0.0;
    std::vector<double> hr(2 * (size_t)n);
    for (int it = 0; it < niter; it++) {
        HIPCHK(launch_lu_resid(c->lu.A, n, x, p, r, c->st));
        HIPCHK(hipMemcpyAsync(hr.data(), r, sizeof(double) * 2 * n, hipMemcpyDeviceToHost, c->st));
        HIPCHK(hipStreamSynchronize(c->st));
        double ss = 0.0;
        for (int i = 0; i < n; i++) ss += hr[2 * i] * hr[2 * i] + hr[2 * i + 1] * hr[2 * i + 1];
        serr = std::sqrt(ss) / (double)n;
        if (int rc = lu_solve_dev(c, r, 1)) return rc;
        HIPCHK(launch_zaxpby(-1.0, 0.0, r, 1.0, 0.0, x, n, c->st));
    }
    HIPCHK(hipMemcpyAsync(anp, x, sizeof(double) * 2 * n, hipMemcpyDeviceToHost, c->st));
    HIPCHK(hipStreamSynchronize(c->st));
    if (solution_error) *solution_error = serr;
    return 0;
}

int mstm_hip_sphereinteraction(mstm_hip_ctx *c, int nrhs, const double *ain, double *aout, const int *con_tran,
                               const int *mie_mult, int use_fft, int prec, const int *rhs_list,
                               int skip_external_translation)
{
    if (!c || !c->nsph) return fail(c, MSTM_HIP_ESTATE, "sphereinteraction: no spheres");
    if (nrhs < 1 || !ain || !aout || !con_tran || !mie_mult) return fail(c, MSTM_HIP_EARG, "sphereinteraction: args");
    HIPCHK(hipSetDevice(c->device));
    const size_t V = 2 * (size_t)c->neqns;
    // A column left out of rhs_list gets no translation (mstm-modules-33.f90:
    // 6507; fft_translation-5.f90:457, 609, 619), and skip_external_translation
    // drops the external translation of every column (mstm-scatprops-26.f90:
    // 101): with no host spheres or plane boundaries those columns are zero
    // after the Mie or conjugation post-step.
    std::vector<int> cols;
    for (int r = 0; r < nrhs; r++) {
        if (!skip_external_translation && (!rhs_list || rhs_list[r])) cols.push_back(r);
        else memset(aout + V * r, 0, sizeof(double) * V);
    }
    double *din = c->d_kv + V * KV_ST, *dout = c->d_kv + V * KV_PW;  // up to four columns per product
    for (size_t q0 = 0; q0 < cols.size(); q0 += 4) {
        const int nr = (int)std::min<size_t>(4, cols.size() - q0);
        int flags[4] = {0, 0, 0, 0};
        for (int q = 0; q < nr; q++) {
            const int r = cols[q0 + q];
            flags[q] = (con_tran[r] ? 1 : 0) | (mie_mult[r] ? 2 : 0);
            HIPCHK(hipMemcpyAsync(din + V * q, ain + V * r, sizeof(double) * V, hipMemcpyHostToDevice, c->st));
        }
        int rc = matvec(c, nr, din, dout, flags, prec, use_fft);
        if (rc) return rc;
        for (int q = 0; q < nr; q++)
            HIPCHK(hipMemcpyAsync(aout + V * cols[q0 + q], dout + V * q, sizeof(double) * V, hipMemcpyDeviceToHost,
                                  c->st));
        HIPCHK(hipStreamSynchronize(c->st));  // din is refilled next
    }
    HIPCHK(hipStreamSynchronize(c->st));
    collect_events(c);
    return 0;
}

// Scratch bytes of one direct product of nr (2 or 4) columns: staged input
// and output columns (nr x neqns complex FP64 each), the padded input and the
// per-block partial sums at the table precision; each part 256-B aligned.
static size_t noalloc_layout(const mstm_hip_ctx *c, int nr, int prec, int G, size_t off[4])
{
    auto al = [](size_t x) { return (x + 255) / 256 * 256; };
    const size_t esz = prec == MSTM_HIP_FP64 ? sizeof(double) : sizeof(float);
    const size_t nbp = (size_t)c->Lmax * (c->Lmax + 2);
    const size_t vcol = sizeof(double) * 2 * (size_t)c->neqns;
    const size_t sz[4] = {vcol * nr, vcol * nr, esz * 2 * nr * 2 * (size_t)c->npad * nbp,
                          esz * 2 * (size_t)c->nblocks * G * nr * 2 * c->npad * nbp};
    size_t o = 0;
    for (int q = 0; q < 4; q++) {
        off[q] = o;
        o += al(sz[q]);
    }
    return o;
}

int mstm_hip_sphereinteraction_noalloc(mstm_hip_ctx *c, int nrhs, const double *ain, double *aout, const int *con_tran,
                                       const int *mie_mult, int use_fft, int prec, const int *rhs_list,
                                       int skip_external_translation)
{
    if (!c || !c->nsph) return fail(c, MSTM_HIP_ESTATE, "sphereinteraction_noalloc: no spheres");
    if (nrhs < 1 || !ain || !aout || !con_tran || !mie_mult)
        return fail(c, MSTM_HIP_EARG, "sphereinteraction_noalloc: args");
    if (use_fft) return fail(c, MSTM_HIP_EUNSUP, "sphereinteraction_noalloc: direct operator only");
    if (prec != MSTM_HIP_FP64 && prec != MSTM_HIP_FP32)
        return fail(c, MSTM_HIP_EARG, "sphereinteraction_noalloc: precision %d", prec);
    HIPCHK(hipSetDevice(c->device));
    const int nr = nrhs > 2 ? 4 : 2;
    size_t off[4];
    // the workgroups per tile of the context's products, fewer if their
    // partials would not fit (the sums are the same)
    int G = c->tgroups;
    size_t need = noalloc_layout(c, nr, prec, G, off);
    while (need > MSTM_SCRATCH_BYTES && G > 1) need = noalloc_layout(c, nr, prec, G /= 2, off);
    if (need > MSTM_SCRATCH_BYTES)
        return fail(c, MSTM_HIP_EARG,
                    "sphereinteraction_noalloc: %zu bytes of scratch needed (%d spheres of order %d, %d columns), "
                    "more than the %u-byte device scratch: use mstm_hip_sphereinteraction",
                    need, c->nsph, c->Lmax, nr, (unsigned)MSTM_SCRATCH_BYTES);
    if (!c->dop[prec].ready)
        return fail(c, MSTM_HIP_ESTATE,
                    "sphereinteraction_noalloc: no %s tables (mstm_hip_setup_direct allocates them; this entry "
                    "point does not)", prec == MSTM_HIP_FP64 ? "FP64" : "FP32");
    if (c->device < 0 || c->device >= MSTM_MAX_DEVICES || !g_scratch_ptr[c->device])
        return fail(c, MSTM_HIP_EHIP, "sphereinteraction_noalloc: no device scratch on GPU %d: %s", c->device,
                    hipGetErrorString(c->device >= 0 && c->device < MSTM_MAX_DEVICES ? g_scratch_rc[c->device]
                                                                                      : hipErrorInvalidDevice));
    unsigned char *base = (unsigned char *)g_scratch_ptr[c->device];
    double *din = (double *)(base + off[0]), *dout = (double *)(base + off[1]);
    void *xin = base + off[2], *part = base + off[3];
    const size_t V = 2 * (size_t)c->neqns;
    const bool timing = c->timing;  // timing events may be created on demand: none here
    c->timing = false;
    int rc = 0, cols[4], ncol = 0;
    auto flush = [&]() -> int {
        if (!ncol) return 0;
        int flags[4] = {0, 0, 0, 0};
        for (int q = 0; q < ncol; q++) {
            const int r = cols[q];
            flags[q] = (con_tran[r] ? 1 : 0) | (mie_mult[r] ? 2 : 0);
            HIPCHK(hipMemcpyAsync(din + V * q, ain + V * r, sizeof(double) * V, hipMemcpyHostToDevice, c->st));
        }
        int r2 = direct_matvec_buf(c, ncol, din, dout, flags, prec, xin, part, G);
        if (r2) return r2;
        for (int q = 0; q < ncol; q++)
            HIPCHK(hipMemcpyAsync(aout + V * cols[q], dout + V * q, sizeof(double) * V, hipMemcpyDeviceToHost, c->st));
        HIPCHK(hipStreamSynchronize(c->st));  // din/dout are refilled next
        ncol = 0;
        return 0;
    };
    // rhs_list / skip_external_translation as mstm_hip_sphereinteraction: zero columns
    for (int r = 0; r < nrhs && !rc; r++) {
        if (skip_external_translation || (rhs_list && !rhs_list[r])) {
            memset(aout + V * r, 0, sizeof(double) * V);
            continue;
        }
        cols[ncol++] = r;
        if (ncol == nr) rc = flush();
    }
    if (!rc) rc = flush();
    c->timing = timing;
    return rc;
}

int mstm_hip_cbicg(mstm_hip_ctx *c, int niter, double eps, const double *pnp, double *anp, int use_fft, int *iter,
                   double *errmax)
{
    if (!c || !c->nsph) return fail(c, MSTM_HIP_ESTATE, "cbicg: no spheres");
    if (!pnp || !anp || !iter || !errmax) return fail(c, MSTM_HIP_EARG, "cbicg: null argument");
    HIPCHK(hipSetDevice(c->device));
    c->obs.x_valid = false;  // the solution slot is reused
    const size_t V = 2 * (size_t)c->neqns;
    double *db = c->d_kv + V * KV_B, *dx = c->d_kv + V * KV_X;
    HIPCHK(hipMemcpyAsync(db, pnp, sizeof(double) * V, hipMemcpyHostToDevice, c->st));
    HIPCHK(hipMemcpyAsync(dx, anp, sizeof(double) * V, hipMemcpyHostToDevice, c->st));
    int rc = 0;
    if (niter > 0) {
        rc = bicg2_dev(c, 1, niter, &eps, db, dx, MSTM_HIP_FP64, use_fft, iter, errmax);
    } else if (niter < 0) {
        rc = oos2_dev(c, 1, -niter, &eps, db, dx, use_fft, iter, errmax);  // order of scattering (:785-825)
    } else {
        // niter = 0 (:768-781): anp becomes the host-sphere part of the
        // product, which is zero for external spheres; pnp = 0 returns first
        *iter = 0;
        *errmax = 0.0;
        double bb[2];
        HIPCHK(launch_zdot(db, db, c->neqns, 1, c->d_partials, nullptr, c->st));
        rc = sum_partials(c, 1, bb);
        if (!rc && bb[0] != 0.0) HIPCHK(hipMemsetAsync(dx, 0, sizeof(double) * V, c->st));
    }
    if (rc) return rc;
    HIPCHK(hipMemcpyAsync(anp, dx, sizeof(double) * V, hipMemcpyDeviceToHost, c->st));
    HIPCHK(hipStreamSynchronize(c->st));
    collect_events(c);
    return 0;
}

int mstm_hip_fixedorsoln(mstm_hip_ctx *c, double alpha, double sinc, int dir, double eps, int niter, int solver,
                         int use_fft, double *amnp, double *qeff, double *maxerr, int *maxiter, int *istat,
                         const int *excited_spheres)
{
    if (!c || !c->nsph) return fail(c, MSTM_HIP_ESTATE, "fixedorsoln: no spheres");
    if (dir != 1 && dir != 2) return fail(c, MSTM_HIP_EARG, "fixedorsoln: dir must be 1 or 2");
    if (!maxerr || !maxiter || !istat) return fail(c, MSTM_HIP_EARG, "fixedorsoln: null status argument");
    if (solver != MSTM_HIP_SOLVE_PLAIN && solver != MSTM_HIP_SOLVE_MIXED && solver != MSTM_HIP_SOLVE_LEARNED &&
        solver != MSTM_HIP_SOLVE_FGMRES && solver != MSTM_HIP_SOLVE_LU)
        return fail(c, MSTM_HIP_EUNSUP, "fixedorsoln: solver %d not available", solver);
    if (solver == MSTM_HIP_SOLVE_LU && use_fft)
        return fail(c, MSTM_HIP_EUNSUP, "fixedorsoln: the direct solution uses the direct operator");
    if (!amnp) return fail(c, MSTM_HIP_EARG, "fixedorsoln: amnp is required");
    if (solver == MSTM_HIP_SOLVE_LEARNED && !c->lig.ready)
        return fail(c, MSTM_HIP_ESTATE, "fixedorsoln: the learned solver needs a network (mstm_hip_set_learned)");
    HIPCHK(hipSetDevice(c->device));
    c->obs.x_valid = false;
    const int n = c->neqns;
    const size_t V = 2 * (size_t)n;
    double *pmnp = c->d_kv + V * KV_PM, *x = c->d_kv + V * KV_X, *b = c->d_kv + V * KV_B, *r = c->d_kv + V * KV_R;
    auto t0 = std::chrono::steady_clock::now();
    // excited_spheres (:373-377, 468): spheres left out get no incident field
    bool all_excited = true;
    if (excited_spheres)
        for (int i = 0; i < c->nsph; i++) all_excited = all_excited && excited_spheres[i] != 0;
    if (!all_excited) {
        std::vector<int> m(excited_spheres, excited_spheres + c->nsph);
        for (auto &v : m) v = v != 0;
        HIPCHK(hipMemcpyAsync(c->d_excited, m.data(), sizeof(int) * c->nsph, hipMemcpyHostToDevice, c->st));
        HIPCHK(hipStreamSynchronize(c->st));  // m lives on the host stack
    }
    HIPCHK(launch_planewave(pmnp, 2 * n, c->nsph, c->d_pos, c->d_order, c->d_offset, alpha, sinc, dir, c->rimed, c->st,
                            all_excited ? nullptr : c->d_excited));
    // the network is trained for incidence along +z (beta = 0) on fully
    // excited clusters; niter < 0 is the order-of-scattering series
    const bool lig_on = (solver == MSTM_HIP_SOLVE_LEARNED || solver == MSTM_HIP_SOLVE_FGMRES) && c->lig.ready &&
                        sinc == 0.0 && dir == 1 && all_excited && niter > 0;
    if (lig_on) {
        auto tl = std::chrono::steady_clock::now();
        int rc = lig_predict(c);
        if (rc) return rc;
        HIPCHK(hipStreamSynchronize(c->st));
        c->stats.lig_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - tl).count();
    }
    // b_p = T f_p and x_p = b_p (:471-483) for both polarizations; the two
    // systems are solved together (each with its own scalars)
    for (int p = 0; p < 2; p++)
        HIPCHK(launch_mie_mult(pmnp + V * p, b + V * p, c->nsph, c->d_order, c->d_offset, c->d_mieoff, c->d_an, 1, 0,
                               c->Lmax, c->st));
    HIPCHK(hipMemcpyAsync(x, b, sizeof(double) * 2 * V, hipMemcpyDeviceToDevice, c->st));
    int it[2] = {0, 0}, rc = 0;
    double err[2] = {0, 0};
    const double eps2[2] = {eps, eps};
    if (niter == 0 && solver != MSTM_HIP_SOLVE_LU) {
        // no solve (:513-522): amnp = T f, iterations and error 0
    } else if (niter < 0 && solver != MSTM_HIP_SOLVE_LU) {
        // cbicg's order-of-scattering series from x = b (:785-825), both
        // polarizations together; the solution_method letters of this
        // library other than the direct one all take it
        rc = oos2_dev(c, 2, -niter, eps2, b, x, use_fft, it, err);
    } else if (solver == MSTM_HIP_SOLVE_PLAIN) {
        rc = bicg2_dev(c, 2, niter, eps2, b, x, MSTM_HIP_FP64, use_fft, it, err);
    } else if (solver == MSTM_HIP_SOLVE_LU) {
        // direct_solver with number_iterations = 0 (:491-493): LU of A once,
        // both polarizations back-substituted together; iter = 0
        if (!c->lu.ready) rc = lu_setup(c);
        if (!rc) rc = lu_solve_dev(c, x, 2);
    } else if (solver == MSTM_HIP_SOLVE_MIXED) {
        // the refinement starts from x = 0 (residual b, no product): the
        // reference's start x = b has |r|^2/|b|^2 >> 1 on dense clusters
        HIPCHK(hipMemsetAsync(x, 0, sizeof(double) * 2 * V, c->st));
        rc = refine2_dev(c, 2, niter, eps, b, x, use_fft, it, err, b);
        // a polarization whose refinement stalls is handed to the plain FP64 solver from b
        for (int p = 0; p < 2 && !rc; p++)
            if (err[p] >= eps && it[p] < niter) {
                c->stats.lig_fallbacks++;
                HIPCHK(hipMemcpyAsync(x + V * p, b + V * p, sizeof(double) * V, hipMemcpyDeviceToDevice, c->st));
                int it2 = 0;
                rc = bicg2_dev(c, 1, niter - it[p], &eps, b + V * p, x + V * p, MSTM_HIP_FP64, use_fft, &it2, &err[p]);
                it[p] += it2;
            }
    } else if (solver == MSTM_HIP_SOLVE_LEARNED) {
        // learned start (or x = 0 where the prediction is worse), mixed
        // refinement from it; the plain FP64 solver from b takes over for a
        // polarization whose refinement does not reach eps
        c->stats.lig_solves += 2;
        bool used[2] = {false, false};
        if (lig_on) {
            rc = lig_start2(c, b, x, r, use_fft, used);
            if (rc) return rc;
        } else {
            HIPCHK(hipMemsetAsync(x, 0, sizeof(double) * 2 * V, c->st));
        }
        for (int p = 0; p < 2; p++)
            if (!used[p]) c->stats.lig_fallbacks++;
        // the learned start's residual is an FP32 product: it steers the first
        // inner solve only, and FP64 residuals decide every answer
        rc = refine2_dev(c, 2, niter, eps, b, x, use_fft, it, err, lig_on ? r : b, !lig_on);
        for (int p = 0; p < 2 && !rc; p++)
            if (err[p] >= eps && it[p] < niter) {
                c->stats.lig_fallbacks++;
                HIPCHK(hipMemcpyAsync(x + V * p, b + V * p, sizeof(double) * V, hipMemcpyDeviceToDevice, c->st));
                int it2 = 0;
                rc = bicg2_dev(c, 1, niter - it[p], &eps, b + V * p, x + V * p, MSTM_HIP_FP64, use_fft, &it2, &err[p]);
                it[p] += it2;
            }
    } else {
        for (int p = 0; p < 2 && !rc; p++) {
            rc = fgmres_dev(c, niter, eps, b + V * p, x + V * p, use_fft, lig_on, p, &it[p], &err[p]);
            if (!rc && err[p] >= eps && it[p] < niter) {  // stalled: the plain FP64 solver from b
                c->stats.lig_fallbacks++;
                HIPCHK(hipMemcpyAsync(x + V * p, b + V * p, sizeof(double) * V, hipMemcpyDeviceToDevice, c->st));
                int it2 = 0;
                rc = bicg2_dev(c, 1, niter - it[p], &eps, b + V * p, x + V * p, MSTM_HIP_FP64, use_fft, &it2, &err[p]);
                it[p] += it2;
            }
        }
    }
    if (rc) return rc;
    // istat, maxiter, maxerr are reset per polarization (:471-475): they
    // report the second solve
    *maxiter = it[1];
    *maxerr = err[1];
    *istat = (it[1] > niter || err[1] > eps) ? 1 : 0;
    HIPCHK(hipStreamSynchronize(c->st));
    c->stats.solve_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    HIPCHK(hipMemcpyAsync(amnp, x, sizeof(double) * 2 * V, hipMemcpyDeviceToHost, c->st));
    c->obs.x_valid = true;
    if (qeff) {
        HIPCHK(launch_qeff(x, pmnp, 2 * n, c->nsph, c->d_radius, c->d_order, c->d_offset, c->d_mieoff, c->d_an,
                           c->rimed, c->d_qeff, c->st));
        HIPCHK(hipMemcpyAsync(qeff, c->d_qeff, sizeof(double) * 9 * c->nsph, hipMemcpyDeviceToHost, c->st));
    }
    HIPCHK(hipStreamSynchronize(c->st));
    collect_events(c);
    return 0;
}

int mstm_hip_set_learned(mstm_hip_ctx *c, const float *params, int nparams, int hidden, int nlayers, int Lnet)
{
    if (!c) return MSTM_HIP_EARG;
    HIPCHK(hipSetDevice(c->device));
    release_lig_buffers(c);
    dfree(c->lig.params);
    c->lig.ready = false;
    if (!params) return 0;
    if (hidden <= 0 || hidden > 1024 || nlayers <= 0 || nlayers > 8 || Lnet <= 0 || Lnet > MSTM_MAX_L)
        return fail(c, MSTM_HIP_EARG, "set_learned: bad shape (hidden %d, layers %d, Lnet %d)", hidden, nlayers, Lnet);
    MlpShape s{LIG_NFEAT, hidden, nlayers, 8 * Lnet * (Lnet + 2)};
    if ((size_t)nparams != mlp_nparams(s))
        return fail(c, MSTM_HIP_EARG, "set_learned: expected %zu parameters, got %d", mlp_nparams(s), nparams);
    HIPCHK(dalloc(&c->lig.params, sizeof(float) * nparams));
    HIPCHK(hipMemcpy(c->lig.params, params, sizeof(float) * nparams, hipMemcpyHostToDevice));
    c->lig.s = s;
    c->lig.Lnet = Lnet;
    c->lig.np = nparams;
    c->lig.ready = true;
    return 0;
}

int mstm_hip_lig_features(mstm_hip_ctx *c, float *feat, float *depth)
{
    if (!c || !c->nsph) return fail(c, MSTM_HIP_ESTATE, "lig_features: no spheres");
    if (!feat || !depth) return fail(c, MSTM_HIP_EARG, "lig_features: null output");
    HIPCHK(hipSetDevice(c->device));
    const int n = c->nsph;
    float *df = nullptr, *dd = nullptr;
    HIPCHK(dalloc(&df, sizeof(float) * (size_t)n * LIG_NFEAT));
    HIPCHK(dalloc(&dd, sizeof(float) * (size_t)n));
    hipError_t e = launch_lig_features(n, c->d_pos, c->d_radius, c->d_mre, c->d_mim, c->rimed, df, dd, c->st);
    if (e == hipSuccess) e = hipMemcpyAsync(feat, df, sizeof(float) * (size_t)n * LIG_NFEAT, hipMemcpyDeviceToHost, c->st);
    if (e == hipSuccess) e = hipMemcpyAsync(depth, dd, sizeof(float) * (size_t)n, hipMemcpyDeviceToHost, c->st);
    if (e == hipSuccess) e = hipStreamSynchronize(c->st);
    dfree(df);
    dfree(dd);
    if (e != hipSuccess) return fail(c, MSTM_HIP_EHIP, "lig_features: %s", hipGetErrorString(e));
    return 0;
}

int mstm_hip_lig_samples(mstm_hip_ctx *c, const double *amnp, int Lnet, float *target, float *base)
{
    if (!c || !c->nsph) return fail(c, MSTM_HIP_ESTATE, "lig_samples: no spheres");
    if (!amnp || !target || !base || Lnet <= 0 || Lnet > MSTM_MAX_L) return fail(c, MSTM_HIP_EARG, "lig_samples: args");
    HIPCHK(hipSetDevice(c->device));
    c->obs.x_valid = false;  // the solution slot is reused
    const int n = c->neqns;
    const size_t V = 2 * (size_t)n, row = (size_t)8 * Lnet * (Lnet + 2);
    double *pmnp = c->d_kv + V * KV_PM, *x = c->d_kv + V * KV_X, *b = c->d_kv + V * KV_B;
    float *dt = nullptr, *db = nullptr;
    HIPCHK(dalloc(&dt, sizeof(float) * row * c->nsph));
    HIPCHK(dalloc(&db, sizeof(float) * row * c->nsph));
    hipError_t e = launch_planewave(pmnp, 2 * n, c->nsph, c->d_pos, c->d_order, c->d_offset, 0.0, 0.0, 1, c->rimed, c->st);
    for (int p = 0; p < 2 && e == hipSuccess; p++) {
        e = launch_mie_mult(pmnp + V * p, b, c->nsph, c->d_order, c->d_offset, c->d_mieoff, c->d_an, 1, 0, c->Lmax, c->st);
        if (e == hipSuccess) e = hipMemcpyAsync(x, amnp + V * p, sizeof(double) * V, hipMemcpyHostToDevice, c->st);
        if (e == hipSuccess)
            e = launch_lig_samples(c->nsph, p, c->d_order, c->d_offset, c->d_pos, c->rimed, x, b, Lnet, dt, db, c->st);
        if (e == hipSuccess) e = hipStreamSynchronize(c->st);
    }
    if (e == hipSuccess) e = hipMemcpy(target, dt, sizeof(float) * row * c->nsph, hipMemcpyDeviceToHost);
    if (e == hipSuccess) e = hipMemcpy(base, db, sizeof(float) * row * c->nsph, hipMemcpyDeviceToHost);
    dfree(dt);
    dfree(db);
    if (e != hipSuccess) return fail(c, MSTM_HIP_EHIP, "lig_samples: %s", hipGetErrorString(e));
    return 0;
}

int mstm_hip_lig_guess(mstm_hip_ctx *c, double *x0)
{
    if (!c || !c->nsph) return fail(c, MSTM_HIP_ESTATE, "lig_guess: no spheres");
    if (!c->lig.ready) return fail(c, MSTM_HIP_ESTATE, "lig_guess: no network (mstm_hip_set_learned)");
    if (!x0) return fail(c, MSTM_HIP_EARG, "lig_guess: null output");
    HIPCHK(hipSetDevice(c->device));
    c->obs.x_valid = false;  // the solution slot is reused
    const int n = c->neqns;
    const size_t V = 2 * (size_t)n;
    double *pmnp = c->d_kv + V * KV_PM, *x = c->d_kv + V * KV_X, *b = c->d_kv + V * KV_B;
    auto t0 = std::chrono::steady_clock::now();
    int rc = lig_predict(c);
    if (rc) return rc;
    HIPCHK(launch_planewave(pmnp, 2 * n, c->nsph, c->d_pos, c->d_order, c->d_offset, 0.0, 0.0, 1, c->rimed, c->st));
    for (int p = 0; p < 2; p++) {
        HIPCHK(launch_mie_mult(pmnp + V * p, b, c->nsph, c->d_order, c->d_offset, c->d_mieoff, c->d_an, 1, 0, c->Lmax,
                               c->st));
        HIPCHK(launch_lig_combine(c->nsph, p, c->d_order, c->d_offset, c->d_pos, c->rimed, c->lig.out, c->lig.Lnet,
                                  c->lig.depth, c->lig.params + c->lig.np - 2, b, x, c->st));
        HIPCHK(hipMemcpyAsync(x0 + V * p, x, sizeof(double) * V, hipMemcpyDeviceToHost, c->st));
    }
    HIPCHK(hipStreamSynchronize(c->st));
    c->stats.lig_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    return 0;
}

int mstm_hip_set_inner_solver(mstm_hip_ctx *c, int kind)
{
    if (!c) return MSTM_HIP_EARG;
    if (kind != 0 && kind != 1) return fail(c, MSTM_HIP_EARG, "set_inner_solver: kind %d (0 BiCG, 1 GMRES)", kind);
    c->inner = kind;
    return 0;
}

int mstm_hip_set_graphs(mstm_hip_ctx *c, int on)
{
    if (!c) return MSTM_HIP_EARG;
    c->graphs = on != 0;
    return 0;
}

int mstm_hip_set_refinement_cycles(mstm_hip_ctx *c, int cycles)
{
    if (!c) return MSTM_HIP_EARG;
    if (cycles < 0 || cycles > 100) return fail(c, MSTM_HIP_EARG, "set_refinement_cycles: %d outside 0..100", cycles);
    c->max_ref = cycles;
    return 0;
}

int mstm_hip_set_lu_wait(mstm_hip_ctx *c, int polls)
{
    if (!c) return MSTM_HIP_EARG;
    if (polls < 0) return fail(c, MSTM_HIP_EARG, "set_lu_wait: %d polls", polls);
    c->lu.polls = polls;
    return 0;
}

int mstm_hip_clear(mstm_hip_ctx *c, int clear_tables)
{
    if (!c) return MSTM_HIP_EARG;
    if (clear_tables) {
        release_direct(c, 0);
        release_direct(c, 1);
        release_lu(c);
        if (c->fft) fft_clear(c->fft);
    }
    c->stats = Stats();
    c->lu.solve_ms = 0;
    if (c->fft) fft_reset_stats(c->fft);
    return 0;
}

const char *mstm_hip_stats_names(void)
{
    return "tables_ms_fp64,tables_ms_fp32,tile_ms_fp64,tile_ms_fp32,tile_launches_fp64,tile_launches_fp32,"
           "matvecs_fp64,matvecs_fp32,solve_ms,iters_fp64,iters_fp32,refinements,table_bytes_fp64,table_bytes_fp32,"
           "fft_setup_ms,fft_conv_ms,fft_launches,npad,ntiles,nblocks,lig_solves,lig_fallbacks,lig_ms,lig_err0,"
           "lig_errb,fgmres_steps,tile4_ms_fp64,tile4_ms_fp32,tile4_launches_fp64,tile4_launches_fp32,inner_solver,"
           "obs_orders_ms,obs_merge_ms,obs_scatmat_ms,obs_moments_ms,obs_T,fft_contract_ms_fp32,"
           "fft_contract_launches_fp32,fft_contract_ms_fp64,fft_contract_launches_fp64,tmatrix_ms,tmatrix_solves,"
           "lu_build_ms,lu_factor_ms,lu_solve_ms,obs_fosm_ms";
}

int mstm_hip_stats(const mstm_hip_ctx *c, double *out, int nout)
{
    if (!c || !out) return 0;
    double v[] = {c->stats.tables_ms[0],
                  c->stats.tables_ms[1],
                  c->stats.tile_ms[0],
                  c->stats.tile_ms[1],
                  (double)c->stats.tile_launches[0],
                  (double)c->stats.tile_launches[1],
                  (double)c->stats.matvecs[0],
                  (double)c->stats.matvecs[1],
                  c->stats.solve_ms,
                  (double)c->stats.iters_fp64,
                  (double)c->stats.iters_fp32,
                  (double)c->stats.refinements,
                  c->stats.table_bytes[0],
                  c->stats.table_bytes[1],
                  c->fft ? fft_stat(c->fft, 0) : 0.0,
                  c->fft ? fft_stat(c->fft, 1) : 0.0,
                  c->fft ? fft_stat(c->fft, 2) : 0.0,
                  (double)c->npad,
                  (double)c->ntiles,
                  (double)c->nblocks,
                  (double)c->stats.lig_solves,
                  (double)c->stats.lig_fallbacks,
                  c->stats.lig_ms,
                  c->stats.lig_err0,
                  c->stats.lig_errb,
                  (double)c->stats.fgmres_steps,
                  c->stats.tile4_ms[0],
                  c->stats.tile4_ms[1],
                  (double)c->stats.tile4_launches[0],
                  (double)c->stats.tile4_launches[1],
                  (double)c->inner,
                  c->obs.orders_ms,
                  c->obs.merge_ms,
                  c->obs.scatmat_ms,
                  c->obs.moments_ms,
                  (double)c->obs.T,
                  c->fft ? fft_stat(c->fft, 3) : 0.0,
                  c->fft ? fft_stat(c->fft, 4) : 0.0,
                  c->fft ? fft_stat(c->fft, 5) : 0.0,
                  c->fft ? fft_stat(c->fft, 6) : 0.0,
                  c->obs.tmatrix_ms,
                  (double)c->obs.tm_solves,
                  c->lu.build_ms,
                  c->lu.factor_ms,
                  c->lu.solve_ms,
                  c->obs.fosm_ms};
    int k = std::min(nout, (int)(sizeof v / sizeof v[0]));
    for (int q = 0; q < k; q++) out[q] = v[q];
    return k;
}

}  // extern "C"

// ------------------------------------------------------- observables (host)
// tranordertest (mstm-modules-33.f90:1896-1942) for a real medium index:
// the smallest n (capped at 200, at least lmax) at which the regular
// translation over r of a degree-lmax, m = 1 wave holds all but eps of its
// norm.  vc2 holds C(n,-1;lmax,1|w,0)^2 at n*(2 lmax+1) + w - |n-lmax|.
static int tran_order(double r, double rimed, int lmax, double eps, const std::vector<double> &vc2,
                      std::vector<double> &jw)
{
    const int nlim = 200;
    if (r == 0.0) return lmax;
    const double z = r * rimed;
    sph_bessel_j(nlim + lmax, z, jw.data());
    double sum = 0.0;
    int n;
    for (n = 1; n <= nlim; n++) {
        const int l = lmax, wmin = std::abs(n - l);
        std::complex<double> a = 0.0, b = 0.0;
        for (int w = wmin; w <= n + l; w++) {
            static const std::complex<double> ipow[4] = {{1, 0}, {0, 1}, {-1, 0}, {0, -1}};
            std::complex<double> xw = jw[w] * ipow[w & 3];
            double v2 = vc2[(size_t)n * (2 * l + 1) + (w - wmin)];
            if (((n + l + w) & 1) == 0) a += v2 * xw;
            else b += v2 * xw;
        }
        static const std::complex<double> ipw[4] = {{1, 0}, {0, 1}, {-1, 0}, {0, -1}};
        std::complex<double> cc = std::sqrt((double)(2 * n + 1)) * std::sqrt((double)(2 * l + 1)) * ipw[((n - l) % 4 + 4) % 4];
        a *= cc;
        b *= cc;
        sum += std::norm(a) + std::norm(b);
        if (std::fabs(1.0 - sum) < eps) break;
    }
    return std::max(std::min(n, nlim), lmax);
}

// vcc(n, l, m, w) of axialtrancoefinit for the merge seeds: n <= T, l <= LS;
// entries are filled where the seeds read them (n <= LS, or l one of the
// sphere orders).  Layout ((n (LS+1) + l)(2LS+1) + m+LS)(2LS+1) + w-|n-l|.
static int ensure_vccm(mstm_hip_ctx *c, int T, int LS)
{
    if (c->obs.d_vccm && c->obs.vccm_T == T && c->obs.vccm_LS == LS) return 0;
    dfree(c->obs.d_vccm);
    const int W = 2 * LS + 1;
    std::vector<double> h((size_t)(T + 1) * (LS + 1) * W * W, 0.0);
    std::vector<char> have(LS + 1, 0);
    for (int L : c->order) have[L] = 1;
    for (int n = 1; n <= T; n++)
        for (int l = 1; l <= LS; l++) {
            if (n > LS && !have[l]) continue;
            const long double c1 = sqrtl((long double)(2 * n + 1)) * sqrtl((long double)(2 * l + 1));
            for (int m = -std::min(n, l); m <= std::min(n, l); m++)
                for (int w = std::abs(n - l); w <= n + l; w++) {
                    const long double c2 = -c1 * ((std::abs(m) & 1) ? -1.0L : 1.0L);
                    const int k4 = (n - l + w) & 3;
                    const long double sg = (k4 == 0 || k4 == 1) ? 1.0L : -1.0L;
                    h[(((size_t)n * (LS + 1) + l) * W + (m + LS)) * W + (w - std::abs(n - l))] =
                        (double)(c2 * clebsch(n, -m, l, m, w) * clebsch(n, -1, l, 1, w) * sg);
                }
        }
    HIPCHK(dalloc(&c->obs.d_vccm, sizeof(double) * h.size()));
    HIPCHK(hipMemcpy(c->obs.d_vccm, h.data(), sizeof(double) * h.size(), hipMemcpyHostToDevice));
    c->obs.vccm_T = T;
    c->obs.vccm_LS = LS;
    return 0;
}

// vector-coupling sums of the distribute translation (target degree t <= LS,
// source degree l' <= T): the same coefficients as ensure_vccm with the
// roles of the two degrees exchanged, laid out [l'][t][m + LS][w - |t - l'|]
static int ensure_vccd(mstm_hip_ctx *c, int T, int LS)
{
    if (c->obs.d_vccd && c->obs.vccd_T == T && c->obs.vccd_LS == LS) return 0;
    dfree(c->obs.d_vccd);
    const int W = 2 * LS + 1;
    std::vector<double> h((size_t)(T + 1) * (LS + 1) * W * W, 0.0);
    for (int l = 1; l <= T; l++)
        for (int t = 1; t <= LS; t++) {
            const long double c1 = sqrtl((long double)(2 * t + 1)) * sqrtl((long double)(2 * l + 1));
            for (int m = -std::min(t, l); m <= std::min(t, l); m++)
                for (int w = std::abs(t - l); w <= t + l; w++) {
                    const long double c2 = -c1 * ((std::abs(m) & 1) ? -1.0L : 1.0L);
                    const int k4 = (t - l + w) & 3;
                    const long double sg = (k4 == 0 || k4 == 1) ? 1.0L : -1.0L;
                    h[(((size_t)l * (LS + 1) + t) * W + (m + LS)) * W + (w - std::abs(t - l))] =
                        (double)(c2 * clebsch(t, -m, l, m, w) * clebsch(t, -1, l, 1, w) * sg);
                }
        }
    HIPCHK(dalloc(&c->obs.d_vccd, sizeof(double) * h.size()));
    HIPCHK(hipMemcpy(c->obs.d_vccd, h.data(), sizeof(double) * h.size(), hipMemcpyHostToDevice));
    c->obs.vccd_T = T;
    c->obs.vccd_LS = LS;
    return 0;
}

template <typename P> static int grow(mstm_hip_ctx *c, P **p, size_t &cap, size_t bytes)
{
    if (*p && cap >= bytes) return 0;
    dfree(*p);
    cap = 0;
    HIPCHK(dalloc(p, bytes));
    cap = bytes;
    return 0;
}

// common-origin coefficients for the scattering matrix / moments: the last
// merge (a0 == NULL) or the caller's (T, a0) copied to the device
static int observe_source(mstm_hip_ctx *c, int T, const double *a0, const double **src, int *Tout)
{
    if (!a0) {
        if (!c->obs.a0_T) return fail(c, MSTM_HIP_ESTATE, "no merged coefficients (mstm_hip_merge_to_common_origin)");
        *src = c->obs.d_a0;
        *Tout = c->obs.a0_T;
        return 0;
    }
    if (T < 1 || T > 127) return fail(c, MSTM_HIP_EUNSUP, "common-origin order %d outside 1..127", T);
    const size_t bytes = sizeof(double) * 2 * 4 * (size_t)T * (T + 2);
    if (int rc = grow(c, &c->obs.d_in, c->obs.in_bytes, bytes)) return rc;
    HIPCHK(hipMemcpyAsync(c->obs.d_in, a0, bytes, hipMemcpyHostToDevice, c->st));
    *src = c->obs.d_in;
    *Tout = T;
    return 0;
}

extern "C" {

int mstm_hip_translation_orders(mstm_hip_ctx *c, const double *origin, double eps, int maxt, int *torder, int *tmo)
{
    if (!c || !c->nsph) return fail(c, MSTM_HIP_ESTATE, "translation_orders: no spheres");
    if (maxt < 1 || maxt > 127) return fail(c, MSTM_HIP_EUNSUP, "translation_orders: maxt %d outside 1..127", maxt);
    if (!(eps > 0.0)) return fail(c, MSTM_HIP_EARG, "translation_orders: eps must be > 0");
    HIPCHK(hipSetDevice(c->device));
    auto t0 = std::chrono::steady_clock::now();
    const int n = c->nsph;
    double r0[3] = {0, 0, 0};
    if (origin) {
        for (int d = 0; d < 3; d++) r0[d] = origin[d];
    } else {  // cluster_origin: mean sphere position (mstm-input-37.f90:1166-1174)
        for (int i = 0; i < n; i++)
            for (int d = 0; d < 3; d++) r0[d] += c->pos[3 * i + d];
        for (int d = 0; d < 3; d++) r0[d] /= (double)n;
    }
    std::vector<std::vector<double>> vc2(c->Lmax + 1);
    std::vector<double> jw(200 + c->Lmax + 1);
    c->obs.torder.assign(n, 0);
    int T = std::min(c->Lmax, maxt);
    for (int i = 0; i < n; i++) {
        const int L = c->order[i];
        if (vc2[L].empty()) {
            vc2[L].assign((size_t)201 * (2 * L + 1), 0.0);
            for (int nn = 1; nn <= 200; nn++)
                for (int w = std::abs(nn - L); w <= nn + L; w++) {
                    const double v = (double)clebsch(nn, -1, L, 1, w);
                    vc2[L][(size_t)nn * (2 * L + 1) + (w - std::abs(nn - L))] = v * v;
                }
        }
        const double dx = c->pos[3 * i] - r0[0], dy = c->pos[3 * i + 1] - r0[1], dz = c->pos[3 * i + 2] - r0[2];
        const double rt = std::sqrt(dx * dx + dy * dy + dz * dz);
        c->obs.torder[i] = std::min(tran_order(rt, c->rimed, L, eps, vc2[L], jw), maxt);
        T = std::max(T, c->obs.torder[i]);
    }
    dfree(c->obs.d_torder);
    HIPCHK(dalloc(&c->obs.d_torder, sizeof(int) * n));
    HIPCHK(hipMemcpy(c->obs.d_torder, c->obs.torder.data(), sizeof(int) * n, hipMemcpyHostToDevice));
    for (int d = 0; d < 3; d++) c->obs.r0[d] = r0[d];
    c->obs.T = T;
    c->obs.a0_T = 0;
    if (torder) std::memcpy(torder, c->obs.torder.data(), sizeof(int) * n);
    if (tmo) *tmo = T;
    c->obs.orders_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    return 0;
}

int mstm_hip_set_translation_orders(mstm_hip_ctx *c, const double *origin, const int *torder, int T)
{
    if (!c || !c->nsph) return fail(c, MSTM_HIP_ESTATE, "set_translation_orders: no spheres");
    if (!origin || !torder) return fail(c, MSTM_HIP_EARG, "set_translation_orders: null argument");
    if (T < 1 || T > 127) return fail(c, MSTM_HIP_EUNSUP, "set_translation_orders: T %d outside 1..127", T);
    for (int i = 0; i < c->nsph; i++)
        if (torder[i] < 1 || torder[i] > 127)
            return fail(c, MSTM_HIP_EARG, "set_translation_orders: order %d of sphere %d", torder[i], i + 1);
    HIPCHK(hipSetDevice(c->device));
    c->obs.torder.assign(torder, torder + c->nsph);
    dfree(c->obs.d_torder);
    HIPCHK(dalloc(&c->obs.d_torder, sizeof(int) * c->nsph));
    HIPCHK(hipMemcpy(c->obs.d_torder, torder, sizeof(int) * c->nsph, hipMemcpyHostToDevice));
    for (int d = 0; d < 3; d++) c->obs.r0[d] = origin[d];
    c->obs.T = T;
    c->obs.a0_T = 0;
    return 0;
}

int mstm_hip_merge_to_common_origin(mstm_hip_ctx *c, const double *amnp, double *amnp0)
{
    if (!c || !c->nsph) return fail(c, MSTM_HIP_ESTATE, "merge: no spheres");
    if (!c->obs.T) return fail(c, MSTM_HIP_ESTATE, "merge: no translation orders (mstm_hip_translation_orders)");
    if (c->Lmax > MSTM_MAX_L) return fail(c, MSTM_HIP_EUNSUP, "merge: sphere order %d > %d", c->Lmax, MSTM_MAX_L);
    if (!amnp && !c->obs.x_valid) return fail(c, MSTM_HIP_ESTATE, "merge: no solution on the device (run fixedorsoln)");
    HIPCHK(hipSetDevice(c->device));
    auto t0 = std::chrono::steady_clock::now();
    const int n = c->neqns, T = c->obs.T, b0 = T * (T + 2);
    const size_t V = 2 * (size_t)n;
    const double *src = c->d_kv + V * KV_X;
    if (amnp) {
        double *st = c->d_kv + V * KV_ST;
        HIPCHK(hipMemcpyAsync(st, amnp, sizeof(double) * 2 * V, hipMemcpyHostToDevice, c->st));
        src = st;
    }
    if (int rc = ensure_vccm(c, T, c->Lmax)) return rc;
    const size_t per_group = sizeof(double) * 8 * (size_t)b0;
    int G = std::min(c->nsph, 1024);
    G = (int)std::max<size_t>(1, std::min<size_t>((size_t)G, ((size_t)1 << 30) / per_group));
    if (int rc = grow(c, &c->obs.d_part, c->obs.part_bytes, per_group * G)) return rc;
    if (int rc = grow(c, &c->obs.d_a0, c->obs.a0_bytes, sizeof(double) * 8 * (size_t)b0)) return rc;
    HIPCHK(launch_merge(src, n, c->d_order, c->d_offset, c->obs.d_torder, c->d_pos, c->nsph, T, c->Lmax, c->obs.r0,
                        c->rimed, c->obs.d_vccm, c->obs.d_part, G, c->obs.d_a0, c->st));
    c->obs.a0_T = T;
    if (amnp0) HIPCHK(hipMemcpyAsync(amnp0, c->obs.d_a0, sizeof(double) * 8 * (size_t)b0, hipMemcpyDeviceToHost, c->st));
    HIPCHK(hipStreamSynchronize(c->st));
    c->obs.merge_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    return 0;
}

int mstm_hip_scattering_matrix(mstm_hip_ctx *c, int T, const double *amnp0, int nang, const double *ct,
                               const double *phi, double *sm)
{
    if (!c) return fail(c, MSTM_HIP_EARG, "scattering_matrix: null context");
    if (nang < 1 || !ct || !phi || !sm) return fail(c, MSTM_HIP_EARG, "scattering_matrix: bad arguments");
    HIPCHK(hipSetDevice(c->device));
    auto t0 = std::chrono::steady_clock::now();
    const double *src = nullptr;
    int Tu = 0;
    if (int rc = observe_source(c, T, amnp0, &src, &Tu)) return rc;
    if ((size_t)nang > c->obs.ang_cap) {
        dfree(c->obs.d_ang);
        dfree(c->obs.d_sm);
        c->obs.ang_cap = 0;
        HIPCHK(dalloc(&c->obs.d_ang, sizeof(double) * 2 * nang));
        HIPCHK(dalloc(&c->obs.d_sm, sizeof(double) * 16 * nang));
        c->obs.ang_cap = nang;
    }
    HIPCHK(hipMemcpyAsync(c->obs.d_ang, ct, sizeof(double) * nang, hipMemcpyHostToDevice, c->st));
    HIPCHK(hipMemcpyAsync(c->obs.d_ang + nang, phi, sizeof(double) * nang, hipMemcpyHostToDevice, c->st));
    HIPCHK(launch_scatmat(src, Tu, nang, c->obs.d_ang, c->obs.d_ang + nang, c->rimed, c->obs.d_sm, c->st));
    HIPCHK(hipMemcpyAsync(sm, c->obs.d_sm, sizeof(double) * 16 * nang, hipMemcpyDeviceToHost, c->st));
    HIPCHK(hipStreamSynchronize(c->st));
    c->obs.scatmat_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    return 0;
}

int mstm_hip_asymmetry(mstm_hip_ctx *c, int T, const double *amnp0, double *s00, double *g)
{
    if (!c) return fail(c, MSTM_HIP_EARG, "asymmetry: null context");
    if (!s00 && !g) return fail(c, MSTM_HIP_EARG, "asymmetry: no output");
    HIPCHK(hipSetDevice(c->device));
    auto t0 = std::chrono::steady_clock::now();
    const double *src = nullptr;
    int Tu = 0;
    if (int rc = observe_source(c, T, amnp0, &src, &Tu)) return rc;
    if (c->obs.cg_T != Tu) {
        dfree(c->obs.d_cg);
        dfree(c->obs.d_mom);
        c->obs.cg_T = 0;
        const int W = 2 * Tu + 1;
        std::vector<double> h((size_t)(Tu + 1) * 3 * W * 2 + (size_t)(Tu + 1) * 3 * 2, 0.0);
        double *cgm = h.data(), *cg1 = h.data() + (size_t)(Tu + 1) * 3 * W * 2;
        for (int n = 1; n <= Tu; n++)
            for (int li = 0; li < 3; li++) {
                const int l = n - 1 + li;
                if (l < 1 || l > Tu) continue;
                for (int w = 0; w <= 1; w++) {
                    cg1[(n * 3 + li) * 2 + w] = (double)clebsch(n, -1, l, 1, w);
                    for (int m = -std::min(n, l); m <= std::min(n, l); m++)
                        cgm[((size_t)(n * 3 + li) * W + m + Tu) * 2 + w] = (double)clebsch(n, -m, l, m, w);
                }
            }
        HIPCHK(dalloc(&c->obs.d_cg, sizeof(double) * h.size()));
        HIPCHK(hipMemcpy(c->obs.d_cg, h.data(), sizeof(double) * h.size(), hipMemcpyHostToDevice));
        HIPCHK(dalloc(&c->obs.d_mom, sizeof(double) * 2 * s00_moment_blocks(Tu)));
        c->obs.cg_T = Tu;
    }
    const int nb = s00_moment_blocks(Tu);
    const double *cgm = c->obs.d_cg, *cg1 = c->obs.d_cg + (size_t)(Tu + 1) * 3 * (2 * Tu + 1) * 2;
    HIPCHK(launch_s00_moments(src, Tu, cgm, cg1, c->obs.d_mom, c->st));
    std::vector<double> part(2 * nb);
    HIPCHK(hipMemcpyAsync(part.data(), c->obs.d_mom, sizeof(double) * 2 * nb, hipMemcpyDeviceToHost, c->st));
    HIPCHK(hipStreamSynchronize(c->st));
    double s[2] = {0, 0};
    for (int b = 0; b < nb; b++) {
        s[0] += part[2 * b];
        s[1] += part[2 * b + 1];
    }
    // sign patch and scale of fosmexpansion (mstm-scatprops-26.f90:1930-1948): s00(1,1) keeps its sign
    for (int w = 0; w < 2; w++) s[w] *= 0.5 / c->rimed;
    if (s00) {
        s00[0] = s[0];
        s00[1] = s[1];
    }
    if (g) *g = s[1] / (3.0 * s[0]);
    c->obs.moments_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    return 0;
}

int mstm_hip_fosmexpansion(mstm_hip_ctx *c, int T, const double *amnp0, double *s00, double *s02, double *sp22,
                           double *sm22)
{
    if (!c) return fail(c, MSTM_HIP_EARG, "fosmexpansion: null context");
    if (!s00 || !s02 || !sp22 || !sm22) return fail(c, MSTM_HIP_EARG, "fosmexpansion: null output");
    HIPCHK(hipSetDevice(c->device));
    auto t0 = std::chrono::steady_clock::now();
    const double *src = nullptr;
    int Tu = 0;
    if (int rc = observe_source(c, T, amnp0, &src, &Tu)) return rc;
    if (Tu != T)  // the outputs are sized by T
        return fail(c, MSTM_HIP_EARG, "fosmexpansion: T = %d, the merged coefficients have order %d", T, Tu);
    const int W = 2 * Tu + 1, ldb = 4 * Tu + 2, nb = fosm_blocks(Tu);
    if (c->obs.bc_T != Tu) {
        dfree(c->obs.d_bc);
        dfree(c->obs.d_fpart);
        c->obs.bc_T = 0;
        // bcof(n,l) = sqrt((n+l)!/(n! l!)) by init's recurrence (mstm-modules-33.f90:46-50)
        std::vector<double> bc((size_t)ldb * ldb, 0.0), fnr(2 * (size_t)ldb + 1);
        for (int i = 0; i <= 2 * ldb; i++) fnr[i] = std::sqrt((double)i);
        bc[0] = 1.0;
        for (int n = 0; n < ldb - 1; n++) {
            for (int l = n + 1; l < ldb; l++) {
                bc[(size_t)n * ldb + l] = fnr[n + l] * bc[(size_t)n * ldb + l - 1] / fnr[l];
                bc[(size_t)l * ldb + n] = bc[(size_t)n * ldb + l];
            }
            bc[(size_t)(n + 1) * ldb + n + 1] = fnr[n + n + 2] * fnr[n + n + 1] * bc[(size_t)n * ldb + n] / fnr[n + 1] / fnr[n + 1];
        }
        HIPCHK(dalloc(&c->obs.d_bc, sizeof(double) * (bc.size() + 8 * (size_t)W)));
        HIPCHK(hipMemcpy(c->obs.d_bc, bc.data(), sizeof(double) * bc.size(), hipMemcpyHostToDevice));
        HIPCHK(dalloc(&c->obs.d_fpart, sizeof(double) * (size_t)nb * 8 * W));
        c->obs.bc_T = Tu;
    }
    double *dout = c->obs.d_bc + (size_t)ldb * ldb;
    HIPCHK(launch_fosm(src, Tu, c->obs.d_bc, ldb, c->obs.d_fpart, dout, c->st));
    std::vector<double> e8((size_t)8 * W);
    HIPCHK(hipMemcpyAsync(e8.data(), dout, sizeof(double) * e8.size(), hipMemcpyDeviceToHost, c->st));
    HIPCHK(hipStreamSynchronize(c->st));
    // the reference's sign patch and scale (mstm-scatprops-26.f90:1930-1948):
    // (j,i) with i = 3, 4 and j <= i negated; sm22(3,3) = -sm22(2,2),
    // sp22(3,3) = sp22(2,2); everything times 1/(2 m_medium)
    const size_t nall = (size_t)16 * W;
    std::fill(s00, s00 + nall, 0.0);
    std::fill(s02, s02 + nall, 0.0);
    std::fill(sp22, sp22 + nall, 0.0);
    std::fill(sm22, sm22 + nall, 0.0);
    const double f = 0.5 / c->rimed;
    auto at = [&](double *s, int i, int j, int w) -> double & { return s[((size_t)w * 4 + (j - 1)) * 4 + (i - 1)]; };
    for (int w = 0; w < W; w++) {
        const double *v = e8.data() + w;
        at(s00, 1, 1, w) = f * v[0];
        at(s00, 4, 4, w) = -f * v[(size_t)W];
        at(s02, 2, 1, w) = f * v[2 * (size_t)W];
        at(s02, 1, 2, w) = f * v[3 * (size_t)W];
        at(s02, 3, 4, w) = -f * v[4 * (size_t)W];
        at(s02, 4, 3, w) = f * v[5 * (size_t)W];
        at(sm22, 2, 2, w) = f * v[6 * (size_t)W];
        at(sp22, 2, 2, w) = f * v[7 * (size_t)W];
        at(sm22, 3, 3, w) = -f * v[6 * (size_t)W];
        at(sp22, 3, 3, w) = f * v[7 * (size_t)W];
    }
    c->obs.fosm_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    return 0;
}

int mstm_hip_tmatrix_solution(mstm_hip_ctx *c, double eps, int niter, double conveps, int solver, double *tmat,
                              int64_t tmat_cap, double *sphere_qeff, double *qteff, double *order_log, int *t_order,
                              int *maxiter, double *maxerr, int *istat)
{
    if (!c || !c->nsph) return fail(c, MSTM_HIP_ESTATE, "tmatrix_solution: no spheres");
    if (c->obs.T < 1 || c->obs.torder.size() != (size_t)c->nsph)
        return fail(c, MSTM_HIP_ESTATE, "tmatrix_solution: no translation orders (mstm_hip_translation_orders)");
    if (niter <= 0) return fail(c, MSTM_HIP_EUNSUP, "tmatrix_solution: niter <= 0 not supported");
    if (solver != MSTM_HIP_SOLVE_PLAIN && solver != MSTM_HIP_SOLVE_MIXED)
        return fail(c, MSTM_HIP_EUNSUP, "tmatrix_solution: solver %d not available", solver);
    if (!tmat || !t_order || !maxiter || !maxerr || !istat) return fail(c, MSTM_HIP_EARG, "tmatrix_solution: null argument");
    if (c->Lmax > MSTM_MAX_L)
        return fail(c, MSTM_HIP_EUNSUP, "tmatrix_solution: sphere order %d > %d", c->Lmax, MSTM_MAX_L);
    const int T = c->obs.T;
    int64_t need = 0;
    for (int l = 1; l <= T; l++) need += (int64_t)4 * (2 * l + 1) * l * (l + 2);
    if (tmat_cap < need)
        return fail(c, MSTM_HIP_EARG, "tmatrix_solution: tmat holds %lld complex values, order %d needs %lld",
                    (long long)tmat_cap, T, (long long)need);
    HIPCHK(hipSetDevice(c->device));
    auto t0 = std::chrono::steady_clock::now();
    c->obs.x_valid = false;
    c->obs.a0_T = 0;
    const int n = c->neqns, nsph = c->nsph, bT = T * (T + 2);
    const size_t V = 2 * (size_t)n;
    double *b = c->d_kv + V * KV_B, *x = c->d_kv + V * KV_X;
    if (int rc = ensure_vccm(c, T, c->Lmax)) return rc;
    if (int rc = ensure_vccd(c, T, c->Lmax)) return rc;
    if (int rc = grow(c, &c->obs.d_dist, c->obs.dist_bytes, sizeof(double) * V * 2 * (2 * T + 1))) return rc;
    const size_t per_group = sizeof(double) * 8 * (size_t)bT;
    int G = std::min(nsph, 1024);
    G = (int)std::max<size_t>(1, std::min<size_t>((size_t)G, ((size_t)1 << 30) / per_group));
    if (int rc = grow(c, &c->obs.d_part, c->obs.part_bytes, per_group * G)) return rc;
    if (int rc = grow(c, &c->obs.d_a0, c->obs.a0_bytes, per_group)) return rc;
    if (int rc = grow(c, &c->obs.d_dq, c->obs.dq_bytes, sizeof(double) * 9 * nsph)) return rc;
    // Column pairs solved together (plain solver): the widest block of any
    // degree.  One allocation holds all that a block needs beyond a single
    // pair's (systems, efficiencies, merge of npm pairs at once), after
    // everything a single pair needs: without room for it the pairs go one by one.
    int np = 1, npm = 1;
    double *dq = c->obs.d_dq, *da0 = c->obs.d_a0, *dpart = c->obs.d_part;
    if (solver == MSTM_HIP_SOLVE_PLAIN) {
        if (!c->dop[MSTM_HIP_FP64].ready)
            if (int rc = mstm_hip_setup_direct(c, MSTM_HIP_FP64)) return rc;
        size_t need_blk = 0;
        for (int l = 1; l <= T; l++) {
            BicgBlock k = bicg_block_plan(c, 2 * l + 1);
            need_blk = std::max(need_blk, bicg_block_layout(c, nullptr, k));
            np = std::max(np, k.np);
        }
        npm = (int)std::max<size_t>(1, std::min<size_t>((size_t)np, ((size_t)1 << 28) / (per_group * G)));
        size_t o[4] = {(need_blk + 255) / 256 * 256};  // the block's systems, then efficiencies, merged columns, partials
        o[1] = o[0] + (sizeof(double) * 9 * nsph * np + 255) / 256 * 256;
        o[2] = o[1] + (per_group * np + 255) / 256 * 256;
        o[3] = o[2] + per_group * G * npm;
        if (np > 1 && (!c->obs.d_blk || c->obs.blk_bytes < o[3])) {
            dfree(c->obs.d_blk);
            c->obs.blk_bytes = 0;
            if (dalloc(&c->obs.d_blk, o[3]) == hipSuccess) c->obs.blk_bytes = o[3];
            else {
                (void)hipGetLastError();
                c->obs.d_blk = nullptr;
                np = npm = 1;
            }
        }
        if (np > 1) {
            dq = reinterpret_cast<double *>(c->obs.d_blk + o[0]);
            da0 = reinterpret_cast<double *>(c->obs.d_blk + o[1]);
            dpart = reinterpret_cast<double *>(c->obs.d_blk + o[2]);
        }
    }
    // vol_radius (mstm-input-37.f90:1205-1211): real(4) exponent .333333
    double vr = 0.0;
    for (int i = 0; i < nsph; i++) vr += c->radius[i] * c->radius[i] * c->radius[i];
    vr = std::pow(vr, (double).333333f);
    const double vr2 = vr * vr;
    // the copies of a block land in pinned memory, so that they are
    // asynchronous and the block waits for them only once
    const size_t nq = (size_t)9 * nsph * np, na0 = (size_t)8 * bT * np;
    const size_t pin_need = sizeof(double) * (nq + na0) + sizeof(BicgScal) * 2 * np;
    if (c->obs.pin_bytes < pin_need) {
        if (c->obs.h_pin) hipHostFree(c->obs.h_pin);
        c->obs.h_pin = nullptr;
        c->obs.pin_bytes = 0;
        HIPCHK(hipHostMalloc((void **)&c->obs.h_pin, pin_need, hipHostMallocDefault));
        c->obs.pin_bytes = pin_need;
    }
    double *hq = c->obs.h_pin, *ha0 = c->obs.h_pin + nq;
    BicgScal *hS = reinterpret_cast<BicgScal *>(ha0 + na0);
    std::vector<int> it(2 * (size_t)np);
    std::vector<double> err(2 * (size_t)np);
    std::vector<double> sq((size_t)3 * nsph, 0.0);
    double qt[3] = {0.0, 0.0, 0.0}, qeffold = 0.0;
    int64_t nt = 0;
    int lreach = T;
    *maxiter = 0;
    *maxerr = 0.0;
    *istat = 0;
    c->obs.tm_solves = 0;
    for (int l = 1; l <= T; l++) {
        const int b0 = l * (l + 2);
        HIPCHK(launch_distribute(l, c->d_order, c->d_offset, c->d_pos, nsph, c->Lmax, c->obs.r0, c->rimed,
                                 c->obs.d_vccd, c->obs.d_dist, n, std::min(nsph, 1024), c->st));
        // columns (k0, q = 1) and (k0, q = 2): pairs of independent systems,
        // one or a block of them solved together
        const BicgBlock plan = np > 1 ? bicg_block_plan(c, 2 * l + 1) : BicgBlock{};
        for (int k0 = -l; k0 <= l;) {
            const int nk = np > 1 ? std::min(plan.np, l + 1 - k0) : 1;
            const double *dp = c->obs.d_dist + V * 2 * (k0 + l);
            const double *xs = x;
            std::fill(it.begin(), it.end(), 0);
            std::fill(err.begin(), err.end(), 0.0);
            int rc = 0;
            if (np > 1) {
                BicgBlock k = plan;
                k.np = nk;
                bicg_block_layout(c, c->obs.d_blk, k);
                HIPCHK(launch_mie_mult(dp, k.b, nsph, c->d_order, c->d_offset, c->d_mieoff, c->d_an, 1, 0, c->Lmax,
                                       c->st, 2 * nk, (int64_t)V));
                HIPCHK(hipMemcpyAsync(k.x, k.b, sizeof(double) * 2 * V * nk, hipMemcpyDeviceToDevice, c->st));
                rc = bicg_block(c, k, niter, eps, hS, it.data(), err.data());
                xs = k.x;
            } else {
                HIPCHK(launch_mie_mult(dp, b, nsph, c->d_order, c->d_offset, c->d_mieoff, c->d_an, 1, 0, c->Lmax,
                                       c->st, 2, (int64_t)V));
                const double eps2[2] = {eps, eps};
                if (solver == MSTM_HIP_SOLVE_PLAIN) {
                    HIPCHK(hipMemcpyAsync(x, b, sizeof(double) * 2 * V, hipMemcpyDeviceToDevice, c->st));
                    rc = bicg2_dev(c, 2, niter, eps2, b, x, MSTM_HIP_FP64, 0, it.data(), err.data());
                } else {
                    HIPCHK(hipMemsetAsync(x, 0, sizeof(double) * 2 * V, c->st));
                    rc = refine2_dev(c, 2, niter, eps, b, x, 0, it.data(), err.data(), b);
                    for (int p = 0; p < 2 && !rc; p++)
                        if (err[p] >= eps && it[p] < niter) {
                            c->stats.lig_fallbacks++;
                            HIPCHK(hipMemcpyAsync(x + V * p, b + V * p, sizeof(double) * V, hipMemcpyDeviceToDevice,
                                                  c->st));
                            int it2 = 0;
                            rc = bicg2_dev(c, 1, niter - it[p], &eps, b + V * p, x + V * p, MSTM_HIP_FP64, 0, &it2,
                                           &err[p]);
                            it[p] += it2;
                        }
                }
            }
            if (rc) return rc;
            c->obs.tm_solves += 2 * nk;
            for (int q = 0; q < 2 * nk; q++) {
                *maxiter = std::max(*maxiter, it[q]);
                *maxerr = std::max(*maxerr, err[q]);
                if (it[q] > niter || err[q] > eps) *istat = 1;
            }
            // per-sphere efficiencies of each column (qefficiencyfactors, npol = 1)
            HIPCHK(launch_qeff(xs, dp, 2 * n, nsph, c->d_radius, c->d_order, c->d_offset, c->d_mieoff, c->d_an,
                               c->rimed, dq, c->st, nk));
            HIPCHK(hipMemcpyAsync(hq, dq, sizeof(double) * 9 * nsph * nk, hipMemcpyDeviceToHost, c->st));
            // the columns merged to the origin at order l (target orders min(l, torder_i))
            for (int p = 0; p < nk; p += npm)
                HIPCHK(launch_merge(xs + 2 * V * p, n, c->d_order, c->d_offset, c->obs.d_torder, c->d_pos, nsph, l,
                                    c->Lmax, c->obs.r0, c->rimed, c->obs.d_vccm, dpart, G,
                                    da0 + (size_t)8 * b0 * p, c->st, std::min(npm, nk - p)));
            HIPCHK(hipMemcpyAsync(ha0, da0, sizeof(double) * 8 * b0 * nk, hipMemcpyDeviceToHost, c->st));
            HIPCHK(hipStreamSynchronize(c->st));
            for (int p = 0; p < nk; p++, k0++)
                for (int q = 0; q < 2; q++) {
                    const double *hqp = hq + (size_t)9 * nsph * p;
                    for (int i = 0; i < nsph; i++)
                        for (int e = 0; e < 3; e++) sq[3 * i + e] += hqp[9 * i + 3 * (q + 1) + e];
                    const double *a0 = ha0 + 4 * (size_t)b0 * (2 * p + q);  // [mode][b0] complex
                    const double d1 = -2.0 / vr2 * a0[2 * ((size_t)q * b0 + amn(k0, l, l))];
                    double d3 = 0.0;
                    for (int e = 0; e < 2 * b0; e++) d3 += a0[2 * e] * a0[2 * e] + a0[2 * e + 1] * a0[2 * e + 1];
                    d3 *= 2.0 / vr2;
                    qt[0] += d1;
                    qt[1] += d1 - d3;
                    qt[2] += d3;
                    for (int nn = 1; nn <= l; nn++)
                        for (int m = -nn; m <= nn; m++)
                            for (int h = 0; h < 2; h++) {
                                const size_t e = (size_t)h * b0 + amn(m, nn, l);
                                tmat[2 * nt] = a0[2 * e];
                                tmat[2 * nt + 1] = a0[2 * e + 1];
                                nt++;
                            }
                }
        }
        double qe[2] = {0.0, 0.0};
        for (int i = 0; i < nsph; i++)
            for (int e = 0; e < 2; e++) qe[e] += sq[3 * i + e] * (c->radius[i] * c->radius[i]) / vr2;
        const double converr = qe[0] - qeffold;
        qeffold = qe[0];
        if (order_log) {
            order_log[4 * (l - 1)] = *maxiter;
            order_log[4 * (l - 1) + 1] = qe[0];
            order_log[4 * (l - 1) + 2] = qe[1];
            order_log[4 * (l - 1) + 3] = converr;
        }
        if (conveps > 0.0 && converr < conveps) {
            lreach = l;
            break;
        }
    }
    *t_order = lreach;
    if (sphere_qeff) std::memcpy(sphere_qeff, sq.data(), sizeof(double) * 3 * nsph);
    if (qteff) std::memcpy(qteff, qt, sizeof(qt));
    c->obs.tmatrix_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    collect_events(c);
    return 0;
}

}  // extern "C"
