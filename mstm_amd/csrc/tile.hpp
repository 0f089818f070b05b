// tile.hpp -- pieces shared by the FP32 and FP64 direct tile kernels
// (tile32.hip, tile64.hip).  Work decomposition of a product H.a over all
// sphere pairs (external_to_external_expansion, mstm-modules-33.f90:
// 6390-6525):
//   * spheres are grouped in blocks of S = MSTM_SLOTS; a tile is an ordered
//     block pair (bI <= bJ); per column pair it has two waves;
//   * the first wave computes I <- J, the second J <- I from the same
//     tables; the compact layout of common.hpp makes the reverse direction
//     the same instruction sequence on sign-changed, mode-exchanged sources;
//   * four lanes (a quad) share a slot.  In step s slot k of the forward
//     wave targets I[k] and sources J[(k+s)%S]; slot k of the reverse wave
//     targets J[k] and sources I[(k-s)%S].  A lane's target never changes
//     inside a tile, so it accumulates in registers and writes one partial
//     sum per (target, partner block): no atomics, deterministic order;
//   * G workgroups share a tile (small clusters, G = 2..16): workgroup g
//     takes the steps [g S/G, (g+1) S/G) and writes its own partials;
//   * all waves of the tile copy a step's table group (16 slots) into LDS
//     once and read it there; the next step's group is loaded into registers
//     while the current step computes.
// Lane = slot (16) x (column, mode): a lane keeps its complex values in
// registers and takes every table value from the LDS copy of the step's
// group.  The tables being triangles of symmetric matrices (common.hpp), a
// degree's or block's triangle is read once per pass and each value serves
// both of its places.
// Vectors (xin, partial sums) are in "quad" layout: per column pair and
// sphere the complex values of a lane in a fixed order (cvec), in units of
// 16 bytes (cvec_unit), the units of the four lanes (column, mode) of a
// sphere side by side.
#pragma once
#include <utility>

#include "common.hpp"

template <typename F, int... Is>
__device__ __forceinline__ void sfor_impl(F &&f, std::integer_sequence<int, Is...>)
{
    (f(std::integral_constant<int, Is>{}), ...);
}
template <int N, typename F> __device__ __forceinline__ void static_for(F &&f)
{
    sfor_impl(f, std::make_integer_sequence<int, N>{});
}

typedef float f32x4 __attribute__((ext_vector_type(4)));

template <typename T> struct vec16;
template <> struct vec16<float> {
    typedef f32x4 type;
};
template <> struct vec16<double> {
    typedef double type __attribute__((ext_vector_type(2)));
};

// copy of a step's table group, 16 bytes per thread and load: all of this
// thread's loads are in flight at once.  Each group is read once from HBM
// and, where two workgroups of one XCD share the tile, once more from its L2.
template <typename T, int L, int NT> struct GroupCopy {
    static constexpr int NV = direct_slot_len(L, sizeof(T)) * MSTM_SLOTS * (int)sizeof(T) / 16;
    static constexpr int NQ = (NV + NT - 1) / NT;
    f32x4 r[NQ];
    __device__ __forceinline__ void load(const T *__restrict__ tab, int64_t group)
    {
        const f32x4 *g = reinterpret_cast<const f32x4 *>(tab + group * direct_slot_len(L, sizeof(T)) * MSTM_SLOTS);
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            const int i = threadIdx.x + q * NT;
            if ((q + 1) * NT <= NV || i < NV) r[q] = __builtin_nontemporal_load(&g[i]);
        }
    }
    __device__ __forceinline__ void store(T *__restrict__ grp) const
    {
        f32x4 *d = reinterpret_cast<f32x4 *>(grp);
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            const int i = threadIdx.x + q * NT;
            if ((q + 1) * NT <= NV || i < NV) d[i] = r[q];
        }
    }
};

template <typename T, int L, int NRL> struct TileShape {
    static constexpr int S = MSTM_SLOTS;
    static constexpr int NB = L * (L + 2);
    static constexpr int UC = cvec_unit(L, sizeof(T));
    static constexpr int RP = NRL / 2;  // column pairs of a workgroup
    // complex values per staged sphere and column pair, 64 bytes (one unit of
    // each lane) apart in the LDS banks for the slots of one read
    static constexpr int SPH = 4 * NB + (4 * NB * 2 * (int)sizeof(T) % 256 == 0 ? 64 / (2 * (int)sizeof(T)) : 0);
    // the two source blocks sit in LDS for the whole tile up to order 4
    // (FP64) / 6 (FP32); above, they would leave one workgroup of two waves
    // per CU
    static constexpr bool STAGED = L <= (sizeof(T) == 8 ? 4 : 6);
    // the next step's table group is loaded into registers while the current
    // step computes, where they are not needed to keep the step out of scratch
    static constexpr bool PIPE = sizeof(T) == 4 || L <= 4;
    static constexpr int SRC = STAGED ? 2 * RP * S * SPH : 1;
    static constexpr int GRP = direct_slot_len(L, sizeof(T)) * S;
};

// LEN elements of a slot from element E0 on (the 16-byte chunks that cover
// them); gs: the group at the slot's place in a chunk row
template <typename T, int E0, int LEN> __device__ __forceinline__ void load_span(const T *__restrict__ gs, T *r)
{
    constexpr int VW = 16 / sizeof(T);
    typedef typename vec16<T>::type V;
#pragma unroll
    for (int c = E0 / VW; c <= (E0 + LEN - 1) / VW; c++) {
        const V v = *reinterpret_cast<const V *>(gs + c * VW * MSTM_SLOTS);
#pragma unroll
        for (int q = 0; q < VW; q++) {
            const int e = c * VW + q - E0;
            if (e >= 0 && e < LEN) r[e] = v[q];
        }
    }
}
// y = A b, A symmetric N x N (triangle a), real
template <typename T, int N> __device__ __forceinline__ void symv(const T *a, const cplx<T> (&b)[N], cplx<T> (&y)[N])
{
#pragma unroll
    for (int r = 0; r < N; r++) {
        y[r] = cscale(b[0], a[ctri(r, 0)]);
#pragma unroll
        for (int k = 1; k < N; k++) crfma(y[r], a[ctri(r, k)], b[k]);
    }
}
// the same, A complex (triangle a as re, im pairs)
template <typename T, int N> __device__ __forceinline__ void symz(const T *a, const cplx<T> (&b)[N], cplx<T> (&z)[N])
{
#pragma unroll
    for (int r = 0; r < N; r++) {
        z[r] = cmul(cmk(a[2 * ctri(r, 0)], a[2 * ctri(r, 0) + 1]), b[0]);
#pragma unroll
        for (int k = 1; k < N; k++) cfma(z[r], cmk(a[2 * ctri(r, k)], a[2 * ctri(r, k) + 1]), b[k]);
    }
}

// Copy the tile's two source blocks to LDS (block 0: J, sources of the forward
// waves; block 1: I, sources of the reverse waves, odd degrees negated), all
// threads, 16 bytes each; visible after the first step's barrier.  rp0: the
// workgroup's first column pair.
template <typename T, int L, int NRL>
__device__ __forceinline__ void stage_sources(int2 bt, int rp0, const cplx<T> *__restrict__ xin, int npad,
                                              cplx<T> *__restrict__ srcs)
{
    typedef TileShape<T, L, NRL> H;
    typedef typename vec16<T>::type V;
    constexpr int S = H::S, NB = H::NB, UC = H::UC, RP = H::RP, NE = cvec_even(L), VZ = 8 / (int)sizeof(T);
    constexpr int U = 4 * NB / VZ;  // 16-byte chunks of a sphere and column pair, VZ complex values each
#pragma unroll 9
    for (int e = threadIdx.x; e < 2 * RP * S * U; e += 64 * NRL) {
        const int c = e % U, i = (e / U) % S, r = (e / (U * S)) % RP, b = e / (U * S * RP);
        V v = reinterpret_cast<const V *>(xin +
                                          ((int64_t)((rp0 + r) * npad) + (b ? bt.x : bt.y) * S + i) * (4 * NB))[c];
        const int idx = c * VZ / (4 * UC) * UC;  // of the chunk's first value
        if (b) {
#pragma unroll
            for (int q = 0; q < VZ; q++)
                if (idx + (UC == 2 ? q : 0) >= NE) {
                    v[2 * q] = -v[2 * q];
                    v[2 * q + 1] = -v[2 * q + 1];
                }
        }
        reinterpret_cast<V *>(srcs + ((b * RP + r) * S + i) * H::SPH)[c] = v;
    }
}

template <typename T, int L, int NR, int NRL>
__device__ __forceinline__ void tile_wave(int2 bt, int tile, const T *__restrict__ tab, cplx<T> *__restrict__ part,
                                            int npad, int rp, int rpl, bool dir, T *__restrict__ grp,
                                            cplx<T> *__restrict__ srcs, const cplx<T> *__restrict__ xin, int s0, int s1,
                                            int G, int g)
{
    typedef cplx<T> Z;
    typedef TileShape<T, L, NRL> H;
    typedef typename vec16<T>::type V;
    constexpr int S = H::S, NB = H::NB, UC = H::UC, VW = 16 / (int)sizeof(T), YN = L * (L + 3) / 2;
    const int lane = threadIdx.x & 63, kslot = lane >> 2, j = lane & 3, md = lane & 1;
    const bool diag = bt.x == bt.y;

    Z W[NB];  // (a_k, b_k) / 2 of the result
#pragma unroll
    for (int q = 0; q < NB; q++) W[q] = cmk((T)0, (T)0);

    GroupCopy<T, L, 64 * NRL> pre;
    if constexpr (H::PIPE) pre.load(tab, (int64_t)tile * S + s0);
    if constexpr (H::STAGED) stage_sources<T, L, NRL>(bt, rp - rpl, xin, npad, srcs);

#pragma unroll 1
    for (int s = s0; s < s1; s++) {
        __syncthreads();
        if constexpr (!H::PIPE) pre.load(tab, (int64_t)tile * S + s);
        pre.store(grp);
        if constexpr (H::PIPE)
            if (s + 1 < s1) pre.load(tab, (int64_t)tile * S + s + 1);
        __syncthreads();
        if (diag && (dir || s == 0)) continue;
        const int slot = dir ? (kslot - s) & (S - 1) : kslot;
        const int src = dir ? slot : (kslot + s) & (S - 1);
        const T *gs = grp + VW * slot;
        const Z *xl = (H::STAGED ? srcs + ((dir ? H::RP * S : 0) + rpl * S + src) * H::SPH
                                 : xin + ((int64_t)rp * npad + (dir ? bt.x : bt.y) * S + src) * (4 * NB)) +
                      (dir ? j ^ 1 : j) * UC;
        auto x = [&](int n, int k, int b) -> Z {
            const int q = cvec(n, k, b, L);
            const Z v = xl[(q / UC) * 4 * UC + q % UC];
            return !H::STAGED && dir && (n & 1) ? cmk(-v.re, -v.im) : v;
        };
        T c[L + 1], sn[L + 1];  // cos(k phi), sin(k phi)
        {
            T e1[2];
            load_span<T, cax_elem(cax_tot(L), L, sizeof(T)), 2>(gs, e1);
            c[0] = (T)1;
            sn[0] = (T)0;
#pragma unroll
            for (int k = 1; k <= L; k++) {
                c[k] = c[k - 1] * e1[0] - sn[k - 1] * e1[1];
                sn[k] = c[k - 1] * e1[1] + sn[k - 1] * e1[0];
            }
        }
        // Y+, Y- of (n, m); after the axial pass z + z', z - z'
        Z Yp[YN], Ym[YN];
        auto ip = [](int n, int m) { return n * (n + 1) / 2 - 1 + m; };
        // ---- forward rotation, degree by degree
        static_for<L>([&](auto nm) {
            constexpr int n = decltype(nm)::value + 1;
            Z u[n + 1], v[n], y[n + 1], w[n];
            u[0] = x(n, 0, 0);
#pragma unroll
            for (int k = 1; k <= n; k++) {
                const Z a = x(n, k, 0), b = x(n, k, 1);
                u[k] = cmk(c[k] * a.re - sn[k] * b.im, c[k] * a.im + sn[k] * b.re);
                v[k - 1] = cmk(c[k] * b.re - sn[k] * a.im, c[k] * b.im + sn[k] * a.re);
            }
            T e[crot_o(n)], o[n * (n + 1) / 2];
            load_span<T, crot_off(n), crot_o(n)>(gs, e);
            symv<T, n + 1>(e, u, y);
            load_span<T, crot_off(n) + crot_o(n), n *(n + 1) / 2>(gs, o);
            symv<T, n>(o, v, w);
#pragma unroll
            for (int m = 0; m <= n; m++) Yp[ip(n, m)] = y[m];
#pragma unroll
            for (int m = 1; m <= n; m++) Ym[ip(n, m)] = w[m - 1];
        });
        // the back pass reloads its matrices from LDS rather than keeping the
        // forward pass's copies live across the axial products
        asm volatile("" ::: "memory");
        // ---- axial products, block by block
        static_for<L + 1>([&](auto mc) {
            constexpr int m = decltype(mc)::value;
            constexpr int m1 = imx(1, m), N = L - m1 + 1;
            constexpr int NT = N * (N + 1), E0 = cax_elem(cax_off(m, 0, L), L, sizeof(T));
            Z b[N], z[N];
            T a[NT];
            if constexpr (m == 0) {
#pragma unroll
                for (int q = 0; q < N; q++) b[q] = Yp[ip(q + 1, 0)];
                load_span<T, E0, NT>(gs, a);
                symz<T, N>(a, b, z);
#pragma unroll
                for (int q = 0; q < N; q++) Yp[ip(q + 1, 0)] = z[q];
            } else {
                // own mode: p_m = Y+ + Y-; the other mode: q_m = Y+ - Y-.  Both
                // triangles are read by every lane at the same place and the
                // lane's mode picks
                Z b2[N], z2[N];
#pragma unroll
                for (int q = 0; q < N; q++) {
                    b[q] = cadd(Yp[ip(q + m1, m)], Ym[ip(q + m1, m)]);
                    b2[q] = csub(Yp[ip(q + m1, m)], Ym[ip(q + m1, m)]);
                }
                constexpr int step = NT % VW == 0 ? NT / VW * VW * S : 0;
                if constexpr (NT % VW == 0) {
                    load_span<T, E0, NT>(gs + (md ? step : 0), a);
                    symz<T, N>(a, b, z);
                    load_span<T, E0, NT>(gs + (md ? 0 : step), a);
                    symz<T, N>(a, b2, z2);
                } else {
                    T a1[NT];
                    load_span<T, E0, NT>(gs, a);
                    load_span<T, E0 + NT, NT>(gs, a1);
#pragma unroll
                    for (int q = 0; q < NT; q++) {
                        const T own = md ? a1[q] : a[q];
                        a1[q] = md ? a[q] : a1[q];
                        a[q] = own;
                    }
                    symz<T, N>(a, b, z);
                    symz<T, N>(a1, b2, z2);
                }
#pragma unroll
                for (int q = 0; q < N; q++) {
                    Yp[ip(q + m1, m)] = cadd(z[q], z2[q]);
                    Ym[ip(q + m1, m)] = csub(z[q], z2[q]);
                }
            }
        });
        asm volatile("" ::: "memory");
        // ---- back rotation and output phase, degree by degree
        static_for<L>([&](auto nm) {
            constexpr int t = decltype(nm)::value + 1;
            Z za[t + 1], zb[t], P[t + 1], Q[t];
#pragma unroll
            for (int m = 0; m <= t; m++) za[m] = Yp[ip(t, m)];
#pragma unroll
            for (int m = 1; m <= t; m++) zb[m - 1] = Ym[ip(t, m)];
            T e[crot_o(t)], o[t * (t + 1) / 2];
            load_span<T, crot_off(t), crot_o(t)>(gs, e);
            symv<T, t + 1>(e, za, P);
            load_span<T, crot_off(t) + crot_o(t), t *(t + 1) / 2>(gs, o);
            symv<T, t>(o, zb, Q);
            W[cvec(t, 0, 0, L)] = cadd(W[cvec(t, 0, 0, L)], P[0]);
#pragma unroll
            for (int k = 1; k <= t; k++) {
                Z &wa = W[cvec(t, k, 0, L)], &wb = W[cvec(t, k, 1, L)];
                const Z q = Q[k - 1];
                wa.re = fma(c[k], P[k].re, fma(sn[k], q.im, wa.re));
                wa.im = fma(c[k], P[k].im, fma(-sn[k], q.re, wa.im));
                wb.re = fma(c[k], q.re, fma(sn[k], P[k].im, wb.re));
                wb.im = fma(c[k], q.im, fma(-sn[k], P[k].re, wb.im));
            }
        });
    }
    if (diag && dir) return;
    // partial of (target, partner block): forward (-1)^t, reverse with the
    // modes exchanged back (its (-1)^t cancels the table's)
    constexpr int NE = cvec_even(L);
    const int tgt = (dir ? bt.y : bt.x) * S + kslot;
    const int partner = (dir ? bt.x : bt.y) * G + g;  // one partial per (partner block, step group)
    typedef T U __attribute__((ext_vector_type(2 * UC)));
    U *out = reinterpret_cast<U *>(part + (((int64_t)partner * (NR / 2) + rp) * npad + tgt) * (4 * NB)) +
             (dir ? j ^ 1 : j);
#pragma unroll
    for (int q = 0; q < NB; q += UC) {
        U v;
#pragma unroll
        for (int i = 0; i < UC; i++) {
            const bool neg = !dir && q + i >= NE;
            v[2 * i] = neg ? -W[q + i].re : W[q + i].re;
            v[2 * i + 1] = neg ? -W[q + i].im : W[q + i].im;
        }
        out[(q / UC) * 4] = v;
    }
}

// What bounds the tiles (MI355X, 5000 spheres of order 4, 12.5 M pairs):
//   FP32, two columns: 2.77 ms.  A step is about 960 vector instructions: at
//   four cycles each and 2.4 GHz they issue during 89% of the launch (counted,
//   profiles/direct_tile_cfg5_sq_counters.txt); HBM moves 9.7 GB, 3.5 TB/s.
//   With the half tables of the former layout (992 bytes per pair,
//   now 624; phases applied to every coefficient) it was 3.68 ms.  The same
//   step on v_mfma_f32_4x4x1 (one small matrix per slot) ran 3.71 ms: those
//   MFMAs take 8.2 cycles, do not overlap with vector work and cost 8 more at
//   every switch.
//   FP64, two / four columns: 6.3 / 11.8 ms (8.8 / 16.0 before): one wave per
//   SIMD (71 KB of LDS per workgroup of two waves), so latency shows: vector
//   instructions issue during 41-44% of the launch, LDS is active 31-33% of it.
//   Sources read from L2 with two waves per SIMD instead: 14% slower.
//   FP64 orders 5..8 spill less without the register prefetch (order 6,
//   801 spheres, four columns: 2.32 -> 1.61 ms; 20.3 ms with the full tables of
//   the former layout).
// waves per SIMD the compiler schedules for (order 5 in FP32 spills 8 registers
// for its second wave and is 13% faster for it)
template <typename T, int L> constexpr int tile_waves() { return sizeof(T) == 4 && L <= 5 ? 2 : 1; }

// NR columns (2 or 4) of the product, NRL of them per workgroup (two waves
// per column pair).  Four columns run as one workgroup of four waves, or as
// two workgroups of two (NRL = 2) where the staged sources of four columns
// would leave one workgroup per CU.  The two are numbered 8 apart: workgroups
// are dealt to MI355X's 8 XCDs round robin, so they run on one XCD and the
// second reads the table group from its L2.  nq sets of columns (a block
// of BiCG systems; sources, partials and gates one set after the other) are
// further workgroups of that kind: all sets of a unit run side by side.
template <typename T, int L, int NR, int NRL>
__global__ __launch_bounds__(64 * NRL) __attribute__((amdgpu_waves_per_eu(tile_waves<T, L>()))) void tile_kernel(
    const T *__restrict__ tab, const int2 *__restrict__ tiles, int nunits, const T *__restrict__ xin,
    T *__restrict__ part, int npad, int G, int nq, const int *__restrict__ gate)
{
    typedef cplx<T> Z;
    typedef TileShape<T, L, NRL> H;
    typedef typename vec16<T>::type V;
    constexpr int S = H::S, RP = H::RP;
    constexpr int NH = NR / NRL;  // workgroups per (tile, step group)
    int u = blockIdx.x, h = 0;
    if (NH * nq > 1) {
        const int sub = (int)(blockIdx.x / 8) % (NH * nq);
        u = (int)(blockIdx.x / (8 * NH * nq)) * 8 + (int)(blockIdx.x % 8);
        if (u >= nunits) return;  // the grid is padded to whole groups of 8 NH nq
        h = sub % NH;
        const int q = sub / NH;
        const int64_t col = (int64_t)NR * 4 * npad * L * (L + 2);  // one set of sources, or one partial
        xin += q * col;
        part += q * col * (npad / MSTM_SLOTS) * G;
        if (gate) gate += q;
    }
    if (gate && !*gate) return;  // the issuing solver has stopped every system of the set
    const int tile = u / G, g = u - tile * G;
    const int s0 = g * (S / G), s1 = s0 + S / G;
    const int2 bt = tiles[tile];
    const int w = threadIdx.x >> 6;
    __shared__ __attribute__((aligned(16))) T grp[H::GRP];
    __shared__ __attribute__((aligned(16))) T srcs[2 * H::SRC];
    tile_wave<T, L, NR, NRL>(bt, tile, tab, reinterpret_cast<Z *>(part), npad, h * RP + (w >> 1), w >> 1, w & 1, grp,
                            reinterpret_cast<Z *>(srcs), reinterpret_cast<const Z *>(xin), s0, s1, G, g);
}

template <typename T, int L>
static hipError_t tile_launch(const T *tab, const int2 *tiles, int ntiles, const T *x, T *p, int npad, int nr, int G,
                              int nq, hipStream_t st, const int *gate)
{
    constexpr int NRL = tile_cols4(L, sizeof(T));
    const int nu = ntiles * G;
    auto grid = [&](int per) { return dim3((unsigned)(per == 1 ? nu : (nu + 7) / 8 * 8 * per)); };
    if (nr == 2)
        hipLaunchKernelGGL((tile_kernel<T, L, 2, 2>), grid(nq), dim3(128), 0, st, tab, tiles, nu, x, p, npad, G, nq,
                           gate);
    else
        hipLaunchKernelGGL((tile_kernel<T, L, 4, NRL>), grid(nq * (4 / NRL)), dim3(64 * NRL), 0, st, tab, tiles, nu, x,
                           p, npad, G, nq, gate);
    return hipGetLastError();
}

template <typename T>
static hipError_t tile_dispatch(const T *tab, const int2 *tiles, int ntiles, int L, const T *xin, T *partial, int npad,
                                int nr, int G, int nq, hipStream_t st, const int *gate)
{
    if ((nr != 2 && nr != 4) || nq < 1) return hipErrorInvalidValue;
    if (G < 1 || G > MSTM_SLOTS || MSTM_SLOTS % G) return hipErrorInvalidValue;
    switch (L) {
#define CASE(LL)                                                                                                       \
    case LL: return tile_launch<T, LL>(tab, tiles, ntiles, xin, partial, npad, nr, G, nq, st, gate);
#ifdef MSTM_TILE_L_ONLY
        CASE(MSTM_TILE_L_ONLY)
#else
        CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7) CASE(8)
#endif
#undef CASE
    default: return hipErrorInvalidValue;
    }
}
