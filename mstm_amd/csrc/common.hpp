// common.hpp -- shared device/host helpers for the MI355X MSTM hot path.
//
// Coefficient layout (matches MSTM's dense "model 2" packing so the Fortran
// host can pass its arrays straight through, mstm-modules-33.f90:2351-2377):
// a sphere of order L owns 2*L*(L+2) complex values, mode p (L/R helicity)
// major; inside a mode block (m,n) sits at
//     m >= 0 : (n-1)(L+2) + m          m < 0 : (-m-1)(L+2) + n + 1
// Inside kernels vectors are re-indexed "naturally" as nk = n(n+1)+k-1.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define MSTM_MAX_L 10  // largest sphere / node order with a compiled tile kernel
// largest order of a generated translation table (build_slot's per-thread
// arrays are sized by it): sphere orders of the pair tables and the node order
// of the FFT path's sphere<->node tables
#define MSTM_TAB_L 12
#define MSTM_SLOTS 16  // pair slots per tile step (and spheres per block)

#define MSTM_HD __host__ __device__ __forceinline__

template <typename T> struct cplx {
    T re, im;
};
template <typename T> MSTM_HD cplx<T> cmk(T r, T i) { return cplx<T>{r, i}; }
template <typename T> MSTM_HD cplx<T> cadd(cplx<T> a, cplx<T> b) { return {a.re + b.re, a.im + b.im}; }
template <typename T> MSTM_HD cplx<T> csub(cplx<T> a, cplx<T> b) { return {a.re - b.re, a.im - b.im}; }
template <typename T> MSTM_HD cplx<T> cmul(cplx<T> a, cplx<T> b)
{
    return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}
template <typename T> MSTM_HD cplx<T> cscale(cplx<T> a, T s) { return {a.re * s, a.im * s}; }
template <typename T> MSTM_HD cplx<T> cconj(cplx<T> a) { return {a.re, -a.im}; }
// a += b*c
template <typename T> MSTM_HD void cfma(cplx<T> &a, cplx<T> b, cplx<T> c)
{
    a.re = fma(b.re, c.re, a.re);
    a.re = fma(-b.im, c.im, a.re);
    a.im = fma(b.re, c.im, a.im);
    a.im = fma(b.im, c.re, a.im);
}
// a += s*c (real s)
template <typename T> MSTM_HD void crfma(cplx<T> &a, T s, cplx<T> c)
{
    a.re = fma(s, c.re, a.re);
    a.im = fma(s, c.im, a.im);
}
template <typename T> MSTM_HD cplx<T> cdiv(cplx<T> a, cplx<T> b)
{
    T d = b.re * b.re + b.im * b.im;
    return {(a.re * b.re + a.im * b.im) / d, (a.im * b.re - a.re * b.im) / d};
}

MSTM_HD constexpr int imx(int a, int b) { return a > b ? a : b; }
MSTM_HD constexpr int imn(int a, int b) { return a < b ? a : b; }
MSTM_HD constexpr int iab(int a) { return a < 0 ? -a : a; }

// MSTM model-2 address inside one mode block, 0-based
MSTM_HD constexpr int amn(int m, int n, int L) { return m >= 0 ? (n - 1) * (L + 2) + m : (-m - 1) * (L + 2) + n + 1; }
// natural index n(n+1)+k-1
MSTM_HD constexpr int nk(int n, int k) { return n * (n + 1) + k - 1; }
// m of the b-th axial block in the order 0,-1,1,-2,2,...
MSTM_HD constexpr int mblock_m(int b) { return b == 0 ? 0 : ((b & 1) ? -((b + 1) >> 1) : (b >> 1)); }

// ---------------------------------------------------------------------------
// Pair-table layout for a directed translation target order LT <- source LS
// (tables are shared by both directions of an unordered pair).  For each
// axial block m (order 0,-1,1,...,-nmin,nmin), m1 = max(1,|m|):
//   ROT  d^n(m,k), n = m1..max(LT,LS), k = -n..n           (reals)
//   AX   mode p=0,1: A(t,s), t = m1..LT fastest, s = m1..LS (complex)
// each section padded to the vector width VW (reals); then PHI (cos,sin).
// A(t,s) is the axial coefficient act(t,s,p) of axialtrancoefrecurrence
// (mstm-modules-33.f90:1566-1676) built with nmax = LT, lmax = LS.
// ---------------------------------------------------------------------------
MSTM_HD constexpr int pad_to(int x, int v) { return (x + v - 1) / v * v; }
MSTM_HD constexpr int rot_len(int m, int LT, int LS)
{
    int m1 = imx(1, iab(m)), s = 0;
    for (int n = m1; n <= imx(LT, LS); n++) s += 2 * n + 1;
    return s;
}
MSTM_HD constexpr int ax_len(int m, int LT, int LS)  // reals, one mode
{
    int m1 = imx(1, iab(m));
    return 2 * (LT - m1 + 1) * (LS - m1 + 1);
}
MSTM_HD constexpr int sec_len(int m, int LT, int LS, int VW)
{
    return pad_to(rot_len(m, LT, LS), VW) + 2 * pad_to(ax_len(m, LT, LS), VW);
}
MSTM_HD constexpr int sec_off(int b, int LT, int LS, int VW)
{
    int o = 0;
    for (int q = 0; q < b; q++) o += sec_len(mblock_m(q), LT, LS, VW);
    return o;
}
MSTM_HD constexpr int nmblocks(int LT, int LS) { return 2 * imn(LT, LS) + 1; }
MSTM_HD constexpr int phi_off(int LT, int LS, int VW) { return sec_off(nmblocks(LT, LS), LT, LS, VW); }
MSTM_HD constexpr int slot_len(int LT, int LS, int VW) { return phi_off(LT, LS, VW) + VW; }
// ---------------------------------------------------------------------------
// Compact pair-table layout of the direct tiles (LT = LS = L).  Four
// symmetries cut the full table to less than a third:
//   d^n(-m,-k) = (-1)^{m+k} d^n(m,k),  d^n(k,m) = (-1)^{m+k} d^n(m,k)
//   A_{-m}(t,s) of mode p = A_m(t,s) of the other mode (for m = 0 both modes
//   coincide),  A_m(s,t) = (-1)^{t+s} A_m(t,s)
// (d: Wigner d, A: axial coefficients).  Stored are, for n = 1..L,
//   E_n(m,k) = (-1)^m (d(m,k) + (-1)^k d(m,-k)) / 2   (k = 0: (-1)^m d(m,0)),
//   O_n(m,k) = (-1)^m (d(m,k) - (-1)^k d(m,-k)) / 2,
// m, k = 0..n (E) and 1..n (O), and for m = 0..L the blocks
//   B_m(t,s) = (-1)^t A_m(t,s), t, s = max(1,m)..L, of mode 0 and (m > 0) 1:
// all symmetric matrices, so only their triangles (row <= column, column by
// column).  With a_k = x_k + (-1)^k x_{-k}, b_k = x_k - (-1)^k x_{-k} (k > 0),
// a_0 = x_0, a translation runs as
//   u_k = cos(k phi) a_k + i sin(k phi) b_k,  v_k = cos b_k + i sin a_k,
//   Y+ = E u, Y- = O v (degree by degree);  p_m = Y+ + Y-, q_m = Y+ - Y-,
//   z_m = B_m p_m (own mode), z'_m = B_m q_m (other mode) (block by block);
//   P = E (z + z'), Q = O (z - z') (degree by degree; the same matrices),
//   (a_k, b_k of the result) / 2 = (-1)^t (cos P - i sin Q, cos Q - i sin P),
// and for k = 0 a_0 = (-1)^t P_0.  The reverse direction (translation by -r)
// is the same sequence on (-1)^n x with the two modes exchanged, its result
// exchanged back and multiplied by (-1)^t.
// ---------------------------------------------------------------------------
MSTM_HD constexpr int ctri(int i, int j) { return i <= j ? j * (j + 1) / 2 + i : i * (i + 1) / 2 + j; }
// rotation section: degree n holds E_n then O_n
MSTM_HD constexpr int crot_off(int n)
{
    int s = 0;
    for (int q = 1; q < n; q++) s += (q + 1) * (q + 1);
    return s;
}
MSTM_HD constexpr int crot_tot(int L) { return crot_off(L + 1); }
MSTM_HD constexpr int crot_o(int n) { return (n + 1) * (n + 2) / 2; }  // O_n after E_n
// axial section, in complex values: blocks m = L..0 (the small ones first),
// mode 0 then mode 1; then one more complex value (cos phi, sin phi)
MSTM_HD constexpr int cax_blk(int m, int L) { return (L - imx(1, m) + 1) * (L - imx(1, m) + 2) / 2; }
MSTM_HD constexpr int cax_off(int m, int p, int L)
{
    int o = 0;
    for (int q = L; q > m; q--) o += 2 * cax_blk(q, L);
    return o + p * cax_blk(m, L);
}
MSTM_HD constexpr int cax_tot(int L) { return cax_off(0, 1, L); }
// sections as stored: padded to whole 16-byte chunks, the chunks of a group's
// MSTM_SLOTS slots side by side (ilv), so that a slot's four lanes read one
// chunk and a wave MSTM_SLOTS consecutive ones
MSTM_HD constexpr int crot_pad(int L, int elem) { return pad_to(crot_tot(L), 16 / elem); }
MSTM_HD constexpr int direct_slot_len(int L, int elem)
{
    return crot_pad(L, elem) + pad_to(2 * (cax_tot(L) + 1), 16 / elem);
}
// element number of axial value c (real part) inside a slot
MSTM_HD constexpr int cax_elem(int c, int L, int elem) { return crot_pad(L, elem) + 2 * c; }
// order of the (a_k, b_k) values of one mode in the direct tiles' vectors:
// even degrees first, so that the (-1)^n of the reverse direction is a
// compare; per degree a_0, a_1, b_1, a_2, b_2, ...
MSTM_HD constexpr int cvec_even(int L)
{
    int s = 0;
    for (int q = 2; q <= L; q += 2) s += 2 * q + 1;
    return s;
}
MSTM_HD constexpr int cvec_deg(int n, int L)
{
    int s = (n & 1) ? cvec_even(L) : 0;
    for (int q = (n & 1) ? 1 : 2; q < n; q += 2) s += 2 * q + 1;
    return s;
}
MSTM_HD constexpr int cvec(int n, int k, int b, int L) { return cvec_deg(n, L) + (k ? 2 * k - 1 + b : 0); }
// complex values per unit of the direct tiles' vectors: 16 bytes (8 where a
// column of an odd order's FP32 values is no whole number of 16-byte units)
MSTM_HD constexpr int cvec_unit(int L, int elem) { return elem == 8 || (L & 1) ? 1 : 2; }

// columns per workgroup of a four-column product of the direct tiles: all
// four in one workgroup of four waves, or (FP64, and FP32 above order 4)
// two workgroups of two, the staged sources of four columns leaving one
// workgroup per CU
MSTM_HD constexpr int tile_cols4(int L, int elem) { return elem == 4 && L <= 4 ? 4 : 2; }

// interleaved position of element e (multiple-of-VW chunks) of slot k
MSTM_HD constexpr int64_t ilv(int64_t e, int k, int VW) { return ((e / VW) * MSTM_SLOTS + k) * VW + e % VW; }
