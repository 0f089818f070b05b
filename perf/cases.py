"""Performance cases: what a user of this package has it compute, through
its public entry points (mstm_amd.solver.HipContext, mstm_amd.batch.BatchSolver).

Every case is a dict of plain values; its "kind" is the entry point:

  solve    fixedorsoln on a cluster whose operator is set up: one incident
           plane wave, both polarizations, to the reference's |r|^2/|b|^2 < eps
  product  sphereinteraction, one application of I - (A a) for a host program
           that keeps its own solver: host vectors in, host vectors out
  config   a new configuration of a configuration average: sphere data in,
           Mie coefficients, pair tables, mixed solve, scattering matrix out
  tmatrix  tmatrix_solution: the cluster T-matrix, every order to convergence
  lu       fixedorsoln's direct branch, matrix built and factored in the call
  batch    many clusters x many incidences at once

`exact` computes the same quantities in FP64 from the addition theorem written
as an expansion in scalar waves: H_ij = sum_wv C_wv h_w(r) Y_wv, C from
Clebsch-Gordan coefficients, applied as one matrix product, with GMRES to a
residual far below the solver's criterion.  It shares no code and no
factorization (rotation, axial translation, FFT) with the package.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from mstm_amd import geometry
from mstm_amd.batch import BatchSolver
from mstm_amd.solver import (FP32, FP64, FP64_FP32, SOLVE_LEARNED, SOLVE_LU, SOLVE_MIXED, SOLVE_PLAIN, HipContext,
                             scattering_angles)

SOLVERS = {"plain": SOLVE_PLAIN, "mixed": SOLVE_MIXED, "learned": SOLVE_LEARNED}


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # a quick look at a handful of particles: nothing but latency and launches
        dict(name="solve_20", kind="solve", shape="sphere", n=20, x=2.0, spread=0.0, fv=0.10, mr=1.5, mi=0.01,
             beta=0.0, alpha=0.0, solver="plain", fft=False),
        # an everyday cluster of unequal spheres (orders 2 to 6 mixed), oblique incidence, default solver
        dict(name="solve_233_mixed_sizes", kind="solve", shape="sphere", n=233, x=1.3, spread=0.5, fv=0.15, mr=1.6,
             mi=0.0123, beta=0.7, alpha=0.4, solver="plain", fft=False),
        # the default FP64 solver (the reference's own iterates) on a large dense cluster
        dict(name="solve_1501_plain", kind="solve", shape="sphere", n=1501, x=2.0, spread=0.0, fv=0.25, mr=1.31,
             mi=0.0, beta=0.3, alpha=1.0, solver="plain", fft=False),
        # the headline workload: 5000 spheres, learned start, mixed precision
        dict(name="solve_5000_learned", kind="solve", shape="sphere", n=5000, x=2.0, spread=0.0, fv=0.30, mr=1.31,
             mi=0.0, beta=0.0, alpha=0.0, solver="learned", fft=False),
        # FFT path, deep orders: the x = 3 cylinder, node order 9
        dict(name="fft_cylinder_1000", kind="solve", shape="cylinder", n=1000, x=3.0, spread=0.0, fv=0.25, mr=1.6,
             mi=0.02, beta=0.0, alpha=0.0, solver="mixed", fft=True),
        # FFT path, many small spheres: one orientation of a soot-like aggregate
        dict(name="fft_aggregate_2000", kind="solve", shape="fractal", n=2000, x=0.5, spread=0.0, fv=0.0, mr=1.75,
             mi=0.4, beta=1.1, alpha=2.0, solver="mixed", fft=True),
        # a host program with its own BiCG: A p and A^H w in FP64
        dict(name="product_2999_fp64", kind="product", n=2999, x=2.0, spread=0.0, fv=0.25, mr=1.31, mi=0.0,
             precision="fp64", ncol=2),
        # the same at FP32 for two right-hand sides, larger spheres (order 6)
        dict(name="product_801_fp32", kind="product", n=801, x=3.5, spread=0.1, fv=0.20, mr=1.33, mi=0.001,
             precision="fp32", ncol=4),
        # one member of a configuration average: everything is new in each call
        dict(name="config_700", kind="config", n=700, x=1.5, spread=0.0, fv=0.20, mr=1.6, mi=0.0123),
        # random-orientation properties of a cluster: the whole T-matrix
        dict(name="tmatrix_200", kind="tmatrix", n=200, x=1.0, spread=0.0, fv=0.20, mr=1.5, mi=0.01),
        # resonant cluster through the direct solver (8400 equations)
        dict(name="lu_120", kind="lu", n=120, x=2.0, spread=0.0, fv=0.20, mr=1.31, mi=0.01),
        # a data set: clusters of 10 to 200 spheres, 32 incidences each
        dict(name="batch_16", kind="batch", ncl=16, nmin=10, nmax=200, xmin=0.5, xmax=3.0, ndir=32, mr=1.33,
             mi=0.001),
    ]


def draw(rng):
    def logint(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))

    def r2(a, b):
        return round(rng.uniform(a, b), 2)

    kind = rng.choice(["solve", "solve", "solve", "fft", "fft", "product", "product", "config", "tmatrix", "lu",
                       "batch"])
    mr, mi = rng.choice([(1.31, 0.0), (1.33, 0.001), (1.5, 0.01), (1.6, 0.0123)])
    if kind == "solve":
        solver = rng.choice(["plain", "plain", "mixed", "learned"])
        if solver == "learned":  # what the shipped network was trained on
            return dict(kind="solve", shape="sphere", n=logint(200, 4000), x=2.0, spread=0.0, fv=r2(0.2, 0.3), mr=1.31,
                        mi=0.0, beta=0.0, alpha=0.0, solver="learned", fft=False)
        n = logint(20, 1500)
        return dict(kind="solve", shape="sphere", n=n, x=r2(0.5, 2.0), spread=rng.choice([0.0, 0.0, 0.3]),
                    fv=r2(0.05, 0.25), mr=mr, mi=mi, beta=r2(0.0, 1.5), alpha=r2(0.0, 3.0), solver=solver, fft=False)
    if kind == "fft":
        if rng.random() < 0.5:
            return dict(kind="solve", shape="cylinder", n=logint(250, 1000), x=r2(1.0, 3.0), spread=0.0, fv=0.25,
                        mr=1.6, mi=0.02, beta=r2(0.0, 1.5), alpha=r2(0.0, 3.0),
                        solver=rng.choice(["plain", "mixed"]), fft=True)
        return dict(kind="solve", shape="fractal", n=logint(250, 2000), x=r2(0.3, 0.8), spread=0.0, fv=0.0, mr=1.75,
                    mi=0.4, beta=r2(0.0, 1.5), alpha=r2(0.0, 3.0), solver=rng.choice(["plain", "mixed"]), fft=True)
    if kind == "product":
        x = r2(0.5, 3.5)
        return dict(kind="product", n=logint(30, 3000 if x <= 2.0 else 800), x=x, spread=rng.choice([0.0, 0.1]),
                    fv=r2(0.05, 0.25), mr=mr, mi=mi, precision=rng.choice(["fp64", "fp32"]),
                    ncol=rng.choice([1, 2, 4]))
    if kind == "config":
        return dict(kind="config", n=logint(50, 1500), x=r2(0.5, 2.0), spread=rng.choice([0.0, 0.2]),
                    fv=r2(0.05, 0.25), mr=mr, mi=mi)
    if kind == "tmatrix":
        return dict(kind="tmatrix", n=logint(10, 200), x=r2(0.3, 1.0), spread=rng.choice([0.0, 0.2]),
                    fv=r2(0.10, 0.25), mr=mr, mi=mi)
    if kind == "lu":
        return dict(kind="lu", n=logint(10, 120), x=r2(0.5, 2.0), spread=rng.choice([0.0, 0.2]), fv=r2(0.10, 0.25),
                    mr=mr, mi=mi)
    return dict(kind="batch", ncl=rng.randint(3, 16), nmin=10, nmax=logint(30, 200), xmin=0.5, xmax=r2(1.0, 3.0),
                ndir=rng.choice([5, 16, 32]), mr=1.33, mi=0.001)


# ---------------------------------------------------------------------------
# sphere data from the seed
# ---------------------------------------------------------------------------
def _rsa(rng, radius, sample):
    """Random sequential addition, 512 candidates at a time; None if it jams."""
    n, a = len(radius), radius[0]
    pos = np.zeros((n, 3))
    k = 0
    # equal spheres: cells that hold one centre at most, so that a candidate
    # is tested against the cells around it only
    equal = radius[-1] == a
    if equal:
        side = 2.0 * a / math.sqrt(3.0)
        off = np.stack(np.meshgrid(*[np.arange(-2, 3)] * 3, indexing="ij"), -1).reshape(-1, 3)
        half = int(np.abs(sample(np.random.default_rng(0), 4096)).max() * 1.05 / side) + 4
        grid = np.full((2 * half + 1,) * 3, -1, np.int64)
    for _ in range(40 + n // 5):
        c = sample(rng, 512)
        a = radius[k]
        ok = np.ones(len(c), bool)
        if equal:
            q = np.floor(c / side).astype(int) + half
            at = q[:, None] + off[None]
            near = grid[at[..., 0], at[..., 1], at[..., 2]]
            ok = ((near < 0) | (((c[:, None] - pos[near]) ** 2).sum(2) >= 4.0 * a * a)).all(1)
        elif k:
            p, d = pos[:k], (radius[:k] + a) ** 2
            ok = ((c * c).sum(1)[:, None] + (p * p).sum(1)[None] - 2.0 * (c @ p.T) >= d[None]).all(1)
        first = k
        for i in np.flatnonzero(ok):
            if radius[k] != a:
                break  # the candidates were tested for this radius
            if ((pos[first:k] - c[i]) ** 2).sum(1).min(initial=1e300) >= 4.0 * a * a:
                pos[k] = c[i]
                if equal:
                    grid[tuple(q[i])] = k
                k += 1
                if k == n:
                    return pos
    return None


def _cluster(case, seed, n=None, x=None, fv=None):
    """(pos, radius, ri): spheres of size parameter x (spread: relative half
    width of a uniform size distribution) in the case's bounding shape."""
    n, x, fv = n or case["n"], x or case["x"], fv or case["fv"]
    rng = np.random.default_rng([seed, n])
    ri = np.full(n, complex(case["mr"], case["mi"]))
    shape = case.get("shape", "sphere")
    if shape == "fractal":
        return geometry.fractal_aggregate(n, x, 1.8, 1.3, seed=seed, ri=ri[0]).pos, np.full(n, x), ri
    s = case.get("spread", 0.0)
    # sizes in 8 classes, largest first
    radius = x * (1.0 + s * (1.0 - 2.0 * np.floor(8.0 * np.arange(n) / n) / 7.0))
    vol = (radius ** 3).sum() / fv
    a = radius[0]
    for grow in range(40):
        if shape == "cylinder":
            rc = (vol / 3.0) ** (1.0 / 3.0) * 1.03 ** grow

            def sample(r, m):
                rr, th = (rc - a) * np.sqrt(r.random(m)), 2.0 * np.pi * r.random(m)
                return np.stack([rr * np.cos(th), rr * np.sin(th), (4.0 * rc - 2.0 * a) * (r.random(m) - 0.5)], 1)
        else:
            R = vol ** (1.0 / 3.0) * 1.03 ** grow

            def sample(r, m):
                v = r.normal(size=(m, 3))
                return v * ((max(R - a, 0.1 * a) * r.random(m) ** (1.0 / 3.0)) / np.sqrt((v * v).sum(1)))[:, None]

        pos = _rsa(rng, radius, sample)
        if pos is not None:
            p = np.random.default_rng([seed, 7]).permutation(n)  # sizes in no order
            return pos[p], radius[p], ri
    raise RuntimeError("no room for the spheres")


def _batch_clusters(case, seed):
    rng = np.random.default_rng([case["ncl"], case["nmax"]])  # the sizes are the case's, the positions the seed's
    out = []
    for k in range(case["ncl"]):
        n = int(round(math.exp(rng.uniform(math.log(case["nmin"]), math.log(case["nmax"])))))
        if k == 0:
            n = case["nmax"]
        x, fv = rng.uniform(case["xmin"], case["xmax"]), rng.uniform(0.05, 0.30)
        p, r, m = _cluster(dict(case, spread=0.0), seed * 101 + k, n=n, x=x, fv=fv)
        out.append(geometry.Cluster(p, r, m))
    return out


def _vectors(case, seed, neqns):
    """Right-hand sides as a Krylov iteration meets them: dense complex vectors."""
    rng = np.random.default_rng([seed, 11])
    return rng.normal(size=(case["ncol"], neqns)) + 1j * rng.normal(size=(case["ncol"], neqns))


def _con_tran(ncol):
    return [bool(c & 1) for c in range(ncol)]  # A p, A^H w, ...


# ---------------------------------------------------------------------------
# the program: what is in hand before the call, and the call
# ---------------------------------------------------------------------------
def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        b = BatchSolver(0)
        b.set(_batch_clusters(case, seed), geometry.fibonacci_directions(case["ndir"]))
        b.setup()
        return dict(case=case, batch=b)
    pos, radius, ri = _cluster(case, seed)
    ctx = HipContext(0)
    s = dict(case=case, ctx=ctx, pos=pos, radius=radius, ri=ri)
    if kind == "config":
        s["angles"] = scattering_angles(0.0)[1:]
        return s
    ctx.set_spheres(pos, radius, ri)
    if kind == "solve":
        if case["fft"]:
            ctx.node_selection()
            ctx.setup_fft(FP64)
            if case["solver"] != "plain":
                ctx.setup_fft(FP32)
        else:
            ctx.setup_direct(FP64 if case["solver"] == "plain" else FP64_FP32)
        if case["solver"] == "learned":
            ctx.load_learned()
    elif kind == "product":
        ctx.setup_direct(FP64 if case["precision"] == "fp64" else FP32)
        s["ain"] = _vectors(case, seed, ctx.number_eqns)
    elif kind == "tmatrix":
        ctx.setup_direct(FP64)
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "batch":
        b = s["batch"]
        b.solve(eps=1e-6, niter=3000)
        return dict(qeff=b.qeff(), amnp=b.vectors(0))
    ctx = s["ctx"]
    if kind == "solve":
        r = ctx.fixedorsoln(alpha=case["alpha"], sinc=math.sin(case["beta"]), eps=1e-6, niter=10000,
                            solver=SOLVERS[case["solver"]], fft_option=case["fft"])
        return dict(amnp=r["amnp"], qeff=r["qeff"])
    if kind == "product":
        return ctx.sphereinteraction(s["ain"], _con_tran(case["ncol"]),
                                     precision=FP64 if case["precision"] == "fp64" else FP32)
    if kind == "config":
        ctx.set_spheres(s["pos"], s["radius"], s["ri"])
        ctx.setup_direct(FP64_FP32)
        r = ctx.fixedorsoln(eps=1e-6, niter=10000, solver=SOLVE_MIXED)
        ctx.translation_orders()
        ctx.merge_to_common_origin(copy=False)
        return dict(amnp=r["amnp"], qeff=r["qeff"], scatmat=ctx.scattering_matrix(*s["angles"]))
    if kind == "tmatrix":
        r = ctx.tmatrix_solution()
        return dict(tmat=r["tmat"], sqeff=r["sqeff"], qteff=r["qteff"])
    ctx.clear()  # lu: the operator is not kept between calls
    r = ctx.fixedorsoln(solver=SOLVE_LU)
    return dict(amnp=r["amnp"], qeff=r["qeff"])


# ---------------------------------------------------------------------------
# work
# ---------------------------------------------------------------------------
def _order(case, x):
    """Truncation order of a sphere of size parameter x at mie_epsilon 1e-6."""
    return _mie(float(x), complex(case["mr"], case["mi"]))[0]


def _pair(L):
    """(real rotation coefficients, complex axial coefficients) of one pair:
    half of the Wigner rows and axial blocks give the other half by symmetry."""
    rot = sum((m > 0) * n + n + 1 for m in range(L + 1) for n in range(max(1, m), L + 1))
    ax = sum((1 + (m > 0)) * (L - max(1, m) + 1) ** 2 for m in range(L + 1))
    return rot, ax


def work(case):
    kind = case["kind"]
    if kind == "batch":  # dense operators, one FP32 pass of both A p and A^H w for each of 12 iterations
        b = f = 0.0
        for k in range(case["ncl"]):
            n = case["nmin"] * (case["nmax"] / case["nmin"]) ** ((k + 0.5) / case["ncl"])
            L = _order(case, 0.5 * (case["xmin"] + case["xmax"]))
            m = n * L * (L + 2)
            b += 12 * 2 * m * m * 8 + 2 * case["ndir"] * 2 * m * 16
            f += 12 * 2 * 2 * m * m * 8 * 2 * case["ndir"]
        return dict(bytes=b, flops=f)
    n, L = case["n"], _order(case, case["x"])
    neq = 2 * n * L * (L + 2)
    rot, ax = _pair(L)
    pairs = n * (n - 1) / 2
    col = pairs * 2 * 16 * (rot + ax)  # flops of one column of one product
    if kind == "lu":
        return dict(bytes=2.0 * 16 * neq * neq, flops=8.0 * neq ** 3 / 3)
    if kind == "tmatrix":  # orders to about twice the cluster's size parameter, 10 iterations of A p and A^H w each
        T = int(1.6 * case["x"] * (n / case["fv"]) ** (1.0 / 3.0)) + 3
        cols = 2 * T * (T + 2)
        return dict(bytes=10.0 * T * pairs * (rot + 2 * ax) * 8 + 16.0 * cols * neq, flops=20.0 * cols * col)
    if kind == "product":
        e = 8 if case["precision"] == "fp64" else 4
        return dict(bytes=pairs * (rot + 2 * ax) * e + 2.0 * case["ncol"] * neq * 16, flops=case["ncol"] * col)
    # steps to |r|^2/|b|^2 < 1e-6 grow with the size of the cluster
    steps = 8 + 0.012 * n if case.get("solver") in ("mixed", "learned") or kind == "config" else 10 + 0.02 * n
    if case.get("fft"):
        d = 2.0 * case["x"] * 1.6
        cells = max(8.0, n / 1.5) * 8
        LG = math.ceil(d + 1)
        blk = LG * (LG + 2)
        e = 8 if case["solver"] == "plain" else 4
        return dict(bytes=steps * 2 * blk * blk * cells * e, flops=steps * 2 * 2 * 8 * blk * blk * cells)
    e, cols = (8, 4) if case.get("solver") == "plain" else (4, 2)
    return dict(bytes=steps * pairs * (rot + 2 * ax) * e + 2.0 * neq * 16, flops=steps * cols * col)


# ---------------------------------------------------------------------------
# the same quantities in FP64, without the package
# ---------------------------------------------------------------------------
_DEV = "cuda" if torch.cuda.is_available() else "cpu"
_Z = torch.complex128
_PI4 = float(np.float32(np.pi))  # the reference's pi


@functools.lru_cache(maxsize=None)
def _cg(j1, m1, j2, m2, J):
    """<j1 m1 j2 m2 | J m1+m2>, Racah's sum in exact integers."""
    M, fac = m1 + m2, math.factorial
    if abs(M) > J or J < abs(j1 - j2) or J > j1 + j2:
        return 0.0
    num = (2 * J + 1) * fac(J + j1 - j2) * fac(J - j1 + j2) * fac(j1 + j2 - J)
    num *= fac(J + M) * fac(J - M) * fac(j1 - m1) * fac(j1 + m1) * fac(j2 - m2) * fac(j2 + m2)
    s, one = 0, fac(j1 + j2 + J + 2)  # a common multiple large enough for an integer sum
    for k in range(max(0, j2 - J - m1, j1 - J + m2), min(j1 + j2 - J, j1 - m1, j2 + m2) + 1):
        den = (fac(k) * fac(j1 + j2 - J - k) * fac(j1 - m1 - k) * fac(j2 + m2 - k) * fac(J - j2 + m1 + k)
               * fac(J - j1 - m2 + k))
        s += (-1) ** k * (one * one // den)
    return math.copysign(math.sqrt(num * s * s / (fac(j1 + j2 + J + 1) * one ** 4)), s) if s else 0.0


def _amn(m, n, L):
    return (n - 1) * (L + 2) + m if m >= 0 else (-m - 1) * (L + 2) + n + 1


@functools.lru_cache(maxsize=None)
def _coupling(LT, LS):
    """C[wv, target, source] of mode 0 (mode 1: its conjugate); wv = w(w+1)+v."""
    W = LT + LS
    C = np.zeros(((W + 1) ** 2, LT * (LT + 2), LS * (LS + 2)), complex)
    for n in range(1, LS + 1):
        for l in range(1, LT + 1):
            base = -(1j ** (l - n)) * math.sqrt((2 * l + 1) * (2 * n + 1))
            for w in range(abs(n - l), n + l + 1):
                f = base * 1j ** w * _cg(l, -1, n, 1, w)
                for m in range(-n, n + 1):
                    for k in range(-l, l + 1):
                        if abs(m - k) <= w:
                            C[w * (w + 1) + m - k, _amn(k, l, LT), _amn(m, n, LS)] += f * (-1) ** k * _cg(l, -k, n, m, w)
    return torch.from_numpy(C).to(_DEV)


def _waves(d, W, regular):
    """z_w(r) Y_wv(theta, phi) of the vectors d (..., 3): (..., (W+1)^2)."""
    r = torch.linalg.vector_norm(d, dim=-1)
    same = r < 1e-10
    r = torch.where(same, torch.ones_like(r), r)
    ct = d[..., 2] / r
    rho = torch.sqrt(d[..., 0] ** 2 + d[..., 1] ** 2)
    st = rho / r
    on = rho == 0
    rho = torch.where(on, torch.ones_like(rho), rho)
    e1 = torch.complex(torch.where(on, torch.ones_like(rho), d[..., 0] / rho), torch.where(on, torch.zeros_like(rho), d[..., 1] / rho))
    if regular:
        top = W + 20 + int(r.max().item())
        j = [torch.zeros_like(r)] * (W + 1)
        a, b = torch.zeros_like(r), torch.full_like(r, 1e-30)
        for n in range(top, 0, -1):  # downward, scaled by j_0 and j_1
            a, b = b, (2 * n + 1) / r * b - a
            big = b.abs() > 1e200
            sc = torch.where(big, torch.full_like(r, 1e-200), torch.ones_like(r))
            a, b = a * sc, b * sc
            j = [v * sc for v in j]
            if n - 1 <= W:
                j[n - 1] = b
        j0, j1 = torch.sin(r) / r, torch.sin(r) / r ** 2 - torch.cos(r) / r
        lead = j0.abs() > j1.abs()
        k = torch.where(lead, j0 / j[0], j1 / (j[1] if W > 0 else a))
        z = [torch.complex(v * k, torch.zeros_like(r)) for v in j]
    else:
        e = torch.exp(torch.complex(torch.zeros_like(r), r))
        z = [-1j * e / r, -e * torch.complex(r, torch.ones_like(r)) / r ** 2]
        for n in range(2, W + 1):
            z.append((2 * n - 1) / r * z[n - 1] - z[n - 2])
    out = torch.zeros(*r.shape, (W + 1) ** 2, dtype=_Z, device=d.device)
    ph, pmm = torch.ones_like(e1), torch.ones_like(r)
    for m in range(W + 1):
        if m:
            ph = ph * e1
            pmm = pmm * -0.5 * st * math.sqrt((2 * m) * (2 * m - 1)) / m
        p1, p = None, pmm
        for n in range(m, W + 1):
            if n > m:
                p1, p = p, ((2 * n - 1) * ct * p - (math.sqrt((n - 1) ** 2 - m * m) * p1 if n > m + 1 else 0.0)) / math.sqrt(n * n - m * m)
            v = z[n] * p
            out[..., n * (n + 1) + m] = v * ph
            if m:
                out[..., n * (n + 1) - m] = (-1) ** m * v * ph.conj()
    if regular:
        zero = torch.zeros((W + 1) ** 2, dtype=_Z, device=d.device)
        zero[0] = 1.0
        out[same] = zero
    else:
        out[same] = 0.0
    return out


def _riccati(n, x):
    """psi_0..n, xi_0..n of real x."""
    top = n + 30 + int(x)
    p = np.zeros(top + 2)
    p[top] = 1e-250
    for k in range(top, 0, -1):
        p[k - 1] = (2 * k + 1) / x * p[k] - p[k + 1]
        if abs(p[k - 1]) > 1e200:
            p[k - 1:] *= 1e-200
    s0, s1 = math.sin(x), math.sin(x) / x - math.cos(x)
    psi = p[:n + 1] * (s0 / p[0] if abs(s0) > abs(s1) else s1 / p[1])
    chi = np.zeros(max(2, n + 1))
    chi[0], chi[1] = -math.cos(x), -math.cos(x) / x - math.sin(x)
    for k in range(2, n + 1):
        chi[k] = (2 * k - 1) / x * chi[k - 1] - chi[k - 2]
    return psi, psi + 1j * chi[:n + 1]


@functools.lru_cache(maxsize=None)
def _mie(x, m):
    """(order at mie_epsilon 1e-6, a_n, b_n)."""
    top = int(round(x + 4.0 * x ** float(np.float32(1.0) / np.float32(3.0)))) + 5
    psi, xi = _riccati(top, x)
    D, z = 0j, m * x
    Ds = np.zeros(top + 1, complex)
    for n in range(top + 40 + int(abs(z)), 0, -1):
        if n <= top:
            Ds[n] = D
        D = n / z - 1.0 / (D + n / z)
    n = np.arange(1, top + 1)
    fa, fb = Ds[1:] / m + n / x, Ds[1:] * m + n / x
    a = (fa * psi[1:] - psi[:-1]) / (fa * xi[1:] - xi[:-1])
    b = (fb * psi[1:] - psi[:-1]) / (fb * xi[1:] - xi[:-1])
    q = np.cumsum((2 * n + 1) * (a + b).real)
    return int(n[np.abs(1.0 - q / q[-1]) < 1e-6][0]), a, b


class _Cluster:
    """The interaction of a cluster's spheres; vectors are (columns, sphere,
    mode, coefficient) at the largest sphere order, zero above a sphere's own."""

    def __init__(self, pos, radius, ri):
        mies = [_mie(float(x), complex(m)) for x, m in zip(radius, ri)]
        self.radius, self.n = radius, len(radius)
        self.order = np.array([m[0] for m in mies])
        self.L = L = int(self.order.max())
        self.NB, self.W = L * (L + 2), 2 * L
        self.pos = torch.from_numpy(np.ascontiguousarray(pos)).to(_DEV)
        deg = np.zeros(self.NB, int)
        for n in range(1, L + 1):
            for m in range(-n, n + 1):
                deg[_amn(m, n, L)] = n
        a = np.array([np.concatenate([m[1][:o], np.zeros(L - o)]) for m, o in zip(mies, self.order)])
        b = np.array([np.concatenate([m[2][:o], np.zeros(L - o)]) for m, o in zip(mies, self.order)])
        live = deg[None] <= self.order[:, None]
        # helicity form: equal and opposite helicity
        self.same = torch.from_numpy(-0.5 * (a + b)[:, deg - 1] * live).to(_DEV)
        self.flip = torch.from_numpy(-0.5 * (a - b)[:, deg - 1] * live).to(_DEV)
        self.deg, self.live = deg, live
        # compact (package) index of every coefficient, sphere by sphere
        idx = []
        for i, o in enumerate(self.order):
            t = np.zeros((2, o * (o + 2)), int)
            for n in range(1, o + 1):
                for m in range(-n, n + 1):
                    for p in range(2):
                        t[p, _amn(m, n, o)] = (i * 2 + p) * self.NB + _amn(m, n, L)
            idx.append(t.ravel())
        self.index = torch.from_numpy(np.concatenate(idx)).to(_DEV)
        N, NW = self.n, (self.W + 1) ** 2
        self.psi = torch.empty(N, N, NW, dtype=_Z, device=_DEV)
        rows = max(1, int(2.0e9 / (16 * N * NW)))
        for i in range(0, N, rows):
            self.psi[i:i + rows] = _waves(self.pos[i:i + rows, None] - self.pos[None], self.W, False)
        C = _coupling(L, L)
        self.C0 = C.permute(2, 0, 1).reshape(self.NB, -1).contiguous()  # source -> (wv, target)
        par = torch.tensor([(-1.0) ** w for w in range(self.W + 1) for _ in range(2 * w + 1)], device=_DEV)
        self.C0t = (C * par[:, None, None]).permute(1, 0, 2).reshape(self.NB, -1).contiguous()

    def full(self, v):
        out = torch.zeros(v.shape[0], self.n * 2 * self.NB, dtype=_Z, device=_DEV)
        out[:, self.index] = v
        return out.view(-1, self.n, 2, self.NB)

    def compact(self, v):
        return v.reshape(v.shape[0], -1)[:, self.index]

    def translate(self, x, C0):
        R, N, NB = x.shape[0], self.n, self.NB
        out = torch.zeros_like(x)
        for p in range(2):
            t = (x[:, :, p] @ (C0 if p == 0 else C0.conj())).view(R, N, -1, NB)  # (R, j, wv, target)
            t = t.permute(1, 2, 0, 3).reshape(-1, R * NB)
            out[:, :, p] = (self.psi.view(N, -1) @ t).view(N, R, NB).permute(1, 0, 2)
        return out

    def mie(self, x):
        return self.same[None, :, None] * x + self.flip[None, :, None] * x.flip(2)

    def apply(self, x):
        return self.mie(self.translate(x, self.C0))

    def adjoint(self, x):
        return self.translate(self.mie(x.conj()), self.C0t).conj()

    def solve(self, b, tol=1e-9):
        """x - T H x = b for every column, GMRES without restart."""
        shape, R = b.shape, b.shape[0]
        b = b.reshape(R, -1)
        nb = torch.linalg.vector_norm(b, dim=1)
        V, H = [b / nb[:, None]], torch.zeros(R, 401, 400, dtype=_Z, device=_DEV)
        for k in range(400):
            w = V[k] - self.apply(V[k].view(shape)).reshape(R, -1)
            for _ in range(2):
                for i, v in enumerate(V):
                    h = (v.conj() * w).sum(1)
                    H[:, i, k] += h
                    w = w - h[:, None] * v
            H[:, k + 1, k] = torch.linalg.vector_norm(w, dim=1).to(_Z)
            V.append(w / H[:, k + 1, k].abs().clamp_min(1e-300)[:, None])
            if k % 5 == 4:
                A = H[:, :k + 2, :k + 1].cpu().numpy()
                ys, res = [], 0.0
                for r in range(R):
                    e = np.zeros(k + 2, complex)
                    e[0] = 1.0
                    y = np.linalg.lstsq(A[r], e, rcond=None)[0]
                    res = max(res, np.linalg.norm(e - A[r] @ y))
                    ys.append(y)
                if res < tol:
                    y = torch.from_numpy(np.array(ys)).to(_DEV) * nb[:, None]
                    return sum(y[:, i, None] * V[i] for i in range(k + 1)).view(shape)
        raise RuntimeError("GMRES did not converge")

    def plane_wave(self, beta, alpha):
        """Incident field of both polarizations at the spheres, (2, n, 2, NB)."""
        d1 = _wigner1(math.cos(beta), self.L)
        f = np.zeros((2, 2, self.NB), complex)
        for n in range(1, self.L + 1):
            for m in range(-n, n + 1):
                fnm, c = math.sqrt((2 * n + 1) / 2.0) / 4.0, 4.0 * 1j ** (n + 1)
                dm, dp = d1[n, -1, m], d1[n, 1, m]
                t1, t2 = -fnm * (dp - dm), -fnm * (dm + dp)
                for p in range(2):
                    v = c * 0.5 * (t1 + (t2 if p == 0 else -t2)) * np.exp(-1j * m * alpha)
                    f[0, p, _amn(m, n, self.L)] = -v
                    f[1, p, _amn(m, n, self.L)] = (1j if p == 0 else -1j) * v
        k = torch.tensor([math.sin(beta) * math.cos(alpha), math.sin(beta) * math.sin(alpha), math.cos(beta)],
                         dtype=torch.float64, device=_DEV)
        ph = torch.exp(1j * (self.pos @ k))
        live = torch.from_numpy(self.live).to(_DEV)
        return torch.from_numpy(f).to(_DEV)[:, None] * (ph[:, None] * live)[None, :, None]

    def efficiencies(self, a, f):
        """(column, n, 3): extinction, absorption and incident-flux efficiency
        of every sphere; a scattered, f incident coefficients, one column each."""
        out = torch.zeros(a.shape[0], self.n, 3, dtype=torch.float64, device=_DEV)
        # exciting field of every sphere (the Mie matrices are inverted in TE/TM form)
        p, m = a[:, :, 0] + a[:, :, 1], a[:, :, 0] - a[:, :, 1]
        live = torch.from_numpy(self.live).to(_DEV)
        ds = torch.where(live, self.same + self.flip, 1.0)
        dd = torch.where(live, self.same - self.flip, 1.0)
        p, m = p / ds, m / dd
        g = torch.stack([0.5 * (p + m), 0.5 * (p - m)], 2)
        w = {}
        for x in set(self.radius.tolist()):
            psi, xi = _riccati(self.L, x)
            n = np.arange(1, self.L + 1)
            w[x] = (psi[1:], psi[:-1] - n * psi[1:] / x, xi[1:], xi[:-1] - n * xi[1:] / x)
        psi, dpsi, xi, dxi = (torch.from_numpy(np.array([w[x][k][self.deg - 1] for x in self.radius.tolist()])).to(_DEV) for k in range(4))
        for s in range(2):
            for t in range(2):
                e = 1.0 if s == t else -1.0
                aam = 1j * (dxi * xi.conj() - e * xi * dxi.conj())
                ggm = 1j * (dpsi * psi - e * psi * dpsi)
                agm = 1j * (dxi * psi - e * xi * dpsi) * (1.0 + e)
                As, Gs, Fs, At, Gt, Ft = a[:, :, s], g[:, :, s], f[:, :, s], a[:, :, t], g[:, :, t], f[:, :, t]
                out[..., 0] += (agm * As * Ft.conj()).real.sum(2)
                out[..., 1] += (aam * As * At.conj() + ggm * Gs * Gt.conj() + agm * As * Gt.conj()).real.sum(2)
                out[..., 2] += (ggm * Fs * Ft.conj()).real.sum(2)
        return out * torch.from_numpy(2.0 / self.radius ** 2).to(_DEV)[None, :, None]

    def qeff(self, a, f):
        q = self.efficiencies(a, f)
        return torch.stack([0.5 * (q[0] + q[1]), q[0], q[1]], 1).cpu().numpy()

    def scattering_matrix(self, a, ct, phi):
        """Mueller elements from the sum of the spheres' far fields."""
        L, out = self.L, np.zeros((len(ct), 16))
        em = torch.stack([a[:, :, 0] + a[:, :, 1], a[:, :, 0] - a[:, :, 1]], 2)
        for q in range(len(ct)):
            st = math.sqrt(1.0 - ct[q] ** 2)
            k = torch.tensor([st * math.cos(phi[q]), st * math.sin(phi[q]), ct[q]], dtype=torch.float64, device=_DEV)
            far = (em * torch.exp(-1j * (self.pos @ k))[None, :, None, None]).sum(1).cpu().numpy()
            d1, S = _wigner1(ct[q], L), np.zeros(4, complex)
            for n in range(1, L + 1):
                fnm = math.sqrt((2 * n + 1) / 2.0) / 4.0
                for m in range(-n, n + 1):
                    dm, dp = d1[n, -1, m], d1[n, 1, m]
                    tau = (-fnm * (dp - dm), -fnm * (dm + dp))
                    ph = (-1j) ** n * np.exp(1j * m * phi[q])
                    for p in range(2):
                        u, v = far[0, p, _amn(m, n, L)], -far[1, p, _amn(m, n, L)]
                        S += ph * np.array([tau[1 - p] * v, 1j * tau[p] * u, 1j * tau[p] * v, tau[1 - p] * u])
            S *= 4.0 / math.sqrt(2.0 / _PI4)
            P = np.outer(S, S.conj())
            f = np.zeros((4, 4))
            f[0] = [(P[0, 0] + P[1, 1] + P[2, 2] + P[3, 3]).real, (-P[0, 0] + P[1, 1] - P[2, 2] + P[3, 3]).real,
                    2 * (P[1, 2] + P[0, 3]).real, -2 * (P[1, 2] - P[0, 3]).imag]
            f[1] = [(-P[0, 0] + P[1, 1] + P[2, 2] - P[3, 3]).real, (P[0, 0] + P[1, 1] - P[2, 2] - P[3, 3]).real,
                    -2 * (P[1, 2] - P[0, 3]).real, -2 * (P[1, 2] + P[0, 3]).imag]
            f[2] = [2 * (P[1, 3] + P[0, 2]).real, -2 * (P[1, 3] - P[0, 2]).real, 2 * (P[0, 1] + P[2, 3]).real,
                    2 * (P[1, 0] + P[3, 2]).imag]
            f[3] = [-2 * (P[3, 1] + P[0, 2]).imag, -2 * (P[3, 1] - P[0, 2]).imag, 2 * (P[0, 1] - P[2, 3]).imag,
                    2 * (P[0, 1] - P[2, 3]).real]
            out[q] = f.T.ravel() / (4.0 * _PI4)
        return out


def _wigner1(ct, L):
    """d^n_{k m} for k = -1, 1 as {(n, k, m): value}, Wigner's explicit sum."""
    c, s = math.sqrt(max(0.0, 0.5 * (1.0 + ct))), math.sqrt(max(0.0, 0.5 * (1.0 - ct)))
    fac, out = math.factorial, {}
    for n in range(1, L + 1):
        for k in (-1, 1):
            for m in range(-n, n + 1):
                v = 0.0
                for t in range(max(0, k - m), min(n + k, n - m) + 1):
                    v += ((-1) ** (m - k + t) * c ** (2 * n + k - m - 2 * t) * s ** (m - k + 2 * t)
                          / (fac(n + k - t) * fac(t) * fac(m - k + t) * fac(n - m - t)))
                out[n, k, m] = v * math.sqrt(fac(n + k) * fac(n - k) * fac(n + m) * fac(n - m))
    return out


def _tmatrix(cl):
    """T-matrix about the mean sphere position, orders until the extinction
    gained by an order is below 1e-6."""
    r0 = cl.pos.mean(0)
    vr2 = float((cl.radius ** 3).sum()) ** (2.0 * float(np.float32(0.333333)))
    live = torch.from_numpy(cl.live).to(_DEV)
    rad2 = torch.from_numpy(cl.radius ** 2).to(_DEV)
    tmat, sq, qt, old = [], torch.zeros(cl.n, 3, dtype=torch.float64, device=_DEV), np.zeros(3), 0.0
    for l in range(1, 60):
        nb, W = l * (l + 2), l + cl.L
        out_w = _waves(cl.pos - r0, W, True)
        back = _waves(r0 - cl.pos, W, True)
        Co, Cb = _coupling(cl.L, l), _coupling(l, cl.L)
        cols = [(k, q) for k in range(-l, l + 1) for q in (1, 2)]
        src = [_amn(k, l, l) for k, _ in cols]
        f = torch.zeros(len(cols), cl.n, 2, cl.NB, dtype=_Z, device=_DEV)
        A = torch.einsum("iw,wtc->cit", out_w, Co[:, :, src])
        B = torch.einsum("iw,wtc->cit", out_w, Co[:, :, src].conj())
        sg = torch.tensor([0.5 if q == 1 else -0.5 for _, q in cols], device=_DEV)
        f[:, :, 0], f[:, :, 1] = 0.5 * A, sg[:, None, None] * B
        f *= live[None, :, None]
        a = cl.solve(cl.mie(f))
        sq += cl.efficiencies(a, f).sum(0)
        far = [torch.einsum("cit,itk->ck", a[:, :, p], torch.einsum("iw,wkt->itk", back, Cb if p == 0 else Cb.conj())) for p in range(2)]
        em = torch.stack([far[0] + far[1], far[0] - far[1]], 1).cpu().numpy()
        order = [_amn(m, n, l) for n in range(1, l + 1) for m in range(-n, n + 1)]
        for c, (k, q) in enumerate(cols):
            d1, d3 = -2.0 / vr2 * em[c, q - 1, _amn(k, l, l)].real, 2.0 / vr2 * (np.abs(em[c]) ** 2).sum()
            qt += [d1, d1 - d3, d3]
            tmat.append(em[c][:, order].T.ravel())
        ext = float((sq[:, 0] * rad2).sum()) / vr2
        if ext - old < 1e-6:
            break
        old = ext
    return dict(tmat=np.concatenate(tmat), sqeff=sq.cpu().numpy(), qteff=qt)


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        q, am = [], []
        for c in _batch_clusters(case, seed):
            cl = _Cluster(c.pos, c.radius, c.ri)
            f = torch.cat([cl.plane_wave(b, a) for b, a in geometry.fibonacci_directions(case["ndir"])])
            a = cl.solve(cl.mie(f))
            am.append(cl.compact(a).cpu().numpy())
            xg2 = float((cl.radius ** 3).sum()) ** (2.0 * float(np.float32(0.333333)))
            w = torch.from_numpy(cl.radius ** 2 / xg2).to(_DEV)
            e = (cl.efficiencies(a, f) * w[None, :, None]).sum(1).cpu().numpy().reshape(-1, 2, 3)
            e[..., 2] += e[..., 0] - e[..., 1]
            q.append(np.stack([0.5 * (e[:, 0] + e[:, 1]), e[:, 0], e[:, 1]], 1))
        return dict(qeff=np.array(q), amnp=am)
    cl = _Cluster(*_cluster(case, seed))
    if kind == "product":
        x = cl.full(torch.from_numpy(_vectors(case, seed, len(cl.index))).to(_DEV))
        ct = _con_tran(case["ncol"])
        y = torch.stack([(cl.adjoint if c else cl.apply)(x[k:k + 1])[0] for k, c in enumerate(ct)])
        return cl.compact(y).cpu().numpy()
    if kind == "tmatrix":
        return _tmatrix(cl)
    f = cl.plane_wave(case.get("beta", 0.0), case.get("alpha", 0.0))
    a = cl.solve(cl.mie(f), 1e-13 if kind == "lu" else 1e-7 if cl.n > 2500 else 1e-9)
    out = dict(amnp=cl.compact(a).cpu().numpy(), qeff=cl.qeff(a, f))
    if kind == "config":
        out["scatmat"] = cl.scattering_matrix(a, *scattering_angles(0.0)[1:])
    return out
