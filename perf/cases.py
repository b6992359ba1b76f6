"""Measured work of the filtered-Lanczos path.

Each case is one call that a program using this framework makes: a Chebyshev
solve with the mass matrix, a product with the stiffness, a polynomial filter
applied to a Lanczos vector, density-of-states moments on a block of columns,
a whole eigensolve.  The bodies are the seeded meshes of
``normalmodes_amd.workloads``: Delaunay balls ("ball", homogeneous) and
sliver-free layered balls ("layered", solid; "fluid", with a fluid outer
core).  ``n_tets`` is the number of tetrahedra asked for, ``porder`` the
polynomial order (P1 / P2).

The matrices of a body are the plan a program keeps; the seed draws the
vectors (right-hand sides, Lanczos vectors, the solver's start vectors), and
for whole eigensolves the body's shear speed too.
"""
from __future__ import annotations

import ctypes
import functools
import math

import numpy as np
import torch

from normalmodes_amd import driver
from normalmodes_amd import pevsl as pv
from normalmodes_amd.assemble import assemble
from normalmodes_amd.mesh import ball_mesh, stuffed_ball_mesh
from normalmodes_amd.models import homogeneous, three_layer, three_layer_solid

MESH_SEED = 1019
PRECISION = {"fp64": pv.FP64, "fp32": pv.FP32_FILTER, "fp32a": pv.FP32_FILTER_A}


def listed():
    return [
        # The reference's smallest demo (CONST3k: P1, 1 821 DoF): one B-solve on
        # device vectors, as a serving loop or a captured region calls it.
        dict(name="bsolve_p1_2k", op="bsolve", body="ball", n_tets=2900, porder=1, tune="1"),
        # The same solve on the 52k-DoF homogeneous ball (the C1 workload; the
        # reference's fluid-solid demos hold 44k-62k DoF).
        dict(name="bsolve_52k", op="bsolve", body="ball", n_tets=12000, porder=2, tune="1"),
        # and at the size of the headline workload (1.9M DoF); autotuning takes
        # over 10 s there, so a program that solves a few bands skips it.
        dict(name="bsolve_1900k", op="bsolve", body="layered", n_tets=450000, porder=2, tune=""),
        # A~ x on host vectors: the callback an unmodified pEVSL driver makes
        # once per Lanczos step.
        dict(name="stiffness_52k", op="matvec", body="ball", n_tets=12000, porder=2, tune="1"),
        # The inner loop of the reference's single-vector ChebLanNr: the filter
        # polynomial of one band applied to one Lanczos vector.
        dict(name="filter_p2_11k", op="filter", body="layered", n_tets=2000, porder=2, tune="1", lo=0.10, hi=0.16,
             precision="fp64"),
        dict(name="filter_440k", op="filter", body="layered", n_tets=100000, porder=2, tune="", lo=0.15, hi=0.30,
             precision="fp64"),
        # Fluid outer core (the reference's Mtopo / RTMDWAK demos): the filter
        # through the Schur-complement operator with its inner pressure solve.
        dict(name="fluid_filter_63k", op="filter", body="fluid", n_tets=12000, porder=2, tune="", lo=0.15, hi=0.30,
             precision="fp64"),
        # Density of states before slicing the spectrum: 16 columns is the
        # slicer's default, degree 50 its smallest expansion.
        dict(name="moments16_56k", op="moments", body="layered", n_tets=12000, porder=2, tune="1,16", nvec=16, mdeg=50,
             precision="fp64"),
        # FP32 filter (values of A~ and B~ in FP32, FP64 accumulation), 8 columns.
        dict(name="moments8_fp32_440k", op="moments", body="layered", n_tets=100000, porder=2, tune="", nvec=8, mdeg=8,
             precision="fp32a"),
        # The headline's block width (4 columns) at the headline's size.
        dict(name="moments4_1900k", op="moments", body="layered", n_tets=450000, porder=2, tune="", nvec=4, mdeg=2,
             precision="fp64"),
        # A whole eigensolve, block width 4, of a small body (the test ball).
        dict(name="solve_block4_2k", op="solve", body="ball", n_tets=300, porder=2, tune="1,4", block=4, lo=1.0,
             hi=12.0),
    ]


def draw(rng):
    op = rng.choice(["bsolve", "bsolve", "matvec", "filter", "filter", "fluid", "moments", "moments", "moments", "solve"])
    size = lambda lo, hi: int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))  # noqa: E731
    if op == "bsolve":
        return dict(op=op, body=rng.choice(["ball", "layered"]), n_tets=size(250, 300000), porder=rng.choice([1, 2, 2]),
                    tune="")
    if op == "matvec":
        return dict(op=op, body=rng.choice(["ball", "layered"]), n_tets=size(250, 60000), porder=rng.choice([1, 2, 2]),
                    tune=rng.choice(["", "1"]))
    if op == "filter" or op == "fluid":
        lo = rng.uniform(0.05, 0.5)
        return dict(op="filter", body="fluid" if op == "fluid" else "layered",
                    n_tets=size(7000, 40000) if op == "fluid" else size(500, 100000), porder=2, tune="", lo=lo,
                    hi=lo + rng.uniform(0.08, 0.2),
                    precision="fp64" if op == "fluid" else rng.choice(["fp64", "fp64", "fp32", "fp32a"]))
    if op == "moments":
        nvec = rng.choice([1, 2, 4, 8, 16])
        n_tets = size(500, 120000)
        return dict(op=op, body="layered", n_tets=n_tets, porder=rng.choice([1, 2, 2]), nvec=nvec,
                    mdeg=max(2, min(60, 400000 // n_tets)), tune=f"{nvec}" if n_tets < 20000 and nvec > 1 else "",
                    precision=rng.choice(["fp64", "fp64", "fp32", "fp32a"]))
    return dict(op="solve", body="ball", n_tets=size(250, 400), porder=2, tune="1", block=rng.choice([1, 2, 4]),
                lo=rng.uniform(0.8, 2.0), hi=rng.uniform(9.0, 13.0))


# --- bodies and plans -------------------------------------------------------
@functools.lru_cache(maxsize=2)
def _body(body, n_tets, porder):
    if body == "ball":
        return assemble(ball_mesh(n_tets, porder=porder, seed=MESH_SEED), homogeneous())
    if body == "layered":
        return assemble(stuffed_ball_mesh(n_tets, porder=porder, seed=MESH_SEED), three_layer_solid())
    model = three_layer(6371.0)
    mesh = stuffed_ball_mesh(n_tets, porder=porder, seed=MESH_SEED, interfaces=model.interfaces, scale=model.radius)
    return assemble(mesh, model, job=1)


def _problem(case, seed=None):
    if case["op"] == "solve" and seed is not None:  # another shear speed (by up to 3%): another body
        vs = 1.0 + 0.03 * float(np.random.default_rng(seed).random())
        return assemble(ball_mesh(case["n_tets"], porder=case["porder"], seed=MESH_SEED), homogeneous(vs=vs))
    return _body(case["body"], case["n_tets"], case["porder"])


def _top(case):
    """An upper end of the pencil's spectrum, from the mesh width: the largest
    eigenvalue of the stuffed meshes is at most 1000 (P2) or 210 (P1) times
    (vp/h)^2, vp = 11."""
    h = _problem(case).mesh.h
    return (1200.0 if case["porder"] == 2 else 260.0) * 121.0 / h ** 2


def _interval(case):
    top = _top(case)
    if case["op"] == "moments":
        return np.array([0.1 * top, 0.2 * top, -1e-3 * top, top])
    return np.array([case["lo"] * top, case["hi"] * top, -1e-3 * top, top])


class _State:
    """The handles a program keeps, freed with the object."""

    def __init__(self):
        self.op = self.mv = self.h = self.pol = None

    def __del__(self):
        if self.pol:
            pv.pevsl_freepol(self.pol)
        if self.h:
            pv.pevsl_finish(self.h)
        if self.mv:
            self.mv.free()


def _solver(mv, seed, precision):
    h = pv.pevsl_start(0)
    pv.pevsl_setprobsizes(h, mv.n, mv.n, -1)
    pv.pevsl_set_seed(h, seed)
    pv.pevsl_setbmv(h, mv.matB)
    pv.pevsl_setbsol_chebiter(h, 2, mv.chebB)
    if mv.fs is not None:
        pv.pevsl_setamv_fs(h, mv.fs.matAd, mv.fs.matE, mv.fs.matET, mv.fs.chebAp, mv.d, mv.fs.dp)
    else:
        pv.pevsl_setamv_dad(h, mv.matA, mv.d)
    pv.pevsl_set_geneig(h)
    if precision != "fp64":
        pv.pevsl_set_precision(h, PRECISION[precision])
    return h


def _vector(n, seed):
    return np.random.default_rng(seed).standard_normal(n)


def prepare(case, seed):
    P = _problem(case, seed)
    s = _State()
    s.op = case["op"]
    tune = tuple(int(k) for k in case["tune"].split(",") if k)
    # bounds of B~ to four digits: enough for the Chebyshev degree
    bounds = (200, 200, 1e-4)
    if case["body"] == "fluid":
        s.mv = driver.setupmatvec_fs(P, bdeg="auto", bounds=bounds, ap_bounds=bounds, tune=tune)
    else:
        s.mv = driver.setupmatvec(P, porder=case["porder"], bdeg="auto", bounds=bounds, tune=tune)
    if s.op == "solve":
        s.interval, s.block, s.seed = (case["lo"], case["hi"]), case["block"], seed
        return s
    if s.op == "bsolve":
        s.b = torch.from_numpy(_vector(P.n, seed)).cuda()
        s.x = torch.zeros_like(s.b)
        return s
    s.h = _solver(s.mv, seed, case.get("precision", "fp64"))
    if s.op == "moments":
        s.xintv, s.mdeg, s.nvec = _interval(case), case["mdeg"], case["nvec"]
        return s
    s.z = _vector(P.n, seed)
    if s.op == "filter":
        s.pol = pv.pevsl_findpol(_interval(case), 0.8, 0.7)
    return s


def run(s):
    if s.op == "bsolve":
        rc = pv._lib().nmg_chebiter_noalloc(ctypes.c_int(2), ctypes.c_void_p(s.b.data_ptr()),
                                            ctypes.c_void_p(s.x.data_ptr()), ctypes.c_int64(s.mv.chebB),
                                            ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        if rc:
            raise RuntimeError(pv._lib().nmg_last_error().decode())
        return s.x
    if s.op == "matvec":
        return pv.apply(s.h, 0, s.z)
    if s.op == "filter":
        return pv.filter_apply(s.h, s.pol, s.z)
    if s.op == "moments":
        mu, count = pv.kpmdos(s.h, s.mdeg, s.nvec, s.xintv)
        return {"mu": mu, "count": count}
    r = driver.apply_pevsl(s.mv, interval=s.interval, block=s.block, seed=s.seed, vectors=False, residual_check=False)
    return {"lam": r.lam}


# --- what a pass cannot do without ------------------------------------------
def _poly(case):
    pol = pv.pevsl_findpol(_interval(case), 0.8, 0.7)
    try:
        return pv.pol_info(pol)
    finally:
        pv.pevsl_freepol(pol)


def work(case):
    """Matrix entries once per product (3x3 blocks of the stiffness 76 bytes,
    mass entries 12 bytes, other entries 12), block vectors once per operand;
    Chebyshev degrees 30 (P1) and 60 (P2) of the mass solve, 60 of the
    pressure solve."""
    P = _problem(case)
    n, op = P.n, case["op"]
    k = case.get("nvec", 1) if op == "moments" else case.get("block", 1)
    deg = 30 if case["porder"] == 1 else 60
    mb = P.B.val.size / 3.0
    ma = (P.Ad if case["body"] == "fluid" else P.A).val.size / 9.0
    small = case.get("precision", "fp64") != "fp64"
    bsolve = (deg * (mb * (8.0 if small else 12.0) + 32.0 * n * k), deg * (6.0 * mb + 18.0 * n / 3.0) * k)
    prod = (ma * (40.0 if case.get("precision") == "fp32a" else 76.0) + 48.0 * n * k, 18.0 * ma * k)
    if case["body"] == "fluid":
        e = P.E.val.size + P.ET.val.size
        ap = P.Ap.val.size
        prod = (prod[0] + 12.0 * e + 60 * (12.0 * ap + 32.0 * P.n_p) + 48.0 * n, prod[1] + 2.0 * e + 120.0 * ap)
    if op == "bsolve":
        reps = (1, 0)
    elif op == "matvec":
        return dict(bytes=ma * 76.0 + 16.0 * n, flops=18.0 * ma)
    elif op == "filter":
        d = _poly(case).deg
        reps = (d, d)
    elif op == "moments":
        reps = (case["mdeg"], case["mdeg"])
    else:
        # block steps x filter degree of the recurrence that finds these bands
        steps = 120 // k
        reps = (steps * 30, steps * 30)
    return dict(bytes=reps[0] * bsolve[0] + reps[1] * prod[0], flops=reps[0] * bsolve[1] + reps[1] * prod[1])


# --- the same results in plain torch, FP64 ----------------------------------
def _csr(M, ncol, dl, dr):
    """diag(dl) M diag(dr) as a sparse CSR tensor on the GPU."""
    rp = torch.from_numpy(np.ascontiguousarray(M.rowptr, dtype=np.int64)).cuda()
    col = torch.from_numpy(np.ascontiguousarray(M.col, dtype=np.int64)).cuda()
    val = torch.from_numpy(np.ascontiguousarray(M.val, dtype=np.float64)).cuda()
    row = torch.repeat_interleave(torch.arange(rp.numel() - 1, device="cuda"), rp[1:] - rp[:-1])
    val = val * dl[row] * dr[col]
    return torch.sparse_csr_tensor(rp, col, val, size=(rp.numel() - 1, ncol))


def _diag(M):
    rows = np.repeat(np.arange(M.rowptr.size - 1), np.diff(M.rowptr))
    d = np.zeros(M.rowptr.size - 1)
    on = rows == M.col
    d[rows[on]] = M.val[on]
    return torch.from_numpy(d).cuda()


def _cg(M, b, steps=400):
    """M^-1 b, every column by conjugate gradients to rounding."""
    x = torch.zeros_like(b)
    r, p = b.clone(), b.clone()
    rr = (r * r).sum(0)
    stop = 1e-32 * rr
    for i in range(steps):
        q = M @ p
        a = rr / (p * q).sum(0).clamp_min(1e-300)
        x += a * p
        r -= a * q
        new = (r * r).sum(0)
        if i % 10 == 9 and bool((new <= stop).all()):
            break
        p = r + (new / rr.clamp_min(1e-300)) * p
        rr = new
    return x


def _operators(case):
    """x -> A~ x and x -> B~^-1 x on blocks of columns."""
    P = _problem(case)
    d = _diag(P.B).rsqrt()
    B = _csr(P.B, P.n, d, d)
    if case["body"] != "fluid":
        A = _csr(P.A, P.n, d, d)
        return (lambda x: A @ x), (lambda x: _cg(B, x))
    one = torch.ones(P.n_p, dtype=torch.float64, device="cuda")
    dp = (-_diag(P.Ap)).rsqrt()
    Ad = _csr(P.Ad, P.n, d, d)
    E, ET = _csr(P.E, P.n_p, d, one), _csr(P.ET, P.n, one, d)
    Ap = _csr(P.Ap, P.n_p, -dp, dp)
    # D (Ad - E Ap^-1 ET) D with -Ap^-1 = Dp Ap~^-1 Dp
    return ((lambda x: Ad @ x + E @ (dp[:, None] * _cg(Ap, dp[:, None] * (ET @ x)))), (lambda x: _cg(B, x)))


def _rademacher(n, k, seed):
    """The start block of the moments: signs of the solver's seeded hash."""
    u = np.uint64
    with np.errstate(over="ignore"):
        z = u(seed ^ 0xD1B54A32D192ED03) * u(0x9E3779B97F4A7C15) + np.arange(n * k, dtype=u) + u(0x632BE59BD9B4E019)
        z = (z ^ (z >> u(30))) * u(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> u(27))) * u(0x94D049BB133111EB)
        z = z ^ (z >> u(31))
    v = (z >> u(11)).astype(np.float64) * (2.0 / 9007199254740992.0) - 1.0
    return np.where(v < 0.0, -1.0, 1.0).reshape(n, k)


def _count(mu, xintv):
    """Jackson-damped count of eigenvalues in [a, b] from trace moments."""
    a, b, lmin, lmax = xintv
    cc, dd = 0.5 * (lmax + lmin), 0.5 * (lmax - lmin)
    ta, tb = (math.acos(min(1.0, max(-1.0, (x - cc) / dd))) for x in (a, b))
    m = mu.size - 1
    k = np.arange(m + 1)
    al = math.pi / (m + 2)
    g = ((m + 2 - k) * np.cos(k * al) + np.sin(k * al) / math.tan(al)) / (m + 2)
    integral = np.where(k == 0, ta - tb, (np.sin(k * ta) - np.sin(k * tb)) / np.maximum(k, 1))
    return float(np.sum(np.where(k == 0, 1.0, 2.0) * g * mu * integral) / math.pi)


def exact(case, seed):
    P = _problem(case, seed)
    op = case["op"]
    if op == "solve":
        if P.n > 3000:
            return None  # dense reference only for the smallest bodies
        dense = lambda M: torch.sparse_csr_tensor(  # noqa: E731
            torch.from_numpy(np.asarray(M.rowptr, dtype=np.int64)), torch.from_numpy(np.asarray(M.col, dtype=np.int64)),
            torch.from_numpy(M.val), size=(P.n, P.n)).to_dense()
        A, B = dense(P.A), dense(P.B)
        L = torch.linalg.cholesky(B)
        T = torch.linalg.solve_triangular(L, torch.linalg.solve_triangular(L, A, upper=False).T, upper=False)
        lam = torch.linalg.eigvalsh(0.5 * (T + T.T))
        return {"lam": lam[(lam >= case["lo"]) & (lam <= case["hi"])].numpy()}
    if op == "bsolve":
        d = _diag(P.B).rsqrt()
        return _cg(_csr(P.B, P.n, d, d), torch.from_numpy(_vector(P.n, seed)).cuda()[:, None])[:, 0]
    amul, bsol = _operators(case)
    if op == "matvec":
        return amul(torch.from_numpy(_vector(P.n, seed)).cuda()[:, None])[:, 0].cpu().numpy()
    xintv = _interval(case)
    if op == "moments":
        k, mdeg = case["nvec"], case["mdeg"]
        v0 = torch.from_numpy(_rademacher(P.n, k, seed)).cuda()
        cc, dd = 0.5 * (xintv[3] + xintv[2]), 0.5 * (xintv[3] - xintv[2])
        vm, v = None, v0
        mu = [float((v0 * v0).sum()) / k]
        for j in range(1, mdeg + 1):
            w = (amul(bsol(v)) - cc * v) * ((1.0 if j == 1 else 2.0) / dd)
            vm, v = v, w if vm is None else w - vm
            mu.append(float((v0 * v).sum()) / k)
        mu = np.array(mu)
        return {"mu": mu, "count": _count(mu, xintv)}
    p = _poly(case)
    vm, v = None, torch.from_numpy(_vector(P.n, seed)).cuda()[:, None]
    y = p.mu[0] * v
    for j in range(1, p.deg + 1):
        w = (amul(bsol(v)) - p.cc * v) * ((1.0 if j == 1 else 2.0) / p.dd)
        vm, v = v, w if vm is None else w - vm
        y = y + p.mu[j] * v
    return y[:, 0].cpu().numpy()
