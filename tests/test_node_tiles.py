"""Node tiles: the host layout on the CPU (every entry once, sums as the
kernel forms them) and the products on the GPU against scipy, at tile edges,
empty and long rows, every column count, value and vector type."""
import ctypes

import numpy as np
import pytest
import scipy.sparse as sp

from normalmodes_amd import pevsl as pv

_i64p, _i32p, _u16p = (ctypes.POINTER(t) for t in (ctypes.c_int64, ctypes.c_int32, ctypes.c_uint16))


# node counts from which K columns of 3x3 blocks, and of scalar masses, take the tiles
def _on_tiles(kind, nb, K):
    return nb >= ((65536 if K == 1 else 1024) if kind == "bsr" else (1 if K >= 8 else 2048))


def _pattern(nb, seed, band=60, long_row=0):
    """A ragged node pattern: 0 to 30 local columns per row, some rows without
    a diagonal, a few far columns, optionally one row of `long_row` columns."""
    rng = np.random.default_rng(seed)
    rows, cols = [], []
    for r in range(nb):
        n = int(rng.integers(0, 31)) if r % 7 else 0
        c = np.clip(r + rng.integers(-band, band + 1, n), 0, nb - 1)
        if r % 11 == 0:
            c = np.append(c, rng.integers(0, nb, 2))
        if r % 3:
            c = np.append(c, r)
        if long_row and r == nb // 2:
            c = np.append(c, rng.choice(nb, min(long_row, nb), replace=False))
        c = np.unique(c)
        rows.append(np.full(c.size, r))
        cols.append(c)
    rows, cols = np.concatenate(rows), np.concatenate(cols)
    M = sp.csr_matrix((rng.standard_normal(rows.size), (rows, cols)), shape=(nb, nb))
    M.sort_indices()
    return M


def _layout(M, rows, cap, waves, pack):
    rp, ci = M.indptr.astype(np.int64), M.indices.astype(np.int32)
    sz = np.zeros(6, dtype=np.int64)

    def call(*out):
        p = [None if o is None else o.ctypes.data_as(t)
             for o, t in zip(out, (_i32p, _i32p, _u16p, _u16p, _i32p))]
        pv._check(pv._lib().nmg_node_tiles_host(
            ctypes.c_int64(M.shape[0]), rp.ctypes.data_as(_i64p), ci.ctypes.data_as(_i32p), ctypes.c_int(rows),
            ctypes.c_int(cap), ctypes.c_int(waves), ctypes.c_int(pack), sz.ctypes.data_as(_i64p), *p))

    call(None, None, None, None, None)
    nt, quads, nl, spt, mx, ex = (int(v) for v in sz)
    if nt == 0:
        return None
    units = np.zeros((nt, waves, 8), dtype=np.int32)
    lists = np.zeros(nl, dtype=np.int32)
    lrow = np.zeros((nt * spt, 16), dtype=np.uint16)
    eidx, perm = np.zeros(64 * quads, dtype=np.uint16), np.zeros(64 * quads, dtype=np.int32)
    call(units, lists, lrow, eidx, perm)
    return dict(units=units, lists=lists, lrow=lrow, eidx=eidx, perm=perm, spt=spt, max_nodes=mx, max_extra=ex)


def _product(M, L, x, pack):
    """y = M x in the tiles' order: per unit, quads of four entries of 16 rows,
    x through the tile's list; later parts of a slice added to its first."""
    y = np.full((M.shape[0], x.shape[1]), np.nan)
    seen = np.zeros(M.nnz, dtype=int)
    assert L["max_extra"] <= L["units"].shape[1] - L["spt"]  # short tiles included
    for tile in L["units"]:
        for w, (lst, nodes, row0, own, q0, nq, sl, part) in enumerate(tile):
            if sl < 0:
                continue
            xs = x[L["lists"][lst:lst + nodes]]
            part, parts, slot = part & 255, (part >> 8) & 255, part >> 16
            assert part < parts and slot + parts - 1 <= L["max_extra"] and nodes <= L["max_nodes"]
            acc = np.zeros((16, x.shape[1]))
            for q in range(q0, q0 + nq):
                for j in range(16):
                    for e in range(4):
                        k = L["perm"][64 * q + 4 * j + e]
                        if k < 0:
                            continue
                        at = 64 * q + 4 * j + e if pack == 1 else 128 * (q // 2) + 2 * (4 * j + e) + q % 2
                        acc[j] += M.data[k] * xs[L["eidx"][at]]
                        seen[k] += 1
            rows = L["lrow"][sl].astype(int)
            for j in np.flatnonzero(rows != 0xffff):
                r = row0 + rows[j]
                assert L["lists"][lst + own + rows[j]] == r      # the row's own x
                y[r] = acc[j] if part == 0 else y[r] + acc[j]
    assert (seen == 1).all()
    return y


@pytest.mark.parametrize("nb,rows,cap,waves,pack,long_row", [
    (1, 16, 100, 16, 2, 0), (15, 16, 100, 8, 1, 0), (16, 16, 100, 16, 1, 0), (17, 16, 100, 16, 2, 0),
    (300, 128, 700, 16, 2, 0), (300, 96, 150, 8, 1, 0), (130, 128, 700, 8, 1, 90), (257, 192, 260, 16, 2, 250),
    (260, 48, 120, 16, 2, 0)])
def test_layout_forms_the_product(nb, rows, cap, waves, pack, long_row):
    M = _pattern(nb, nb + rows, long_row=long_row)
    L = _layout(M, rows, cap, waves, pack)
    x = np.random.default_rng(1).standard_normal((nb, 2))
    # both sides sum at most 300 terms: (300 + 3) eps of the absolute sum
    bound = 303 * np.finfo(float).eps * (abs(M) @ abs(x)) + 1e-300
    assert (abs(_product(M, L, x, pack) - M @ x) <= bound).all()


@pytest.mark.parametrize("pack", [1, 2])
def test_padding_reads_no_node(pack):
    """Slots that pad a row point at the zero, not at a node of the list."""
    L = _layout(_pattern(300, 7), 96, 700, 16, pack)
    pad = L["perm"].reshape(-1, 64) < 0
    idx = L["eidx"].reshape(-1, 64) if pack == 1 else L["eidx"].reshape(-1, 64, 2).transpose(0, 2, 1).reshape(-1, 64)
    assert pad.any() and (idx[pad] == 0xffff).all() and (idx[~pad] < L["max_nodes"]).all()


def test_layout_refuses_what_a_tile_cannot_hold():
    M = _pattern(200, 3, long_row=150)
    assert _layout(M, 64, 100, 16, 2) is None          # one row references more than 100 nodes
    assert _layout(M, 256, 700, 8, 1) is None          # more slices than wavefronts
    assert _layout(M, 64, 160, 16, 2) is not None


_LIMITED = '''
import ctypes, resource
import numpy as np
from normalmodes_amd import pevsl as pv
lib, p = pv._lib(), lambda a: a.ctypes.data_as(ctypes.c_void_p)

def lay(nb, rp, ci, sz):
    return lib.nmg_node_tiles_host(ctypes.c_int64(nb), p(rp), p(ci), 128, 700, 16, 2, p(sz), None, None, None, None, None)

nb = 1 << 20
rp, ci = np.arange(nb + 1, dtype=np.int64), np.arange(nb, dtype=np.int32)
sz = np.zeros(6, dtype=np.int64)
assert lay(4096, rp, ci, sz) == 0            # the threads and their heaps are there
used = int(open("/proc/self/statm").read().split()[0]) * resource.getpagesize()
seen = []
for mb in list(range(1, 65, 3)) + [1024]:
    resource.setrlimit(resource.RLIMIT_AS, (used + (mb << 20), resource.RLIM_INFINITY))
    seen.append(lay(nb, rp, ci, sz))
print(sorted(set(seen)), seen[0], seen[-1])
'''


def test_layout_without_memory_is_an_error():
    """Host memory that runs out while tiles are laid out, in one of the threads
    or outside, is an error of the call (NMG_ENOMEM), not the end of the process."""
    import subprocess
    import sys
    from pathlib import Path
    r = subprocess.run([sys.executable, "-c", _LIMITED], capture_output=True, text=True, timeout=120,
                       cwd=Path(__file__).resolve().parent.parent)
    assert r.returncode == 0, r.stderr[-800:]
    kinds, first, last = r.stdout.strip().rsplit(" ", 2)
    assert first != "0" and last == "0" and kinds == f"[{min(int(first), 0)}, {max(int(first), 0)}]", r.stdout


def _handles(M, kind, seed):
    """The DoF matrix of a node pattern: mass (x) I3, or random 3x3 blocks."""
    if kind == "mass":
        D = sp.kron(M, sp.identity(3), format="csr")
    else:
        rng = np.random.default_rng(seed)
        D = sp.bsr_matrix((rng.standard_normal((M.nnz, 3, 3)), M.indices, M.indptr), shape=(3 * M.shape[0],) * 2)
        D = D.tocsr()
    D.sort_indices()
    m = pv.csr_create(D.indptr, D.indices, D.data)
    assert pv.csr_info(m)["layout"] == ("mass3" if kind == "mass" else "bsr3")
    return D, m


@pytest.mark.gpu
@pytest.mark.parametrize("kind,nb,long_row", [
    ("mass", 2048, 0), ("mass", 2049, 0), ("mass", 6000, 300), ("mass", 40000, 0), ("mass", 3000, 1500), ("mass", 40, 0),
    ("mass", 20480, 0), ("mass", 20481, 0), ("bsr", 1024, 0), ("bsr", 1025, 300), ("bsr", 30000, 0), ("bsr", 66000, 0)])
def test_products(kind, nb, long_row):
    """A x (or B x) on 1 to 64 columns, FP64 and FP32 values."""
    M = _pattern(nb, nb, long_row=long_row)
    D, m = _handles(M, kind, 5)
    n = D.shape[0]
    h = ch = None
    try:
        ch = pv.pevsl_setup_chebiter(0.5, 1.5, 1, m)        # lays the tiles out
        h = pv.pevsl_start(0)
        pv.pevsl_setprobsizes(h, n, n, -1)
        pv.pevsl_setbmv(h, m)
        pv.pevsl_setbsol_chebiter(h, 2, ch)
        pv.pevsl_setamv(h, m)
        rng = np.random.default_rng(2)
        aD = abs(D)
        most = int(np.diff(D.indptr).max())
        eps = np.finfo(float).eps
        for K in (1, 2, 4, 8, 16, 32, 64):
            refused = long_row + 1 >= 1400 or (long_row >= 700 and K * 8 > 16)
            assert (pv.product_route(m, K)[0] > 0) == (_on_tiles(kind, nb, K) and not refused)
            X = rng.standard_normal((K, n))
            tol = 2 * (most + 3) * eps * (aD @ abs(X).T).T + 1e-300
            assert (abs(pv.apply_block(h, 1, X) - (D @ X.T).T) <= tol).all(), K
        pv.pevsl_set_precision(h, pv.FP32_FILTER)
        for K in (1, 4):  # FP32 values: one rounding of 2^-24 per entry
            X = rng.standard_normal((K, n))
            tol = (2 * (most + 3) * eps + 2.0 ** -24) * (aD @ abs(X).T).T + 1e-300
            assert (abs(pv.apply_block(h, 0, X) - (D @ X.T).T) <= tol).all(), K
    finally:
        if h:
            pv.pevsl_finish(h)
        if ch:
            pv.pevsl_chebiter_free(ch)
        pv.csr_free(m)


@pytest.mark.gpu
@pytest.mark.parametrize("kind,nb", [("mass", 2100), ("mass", 21000), ("bsr", 1100), ("bsr", 66000)])
def test_non_finite_x(kind, nb):
    """Infinities and NaN in x reach the rows that reference them and no others:
    finite results to the bound, the others of the same kind as scipy's."""
    M = _pattern(nb, nb)
    D, m = _handles(M, kind, 5)
    n = D.shape[0]
    h = ch = None
    try:
        ch = pv.pevsl_setup_chebiter(0.5, 1.5, 1, m)
        h = pv.pevsl_start(0)
        pv.pevsl_setprobsizes(h, n, n, -1)
        pv.pevsl_setbmv(h, m)
        pv.pevsl_setbsol_chebiter(h, 2, ch)
        pv.pevsl_setamv(h, m)
        rng = np.random.default_rng(12)
        most, eps = int(np.diff(D.indptr).max()), np.finfo(float).eps
        for K in (1, 2, 4, 16):
            X = rng.standard_normal((K, n))
            for c in range(K):
                X[c, rng.integers(0, n, 40)] = rng.choice([np.inf, -np.inf, np.nan], 40)
            X[:, 0] = np.nan
            with np.errstate(invalid="ignore"):
                want, scale = (D @ X.T).T, (abs(D) @ np.where(np.isfinite(X), abs(X), 0.0).T).T
            got = pv.apply_block(h, 1, X)
            ok = np.isfinite(want)
            assert not ok.all() and (np.isfinite(got) == ok).all()
            assert (abs(got[ok] - want[ok]) <= 2 * (most + 3) * eps * scale[ok] + 1e-300).all()
            assert np.array_equal(got[~ok], want[~ok], equal_nan=True)
    finally:
        if h:
            pv.pevsl_finish(h)
        if ch:
            pv.pevsl_chebiter_free(ch)
        pv.csr_free(m)


@pytest.mark.gpu
@pytest.mark.parametrize("nb,long_row", [(2048, 0), (6001, 300), (36000, 0)])
def test_chebyshev_steps(nb, long_row):
    """The fused step on a mass pattern: `deg` steps against the recurrence in
    numpy, FP64 and FP32 iterates, 1 to 16 columns."""
    M = _pattern(nb, nb + 1, long_row=long_row)
    M = M * 0.02 + sp.identity(nb) * 2.0                    # well conditioned, not symmetric
    M.sort_indices()
    D, m = _handles(M.tocsr(), "mass", 5)
    n, deg, lo, hi = D.shape[0], 5, 1.0, 3.0
    h = ch = None
    try:
        ch = pv.pevsl_setup_chebiter(lo, hi, deg, m)
        h = pv.pevsl_start(0)
        pv.pevsl_setprobsizes(h, n, n, -1)
        pv.pevsl_setbmv(h, m)
        pv.pevsl_setbsol_chebiter(h, 2, ch)
        pv.pevsl_setamv(h, m)
        pv.pevsl_set_geneig(h)
        th, sg = 0.5 * (lo + hi), (lo + hi) / (hi - lo)

        def ref(b):
            xm, xk, w = np.zeros_like(b), b / th, 2.0
            for _ in range(deg):
                w = 1.0 / (1.0 - w / (4.0 * sg * sg))
                xm, xk = xk, xm + w * (xk - xm + (b - D @ xk) / th)
            return xk

        rng = np.random.default_rng(4)
        for prec, rel in ((pv.FP64, 1e-13), (pv.FP32_FILTER, 1e-6), (pv.FP32_BSOLVE, 4e-6)):
            if prec != pv.FP64:
                pv.pevsl_set_precision(h, prec)
            for K in (1, 2, 4, 8, 16):
                X = rng.standard_normal((K, n))
                want = ref(X.T).T
                got = pv.apply_block(h, 2, X)
                assert np.linalg.norm(got - want) <= rel * np.linalg.norm(want), (prec, K)
    finally:
        if h:
            pv.pevsl_finish(h)
        if ch:
            pv.pevsl_chebiter_free(ch)
        pv.csr_free(m)


def _solver(n, m, ch):
    h = pv.pevsl_start(0)
    pv.pevsl_setprobsizes(h, n, n, -1)
    pv.pevsl_setbmv(h, m)
    pv.pevsl_setbsol_chebiter(h, 2, ch)
    pv.pevsl_setamv(h, m)
    return h


@pytest.mark.gpu
@pytest.mark.parametrize("kind,nb", [("mass", 21000), ("bsr", 3000)])
def test_tiles_that_do_not_fit(kind, nb):
    """Where the tiles' memory does not suffice, set-up succeeds and products run
    on the row kernels: no tiles, part of their tables, all but the last, and
    room for the FP64 values but not for their FP32 copy."""
    M = _pattern(nb, nb)
    D, m = _handles(M, kind, 5)
    n, K = D.shape[0], 4
    h = ch = None
    X = np.random.default_rng(2).standard_normal((K, n))
    want, scale = (D @ X.T).T, (abs(D) @ abs(X).T).T
    tol = 2 * (int(np.diff(D.indptr).max()) + 3) * np.finfo(float).eps * scale + 1e-300
    try:
        pv.set_tile_memory(m, 0)
        ch = pv.pevsl_setup_chebiter(0.5, 1.5, 1, m)
        h = _solver(n, m, ch)

        def check(tiles):
            assert (pv.product_route(m, K)[0] > 0) == tiles
            assert (abs(pv.apply_block(h, 1, X) - want) <= tol).all()

        check(False)
        lo, hi = 0, 1 << 30
        while hi - lo > 1:                                  # the least memory that holds them
            mid = (lo + hi) // 2
            pv.set_tile_memory(m, mid)
            lo, hi = (lo, mid) if pv.product_route(m, K)[0] else (mid, hi)
        for limit, tiles in ((hi, True), (hi - 1, False), (hi // 2, False), (1 << 12, False), (hi, True)):
            pv.set_tile_memory(m, limit)
            check(tiles)
        pv.pevsl_set_precision(h, pv.FP32_FILTER)           # no room for FP32 values
        got = pv.apply_block(h, 0, X)
        assert (abs(got - want) <= tol + 2.0 ** -24 * scale).all()
        pv.set_tile_memory(m, -1)
        assert pv.product_route(m, K)[0] > 0
    finally:
        if h:
            pv.pevsl_finish(h)
        if ch:
            pv.pevsl_chebiter_free(ch)
        pv.csr_free(m)


@pytest.mark.gpu
def test_tuned_source_of_a_scaled_copy():
    """Tuning a 3x3-block matrix leaves it without tile values (a scaled copy
    brings its own); they are there once the matrix itself is an operator.  The
    copy's products see the scaling, and the source's do not."""
    nb, K = 2000, 4
    D, m = _handles(_pattern(nb, 4), "bsr", 6)
    n = D.shape[0]
    rng = np.random.default_rng(3)
    d, X = rng.uniform(0.5, 2.0, n), rng.standard_normal((K, n))
    h, g = pv.pevsl_start(0), pv.pevsl_start(0)
    try:
        for s in (h, g):
            pv.pevsl_setprobsizes(s, n, n, -1)
        pv.csr_autotune(m, 1, 2)
        assert pv.product_route(m, K)[0] == 0
        pv.pevsl_setamv_dad(h, m, d)
        assert pv.product_route(m, K)[0] == 0
        pv.pevsl_setamv(g, m)
        assert pv.product_route(m, K)[0] > 0
        eps = 2 * (int(np.diff(D.indptr).max()) + 5) * np.finfo(float).eps
        for s, e in ((h, d), (g, np.ones(n))):
            want, scale = e * (D @ (e * X).T).T, e * (abs(D) @ (e * abs(X)).T).T
            assert (abs(pv.apply_block(s, 0, X) - want) <= eps * scale + 1e-300).all()
        pv.csr_autotune(m, 2, 2)                            # in use: the values stay
        assert pv.product_route(m, K)[0] > 0
    finally:
        pv.pevsl_finish(h)
        pv.pevsl_finish(g)
        pv.csr_free(m)


@pytest.mark.gpu
def test_solvers_of_several_threads_share_a_matrix():
    """Solvers in four threads set up solves, tiles and FP32 values of one matrix
    at the same time and work with them at once."""
    import threading
    nb, deg, lo, hi = 6000, 6, 1.0, 3.0
    M = (_pattern(nb, 8) * 0.02 + sp.identity(nb) * 2.0).tocsr()
    M.sort_indices()
    A, a = _handles(_pattern(1500, 9), "bsr", 5)
    D, m = _handles(M, "mass", 5)
    n, na = D.shape[0], A.shape[0]
    th, sg = 0.5 * (lo + hi), (lo + hi) / (hi - lo)
    eps, go, failed = 2.0 ** -23, threading.Barrier(4), []

    def ref(b):
        xm, xk, w = np.zeros_like(b), b / th, 2.0
        for _ in range(deg):
            w = 1.0 / (1.0 - w / (4.0 * sg * sg))
            xm, xk = xk, xm + w * (xk - xm + (b - D @ xk) / th)
        return xk

    def work(i):
        try:
            rng = np.random.default_rng(i)
            X, Y, d = rng.standard_normal((4, n)), rng.standard_normal((4, na)), rng.uniform(0.5, 2.0, na)
            want, wanta = ref(X.T).T, d * (A @ (d * Y).T).T
            go.wait()
            ch = pv.pevsl_setup_chebiter(lo, hi, deg, m)
            h, g = _solver(n, m, ch), pv.pevsl_start(0)
            pv.pevsl_set_geneig(h)
            pv.pevsl_setprobsizes(g, na, na, -1)
            pv.pevsl_setamv_dad(g, a, d)
            if i % 2:
                pv.pevsl_set_precision(h, pv.FP32_FILTER)
            for _ in range(3):
                got, gota = pv.apply_block(h, 2, X), pv.apply_block(g, 0, Y)
                # FP32 values: 2^-24 each, at most doubled by the recurrence
                assert np.linalg.norm(got - want) <= (eps if i % 2 else 1e-13) * np.linalg.norm(want)
                assert np.linalg.norm(gota - wanta) <= 1e-13 * np.linalg.norm(wanta)
            pv.pevsl_finish(h)
            pv.pevsl_finish(g)
            pv.pevsl_chebiter_free(ch)
        except BaseException as e:  # noqa: BLE001 - reported below
            failed.append((i, e))

    ts = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    try:
        for t in ts:
            t.start()
        for t in ts:
            t.join()
        assert not failed, failed
        assert pv.product_route(m, 4)[0] > 0 and pv.product_route(a, 4)[0] == 0
    finally:
        pv.csr_free(m)
        pv.csr_free(a)


@pytest.mark.gpu
@pytest.mark.parametrize("nb,kind,band,long_row", [
    (1024, "bsr", 60, 0), (3001, "bsr", 60, 300), (66000, "bsr", 60, 0)])
def test_filter_steps(nb, kind, band, long_row):
    """The fused filter step: whole filters of low degree on 1 to 16 columns with
    a polynomial of its own each, FP64 and FP32 values, against the recurrence
    in numpy; after non-finite columns, so that a first step that read the work
    of the last call would show."""
    M = _pattern(nb, nb + 2, band=band, long_row=long_row)
    D, m = _handles(M, kind, 5)
    pv.csr_free(m)
    D = (D * (1.0 / abs(D).sum(1).max())).tocsr()           # the spectrum lies in [-1, 1]
    D.sort_indices()
    m = pv.csr_create(D.indptr, D.indices, D.data)
    n, eps, most = D.shape[0], np.finfo(float).eps, int(np.diff(D.indptr).max())
    ch = pv.pevsl_setup_chebiter(0.5, 1.5, 1, m)
    h = _solver(n, m, ch)
    pols = [pv.pevsl_findpol(np.array([lo, hi, -1.2, 1.1]), 0.8, 0.7)
            for lo, hi in ((0.2, 1.0), (-0.3, 0.3), (-1.2, -0.4), (0.4, 1.0))]
    info = [pv.pol_info(p) for p in pols]
    assert [p.deg for p in info] == [3, 6, 2, 4]

    def ref(p, v, absolute=False):
        """p(D) v, or the sum of the absolute values that its rounding scales with."""
        A, c, s = (abs(D), abs(p.cc), 1.0) if absolute else (D, p.cc, -1.0)
        mu = abs(p.mu) if absolute else p.mu
        vm, vk, y = np.zeros_like(v), v, mu[0] * v
        for k in range(1, p.deg + 1):
            vm, vk = vk, (1.0 if k == 1 else 2.0) / p.dd * (A @ vk + s * c * vk) + s * vm
            y = y + mu[k] * vk
        return y

    try:
        rng = np.random.default_rng(11)
        for prec, unit in ((pv.FP64, 0.0), (pv.FP32_FILTER_A, 2.0 ** -24)):
            pv.pevsl_set_precision(h, prec)
            for K in (1, 2, 4, 8, 16):
                assert (pv.product_route(m, K)[0] > 0) == _on_tiles(kind, nb, K)
                X = rng.standard_normal((K, n))
                mine = [c * 7 % 4 for c in range(K)]        # neighbours differ
                pv.filter_apply_block(h, [pols[i] for i in mine], np.full((K, n), np.nan))
                got = pv.filter_apply_block(h, [pols[i] for i in mine], X)
                for c in range(K):
                    p = info[mine[c]]
                    tol = (p.deg + 1) * (2 * (most + 6) * eps + unit) * ref(p, abs(X[c]), True)
                    assert (abs(got[c] - ref(p, X[c])) <= tol).all(), (prec, K, c)
            if _on_tiles(kind, nb, 1):                      # the single-vector filter's scalar mu
                pv.filter_apply(h, pols[0], np.full(n, np.nan))
                for p, i in zip(pols, info):
                    x = rng.standard_normal(n)
                    tol = (i.deg + 1) * (2 * (most + 6) * eps + unit) * ref(i, abs(x), True)
                    assert (abs(pv.filter_apply(h, p, x) - ref(i, x)) <= tol).all()
    finally:
        for p in pols:
            pv.pevsl_freepol(p)
        pv.pevsl_finish(h)
        pv.pevsl_chebiter_free(ch)
        pv.csr_free(m)


@pytest.mark.gpu
@pytest.mark.parametrize("long_row", [0, 1000, 1398])
def test_lists_near_the_largest(long_row):
    """Node lists of up to 1400 nodes: more than 64 KB of LDS at two columns; with
    a row of more than 700 nodes there is no second cut, and four columns take
    the first, with up to 134 KB."""
    nb = 36000
    M = _pattern(nb, 5, band=1000, long_row=long_row)
    M = M.tolil()
    if long_row:                                            # exactly that many, and its own node
        r = nb // 2
        M[r, :] = 0.0
        M[r, np.arange(r, r + long_row)] = 1.0
    M = M.tocsr()
    M.eliminate_zeros()
    M.sort_indices()
    assert _layout(M, 144, 1400, 16, 2)["max_nodes"] > 1390
    assert (_layout(M, 144, 700, 16, 2) is None) == (long_row > 0)
    D, m = _handles(M, "mass", 5)
    n = D.shape[0]
    ch = pv.pevsl_setup_chebiter(0.5, 1.5, 1, m)
    h = _solver(n, m, ch)
    rng, most = np.random.default_rng(2), int(np.diff(D.indptr).max())
    try:
        for K in (1, 2, 4, 8, 16):
            assert pv.product_route(m, K)[0] == (2 if K >= 4 and not long_row else 1)
            X = rng.standard_normal((K, n))
            tol = 2 * (most + 3) * np.finfo(float).eps * (abs(D) @ abs(X).T).T + 1e-300
            assert (abs(pv.apply_block(h, 1, X) - (D @ X.T).T) <= tol).all(), K
    finally:
        pv.pevsl_finish(h)
        pv.pevsl_chebiter_free(ch)
        pv.csr_free(m)
