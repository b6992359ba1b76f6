"""One-launch Chebyshev solves of small scalar-mass systems: against the
recurrence in numpy and against the step-by-step kernels (a layout set by hand
turns the one-launch form off), at one node, empty and long rows, the sizes
around its limits, 1 to 64 columns, FP64 and FP32 values."""
import ctypes

import numpy as np
import pytest
import scipy.sparse as sp

from normalmodes_amd import pevsl as pv

gpu = pytest.mark.gpu


def _mass(nb, per_row, seed, long_row=0):
    rng = np.random.default_rng(seed)
    rows, cols = [], []
    for r in range(nb):
        n = 0 if r % 9 == 4 else int(rng.integers(0, per_row + 1))
        c = np.unique(rng.integers(0, nb, n + (long_row if r == nb // 3 else 0)))
        rows.append(np.full(c.size, r))
        cols.append(c)
    rows, cols = np.concatenate(rows), np.concatenate(cols)
    M = sp.csr_matrix((0.4 / max(per_row, 1) * rng.standard_normal(rows.size), (rows, cols)), shape=(nb, nb))
    M = (M + sp.diags(np.where(np.arange(nb) % 9 == 4, 0.0, 2.0))).tocsr()
    M.eliminate_zeros()
    M.sort_indices()
    return M


def _layout(M):
    rp, ci = M.indptr.astype(np.int64), M.indices.astype(np.int32)
    sz, c = np.zeros(2, dtype=np.int64), ctypes

    def call(*out):
        pv._check(pv._lib().nmg_small_layout_host(
            c.c_int64(M.shape[0]), *(a.ctypes.data_as(c.c_void_p) for a in (rp, ci, sz)),
            *(None if o is None else o.ctypes.data_as(c.c_void_p) for o in out)))

    call(None, None, None, None)
    quads, slices = (int(v) for v in sz)
    if quads == 0:
        return None
    out = (np.zeros(32, np.uint32), np.zeros((16, slices, 16), np.uint16), np.zeros((16, quads, 64), np.uint16),
           np.zeros((16, quads, 64), np.int32))
    call(*out)
    return out


@pytest.mark.parametrize("nb,per_row,long_row,fits", [
    (1, 1, 0, True), (16, 6, 0, True), (17, 6, 0, True), (555, 28, 0, True), (300, 60, 0, True), (700, 40, 400, None),
    (4096, 3, 0, True), (4097, 3, 0, False), (3000, 40, 0, False)])
def test_small_layout(nb, per_row, long_row, fits):
    """The host layout: every row in one place, its entries once each in the
    slots of its lanes and slice, everything else padding at the zero."""
    M = _mass(nb, per_row, nb, long_row)
    L = _layout(M)
    if fits is not None:
        assert (L is not None) == fits
    if L is None:
        return
    ends, rows, eidx, perm = L
    quads = perm.shape[1]
    assert quads in (8, 16, 24) and rows.shape[1] <= 16
    pad = perm < 0
    assert (eidx[pad] == nb).all() and (eidx[~pad] == M.indices[perm[~pad]]).all()
    assert (np.bincount(perm[~pad], minlength=M.nnz) == 1).all()
    assert (np.sort(rows[rows != 0xffff]) == np.arange(nb)).all()
    for w in range(16):
        last = [q for q in range(32) if ends[w] >> q & 1]
        assert not ends[16 + w] & ~ends[w] and all(q < quads for q in last)
        q0 = 0
        for i, q in enumerate(last):
            lanes = 16 if ends[16 + w] >> q & 1 else 4
            for lane in range(64):
                ks = perm[w, q0:q + 1, lane]
                r = rows[w, i, lane // lanes * lanes // 4]
                assert (M.indptr[r] <= ks[ks >= 0]).all() and (ks[ks >= 0] < M.indptr[r + 1]).all() if r != 0xffff \
                    else (ks < 0).all()
            q0 = q + 1
        assert (perm[w, q0:] < 0).all() and (rows[w, len(last):] == 0xffff).all()


# (nodes, entries per row): one slot per wavefront, a whole and a broken slice,
# both sides of each register size (8, 16, 24 quads) and sizes too large
@gpu
@pytest.mark.parametrize("nb,per_row,long_row", [
    (1, 1, 0), (15, 6, 0), (16, 6, 0), (17, 6, 0), (555, 28, 0), (614, 15, 0), (700, 40, 400), (1100, 28, 0),
    (2300, 12, 0), (4096, 3, 0), (4097, 3, 0), (3000, 40, 0)])
def test_small_solve(nb, per_row, long_row):
    M = _mass(nb, per_row, nb, long_row)
    D = sp.kron(M, sp.identity(3), format="csr")
    D.sort_indices()
    n, lo, hi = D.shape[0], 1.0, 3.0
    th, sg = 0.5 * (lo + hi), (lo + hi) / (hi - lo)

    def ref(b, deg):
        xm, xk, w = np.zeros_like(b), b / th, 2.0
        for _ in range(deg):
            w = 1.0 / (1.0 - w / (4.0 * sg * sg))
            xm, xk = xk, xm + w * (xk - xm + (b - D @ xk) / th)
        return xk

    m = pv.csr_create(D.indptr, D.indices, D.data)
    rng = np.random.default_rng(2)
    handles = []
    try:
        if pv.csr_info(m)["layout"] != "mass3":
            pytest.skip("the pattern reads as 3x3 blocks")
        for deg in (1, 2, 9):
            ch = pv.pevsl_setup_chebiter(lo, hi, deg, m)
            handles.append((pv.pevsl_chebiter_free, ch))
            h = pv.pevsl_start(0)
            handles.insert(0, (pv.pevsl_finish, h))
            pv.pevsl_setprobsizes(h, n, n, -1)
            pv.pevsl_setbmv(h, m)
            pv.pevsl_setbsol_chebiter(h, 2, ch)
            pv.pevsl_setamv(h, m)
            pv.pevsl_set_geneig(h)
            for K in (1, 2, 4, 16, 64):
                assert pv.product_route(m, K)[1] == (_layout(M) is not None)
                X = rng.standard_normal((K, n))
                want = ref(X.T, deg).T
                got = pv.apply_block(h, 2, X)
                assert np.linalg.norm(got - want) <= 1e-13 * np.linalg.norm(want), (deg, K)
            x = rng.standard_normal(n)
            one = pv.pevsl_chebiter(2, x, ch)
            assert np.linalg.norm(one - ref(x, deg)) <= 1e-13 * np.linalg.norm(one)
            pv.set_kernel_map(m, 32)                       # by hand: step by step
            assert not pv.product_route(m, 1)[1]
            step = pv.pevsl_chebiter(2, x, ch)
            pv.set_kernel_map(m, 0)
            assert np.linalg.norm(one - step) <= 1e-14 * deg * np.linalg.norm(step)
            pv.pevsl_set_precision(h, pv.FP32_FILTER)      # FP32 values: 2^-24 each, grown by the recurrence
            got = pv.apply_block(h, 2, X)
            assert np.linalg.norm(got - want) <= 2.0 ** -22 * np.linalg.norm(want)
    finally:
        for f, v in handles:
            f(v)
        pv.csr_free(m)


def _open(n, m, ch, graphs=False):
    h = pv.pevsl_start(0)
    pv.pevsl_setprobsizes(h, n, n, -1)
    pv.pevsl_setbmv(h, m)
    pv.pevsl_setbsol_chebiter(h, 2, ch)
    pv.pevsl_setamv(h, m)
    pv.pevsl_set_geneig(h)
    pv.set_graphs(h, graphs)
    return h


@gpu
@pytest.mark.parametrize("nb", [300, 2300])
def test_graphs_belong_to_one_solve(nb):
    """A graph captured from one Chebyshev solve is not replayed for another
    with the same bounds and degree (which may lie where the freed one lay),
    nor after the solve's refinement changed."""
    D = sp.kron(_mass(nb, 12, nb), sp.identity(3), format="csr")
    D.sort_indices()
    n, lo, hi, deg = D.shape[0], 1.0, 3.0, 12
    m = pv.csr_create(D.indptr, D.indices, D.data)
    rng = np.random.default_rng(3)
    ch = pv.pevsl_setup_chebiter(lo, hi, deg, m)
    eager, graph = _open(n, m, ch), _open(n, m, ch, graphs=True)
    try:
        for K in (1, 2):
            for new in ("first", "another solve", "one coarse pass", "no passes"):
                if new == "another solve":
                    pv.pevsl_chebiter_free(ch)
                    ch = pv.pevsl_setup_chebiter(lo, hi, deg, m)
                    for h in (eager, graph):
                        pv.pevsl_setbsol_chebiter(h, 2, ch)
                elif new == "one coarse pass":
                    pv.chebiter_set_refine(ch, 1, 1)
                elif new == "no passes":
                    pv.chebiter_set_refine(ch, 0)
                before = pv.graph_stats(graph)[1]
                for i in range(4):  # eager first use, capture, replays
                    X = rng.standard_normal((K, n))
                    want, got = pv.apply_block(eager, 2, X), pv.apply_block(graph, 2, X)
                    assert np.linalg.norm(got - want) <= 1e-15 * np.linalg.norm(want), (K, new, i)
                    assert pv.graph_stats(graph)[1] - before == max(0, i - 1), (K, new, i)
    finally:
        pv.pevsl_finish(eager)
        pv.pevsl_finish(graph)
        pv.pevsl_chebiter_free(ch)
        pv.csr_free(m)


class _Hip:
    """The HIP runtime that the library is linked to."""

    def __init__(self):
        pv._lib()
        self.h = ctypes.CDLL("libamdhip64.so")

    def __getattr__(self, name):
        def call(*args):
            assert getattr(self.h, name)(*args) == 0, name
        return call


@gpu
@pytest.mark.parametrize("nb", [300, 2300])
def test_captured_solve_outlives_its_handle(nb):
    """A caller's own graph of nmg_chebiter_noalloc holds the matrix and the
    caller's vectors only: replayed on new inputs after the solve's handle was
    freed and another solve was set up, with eager solves in between."""
    D = sp.kron(_mass(nb, 12, nb), sp.identity(3), format="csr")
    D.sort_indices()
    n, vp = D.shape[0], ctypes.c_void_p
    lib, hip, rng = pv._lib(), _Hip(), np.random.default_rng(6)
    m = pv.csr_create(D.indptr, D.indices, D.data)
    ch = pv.pevsl_setup_chebiter(1.0, 3.0, 20, m)
    b, x, s, g, ex = vp(), vp(), vp(), vp(), vp()
    for p in (b, x):
        hip.hipMalloc(ctypes.byref(p), ctypes.c_size_t(8 * n))
    hip.hipStreamCreate(ctypes.byref(s))

    def replay(want_of):
        v, out = rng.standard_normal(n), np.empty(n)
        hip.hipMemcpy(b, v.ctypes.data_as(vp), ctypes.c_size_t(8 * n), 1)
        hip.hipGraphLaunch(ex, s)
        hip.hipStreamSynchronize(s)
        hip.hipMemcpy(out.ctypes.data_as(vp), x, ctypes.c_size_t(8 * n), 2)
        want = pv.pevsl_chebiter(2, v, want_of)
        assert np.linalg.norm(out - want) <= 1e-15 * np.linalg.norm(want)

    def noalloc():
        pv._check(lib.nmg_chebiter_noalloc(ctypes.c_int(2), b, x, ctypes.c_int64(ch), s))

    try:
        noalloc()
        hip.hipStreamSynchronize(s)
        hip.hipStreamBeginCapture(s, 1)                    # thread local
        noalloc()
        hip.hipStreamEndCapture(s, ctypes.byref(g))
        hip.hipGraphInstantiate(ctypes.byref(ex), g, None, None, ctypes.c_size_t(0))
        for _ in range(3):
            replay(ch)
        pv.pevsl_chebiter_free(ch)
        others = [pv.pevsl_setup_chebiter(0.5, 7.0, 20, m) for _ in range(3)]
        ch = pv.pevsl_setup_chebiter(1.0, 3.0, 20, m)
        for _ in range(3):
            replay(ch)
        for o in others:
            pv.pevsl_chebiter_free(o)
        hip.hipGraphExecDestroy(ex)
        hip.hipGraphDestroy(g)
    finally:
        hip.hipFree(b)
        hip.hipFree(x)
        hip.hipStreamDestroy(s)
        pv.pevsl_chebiter_free(ch)
        pv.csr_free(m)


@gpu
@pytest.mark.parametrize("lo,hi,deg", [
    (1.0, 3.0, 1500), (1e-3, 1.0, 400), (1e-6, 1.0, 2500), (0.999, 1.0, 3), (1e-4, 1.0, 8192), (1e-4, 1.0, 8500),
    (1e-8, 1.0, 8500)])
def test_small_solve_weights(lo, hi, deg):
    """The one-launch solve's step weights, up to and beyond the 8192 held, from
    ill- to well-conditioned bounds (1e-8 with 8500 steps: not settled by then, so
    step by step), against the recurrence: diagonal systems, whose every entry is one polynomial of
    its eigenvalue."""
    nb = 4096 if deg == 8500 else 48
    lam = np.linspace(lo, hi, nb)
    D = sp.kron(sp.diags(lam), sp.identity(3), format="csr")
    th, sg = 0.5 * (lo + hi), (lo + hi) / (hi - lo)
    rng = np.random.default_rng(8)
    b = rng.standard_normal(3 * nb)
    xm, xk, w = np.zeros(3 * nb, np.longdouble), b / np.longdouble(th), np.longdouble(2.0)
    d = np.repeat(lam, 3).astype(np.longdouble)
    for _ in range(deg):
        w = 1 / (1 - w / (4 * np.longdouble(sg) ** 2))
        xm, xk = xk, xm + w * (xk - xm + (b - d * xk) / np.longdouble(th))
    m = pv.csr_create(D.indptr, D.indices, D.data)
    ch = pv.pevsl_setup_chebiter(lo, hi, deg, m)
    try:
        assert pv.csr_info(m)["layout"] == "mass3"
        got = pv.pevsl_chebiter(2, b, ch)
        pv.set_kernel_map(m, 32)                           # by hand: step by step
        step = pv.pevsl_chebiter(2, b, ch)
        err = [float(np.linalg.norm(v - xk) / np.linalg.norm(xk)) for v in (got, step)]
        # rounding of the iteration itself grows with deg and the condition
        assert err[0] <= 2.0 * err[1] + 1e-15 * min(deg, hi / lo), err
    finally:
        pv.pevsl_chebiter_free(ch)
        pv.csr_free(m)


@gpu
@pytest.mark.parametrize("nb", [200, 900])
def test_non_finite_stays_in_its_component(nb):
    """Two systems that do not touch, numbered alternately: an infinity or NaN
    in the right-hand side of one leaves the other's solution as it is."""
    M = _mass(nb, 12, nb)
    two = sp.kron(M, sp.identity(2), format="csr")           # node 2r and 2r + 1: M twice
    assert _layout(two) is not None
    D = sp.kron(two, sp.identity(3), format="csr")
    D.sort_indices()
    n = D.shape[0]
    m = pv.csr_create(D.indptr, D.indices, D.data)
    ch = pv.pevsl_setup_chebiter(1.0, 3.0, 9, m)
    h = _open(n, m, ch)
    rng = np.random.default_rng(9)
    even = np.repeat(np.arange(2 * nb) % 2 == 0, 3)
    try:
        for K in (1, 2, 4):
            X = rng.standard_normal((K, n))
            want = pv.apply_block(h, 2, X)
            for side, bad in ((even, np.inf), (~even, np.nan)):
                Y = X.copy()
                Y[:, side] = bad                             # node 0 (and the last) among them
                got = pv.apply_block(h, 2, Y)
                assert (got[:, ~side] == want[:, ~side]).all() and not np.isfinite(got[:, side]).all()
    finally:
        pv.pevsl_finish(h)
        pv.pevsl_chebiter_free(ch)
        pv.csr_free(m)


@gpu
def test_layouts_set_by_hand_come_first():
    """On a tuned small matrix: a refused layout call changes no route, and a
    layout set by hand for a width (the single-column map among them, whatever
    width the call names) turns the one-launch solve of that width off."""
    D = sp.kron(_mass(600, 14, 600), sp.identity(3), format="csr")
    D.sort_indices()
    m = pv.csr_create(D.indptr, D.indices, D.data)
    ch = pv.pevsl_setup_chebiter(1.0, 3.0, 9, m)
    widths = (1, 2, 4)

    def routes():
        return [pv.product_route(m, K)[1] for K in widths]

    try:
        for K in widths:
            pv.csr_autotune(m, K, 2)
        assert routes() == [True] * 3
        for refused in (lambda: pv.set_kernel_map(m, 32, 3, 1), lambda: pv.set_kernel_map(m, 32, 4, 5),
                        lambda: pv.set_kernel_map(m, 7, 1, 1), lambda: pv.set_kernel_map(m, 0, 2, 64),
                        lambda: pv.set_tiling(m, 2, 1, 1), lambda: pv.set_tiling(m, 4, 10 ** 6, 1),
                        lambda: pv.set_tiling(m, 1, 500, 9), lambda: pv.set_tiled_wide(m, 4, 10 ** 6, 4),
                        lambda: pv.set_tiled_wide(m, 2, 1, 4), lambda: pv.set_wide(m, 2, 5),
                        lambda: pv.set_row_pipeline(m, 16, 2), lambda: pv.set_row_groups(m, 3)):
            with pytest.raises(pv.PevslError):
                refused()
            assert routes() == [True] * 3
        x = np.random.default_rng(1).standard_normal(D.shape[0])
        tuned = pv.pevsl_chebiter(2, x, ch)
        pv.set_kernel_map(m, 32, 4, 2)
        assert routes() == [False, True, False]
        hand = pv.pevsl_chebiter(2, x, ch)
        assert np.linalg.norm(hand - tuned) <= 1e-13 * np.linalg.norm(tuned)
        pv.set_kernel_map(m, 0, 4, 0)
        pv.set_kernel_map(m, 0, 1, 0)                      # what the tuner chose for one column, too
        pv.set_row_groups(m, 0)
        pv.set_tiling(m, 1, 0)
        assert routes() == [True] * 3
        pv.set_wide(m, 2, 8)
        assert routes() == [True, False, True]
        pv.set_wide(m, 2, 0)
        pv.set_kernel_map(m, 0, 2, 0)                      # the tuner's rows per wavefront go too
        pv.set_row_groups(m, 2)
        assert routes() == [False, True, True]
    finally:
        pv.pevsl_chebiter_free(ch)
        pv.csr_free(m)


@gpu
def test_many_bounds_on_one_matrix():
    """A matrix keeps the weights of 64 different solves, those set up again
    counting once; further ones run step by step.  All follow the recurrence."""
    D = sp.kron(_mass(200, 10, 3), sp.identity(3), format="csr")
    D.sort_indices()
    m = pv.csr_create(D.indptr, D.indices, D.data)
    b, lo, deg = np.random.default_rng(1).standard_normal(D.shape[0]), 1.0, 9
    try:
        for i in range(80):
            hi = 3.0 + 1e-3 * i
            th, sg = 0.5 * (lo + hi), (lo + hi) / (hi - lo)
            xm, xk, w = np.zeros_like(b), b / th, 2.0
            for _ in range(deg):
                w = 1.0 / (1.0 - w / (4.0 * sg * sg))
                xm, xk = xk, xm + w * (xk - xm + (b - D @ xk) / th)
            for _ in range(2):
                ch = pv.pevsl_setup_chebiter(lo, hi, deg, m)
                x = pv.pevsl_chebiter(2, b, ch)
                pv.pevsl_chebiter_free(ch)
                assert np.linalg.norm(x - xk) <= 1e-13 * np.linalg.norm(xk), i
    finally:
        pv.csr_free(m)
