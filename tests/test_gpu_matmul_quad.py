"""The quad-union kernel of SO_LAYOUT_RBM (csrc/matmul_quad.hip), forced, at the edges of its tiles: rows in quads of
4 and blocks of up to 64, tiles of 256 X rows, slabs of 64 dense columns in groups of 4, chunks of 16 steps in units of
4, every rows-per-workgroup and K-split choice.

Bound: max|y - ref| <= 1e-5 * max|ref| against the in-order oracle and the fp64 product, as for the layout's other
kernel (tests/test_gpu_matmul_rbm.py): the same products, summed in another order in fp32."""

import numpy as np
import pytest

from conftest import as_oracle, rel_err, sparse_matrix

import datagen
import hipabi

pytestmark = pytest.mark.gpu
TOL = 1e-5
RBM = hipabi.LAYOUT_ROW | hipabi.LAYOUT_RBM


def quad_matmul(ctx, E, X, bias, act="none", rows=None, split=None):
    m, C = E.m, X.shape[1]
    with ctx.tuning(SPARSEOPS_MATMUL_QUAD="1", SPARSEOPS_MATMUL_QUAD_ROWS=rows, SPARSEOPS_MATMUL_QUAD_SPLIT=split):
        dE = ctx.upload_ellpack(E.Wd, E.idx, E.nnz, E.m, E.n, E.r, RBM)
        dX, dY, dB = ctx.array(X), ctx.empty((m, C)), ctx.array(bias) if bias is not None else None
        outs = []
        for _ in range(2):
            dY.upload(np.full((m, C), np.nan, np.float32))
            ctx.matmul(dE, dX, C, dB, dY, act)
            assert ctx.last_kernel() == "quad"
            outs.append(dY.download())
        for a in (dX, dY, dB):
            if a is not None:
                a.free()
        dE.free()
    assert np.array_equal(outs[0], outs[1], equal_nan=True)
    return outs[0]


@pytest.mark.parametrize("m,n,C,sp", [
    (1, 1, 4, .0), (3, 2, 5, .0), (4, 255, 7, .5), (5, 256, 63, .5), (63, 257, 64, .9), (64, 300, 65, .7), (65, 511, 66, .3),
    (130, 513, 67, .95), (129, 1025, 130, .8), (300, 700, 256, .5), (257, 2100, 101, .6), (17, 4096, 12, .99), (1000, 512, 32, .0)])
@pytest.mark.parametrize("rows,split", [(None, None), (4, 1), (2, 3), (0, 2)])
def test_quad_shapes(ctx, oracle, m, n, C, sp, rows, split):
    rng = np.random.default_rng(m * 31 + n * 7 + C)
    W = sparse_matrix(rng, m, n, sp)
    X = rng.standard_normal((n, C)).astype(np.float32)
    b = rng.standard_normal(m).astype(np.float32)
    E = datagen.encode_dense(W)
    Y = quad_matmul(ctx, E, X, b, "relu" if split == 3 else "none", rows, split)
    ref = W.astype(np.float64) @ X + b[:, None]
    assert rel_err(Y, np.maximum(ref, 0) if split == 3 else ref) <= TOL
    assert rel_err(Y, oracle.matmul(as_oracle(E), X, b, "relu" if split == 3 else "none")) <= TOL


def test_quad_multiply_adds_are_fused_and_keep_subnormals(ctx, oracle):
    """Rows i of a quad with nonzeros in columns i and i + 4: union steps of one quarter of one chunk, so an output is
    one chain of two multiply-adds, and its bits are the in-order oracle's (fmaf) -- with weights, X and results below
    the normal range, and with second products that nearly cancel the first."""
    rng = np.random.default_rng(5)
    m, n, C = 512, 8, 64
    rows = np.arange(m)
    W = np.zeros((m, n), np.float32)
    for k in (0, 4):
        W[rows, rows % 4 + k] = np.ldexp(rng.uniform(1, 2, m), rng.integers(-148, 10, m))
    X = np.ldexp(rng.uniform(-2, 2, (n, C)), rng.integers(-148, 10, (n, C))).astype(np.float32)
    W[::2, :] = np.where(W[::2] != 0, rng.uniform(1, 2, (m // 2, n)), 0)
    X[4:, ::2] = -X[:4, ::2]
    W[::8, 4] = W[::8, 0] * np.float32(1 + 2.0 ** -22)
    E = datagen.encode_dense(W)
    want = oracle.matmul(as_oracle(E), X, None, "none")
    tiny = np.float32(np.finfo(np.float32).tiny)
    for a in (E.Wd, X, want):
        assert ((a != 0) & (np.abs(a) < tiny)).sum() > 10
    fused = W.astype(np.float64) @ X                       # products are exact here: what separate roundings would change
    assert (want != (W[rows, rows % 4, None] * X[rows % 4] + W[rows, rows % 4 + 4, None] * X[rows % 4 + 4])).sum() > 100
    assert np.abs(want - fused).max() <= 2.0 ** -23 * np.abs(fused).max()
    assert np.array_equal(quad_matmul(ctx, E, X, None), want)


def test_quad_unordered_repeated_and_special_values(ctx, oracle):
    """Reversed rows, a column that a row names twice, empty rows, a dense row; and an infinity in X reaches exactly
    the rows that use it, although a quad's other rows meet it with a zero weight."""
    rng = np.random.default_rng(11)
    m, n, C = 140, 600, 70
    W = sparse_matrix(rng, m, n, .8)
    W[7], W[9] = 0, rng.standard_normal(n)
    E = datagen.encode_dense(W)
    for i in range(0, m, 2):
        c = int(E.nnz[i])
        E.Wd[i, :c], E.idx[i, :c] = E.Wd[i, :c][::-1].copy(), E.idx[i, :c][::-1].copy()
    c = int(E.nnz[20])
    E.idx[20, 1] = E.idx[20, 0]
    Wd = np.zeros((m, n))
    for i in range(m):
        np.add.at(Wd[i], E.idx[i, :E.nnz[i]], E.Wd[i, :E.nnz[i]].astype(np.float64))
    X = rng.standard_normal((n, C)).astype(np.float32)
    assert rel_err(quad_matmul(ctx, E, X, None), Wd @ X) <= TOL
    X[0, :], X[17, 3], X[300, 5] = np.inf, -np.inf, np.nan
    E = datagen.encode_dense(W)
    for split in (1, 3):
        Y = quad_matmul(ctx, E, X, None, split=split)
        Yo = oracle.matmul(as_oracle(E), X, None)
        assert np.array_equal(np.isnan(Y), np.isnan(Yo)) and np.array_equal(np.isinf(Y), np.isinf(Yo))
        fin = np.isfinite(Yo)
        assert np.array_equal(Y[np.isinf(Yo)], Yo[np.isinf(Yo)])
        assert np.abs(Y[fin] - Yo[fin]).max() <= TOL * np.abs(Yo[fin]).max()


@pytest.mark.parametrize("C", [4, 5, 66, 131])
@pytest.mark.parametrize("n,sp", [(40, .5), (700, .8), (2100, .4)])
def test_quad_outputs_that_meet_a_foreign_infinity(ctx, C, n, sp):
    """Every column of X has an infinity in a row that half of the matrix's rows do not use: those outputs, NaN as computed
    with the quad's other rows, are computed again from the row's own nonzeros (up to 1260 of them, 16 lanes a row, groups
    of four columns, the last group past the end of X's rows), to the same bound."""
    rng = np.random.default_rng(n + C)
    m = 90
    W = sparse_matrix(rng, m, n, sp)
    j = n // 2
    W[:, j] = np.where(np.arange(m) % 3 == 1, 0, 2)
    W[17] = 0
    X = rng.standard_normal((n, C)).astype(np.float32)
    b = rng.standard_normal(m).astype(np.float32)
    E = datagen.encode_dense(W)
    X[j] = 0
    ref = W.astype(np.float64) @ X + b[:, None]
    X[j] = np.where(np.arange(C) % 2, np.inf, -np.inf)
    Y = quad_matmul(ctx, E, X, b)
    uses = W[:, j] != 0
    assert np.array_equal(Y[uses], np.repeat(X[j][None], uses.sum(), axis=0))
    assert rel_err(Y[~uses], ref[~uses]) <= TOL


def test_quad_in_a_launch_graph(ctx, oracle):
    """so_matmul_reserve sizes the workspace of a K split ahead of a recording; replays give the eager launch's bits."""
    rng = np.random.default_rng(3)
    W = sparse_matrix(rng, 300, 1100, .7)
    E = datagen.encode_dense(W)
    C = 40
    with ctx.tuning(SPARSEOPS_MATMUL_QUAD="1", SPARSEOPS_MATMUL_QUAD_SPLIT="4"):
        dE = ctx.upload_ellpack(E.Wd, E.idx, E.nnz, E.m, E.n, E.r, RBM)
        dX, dY = ctx.empty((1100, C)), ctx.empty((300, C))
        ctx.matmul_reserve(dE, C)
        ctx.graph_begin()
        ctx.matmul(dE, dX, C, None, dY, "tanh")
        assert ctx.last_kernel() == "quad"
        g = ctx.graph_end()
        for _ in range(3):
            X = rng.standard_normal((1100, C)).astype(np.float32) * 0.1
            dX.upload(X)
            ctx.matmul(dE, dX, C, None, dY, "tanh")
            eager = dY.download()
            ctx.fill_zero(dY)
            ctx.sync()
            ctx.graph_launch(g)
            assert np.array_equal(dY.download(), eager)
            # tanh's slope is at most 1: the sums' bound carries over, plus the device tanhf's 1e-6
            pre = np.abs(oracle.matmul(as_oracle(E), X, None)).max()
            assert np.abs(eager - np.tanh(W.astype(np.float64) @ X)).max() <= TOL * pre + 1e-6
        ctx.graph_free(g)
        for a in (dX, dY):
            a.free()
        dE.free()


@pytest.mark.parametrize("m,n,per_row,quads", [(65536, 65536, 10, False), (2048, 16384, 16, False), (2048, 16384, 60, False),
                                               (2048, 16384, 400, True), (300, 9000, 3, True)])
def test_very_sparse_matrices_do_without_the_quads(ctx, oracle, m, n, per_row, quads):
    """Few nonzeros per (quad, 256 columns): the copy would be many times the matrix.  By the table's size alone, by the
    chunks counted, and not: dense enough, too small to matter.  The handle works either way, forced or not."""
    rng = np.random.default_rng(per_row)
    idx = np.sort(rng.choice(n // per_row, (m, per_row)).astype(np.uint32) + np.arange(per_row, dtype=np.uint32) * (n // per_row), axis=1)
    Wd, nnz = rng.standard_normal((m, per_row)).astype(np.float32), np.full(m, per_row, np.uint32)
    X = rng.standard_normal((n, 8)).astype(np.float32)
    dE = ctx.upload_ellpack(Wd, idx, nnz, m, n, per_row, RBM)
    dX, dY = ctx.array(X), ctx.empty((m, 8))
    ref = (Wd[:, :, None].astype(np.float64) * X[idx]).sum(axis=1)
    for forced in (None, "1"):
        with ctx.tuning(SPARSEOPS_MATMUL_QUAD=forced):
            ctx.matmul_reserve(dE, 8)
            ctx.matmul(dE, dX, 8, None, dY)
            assert forced is None or (ctx.last_kernel() == "quad") == quads
            assert rel_err(dY.download(), ref) <= TOL
    for a in (dX, dY, dE):
        a.free()


@pytest.mark.parametrize("forced", [None, "SPARSEOPS_MATMUL_QUAD", "SPARSEOPS_MATMUL_RBM"])
def test_no_columns(ctx, forced):
    """A matrix without columns has no row of X to read: the layout's kernels, which read ahead, are not for it."""
    b = np.linspace(-1, 1, 300).astype(np.float32)
    E = datagen.encode_dense(np.zeros((300, 0), np.float32))
    with ctx.tuning(**({forced: "1"} if forced else {})):
        dE = ctx.upload_ellpack(E.Wd, E.idx, E.nnz, 300, 0, E.r, RBM)
        dX, dB = ctx.empty((4,)), ctx.array(b)
        for C in (1, 64, 130):
            dY = ctx.array(np.full((300, C), np.nan, np.float32))
            ctx.matmul_reserve(dE, C)
            ctx.matmul(dE, dX, C, dB, dY, "relu")
            assert ctx.last_kernel() in ("row", "shared")
            assert np.array_equal(dY.download(), np.repeat(np.maximum(b, 0)[:, None], C, axis=1))
            dY.free()
        for a in (dX, dB, dE):
            a.free()


def test_recording_without_a_reservation(oracle):
    """A launch that is too small for the row-block-merged kernel can be recorded on a context that has no workspace yet;
    with the reservation it is recorded on the kernel that an eager launch takes."""
    rng = np.random.default_rng(9)
    E = datagen.encode_dense(sparse_matrix(rng, 512, 4000, .6))
    C = 16
    X = rng.standard_normal((4000, C)).astype(np.float32)
    c = hipabi.Context()
    dE = c.upload_ellpack(E.Wd, E.idx, E.nnz, E.m, E.n, E.r, RBM)
    dX, dY = c.array(X), c.empty((512, C))
    want = oracle.matmul(as_oracle(E), X, None)
    for reserved in (False, True):
        if reserved:
            c.matmul_reserve(dE, C)
        c.graph_begin()
        try:
            c.matmul(dE, dX, C, None, dY)
            assert c.last_kernel() == ("quad" if reserved else "row")
        finally:
            g = c.graph_end()
        for _ in range(2):
            c.fill_zero(dY)
            c.graph_launch(g)
            Y = dY.download()
            assert rel_err(Y, want) <= TOL
        c.graph_free(g)
    c.matmul(dE, dX, C, None, dY)
    assert np.array_equal(dY.download(), Y) and not np.array_equal(Y, want)      # another order of summation than the oracle's
    for a in (dX, dY, dE):
        a.free()
    c.close()


def test_reserved_workspace_stays_reserved():
    """A matrix that needs more counters and smaller partial tiles than the one reserved before it: both can be recorded."""
    rng = np.random.default_rng(6)
    C = 64
    c = hipabi.Context()
    cases = [(3840, 2100, "4", "8"), (4400, 600, "0", "2")]        # 60 tiles of 8 x 16 KB; 1100 of 2 x 1 KB
    handles = []
    for m, n, rows, split in cases:
        E = datagen.encode_dense(sparse_matrix(rng, m, n, .97))
        handles.append((c.upload_ellpack(E.Wd, E.idx, E.nnz, E.m, E.n, E.r, RBM), c.array(rng.standard_normal((n, C)).astype(np.float32)), c.empty((m, C))))
    for (m, n, rows, split), (dE, _, _) in zip(cases, handles):
        with c.tuning(SPARSEOPS_MATMUL_QUAD="1", SPARSEOPS_MATMUL_QUAD_ROWS=rows, SPARSEOPS_MATMUL_QUAD_SPLIT=split):
            c.matmul_reserve(dE, C)
    for (m, n, rows, split), (dE, dX, dY) in zip(cases, handles):
        with c.tuning(SPARSEOPS_MATMUL_QUAD="1", SPARSEOPS_MATMUL_QUAD_ROWS=rows, SPARSEOPS_MATMUL_QUAD_SPLIT=split):
            c.graph_begin()
            try:
                c.matmul(dE, dX, C, None, dY)
            finally:
                g = c.graph_end()
            c.matmul(dE, dX, C, None, dY)
            eager = dY.download()
            c.fill_zero(dY)
            c.graph_launch(g)
            assert np.array_equal(dY.download(), eager)
            c.graph_free(g)
    for h in handles:
        for a in h:
            a.free()
    c.close()


@pytest.mark.parametrize("kernel", ["SPARSEOPS_MATMUL_QUAD", "SPARSEOPS_MATMUL_RBM"])
def test_recorded_graph_outlives_its_workspace(ctx, kernel):
    """A larger launch makes the context's workspace grow; a graph recorded before keeps the one it was recorded with, so
    its replays still give the eager launch's bits, and leave alone what was allocated since."""
    rng = np.random.default_rng(5)
    C = 40
    small, large = (datagen.encode_dense(sparse_matrix(rng, m, n, .7)) for m, n in ((300, 1100), (900, 3000)))
    with ctx.tuning(**{kernel: "1", "SPARSEOPS_MATMUL_QUAD_SPLIT": "4", "SPARSEOPS_MATMUL_RBM_SPLIT": "4"}):
        dS, dL = (ctx.upload_ellpack(E.Wd, E.idx, E.nnz, E.m, E.n, E.r, RBM) for E in (small, large))
        dX, dY = ctx.array(rng.standard_normal((1100, C)).astype(np.float32)), ctx.empty((300, C))
        ctx.matmul(dS, dX, C, None, dY, "relu")
        assert ctx.last_kernel() == ("quad" if "QUAD" in kernel else "merged")
        eager = dY.download()
        ctx.graph_begin()
        ctx.matmul(dS, dX, C, None, dY, "relu")
        g = ctx.graph_end()
        arrays = [dX, dY]
        for Cl in (64, 700, 5000):
            Xl = ctx.array(rng.standard_normal((3000, Cl)).astype(np.float32))
            Yl = ctx.empty((900, Cl))
            ctx.matmul(dL, Xl, Cl, None, Yl, "none")
            Y0 = Yl.download()
            filler = [ctx.array(np.full(1 << k, 3, np.float32)) for k in range(10, 22)]
            for _ in range(3):
                ctx.fill_zero(dY)
                ctx.graph_launch(g)
                assert np.array_equal(dY.download(), eager)
            assert all((f.download() == 3).all() for f in filler)
            ctx.matmul(dL, Xl, Cl, None, Yl, "none")
            assert np.array_equal(Yl.download(), Y0)
            arrays += [Xl, Yl] + filler
        ctx.graph_free(g)
        for a in arrays + [dS, dL]:
            a.free()


@pytest.mark.parametrize("m,n,C,sp", [(1, 64, 1, .0), (5, 4097, 3, .5), (16, 70, 1, .0), (130, 513, 2, .5), (257, 700, 3, .7), (1000, 1025, 1, .8),
                                      (65, 50000, 2, .99), (4100, 300, 3, .3)])
@pytest.mark.parametrize("act", ["none", "relu", "sigmoid", "tanh"])
@pytest.mark.parametrize("idx16", [False, True])
def test_few_columns_on_the_matvec_kernel(ctx, oracle, m, n, C, sp, act, idx16):
    """One to three columns: a row over the lanes of a wave or a part of one, x in LDS or not, an infinity in X in the rows
    that use it only.  The activations' slopes are at most 1: the sums' bound carries over, plus the device functions' 1e-6."""
    rng = np.random.default_rng(m + n)
    W = sparse_matrix(rng, m, n, sp)
    if m > 4:
        W[m // 2] = 0
    W[0, 0] = 1.0
    E = datagen.encode_dense(W)
    X = rng.standard_normal((n, C)).astype(np.float32)
    b = rng.standard_normal(m).astype(np.float32)
    dE = ctx.upload_ellpack(E.Wd, E.idx, E.nnz, E.m, E.n, E.r, RBM | (hipabi.LAYOUT_IDX16 if idx16 else 0))
    dX, dY, dB = ctx.array(X), ctx.empty((m, C)), ctx.array(b)
    pre = np.abs(W.astype(np.float64) @ X + b[:, None]).max()
    for special in (False, True):
        if special:
            X[0, C - 1] = np.inf
            dX.upload(X)
        dY.upload(np.full((m, C), np.nan, np.float32))
        ctx.matmul(dE, dX, C, dB, dY, act)
        assert ctx.last_kernel() == "vector"
        Y, Yo = dY.download(), oracle.matmul(as_oracle(E), X, b, act)
        fin = np.isfinite(Yo)
        assert np.array_equal(Y[~fin], Yo[~fin], equal_nan=True)
        assert np.abs(Y[fin] - Yo[fin]).max(initial=0.0) <= TOL * pre + 1e-6
    for a in (dX, dY, dB):
        a.free()
    dE.free()
