"""The narrow kernel of SO_LAYOUT_RBM (csrc/matmul_narrow.hip): up to 32 dense columns, or slabs of 16 and 32, forced, at the edges of its column
groups (4, 8, 16, 32), its copy of X (4096 and 10 240 groups of four values; rows of no multiple of four), its chunks of 16
steps and batches of 4 chunks, its tiles of 256 columns and 4 rows and its quads per workgroup (more than 1024 rows: two); and
which calls it takes by itself.

Bound: max|y - ref| <= 1e-5 * max|ref|, as for the layout's other kernels (tests/test_gpu_matmul_quad.py)."""
import numpy as np
import pytest

from conftest import as_oracle, rel_err, sparse_matrix

import datagen
import hipabi

pytestmark = pytest.mark.gpu
TOL = 1e-5
RBM = hipabi.LAYOUT_ROW | hipabi.LAYOUT_RBM


def narrow_matmul(ctx, E, X, bias, act="none", at=0):
    """`at`: floats by which X and Y are off a 16-byte boundary."""
    m, (n, C) = E.m, X.shape
    dE = ctx.upload_ellpack(E.Wd, E.idx, E.nnz, E.m, E.n, E.r, RBM)
    flat = ctx.array(np.concatenate([np.full(at, np.nan, np.float32), X.ravel(), np.full(4, np.nan, np.float32)]))
    out, dB = ctx.array(np.full(at + m * C + 4, 7.0, np.float32)), ctx.array(bias) if bias is not None else None
    with ctx.tuning(SPARSEOPS_MATMUL_NARROW="1"):
        for _ in range(2):
            ctx.matmul(dE, flat.offset(at), C, dB, out.offset(at), act)
            assert ctx.last_kernel() == "narrow"
    Y = out.download()
    assert (Y[:at] == 7.0).all() and (Y[at + m * C:] == 7.0).all()
    for a in (flat, out, dB, dE):
        if a is not None:
            a.free()
    return Y[at:at + m * C].reshape(m, C)


@pytest.mark.parametrize("m,n,C,sp", [
    (1, 1, 1, .0), (1, 1, 3, .0), (3, 2, 4, .0), (4, 255, 5, .5), (5, 256, 8, .5), (63, 257, 9, .5), (64, 300, 16, .7), (65, 511, 17, .3), (130, 513, 31, .95),
    (129, 1025, 32, .8), (300, 10240, 4, .9), (20, 10240, 3, .5), (17, 5120, 8, .99), (40, 2560, 13, .2), (1000, 1280, 30, .6), (1025, 700, 2, .5),
    (2049, 600, 7, .9), (10, 2560, 36, .5), (77, 1280, 64, .6), (130, 900, 100, .7), (500, 513, 132, .9), (4097, 512, 12, .7), (16400, 300, 6, .9), (33000, 260, 4, .97)])
@pytest.mark.parametrize("at", [0, 1])
def test_narrow_shapes(ctx, oracle, m, n, C, sp, at):
    rng = np.random.default_rng(m * 31 + n * 7 + C)
    W = sparse_matrix(rng, m, n, sp)
    if m > 8:
        W[4:8] = 0                                   # a quad without nonzeros
    X = rng.standard_normal((n, C)).astype(np.float32)
    b = rng.standard_normal(m).astype(np.float32)
    E = datagen.encode_dense(W)
    ref = W.astype(np.float64) @ X + b[:, None]
    assert rel_err(narrow_matmul(ctx, E, X, b, "none", at), ref) <= TOL
    assert rel_err(narrow_matmul(ctx, E, X, None, "relu", at), np.maximum(ref - b[:, None], 0)) <= TOL
    # slopes of at most 1: the sums' bound carries over, plus the device functions' 1e-6
    Y, want = narrow_matmul(ctx, E, X, b, "tanh", at), oracle.matmul(as_oracle(E), X, b, "tanh")
    assert np.abs(Y - want).max() <= TOL * np.abs(ref).max() + 1e-6


@pytest.mark.parametrize("C", [3, 8, 14, 32])
def test_values_that_are_not_finite(ctx, oracle, C):
    """A zero weight in the union times an infinity or a NaN leaves nothing behind; a nonzero one does."""
    rng = np.random.default_rng(C)
    W = sparse_matrix(rng, 203, 300, .8)
    E = datagen.encode_dense(W)
    X = rng.standard_normal((300, C)).astype(np.float32)
    X[7, C - 1], X[100, 0], X[299, 1] = np.inf, np.nan, -np.inf
    b = rng.standard_normal(203).astype(np.float32)
    Y, want = narrow_matmul(ctx, E, X, b), oracle.matmul(as_oracle(E), X, b)
    fin = np.isfinite(want)
    assert np.array_equal(Y[~fin], want[~fin], equal_nan=True) and fin.any() and not fin.all()
    assert np.abs(Y[fin] - want[fin]).max() <= TOL * np.abs(want[fin]).max()


@pytest.mark.parametrize("C,n", [(36, 300), (100, 300), (36, 1300), (100, 1300), (64, 2560)])
def test_values_that_are_not_finite_in_slabs(ctx, oracle, C, n):
    """The same with more than 32 columns: slabs of 16 or 32 where n rows of 32 columns fit into LDS, else of 16, the last of them partial;
    in its last column, in one before it and in another slab."""
    rng = np.random.default_rng(C)
    W = sparse_matrix(rng, 203, n, .8)
    E = datagen.encode_dense(W)
    X = rng.standard_normal((n, C)).astype(np.float32)
    X[7, C - 1], X[9, C - 3], X[n - 1, C // 2], X[100, 1] = np.inf, -np.inf, np.nan, np.inf
    b = rng.standard_normal(203).astype(np.float32)
    Y, want = narrow_matmul(ctx, E, X, b), oracle.matmul(as_oracle(E), X, b)
    fin = np.isfinite(want)
    assert np.array_equal(Y[~fin], want[~fin], equal_nan=True) and fin.any() and not fin.all()
    assert np.abs(Y[fin] - want[fin]).max() <= TOL * np.abs(want[fin]).max()


@pytest.mark.parametrize("m,n,C,sp", [(2847, 1952, 8, .6), (1067, 900, 28, .6), (256, 1136, 36, .7), (2000, 1500, 3, .5)])
def test_time_with_values_that_are_not_finite(ctx, m, n, C, sp):
    """An infinity in every column: groups of four columns of four rows are computed again at a time, not output by output."""
    rng = np.random.default_rng(3)
    E = datagen.encode_dense(sparse_matrix(rng, m, n, sp))
    X = rng.standard_normal((n, C)).astype(np.float32)
    dE, dX, dY = ctx.upload_ellpack(E.Wd, E.idx, E.nnz, E.m, E.n, E.r, RBM), ctx.array(X), ctx.empty((m, C))

    def shortest():
        ms = []
        for _ in range(5):
            ctx.timer_begin()
            for _ in range(10):
                ctx.matmul(dE, dX, C, None, dY)
            ms.append(ctx.timer_end())
        return min(ms)
    with ctx.tuning(SPARSEOPS_MATMUL_NARROW="1"):
        shortest()
        before = shortest()
        X[rng.integers(0, n, C), np.arange(C)] = np.inf
        dX.upload(X)
        assert shortest() <= 6.5 * before
    for a in (dX, dY, dE):
        a.free()


@pytest.mark.parametrize("C,want", [(65535 * 16, "narrow"), (65535 * 16 + 4, None), (2 ** 20, None)])
def test_very_wide(ctx, C, want):
    """A grid has at most 65 535 workgroups in y: slabs of 16 columns, all that fit beside more than 1280 rows of X, end at 1 048 560."""
    n, cols = 1281, np.array([0, 700, 1280], np.uint32)
    Wd = np.array([[1.5, -2.0, 0.75]], np.float32)
    rows = np.random.default_rng(C).standard_normal((3, C)).astype(np.float32)
    dE, dX, dY = ctx.upload_ellpack(Wd, cols[None], np.array([3], np.uint32), 1, n, 3, RBM), ctx.empty((n, C)), ctx.empty((1, C))
    ctx.fill_zero(dX)
    for k, x in zip(cols, rows):
        ctx._ck(ctx.lib.so_h2d(ctx.h, dX.ptr + 4 * int(k) * C, hipabi._ptr(x), x.nbytes))
    with ctx.tuning(SPARSEOPS_MATMUL_NARROW="1"):
        ctx.matmul(dE, dX, C, None, dY)
        assert (ctx.last_kernel() == "narrow") == (want == "narrow")
    assert rel_err(dY.download(), Wd.astype(np.float64) @ rows) <= TOL
    for a in (dX, dY, dE):
        a.free()


def test_rows_in_any_order(ctx, oracle):
    """Columns of a row unordered and named twice: two steps of the union."""
    rng = np.random.default_rng(2)
    m, n, r = 90, 700, 40
    idx = rng.integers(0, n, (m, r)).astype(np.uint32)
    idx[:, 1] = idx[:, 0]
    Wd, nnz = rng.standard_normal((m, r)).astype(np.float32), np.full(m, r, np.uint32)
    X = rng.standard_normal((n, 10)).astype(np.float32)
    ref = (Wd[:, :, None].astype(np.float64) * X[idx]).sum(axis=1)
    dE, dX, dY = ctx.upload_ellpack(Wd, idx, nnz, m, n, r, RBM), ctx.array(X), ctx.empty((m, 10))
    with ctx.tuning(SPARSEOPS_MATMUL_NARROW="1"):
        ctx.matmul(dE, dX, 10, None, dY)
        assert ctx.last_kernel() == "narrow"
    assert rel_err(dY.download(), ref) <= TOL
    for a in (dX, dY, dE):
        a.free()


@pytest.mark.parametrize("m,n,C,sp,want", [(2000, 1500, 8, .6, True), (2000, 1500, 33, .6, False), (2000, 1500, 64, .6, False), (84, 692, 148, .5, True), (84, 692, 149, .5, False), (2000, 2600, 16, .6, False), (2000, 600, 30, .97, False),
                                           (2000, 1500, 3, .5, True), (300, 1500, 3, .5, False), (2000, 1500, 1, .5, False),
                                           (2126, 531, 17, .85, False), (4, 1792, 3780, .8, False), (12, 2172, 1860, .7, False)])
def test_which_calls_take_it(ctx, m, n, C, sp, want):
    """Also while a graph is recorded (no workspace is needed), whose replays give the same bits."""
    rng = np.random.default_rng(m + n)
    W = sparse_matrix(rng, m, n, sp)
    E = datagen.encode_dense(W)
    X = rng.standard_normal((n, C)).astype(np.float32)
    dE, dX, dY = ctx.upload_ellpack(E.Wd, E.idx, E.nnz, E.m, E.n, E.r, RBM), ctx.array(X), ctx.empty((m, C))
    ctx.matmul_reserve(dE, C)
    ctx.matmul(dE, dX, C, None, dY)
    assert (ctx.last_kernel() == "narrow") == want
    Y = dY.download()
    assert rel_err(Y, W.astype(np.float64) @ X) <= TOL
    ctx.graph_begin()
    try:
        ctx.matmul(dE, dX, C, None, dY)
    finally:
        g = ctx.graph_end()
    for _ in range(3):
        ctx.fill_zero(dY)
        ctx.graph_launch(g)
        assert np.array_equal(dY.download(), Y)
    ctx.graph_free(g)
    for name in ("SPARSEOPS_MATMUL_NARROW", "SPARSEOPS_MATMUL_QUAD", "SPARSEOPS_MATMUL_RBM"):
        with ctx.tuning(**{name: "0"}):
            ctx.matmul(dE, dX, C, None, dY)
            assert ctx.last_kernel() != "narrow"
    for a in (dX, dY, dE):
        a.free()


@pytest.mark.parametrize("m,n,C,sp,want", [(979, 223, 19, .57, False), (7064, 109, 31, .7, False), (123, 168, 23, .54, False), (3280, 171, 19, .89, False), (8815, 295, 29, .48, True),
                                           (2818, 728, 32, .42, True), (979, 223, 8, .57, True)])
def test_wide_slabs_of_small_launches(ctx, m, n, C, sp, want):
    """17 to 32 columns: launches of 3.4 to 4.6 us on the columns or row kernel took up to a fifth longer here; those of 7.6 and more stay."""
    rng = np.random.default_rng(m + n)
    W = sparse_matrix(rng, m, n, sp)
    E = datagen.encode_dense(W)
    X = rng.standard_normal((n, C)).astype(np.float32)
    dE, dX, dY = ctx.upload_ellpack(E.Wd, E.idx, E.nnz, E.m, E.n, E.r, RBM), ctx.array(X), ctx.empty((m, C))
    ctx.matmul_reserve(dE, C)
    ctx.matmul(dE, dX, C, None, dY)
    assert (ctx.last_kernel() == "narrow") == want
    assert rel_err(dY.download(), W.astype(np.float64) @ X) <= TOL
    for a in (dX, dY, dE):
        a.free()
