"""The quad-union copy's kernel with X in LDS a part at a time (csrc/matmul_narrow.hip), forced, with slabs of 16 and 32 columns: at the edges of its
parts (1280 and 512 rows of X), its slabs, its chunks of 16 steps and batches of 4 chunks, its quads per workgroup; with C of no multiple of four, whose
last groups overhang X; and which calls it takes by itself.

Bound: max|y - ref| <= 1e-5 * max|ref|, as for the layout's other kernels (tests/test_gpu_matmul_quad.py)."""
import numpy as np
import pytest

from conftest import as_oracle, rel_err, sparse_matrix

import datagen
import hipabi

pytestmark = pytest.mark.gpu
TOL = 1e-5
RBM = hipabi.LAYOUT_ROW | hipabi.LAYOUT_RBM


def slabs_matmul(ctx, E, X, bias, slab, act="none", at=0):
    """`at`: floats by which X and Y are off a 16-byte boundary.  X ends right before a NaN, Y before a value that has to stay."""
    m, (n, C) = E.m, X.shape
    dE = ctx.upload_ellpack(E.Wd, E.idx, E.nnz, E.m, E.n, E.r, RBM)
    flat = ctx.array(np.concatenate([np.full(at, np.nan, np.float32), X.ravel(), np.full(4, np.nan, np.float32)]))
    out, dB = ctx.array(np.full(at + m * C + 4, 7.0, np.float32)), ctx.array(bias) if bias is not None else None
    with ctx.tuning(SPARSEOPS_MATMUL_SLABS=slab):
        for _ in range(2):
            ctx.matmul(dE, flat.offset(at), C, dB, out.offset(at), act)
            assert ctx.last_kernel() == "slabs"
    Y = out.download()
    assert (Y[:at] == 7.0).all() and (Y[at + m * C:] == 7.0).all()
    for a in (flat, out, dB, dE):
        if a is not None:
            a.free()
    return Y[at:at + m * C].reshape(m, C)


@pytest.mark.parametrize("m,n,C,sp", [
    (1, 1, 4, .0), (3, 2, 5, .0), (5, 511, 4, .5), (20, 512, 7, .5), (63, 513, 16, .5), (64, 1023, 17, .7), (65, 1024, 33, .3), (130, 1025, 31, .95), (4, 2048, 6, .5),
    (129, 2049, 32, .8), (300, 4100, 13, .9), (20, 10240, 19, .5), (17, 5120, 40, .99), (40, 2560, 69, .2), (1000, 1280, 30, .6), (1025, 700, 45, .5),
    (2049, 1600, 50, .9), (77, 1280, 64, .6), (130, 3000, 101, .7), (500, 513, 131, .9), (4097, 512, 22, .7), (16400, 300, 10, .9)])
@pytest.mark.parametrize("slab", ["4", "8"])
@pytest.mark.parametrize("at", [0, 1])
def test_slabs_shapes(ctx, oracle, m, n, C, sp, slab, at):
    rng = np.random.default_rng(m * 31 + n * 7 + C)
    W = sparse_matrix(rng, m, n, sp)
    if m > 8:
        W[4:8] = 0                                   # a quad without nonzeros
        W[8:12, :n // 2] = 0                         # and one without any in its first parts
    X = rng.standard_normal((n, C)).astype(np.float32)
    b = rng.standard_normal(m).astype(np.float32)
    E = datagen.encode_dense(W)
    ref = W.astype(np.float64) @ X + b[:, None]
    assert rel_err(slabs_matmul(ctx, E, X, b, slab, "none", at), ref) <= TOL
    assert rel_err(slabs_matmul(ctx, E, X, None, slab, "relu", at), np.maximum(ref - b[:, None], 0)) <= TOL
    # slopes of at most 1: the sums' bound carries over, plus the device functions' 1e-6
    Y, want = slabs_matmul(ctx, E, X, b, slab, "tanh", at), oracle.matmul(as_oracle(E), X, b, "tanh")
    assert np.abs(Y - want).max() <= TOL * np.abs(ref).max() + 1e-6


@pytest.mark.parametrize("slab", ["4", "8"])
@pytest.mark.parametrize("n,C", [(300, 5), (1300, 36), (2560, 101)])
def test_values_that_are_not_finite(ctx, oracle, n, C, slab):
    """A zero weight in the union times an infinity or a NaN leaves nothing behind; a nonzero one does."""
    rng = np.random.default_rng(C)
    W = sparse_matrix(rng, 203, n, .8)
    E = datagen.encode_dense(W)
    X = rng.standard_normal((n, C)).astype(np.float32)
    X[7, C - 1], X[9, C - 3], X[n - 1, C // 2], X[100, 1], X[n - 1, C - 1] = np.inf, -np.inf, np.nan, np.inf, np.inf
    b = rng.standard_normal(203).astype(np.float32)
    Y, want = slabs_matmul(ctx, E, X, b, slab), oracle.matmul(as_oracle(E), X, b)
    fin = np.isfinite(want)
    assert np.array_equal(Y[~fin], want[~fin], equal_nan=True) and fin.any() and not fin.all()
    assert np.abs(Y[fin] - want[fin]).max() <= TOL * np.abs(want[fin]).max()


def test_rows_in_any_order(ctx):
    """Columns of a row unordered and named twice: two steps of the union."""
    rng = np.random.default_rng(2)
    m, n, r = 90, 1500, 40
    idx = rng.integers(0, n, (m, r)).astype(np.uint32)
    idx[:, 1] = idx[:, 0]
    Wd, nnz = rng.standard_normal((m, r)).astype(np.float32), np.full(m, r, np.uint32)
    X = rng.standard_normal((n, 10)).astype(np.float32)
    ref = (Wd[:, :, None].astype(np.float64) * X[idx]).sum(axis=1)
    for slab in ("4", "8"):
        assert rel_err(slabs_matmul(ctx, datagen.EllpackHost(m, n, r, Wd, idx, nnz), X, None, slab), ref) <= TOL


@pytest.mark.parametrize("m,n,C,sp,want", [(84, 692, 149, .5, True), (12, 1238, 173, .55, True), (2000, 2600, 16, .6, True), (17, 1090, 28, .67, True),
                                           (300, 300, 300, .9, False), (2000, 1500, 8, .6, False), (40, 4000, 83, .78, False), (200, 1500, 3, .5, False)])
def test_which_calls_take_it(ctx, m, n, C, sp, want):
    """By name; forbidding it changes the bits.  Recorded after a reservation, whose replays give the same bits."""
    rng = np.random.default_rng(m + n)
    W = sparse_matrix(rng, m, n, sp)
    E = datagen.encode_dense(W)
    X = rng.standard_normal((n, C)).astype(np.float32)
    dE, dX, dY = ctx.upload_ellpack(E.Wd, E.idx, E.nnz, E.m, E.n, E.r, RBM), ctx.array(X), ctx.empty((m, C))
    ctx.matmul_reserve(dE, C)
    bits = {}
    for slabs in (None, "0", "4", "8"):
        with ctx.tuning(SPARSEOPS_MATMUL_SLABS=slabs):
            ctx.matmul(dE, dX, C, None, dY)
            assert (ctx.last_kernel() == "slabs") == (want if slabs is None else slabs != "0" and C >= 4)
            bits[slabs] = dY.download()
            assert rel_err(bits[slabs], W.astype(np.float64) @ X) <= TOL
    assert (not np.array_equal(bits[None], bits["0"])) == want
    assert not want or np.array_equal(bits[None], bits["4"]) or np.array_equal(bits[None], bits["8"])
    ctx.graph_begin()
    try:
        ctx.matmul(dE, dX, C, None, dY)
    finally:
        g = ctx.graph_end()
    for _ in range(3):
        ctx.fill_zero(dY)
        ctx.graph_launch(g)
        assert np.array_equal(dY.download(), bits[None])
    ctx.graph_free(g)
    for a in (dX, dY, dE):
        a.free()


@pytest.mark.parametrize("m,n,C,sp", [(4, 1187, 3347, .82), (5, 2003, 1119, .84), (4, 1280, 4095, .6), (9, 956, 2264, .67), (35, 944, 1329, .62)])
def test_slabs_of_a_large_x(ctx, m, n, C, sp):
    """X beyond an XCD's L2 (4.7 to 20 MB): slabs, in parts or whole, were up to 1.7 times as slow as what runs without them."""
    rng = np.random.default_rng(m + C)
    W = sparse_matrix(rng, m, n, sp)
    E = datagen.encode_dense(W)
    X = rng.standard_normal((n, C)).astype(np.float32)
    dE, dX, dY = ctx.upload_ellpack(E.Wd, E.idx, E.nnz, E.m, E.n, E.r, RBM), ctx.array(X), ctx.empty((m, C))
    ctx.matmul_reserve(dE, C)
    ctx.matmul(dE, dX, C, None, dY)
    assert ctx.last_kernel() not in ("slabs", "narrow")
    assert rel_err(dY.download(), W.astype(np.float64) @ X) <= TOL
    for a in (dX, dY, dE):
        a.free()


@pytest.mark.parametrize("n,C", [(1279, 5), (1281, 5), (1281, 18), (1281, 39), (2559, 17), (2561, 6), (2561, 35), (3841, 4), (3841, 23), (3839, 50)])
@pytest.mark.parametrize("slab", ["4", "8"])
@pytest.mark.parametrize("m", [3, 90])
def test_last_parts_of_one_row(ctx, m, n, C, slab):
    """One row more or less than parts of 1280 rows: every row of the last part is its first one, and a group that overhangs X is read from four values before its end."""
    rng = np.random.default_rng(m + n + C)
    W = sparse_matrix(rng, m, n, .6)
    W[:, n - 1] = 1 + np.arange(m)
    X = rng.standard_normal((n, C)).astype(np.float32)
    b = rng.standard_normal(m).astype(np.float32)
    ref = W.astype(np.float64) @ X + b[:, None]
    for at in (0, 1, 2, 3):
        assert rel_err(slabs_matmul(ctx, datagen.encode_dense(W), X, b, slab, "none", at), ref) <= TOL
