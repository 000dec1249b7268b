"""The kernel with X in LDS for few dense columns (csrc/matmul_columns.hip), bit for bit against the oracle: one, two and four rows
per wave, rows of no and all columns, groups of 16 entries that end anywhere, row counts no multiple of a workgroup's, four to
sixteen waves, X and Y at any word, the largest X that fits; which launches it is chosen for."""

import numpy as np
import pytest

from conftest import as_oracle, rel_err, sparse_matrix

import datagen
import hipabi

pytestmark = pytest.mark.gpu


def _matrix(rng, m, n, sp):
    W = sparse_matrix(rng, m, n, sp)
    W[m // 2] = 0
    W[m // 3] = rng.standard_normal(n)
    return datagen.encode_dense(W)


def _run(ctx, E, X, bias, act, off=0, layouts=hipabi.LAYOUT_ROW, **tuning):
    n, C = X.shape
    dE = ctx.upload_ellpack(E.Wd, E.idx, E.nnz, E.m, E.n, E.r, layouts)
    dX, dY, dB = ctx.empty((n * C + off,)), ctx.empty((E.m * C + off,)), ctx.array(bias) if bias is not None else None
    dX.upload(np.concatenate([np.full(off, np.nan, np.float32), X.ravel()]))
    dY.upload(np.full(E.m * C + off, np.float32(7.5)))

    class At:
        def __init__(self, a):
            self.ptr = a.ptr + 4 * off

    with ctx.tuning(**tuning):
        ctx.matmul(dE, At(dX), C, dB, At(dY), act)
    kernel, Y = ctx.last_kernel(), dY.download()
    assert (Y[:off] == 7.5).all()
    for a in (dE, dX, dY) + ((dB,) if dB else ()):
        a.free()
    return kernel, Y[off:].reshape(E.m, C)


@pytest.mark.parametrize("m,n,sp", [(1, 1, 0.), (3, 17, .2), (67, 129, .6), (1000, 512, .0), (1500, 600, .8), (4099, 300, .9), (33, 2400, .5)])
@pytest.mark.parametrize("C", [1, 4, 15, 16, 17, 32, 33, 64])
def test_bits(ctx, oracle, m, n, sp, C):
    if (n + 1) * C * 4 > 160 * 1024:
        C = 160 * 1024 // 4 // (n + 1)                       # the largest X that fits
    rng = np.random.default_rng(m + n + C)
    E = _matrix(rng, m, n, sp)
    X, b = rng.standard_normal((n, C)).astype(np.float32), rng.standard_normal(m).astype(np.float32)
    for bias, act, off in ((b, "none", 0), (None, "relu", 1), (b, "none", 3)):
        kernel, Y = _run(ctx, E, X, bias, act, off, SPARSEOPS_MATMUL_COLUMNS="1")
        assert kernel == "columns" and np.array_equal(Y, oracle.matmul(as_oracle(E), X, bias, act))
    assert rel_err(_run(ctx, E, X, b, "tanh", SPARSEOPS_MATMUL_COLUMNS="1")[1], oracle.matmul(as_oracle(E), X, b, "tanh")) <= 1e-6


def test_rows_in_any_order_and_values_that_are_not_finite(ctx, oracle):
    rng = np.random.default_rng(3)
    E = _matrix(rng, 200, 90, .5)
    for i in range(200):
        p = rng.permutation(int(E.nnz[i]))
        E.Wd[i, :len(p)], E.idx[i, :len(p)] = E.Wd[i, p], E.idx[i, p]
    X = rng.standard_normal((90, 20)).astype(np.float32)
    X[5], X[17, 3], X[0, 0], X[60] = np.inf, np.nan, -np.inf, 1e-42
    kernel, Y = _run(ctx, E, X, None, "none", SPARSEOPS_MATMUL_COLUMNS="1")
    assert kernel == "columns" and np.array_equal(Y, oracle.matmul(as_oracle(E), X, None, "none"), equal_nan=True)


@pytest.mark.parametrize("m,n,C,sp,layouts,kernel", [
    (1000, 512, 32, .0, hipabi.LAYOUT_ROW, "columns"), (300, 400, 64, .5, hipabi.LAYOUT_ROW, "columns"), (300, 400, 65, .5, hipabi.LAYOUT_ROW, "row"),
    (2000, 150, 8, .85, hipabi.LAYOUT_ROW, "row"), (100, 900, 60, .5, hipabi.LAYOUT_ROW, "shared"),
    (1771, 719, 18, .9, hipabi.LAYOUT_ROW | hipabi.LAYOUT_RBM, "columns"), (200, 2300, 11, .53, hipabi.LAYOUT_ROW | hipabi.LAYOUT_RBM, "quad")])
def test_chosen(ctx, m, n, C, sp, layouts, kernel):
    rng = np.random.default_rng(9)
    E = datagen.encode_dense(sparse_matrix(rng, m, n, sp))
    assert _run(ctx, E, rng.standard_normal((n, C)).astype(np.float32), None, "none", layouts=layouts)[0] == kernel


@pytest.mark.parametrize("m,n,C,mean,longest,layouts,kernel", [
    (50000, 600, 64, 8, 64, hipabi.LAYOUT_ROW, "row"), (200000, 600, 64, 5, 48, hipabi.LAYOUT_ROW, "row"), (16000, 600, 60, 2, 48, hipabi.LAYOUT_ROW, "row"),
    (100000, 2000, 16, 6, 64, hipabi.LAYOUT_ROW, "columns"), (4096, 600, 64, 150, 190, hipabi.LAYOUT_ROW, "columns"), (5000, 600, 64, 8, 600, hipabi.LAYOUT_ROW, "columns"),
    (20000, 600, 64, 60, 64, hipabi.LAYOUT_ROW | hipabi.LAYOUT_RBM, "quad")])
def test_chosen_by_rows_and_not_by_the_longest_alone(ctx, oracle, m, n, C, mean, longest, layouts, kernel):
    """Many short rows and a long one: every workgroup copies X for its few rows, which the row kernel's few gathers undercut.
    With the RBM layout too, whose kernels are compared with the one that would run in their place."""
    rng = np.random.default_rng(m + C)
    step = n // longest
    first = rng.integers(0, step, m).astype(np.uint32)
    nnz = np.clip(rng.poisson(mean, m), 0, longest).astype(np.uint32)
    nnz[m // 2] = longest
    held = np.arange(longest, dtype=np.uint32)[None, :] < nnz[:, None]
    idx = np.where(held, first[:, None] + np.arange(longest, dtype=np.uint32) * step, 0).astype(np.uint32)
    Wd = np.where(held, rng.standard_normal((m, longest), dtype=np.float32), np.float32(0))
    E = datagen.EllpackHost(m, n, longest, Wd, idx, nnz)
    X = rng.standard_normal((n, C)).astype(np.float32)
    taken, Y = _run(ctx, E, X, None, "none", layouts=layouts)
    want = oracle.matmul(as_oracle(E), X, None, "none")
    assert taken == kernel
    assert np.array_equal(Y, want) if layouts == hipabi.LAYOUT_ROW else rel_err(Y, want) <= 1e-5
