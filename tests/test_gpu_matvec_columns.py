"""so_matmul at two and three columns on the matvec kernel: all columns at once where their workgroups would not fit the chip side by side, in turn otherwise and
where they do not fit LDS together; the bits of each column by itself, at every number of lanes per row, with empty rows, rows of one, and an infinity that only its
column and rows meet."""
import numpy as np
import pytest

import hipabi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = hipabi.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("idx16", [False, True])
@pytest.mark.parametrize("m,n,C,r", [(8200, 300, 2, 128), (8195, 301, 2, 128), (4200, 777, 3, 201), (2060, 901, 2, 389), (2100, 1003, 3, 387), (2050, 640, 2, 479), (1400, 5001, 3, 700), (2500, 1234, 3, 385),
                                     (1366, 13000, 3, 700), (1366, 13700, 3, 700), (40, 600, 3, 230), (300, 700, 2, 128), (1360, 3000, 3, 700)])
def test_columns_are_matvecs(ctx, m, n, C, r, idx16):
    rng = np.random.default_rng(m + n)
    nnz = np.full(m, r, np.uint32)
    nnz[rng.random(m) < .3] = rng.integers(2, r)
    nnz[m // 2], nnz[m - 1], nnz[1] = 0, 1, r
    Wd, idx = rng.standard_normal((m, r)).astype(np.float32), np.sort(rng.integers(1, n, (m, r)), axis=1).astype(np.uint32)
    idx[3, 0] = 0
    pad = np.arange(r) >= nnz[:, None]
    Wd[pad], idx[pad] = 0, 0
    X = rng.standard_normal((n, C)).astype(np.float32)
    X[0, 1] = np.inf
    b = rng.standard_normal(m).astype(np.float32)
    dE = ctx.upload_ellpack(Wd, idx, nnz, m, n, r, hipabi.LAYOUT_ROW | hipabi.LAYOUT_RBM | (hipabi.LAYOUT_IDX16 if idx16 else 0))
    dB, dX, dY, dy = ctx.array(b), ctx.array(X), ctx.array(np.full((m, C), np.nan, np.float32)), ctx.empty((m,))
    with ctx.tuning(SPARSEOPS_MATMUL_NARROW="0"):
        ctx.matmul(dE, dX, C, dB, dY, "relu")
    assert ctx.last_kernel() == "vector"
    Y = dY.download()
    for j in range(C):
        dx = ctx.array(np.ascontiguousarray(X[:, j]))
        ctx.matvec(dE, dx, dB, dy, hipabi.LAYOUT_ROW)
        y = dy.download()
        assert np.isinf(y).sum() == (j == 1) and np.array_equal(Y[:, j], np.maximum(y, 0))
        fin = np.isfinite(y)
        xj = np.where(pad | ~np.isfinite(X[idx, j]), 0, X[idx, j]).astype(np.float64)
        ref = (Wd * xj).sum(axis=1)[fin] + b[fin]
        scale = np.abs(Wd * xj).sum(axis=1)[fin] + np.abs(b[fin])
        # a lane adds up to r / (4 G) + 1 products into each of four sums, which then meet in at most nine additions
        assert (np.abs(y[fin] - ref) <= (r / 32 + 10) * 2.0 ** -24 * scale).all()
        dx.free()
    for a in (dB, dX, dY, dy, dE):
        a.free()
