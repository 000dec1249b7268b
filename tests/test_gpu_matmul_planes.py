"""The bf16-planes kernel of SO_LAYOUT_RBM (csrc/matmul_planes.hip), forced, at the edges of its tiles: blocks of 128 rows,
slabs of 64 dense columns, iterations of 64 columns of the matrix, totals that leave the registers every 8 iterations,
every number of workgroups per tile.

Bound: max|y - ref| <= 1e-5 * max|ref| against the in-order oracle and the fp64 product, as for the layout's other kernels
(tests/test_gpu_matmul_rbm.py).  Beside it the error in the 2-norm: with x = hi + mid + lo exactly, the products left out
are 2^-27.5 of |w x| in the 2-norm (2^-24 at most), and a sum that is rounded once per 16 terms over at most 32 roundings, five times that often for
parts 2^-7 as large, once per 512 terms and once per workgroup, each time by at most 2^-24 of a partial sum, is off by less than
(sqrt(32 + n / 512 + 16) + 1) * 2^-24 of the 2-norm when roundings are independent: 2.5 times that is asked.  Output by output, and where roundings are not
independent: test_planes_worst_mantissas and test_planes_one_step_of_the_matrix_cores."""

import numpy as np
import pytest

from conftest import as_oracle, rel_err, sparse_matrix

import datagen
import hipabi

pytestmark = pytest.mark.gpu
TOL = 1e-5
RBM = hipabi.LAYOUT_ROW | hipabi.LAYOUT_RBM


def planes_matmul(ctx, E, X, bias, act="none", split=None):
    m, C = E.m, X.shape[1]
    with ctx.tuning(SPARSEOPS_MATMUL_PLANES="1", SPARSEOPS_MATMUL_PLANES_SPLIT=split):
        dE = ctx.upload_ellpack(E.Wd, E.idx, E.nnz, E.m, E.n, E.r, RBM)
        dX, dY, dB = ctx.array(X), ctx.empty((m, C)), ctx.array(bias) if bias is not None else None
        outs = []
        for _ in range(2):
            dY.upload(np.full((m, C), np.nan, np.float32))
            ctx.matmul(dE, dX, C, dB, dY, act)
            assert ctx.last_kernel() == "planes"
            outs.append(dY.download())
        for a in (dX, dY, dB):
            if a is not None:
                a.free()
        dE.free()
    assert np.array_equal(outs[0], outs[1], equal_nan=True)
    return outs[0]


@pytest.mark.parametrize("m,n,C,sp", [
    (1, 1, 1, .0), (3, 15, 5, .0), (31, 16, 31, .5), (32, 17, 32, .5), (33, 63, 33, .9), (127, 64, 63, .3), (128, 65, 64, .7),
    (129, 511, 65, .5), (300, 512, 130, .8), (257, 513, 200, .6), (64, 1100, 256, .5), (500, 2777, 101, .7)])
@pytest.mark.parametrize("split,act", [(None, "none"), (1, "relu"), (2, "none"), (3, "relu"), (16, "none")])
def test_planes_shapes(ctx, oracle, m, n, C, sp, split, act):
    rng = np.random.default_rng(m * 31 + n * 7 + C)
    W = sparse_matrix(rng, m, n, sp)
    W[rng.integers(m), rng.integers(n)] = 1.5
    X = rng.standard_normal((n, C)).astype(np.float32)
    b = rng.standard_normal(m).astype(np.float32)
    E = datagen.encode_dense(W)
    Y = planes_matmul(ctx, E, X, b, act, split)
    ref = W.astype(np.float64) @ X + b[:, None]
    if act == "relu":
        ref = np.maximum(ref, 0)
    assert rel_err(Y, ref) <= TOL
    assert rel_err(Y, oracle.matmul(as_oracle(E), X, b, act)) <= TOL
    assert np.linalg.norm(Y - ref) <= 2.5 * (np.sqrt(48 + n / 512) + 1) * 2.0 ** -24 * np.linalg.norm(ref)


@pytest.mark.parametrize("n", [1, 16, 100, 512, 2048, 4100])
@pytest.mark.parametrize("split", [1, 3])
def test_planes_worst_mantissas(ctx, n, split):
    """Weights and X that the planes split worst: every product loses 0.99 * 2^-24 of itself, all of one sign, and every sum grows.  Output by output,
    in units of 2^-24 of |w||x|: that, the small products' sums (2^-7 as large, 5 n / 16 additions), 32 additions to the large sums at
    most, n / 512 to the totals, and one per part and for the small sums; each by 1."""
    rng = np.random.default_rng(n)
    m, C, worst = 130, 66, np.float32(1 + 2.0 ** -8 - 2.0 ** -17)
    W = np.where(rng.random((m, n)) < .6, worst, 0).astype(np.float32)
    W[0], W[1, :-1] = worst, 0
    W[1, -1] = worst
    X = np.full((n, C), worst, np.float32)
    X[:, 1::2] *= -1
    W[2] *= np.ldexp(np.float32(1), rng.integers(-20, 20, n).astype(np.int32))
    Y, ref = planes_matmul(ctx, datagen.encode_dense(W), X, None, split=split), W.astype(np.float64) @ X.astype(np.float64)
    bound = 1 + 5 * n / 16 / 128 + min(32, n / 16) + n / 512 + split + 1
    assert (np.abs(Y - ref) <= bound * 2.0 ** -24 * (np.abs(W).astype(np.float64) @ np.abs(X).astype(np.float64))).all()


@pytest.mark.parametrize("spread", [0, 8, 30, 60])
def test_planes_one_step_of_the_matrix_cores(ctx, spread):
    """A v_mfma_f32_32x32x16_bf16 adds 16 products with at most the error of a chain of fmaf, 16 * 2^-24 of sum |w x|: factors of eight significant
    bits, whose other planes are zeros, of very different sizes and both signs, and large ones that cancel."""
    rng = np.random.default_rng(spread)
    m, n, C = 256, 16, 128

    def eight_bits(shape, spread):
        v = rng.integers(128, 256, shape).astype(np.float32) * rng.choice([-1, 1], shape)
        return np.ldexp(v, rng.integers(-spread, spread + 1, shape) - 7).astype(np.float32)
    W, X = eight_bits((m, n), min(spread, 30)), eight_bits((n, C), spread)
    W[:64, 8:] = -W[:64, :8]
    X[8:, :32] = X[:8, :32] * rng.choice([1, 1, 1, 0, 0.5], (8, 32))
    assert not (W.view(np.uint32) & 0xffff).any() and not (X.view(np.uint32) & 0xffff).any()
    Y, ref = planes_matmul(ctx, datagen.encode_dense(W), X, None, split=1), W.astype(np.float64) @ X.astype(np.float64)
    assert (np.abs(Y - ref) <= 16 * 2.0 ** -24 * (np.abs(W).astype(np.float64) @ np.abs(X).astype(np.float64))).all()


@pytest.mark.parametrize("act", ["sigmoid", "tanh"])
def test_planes_epilogues(ctx, oracle, act):
    rng = np.random.default_rng(1)
    W = sparse_matrix(rng, 200, 700, .6)
    X = rng.standard_normal((700, 70)).astype(np.float32) * 0.1
    E = datagen.encode_dense(W)
    Y, Yo = planes_matmul(ctx, E, X, None, act), oracle.matmul(as_oracle(E), X, None, act)
    pre = np.abs(oracle.matmul(as_oracle(E), X, None, "none")).max()
    # the bound of the sums times the slope, and what the device's expf / tanhf differ by (tests/test_gpu_matmul_rbm.py)
    assert np.abs(Y.astype(np.float64) - Yo).max() <= TOL * pre * (0.25 if act == "sigmoid" else 1.0) + 1e-6


@pytest.mark.parametrize("split", [1, 3])
def test_planes_values_that_are_not_finite(ctx, oracle, split):
    """An infinity or a NaN in X reaches exactly the rows that use it, although the others meet it with a zero; sums that
    come near the largest float (where a plane, rounded up, is beyond it) stay finite."""
    rng = np.random.default_rng(11)
    m, n, C = 200, 600, 70
    W = sparse_matrix(rng, m, n, .6)
    X = rng.standard_normal((n, C)).astype(np.float32)
    X[0, :9], X[17, 3], X[300, 5], X[599, 69] = np.inf, -np.inf, np.nan, np.inf
    W[:, 40] = np.where(np.arange(m) % 2 == 0, 1, 0)
    X[:, 20] = 0
    X[40, 20] = 3.4e38                               # to bf16: infinity
    X[:, 21] = 0
    X[40, 21] = 1.7e38                               # to bf16: 2^127
    W[2, 40] = 2
    E = datagen.encode_dense(W)
    Y, Yo = planes_matmul(ctx, E, X, None, split=split), oracle.matmul(as_oracle(E), X, None)
    assert np.isfinite(Yo[:, 20:22]).sum() >= 2 * m - 1 and Yo[2, 21] == np.float32(3.4e38)
    assert np.array_equal(np.isnan(Y), np.isnan(Yo)) and np.array_equal(np.isinf(Y), np.isinf(Yo))
    assert np.array_equal(Y[np.isinf(Yo)], Yo[np.isinf(Yo)])
    for c in range(C):
        fin = np.isfinite(Yo[:, c])
        assert np.abs(Y[fin, c] - Yo[fin, c]).max(initial=0.0) <= TOL * np.abs(Yo[fin, c]).max(initial=0.0)


@pytest.mark.parametrize("exponent", [-60, -109, -112, -126, -140])
def test_planes_values_too_small_for_three_planes(ctx, oracle, exponent):
    """Columns of X with values whose lowest plane would fall below the smallest bf16 are as exact as the others."""
    rng = np.random.default_rng(7)
    m, n, C = 150, 700, 66
    W = sparse_matrix(rng, m, n, .7)
    X = rng.standard_normal((n, C)).astype(np.float32)
    small = np.ldexp(rng.uniform(1, 2, (n, 30)), exponent + rng.integers(0, 3, (n, 30))).astype(np.float32)
    X[:, 10:40] = small
    X[::3, 12] = 0
    X[5, 0] = small[0, 0]                             # one among ordinary values
    E = datagen.encode_dense(W)
    Y = planes_matmul(ctx, E, X, None, split=2)
    Yo = oracle.matmul(as_oracle(E), X, None)
    ref = W.astype(np.float64) @ X.astype(np.float64)
    for c in range(C):
        # a sum of subnormal products is rounded to 2^-149 per term, whatever its size
        assert np.abs(Y[:, c] - ref[:, c]).max() <= TOL * np.abs(ref[:, c]).max() + n * 2.0 ** -149, c
        assert np.abs(Y[:, c] - Yo[:, c]).max() <= TOL * np.abs(Yo[:, c]).max() + n * 2.0 ** -149, c


@pytest.mark.parametrize("split", [1, 2, 3])
@pytest.mark.parametrize("m,n,C", [(130, 640, 66), (200, 705, 130)])
def test_planes_values_of_any_size(ctx, oracle, split, m, n, C):
    """Values around 2^40, 2^104 and the largest float beside ordinary and tiny ones, alone and many in a column, and infinities and NaNs among
    them: the passes that a workgroup takes for them, one, two, three and four; a slab without any beside one with."""
    rng = np.random.default_rng(m + split)
    W = sparse_matrix(rng, m, n, .6)
    W[:, 5] = np.where(np.arange(m) % 2, 0, 2.0 ** -30)
    X = rng.standard_normal((n, C)).astype(np.float32)
    for c, e in ((1, 39), (2, 40), (3, 41), (4, 70), (5, 103), (6, 104), (7, 105), (8, 115), (C - 1, 60)):
        X[rng.integers(n), c] = np.ldexp(np.float32(1.37), e)
        X[0, c] = np.ldexp(np.float32(-1.21), e)
    X[:, 9] = np.ldexp(X[:, 9], 112)                 # sums near 2^117
    X[:, 10] = np.ldexp(X[:, 10], 90)                # values that fit, sums that do not
    X[::2, 11] = np.ldexp(X[::2, 11], -140)          # both ends of the range
    X[1::2, 11] = np.ldexp(X[1::2, 11], 100)
    X[5, 12] = -3.4028235e38                         # the lowest value, times 2^-30 or nothing
    X[n - 1, 13], X[3, 13], X[n // 2, 14], X[9, 14] = np.inf, 1e30, np.nan, 1e-42
    X[:, 15] = np.inf
    X[2, 16], X[n - 2, 16] = np.inf, -np.inf
    E = datagen.encode_dense(W)
    Y, Yo = planes_matmul(ctx, E, X, None, split=split), oracle.matmul(as_oracle(E), X, None)
    assert np.array_equal(np.isnan(Y), np.isnan(Yo)) and np.array_equal(Y[np.isinf(Yo)], Yo[np.isinf(Yo)])
    for c in range(C):
        fin = np.isfinite(Yo[:, c])
        ref = W[fin].astype(np.float64) @ np.where(np.isfinite(X[:, c]), X[:, c], 0).astype(np.float64)
        assert np.abs(Y[fin, c] - ref).max(initial=0.0) <= TOL * np.abs(ref).max(initial=0.0), c


@pytest.mark.parametrize("value,most", [(1e-38, 1.5), (1e25, 1.5), (1e35, 10.0), (np.inf, 10.0), (np.nan, 10.0)])
def test_planes_time_with_such_values(ctx, value, most):
    """One value in every column: tiny and large ones cost nothing, those that the planes do not hold two or three passes more (not a sum
    over the nonzeros per output, a hundred times as long)."""
    rng = np.random.default_rng(6)
    m, n, C = 2048, 2048, 128
    W = sparse_matrix(rng, m, n, .6)
    X = rng.standard_normal((n, C)).astype(np.float32)
    E = datagen.encode_dense(W)
    with ctx.tuning(SPARSEOPS_MATMUL_PLANES="1"):
        dE = ctx.upload_ellpack(E.Wd, E.idx, E.nnz, m, n, E.r, RBM)
        dX, dY = ctx.array(X), ctx.empty((m, C))

        def shortest():
            ms = []
            for _ in range(5):
                ctx.timer_begin()
                for _ in range(10):
                    ctx.matmul(dE, dX, C, None, dY)
                ms.append(ctx.timer_end())
            return min(ms)
        shortest()
        before = shortest()
        X[rng.integers(0, n, C), np.arange(C)] = value
        dX.upload(X)
        assert shortest() <= most * before
    for a in (dX, dY, dE):
        a.free()


def test_planes_left_out(ctx):
    """Weights without room for three planes, stored zeros, rows whose columns do not ascend: the handle does without, whatever is asked."""
    rng = np.random.default_rng(3)
    W = sparse_matrix(rng, 100, 200, .5)
    X = rng.standard_normal((200, 8)).astype(np.float32)
    cases = []
    for value in (1e-35, 1e12, 1e37, np.inf, np.nan):
        V = W.copy()
        V[3, 5] = value
        cases.append(datagen.encode_dense(V))
    E = datagen.encode_dense(W)
    c = int(E.nnz[9])
    E.Wd[9, :c], E.idx[9, :c] = E.Wd[9, :c][::-1].copy(), E.idx[9, :c][::-1].copy()
    cases.append(E)
    E = datagen.encode_dense(W)
    E.Wd[7, 1] = 0                                   # times an infinity in X: NaN
    cases.append(E)
    for E in cases:
        with ctx.tuning(SPARSEOPS_MATMUL_PLANES="1"):
            dE = ctx.upload_ellpack(E.Wd, E.idx, E.nnz, E.m, E.n, E.r, RBM)
            dX, dY = ctx.array(X), ctx.empty((100, 8))
            ctx.matmul(dE, dX, 8, None, dY)
            assert ctx.last_kernel() != "planes"
            dE.free()


@pytest.mark.parametrize("n,want", [(2 ** 24 - 1, True), (2 ** 24, False), (22369664, False)])
def test_planes_very_many_columns(ctx, n, want):
    """192 bytes of planes per column and row tile: beyond 2^32 of them (22 369 600 columns) an offset no longer fits 32 bits, and
    handles do without from 2^24 columns on.  The last columns count."""
    m, r, C = 3, 40, 2
    rng = np.random.default_rng(5)
    idx = np.sort(rng.choice(n - 1, (m, r), replace=False), axis=1).astype(np.uint32)
    idx[:, -1] = n - 1
    Wd = rng.standard_normal((m, r)).astype(np.float32)
    X = rng.standard_normal((n, C)).astype(np.float32)
    ref = (Wd[:, :, None].astype(np.float64) * X[idx]).sum(axis=1)
    with ctx.tuning(SPARSEOPS_MATMUL_PLANES="1"):
        dE = ctx.upload_ellpack(Wd, idx, np.full(m, r, np.uint32), m, n, r, RBM)
        dX, dY = ctx.array(X), ctx.empty((m, C))
        ctx.matmul(dE, dX, C, None, dY)
        assert (ctx.last_kernel() == "planes") == want
        assert rel_err(dY.download(), ref) <= TOL
    for a in (dX, dY, dE):
        a.free()


def test_planes_by_default(ctx, oracle):
    """The dispatch's own choice: a half-full matrix on a wide batch takes the kernel, a batch of ones or a very sparse matrix does not;
    a column's bits do not depend on its neighbours."""
    rng = np.random.default_rng(2)
    m = n = 2048
    X = rng.standard_normal((n, 200)).astype(np.float32)
    for sp, C, want in ((.5, 200, True), (.5, 1, False), (.95, 200, False)):
        W = sparse_matrix(rng, m, n, sp)
        E = datagen.encode_dense(W)
        dE = ctx.upload_ellpack(E.Wd, E.idx, E.nnz, m, n, E.r, RBM)
        x = np.ascontiguousarray(X[:, :C])
        dX, dY = ctx.array(x), ctx.empty((m, C))
        ctx.matmul(dE, dX, C, None, dY)
        assert (ctx.last_kernel() == "planes") == want
        Y = dY.download()
        assert rel_err(Y, W.astype(np.float64) @ x) <= TOL
        if want:
            perm = rng.permutation(C)
            dX.upload(np.ascontiguousarray(x[:, perm]))
            ctx.matmul(dE, dX, C, None, dY)
            assert np.array_equal(dY.download(), Y[:, perm])
        dE.free()


def test_planes_in_a_recorded_graph(ctx):
    """Reserved, recorded and replayed with new inputs; eager launches of another width between the replays."""
    rng = np.random.default_rng(4)
    m, n, C = 400, 1300, 100
    W = sparse_matrix(rng, m, n, .6)
    E = datagen.encode_dense(W)
    with ctx.tuning(SPARSEOPS_MATMUL_PLANES="1"):
        dE = ctx.upload_ellpack(E.Wd, E.idx, E.nnz, m, n, E.r, RBM)
        dX, dY, dZ = ctx.empty((n, C)), ctx.empty((m, C)), ctx.empty((m, 7))
        ctx.matmul_reserve(dE, C)
        ctx.graph_begin()
        ctx.matmul(dE, dX, C, None, dY)
        assert ctx.last_kernel() == "planes"
        g = ctx.graph_end()
        dx = ctx.array(rng.standard_normal((n, 7)).astype(np.float32))
        for _ in range(3):
            X = rng.standard_normal((n, C)).astype(np.float32)
            dX.upload(X)
            ctx.graph_launch(g)
            ctx.sync()
            Y = dY.download()
            ctx.matmul(dE, dX, C, None, dY)
            assert np.array_equal(dY.download(), Y)
            assert rel_err(Y, W.astype(np.float64) @ X) <= TOL
            ctx.matmul(dE, dx, 7, None, dZ)
        ctx.graph_free(g)
        dE.free()
