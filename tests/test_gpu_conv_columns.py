"""The column kernel for small batches (csrc/conv_columns.hip) on plans tuned for the batch, bit for bit against the
oracle: tiles and planes that are no multiple of anything, a window larger than the workgroup, several channel chunks,
rows whose padding columns share a place, strides on 1-wide axes, dilation, empty and dense channels, the residual form,
padding entries that must not turn an infinity in the input into a NaN."""

import numpy as np
import pytest

from conftest import as_oracle, sparse_matrix

import datagen
import hipabi

pytestmark = pytest.mark.gpu

CASES = [  # Cin, Cout, H, W, kernel, stride, pad, dilation, sparsity
    (3, 5, 7, 9, (3, 3), (1, 1), (1, 1), (1, 1), .5), (1, 1, 1, 1, (1, 1), (1, 1), (0, 0), (1, 1), .0), (20, 33, 7, 7, (3, 3), (1, 1), (1, 1), (1, 1), .8),
    (3, 16, 33, 31, (7, 7), (2, 2), (3, 3), (1, 1), .8), (40, 24, 13, 14, (3, 3), (2, 2), (1, 1), (1, 1), .7), (64, 48, 14, 14, (1, 1), (2, 2), (0, 0), (1, 1), .8),
    (7, 6, 12, 20, (3, 2), (1, 3), (2, 0), (2, 1), .3), (5, 9, 17, 5, (1, 5), (3, 1), (0, 2), (1, 1), .5), (600, 20, 7, 7, (3, 3), (1, 1), (1, 1), (1, 1), .9),
    (900, 12, 8, 9, (3, 3), (1, 1), (1, 1), (1, 1), .95), (6, 8, 30, 30, (9, 9), (3, 3), (4, 4), (2, 2), .6)]


@pytest.mark.parametrize("Cin,Cout,H,Wi,k,s,p,d,sp", CASES)
@pytest.mark.parametrize("B", [1, 2, 3, 4])
def test_columns_match_oracle(ctx, oracle, Cin, Cout, H, Wi, k, s, p, d, sp, B):
    from oracle import conv_geom as ocg
    rng = np.random.default_rng(Cin * 31 + Cout + H * 7 + B)
    Wc = sparse_matrix(rng, Cout, Cin * k[0] * k[1], sp)
    if Cout > 4:
        Wc[2] = 0
        Wc[4] = rng.standard_normal(Wc.shape[1])
    E = datagen.encode_dense(Wc)
    g, og = hipabi.conv_geom(Cin, Cout, k[0], k[1], H, Wi, s, p, d), ocg(Cin, Cout, k[0], k[1], H, Wi, s, p, d)
    X = rng.standard_normal((Cin, H, Wi, B)).astype(np.float32)
    R = rng.standard_normal((Cout, g.H_out, g.W_out, B)).astype(np.float32)
    b = rng.standard_normal(Cout).astype(np.float32)
    with ctx.tuning(SPARSEOPS_CONV_COLUMNS="1"):
        dE = ctx.upload_ellpack(E.Wd, E.idx, E.nnz, E.m, E.n, E.r)
        plan = ctx.conv_plan(dE, g)
        ctx.conv_plan_tune(plan, B)
        dX, dY, dB, dR = ctx.array(X), ctx.empty(R.shape), ctx.array(b), ctx.array(R)
        for residual in (None, dR):
            dY.upload(np.full(R.shape, np.nan, np.float32))
            ctx.conv2d(plan, dX, B, dB, dY, "relu", residual=residual)
            assert ctx.last_kernel() == "columns"
            want = oracle.conv2d_pf(as_oracle(E), og, X, B, b, "none")
            want = np.maximum(want if residual is None else want + R, 0)
            assert np.array_equal(dY.download(), want)
        X[0, 0, 0, 0] = np.inf
        dX.upload(X)
        ctx.conv2d(plan, dX, B, dB, dY, "none")
        assert ctx.last_kernel() == "columns"
        want = oracle.conv2d_pf(as_oracle(E), og, X, B, b, "none")
        assert np.array_equal(dY.download(), want, equal_nan=True)
        ctx.conv_plan_free(plan)
        for a in (dX, dY, dB, dR, dE):
            a.free()


@pytest.mark.parametrize("case", [CASES[0], CASES[1], CASES[2], CASES[3], CASES[5], CASES[6], CASES[9]])
@pytest.mark.parametrize("B", [8, 16, 32])
def test_columns_wider_batches(ctx, oracle, case, B):
    """Batches of 8, 16 and 32: tiles of eight, four and two pixels."""
    test_columns_match_oracle(ctx, oracle, *case, B)


# Cin, Cout, H, k, s, sparsity, B, kernel: small images with long rows go to the column kernel, others keep the windowed one
@pytest.mark.parametrize("Cin,Cout,H,k,s,sp,B,kernel", [
    (256, 256, 2, 3, 1, .6, 16, "columns"), (256, 256, 2, 3, 1, .6, 32, "columns"), (128, 128, 4, 3, 1, .6, 16, "columns"),
    (512, 512, 7, 3, 1, .8, 8, "window"), (256, 256, 8, 3, 1, .7, 32, "window"), (128, 128, 12, 3, 1, .8, 16, "window"), (128, 256, 4, 1, 2, .6, 16, "columns")])
def test_columns_or_window(ctx, oracle, Cin, Cout, H, k, s, sp, B, kernel):
    from oracle import conv_geom as ocg
    rng = np.random.default_rng(Cin + H + B)
    E = datagen.encode_dense(sparse_matrix(rng, Cout, Cin * k * k, sp))
    args = Cin, Cout, k, k, H, H, (s, s), (k // 2, k // 2), (1, 1)
    g, og = hipabi.conv_geom(*args), ocg(*args)
    X = rng.standard_normal((Cin, H, H, B)).astype(np.float32)
    dE = ctx.upload_ellpack(E.Wd, E.idx, E.nnz, E.m, E.n, E.r)
    plan = ctx.conv_plan(dE, g)
    want = oracle.conv2d_pf(as_oracle(E), og, X, B, None, "none")
    dX, dY = ctx.array(X), ctx.empty(want.shape)
    for batch, expect in ((B, kernel), (4, None), (B, kernel)):         # and after the plan has been tuned for another batch
        ctx.conv_plan_tune(plan, batch)
        if expect:
            ctx.conv2d(plan, dX, B, None, dY, "none")
            assert ctx.last_kernel() == expect
            assert np.array_equal(dY.download(), want)
    ctx.conv_plan_free(plan)
    for a in (dX, dY, dE):
        a.free()


@pytest.mark.parametrize("Cin,Cout,H,k,s,sp,B,kernel", [
    (11, 4, 120, 1, 1, .5, 32, "window"), (5, 4, 111, 3, 1, .5, 32, "window"), (26, 2, 88, 3, 1, .9, 8, "window"),
    (10, 1, 44, 5, 2, .7, 32, "columns"), (282, 4, 38, 1, 1, .5, 8, "columns")])
def test_columns_or_window_with_few_channels(ctx, oracle, Cin, Cout, H, k, s, sp, B, kernel):
    """Layers of few channels have one channel a wave on large images too: many workgroups of short rows keep the windowed kernel."""
    test_columns_or_window(ctx, oracle, Cin, Cout, H, k, s, sp, B, kernel)


def test_declined_by_estimate_is_not_for_good(ctx, oracle):
    """A plan tuned for a batch of 16 without streams, since the windowed kernel is estimated ahead, gets them when it is tuned
    again under SPARSEOPS_CONV_COLUMNS=1; without the override the estimate decides as before."""
    from oracle import conv_geom as ocg
    rng = np.random.default_rng(61)
    E = datagen.encode_dense(sparse_matrix(rng, 128, 128 * 9, .8))
    args = 128, 128, 3, 3, 12, 12, (1, 1), (1, 1), (1, 1)
    g, og = hipabi.conv_geom(*args), ocg(*args)
    X = rng.standard_normal((128, 12, 12, 16)).astype(np.float32)
    dE = ctx.upload_ellpack(E.Wd, E.idx, E.nnz, E.m, E.n, E.r)
    plan, dX, dY = ctx.conv_plan(dE, g), ctx.array(X), ctx.empty((128, 12, 12, 16))
    want = oracle.conv2d_pf(as_oracle(E), og, X, 16, None, "none")
    for asked, kernel in ((None, "window"), ("1", "columns"), (None, "window"), ("1", "columns")):
        with ctx.tuning(SPARSEOPS_CONV_COLUMNS=asked):
            ctx.conv_plan_tune(plan, 16)
            ctx.conv2d(plan, dX, 16, None, dY, "none")
        assert ctx.last_kernel() == kernel and np.array_equal(dY.download(), want)
    ctx.conv_plan_free(plan)
    for a in (dX, dY, dE):
        a.free()


@pytest.mark.parametrize("Cin,H", [(34, 9), (400, 18)])            # one chunk and several
def test_columns_groups_per_run(ctx, oracle, Cin, H):
    """Runs of no group of 16 entries up to three blocks of eight, one entry more or fewer: what a block, the rest behind it
    and the groups asked for ahead come to."""
    from oracle import conv_geom as ocg
    rng = np.random.default_rng(Cin)
    lengths = [n for k in (0, 1, 6, 7, 8, 9, 15, 16, 17) for n in (16 * k - 1, 16 * k, 16 * k + 1) if n >= 0]
    Wc = np.zeros((len(lengths), Cin * 9), np.float32)
    for row, n in zip(Wc, lengths):
        row[rng.choice(Cin * 9, n, replace=False)] = rng.standard_normal(n)
    E = datagen.encode_dense(Wc)
    args = Cin, len(lengths), 3, 3, H, H, (1, 1), (1, 1), (1, 1)
    g, og = hipabi.conv_geom(*args), ocg(*args)
    X = rng.standard_normal((Cin, H, H, 1)).astype(np.float32)
    with ctx.tuning(SPARSEOPS_CONV_COLUMNS="1"):
        dE = ctx.upload_ellpack(E.Wd, E.idx, E.nnz, E.m, E.n, E.r)
        plan = ctx.conv_plan(dE, g)
        ctx.conv_plan_tune(plan, 1)
        dX, dY = ctx.array(X), ctx.empty((len(lengths), H, H, 1))
        ctx.conv2d(plan, dX, 1, None, dY, "none")
        assert ctx.last_kernel() == "columns"
        assert np.array_equal(dY.download(), oracle.conv2d_pf(as_oracle(E), og, X, 1, None, "none"))
        ctx.conv_plan_free(plan)
        for a in (dX, dY, dE):
            a.free()


@pytest.mark.parametrize("ordered", [True, False])
def test_streams_are_made_once_per_batch_and_kept(ctx, oracle, ordered):
    """Tuning for one small batch after another neither takes away the streams that a recorded graph replays with nor makes
    any again -- also where the kernel does not apply (rows that do not ascend): a second tuning for a batch copies nothing,
    so it is even possible while a graph is being recorded, where a download is refused."""
    from oracle import conv_geom as ocg
    rng = np.random.default_rng(21)
    args = (12, 20, 3, 3, 9, 11, (1, 1), (1, 1), (1, 1))
    g, og = hipabi.conv_geom(*args), ocg(*args)
    E = datagen.encode_dense(sparse_matrix(rng, 20, 12 * 9, .6))
    if not ordered:
        c = int(E.nnz[3])
        E.Wd[3, :c], E.idx[3, :c] = E.Wd[3, :c][::-1].copy(), E.idx[3, :c][::-1].copy()
    dE = ctx.upload_ellpack(E.Wd, E.idx, E.nnz, E.m, E.n, E.r)
    plan = ctx.conv_plan(dE, g)
    runs = []
    for B in (1, 2, 3, 4):
        X = rng.standard_normal((12, 9, 11, B)).astype(np.float32)
        dX, dY = ctx.array(X), ctx.empty((20, g.H_out, g.W_out, B))
        ctx.conv_plan_tune(plan, B)
        ctx.graph_begin()
        try:
            ctx.conv_plan_tune(plan, B)
            ctx.conv2d(plan, dX, B, None, dY, "none")
            if B < 4:
                assert ctx.last_kernel() == ("columns" if ordered else "gather")
        finally:
            graph = ctx.graph_end()
        runs.append((graph, dX, dY, oracle.conv2d_pf(as_oracle(E), og, X, B, None, "none")))
        for graph, _, dY, want in runs:
            ctx.fill_zero(dY)
            ctx.graph_launch(graph)
            assert np.array_equal(dY.download(), want)
    ctx.graph_begin()
    try:
        for B in (1, 4, 2, 3, 1):
            ctx.conv_plan_tune(plan, B)
    finally:
        ctx.graph_free(ctx.graph_end())
    for graph, dX, dY, _ in runs:
        ctx.graph_free(graph)
        dX.free()
        dY.free()
    ctx.conv_plan_free(plan)
    dE.free()


@pytest.mark.parametrize("Cin,Cout,H,Wi,k,s,per_row,kernels", [        # kernels at batch 1, 2 and 3
    (16, 96, 200, 190, 1, 1, 6, "gather gather gather"),               # short rows, many workgroups
    (24, 200, 150, 180, 1, 2, 12, "gather gather gather"), (3, 96, 200, 190, 3, 1, 12, "gather gather gather"),
    (8, 128, 120, 130, 3, 1, 36, "columns gather columns"),            # enough for one entry of the batch, not for a pair
    (16, 64, 120, 130, 3, 1, 90, "columns columns columns"),
    (5, 40, 14, 10, 3, 2, 9, "columns columns columns"), (5, 40, 14, 10, 3, 2, 5, "gather gather gather"),   # one round
    (580, 40, 19, 17, 1, 2, 30, "gather gather gather")])              # one round, a large window for few entries
def test_small_batches_take_the_faster_kernel(ctx, oracle, Cin, Cout, H, Wi, k, s, per_row, kernels):
    """A plan tuned for a small batch keeps to the gather kernel where rows are too short for the column kernel's copy of the
    window, and the two give the same bits."""
    from oracle import conv_geom as ocg
    rng = np.random.default_rng(per_row)
    Wc = np.zeros((Cout, Cin * k * k), np.float32)
    for row in Wc:
        row[rng.permutation(Wc.shape[1])[:per_row]] = rng.standard_normal(per_row)
    E = datagen.encode_dense(Wc)
    g, og = (f(Cin, Cout, k, k, H, Wi, (s, s), (k // 2, k // 2), (1, 1)) for f in (hipabi.conv_geom, ocg))
    dE = ctx.upload_ellpack(E.Wd, E.idx, E.nnz, E.m, E.n, E.r)
    for B, kernel in zip((1, 2, 3), kernels.split()):
        plan = ctx.conv_plan(dE, g)
        ctx.conv_plan_tune(plan, B)
        X = rng.standard_normal((Cin, H, Wi, B)).astype(np.float32)
        dX, dY = ctx.array(X), ctx.empty((Cout, g.H_out, g.W_out, B))
        want = oracle.conv2d_pf(as_oracle(E), og, X, B, None, "none")
        for forced in (None, "0", "1"):
            with ctx.tuning(**({"SPARSEOPS_CONV_COLUMNS": forced} if forced else {})):
                dY.upload(np.full(want.shape, np.nan, np.float32))
                ctx.conv2d(plan, dX, B, None, dY, "none")
                assert ctx.last_kernel() == (kernel if forced is None else "gather" if forced == "0" else "columns")
                assert np.array_equal(dY.download(), want)
        ctx.conv_plan_free(plan)
        dX.free()
        dY.free()
    dE.free()
