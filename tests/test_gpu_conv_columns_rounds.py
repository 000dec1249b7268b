"""The column convolution where its workgroups fill the chip more than once, in sizes that the estimate holds equal, and the line against the gather kernel
there: entries and windows on both sides of it, the bits of the gather kernel."""
import numpy as np
import pytest

import datagen
import hipabi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = hipabi.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("Cin,Cout,H,W,k,s,per_row,B,kernel", [
    (3, 64, 130, 127, 3, 1, 14, 1, "columns"), (3, 64, 130, 127, 3, 1, 13, 1, "gather"), (3, 65, 120, 111, 3, 1, 14, 3, "columns"), (3, 64, 120, 111, 3, 1, 13, 3, "gather"),
    (3, 63, 224, 221, 7, 2, 29, 1, "columns"), (4, 70, 125, 124, 5, 1, 40, 2, "columns"), (4, 64, 125, 124, 5, 1, 39, 2, "gather"),
    (32, 64, 160, 160, 3, 1, 18, 1, "gather"), (8, 150, 118, 120, 3, 1, 15, 1, "columns")])
def test_rounds(ctx, Cin, Cout, H, W, k, s, per_row, B, kernel):
    rng = np.random.default_rng(Cout + per_row + B)
    D = np.zeros((Cout, Cin * k * k), np.float32)
    for row in D:
        row[rng.permutation(D.shape[1])[:per_row]] = rng.standard_normal(per_row)
    E, g = datagen.encode_dense(D), hipabi.conv_geom(Cin, Cout, k, k, H, W, (s, s), (k // 2, k // 2))
    dE = ctx.upload_ellpack(E.Wd, E.idx, E.nnz, E.m, E.n, E.r)
    plan = ctx.conv_plan(dE, g)
    ctx.conv_plan_tune(plan, B)
    dX, dB, dY = ctx.array(rng.standard_normal((Cin, H, W, B)).astype(np.float32)), ctx.array(rng.standard_normal(Cout).astype(np.float32)), ctx.empty((Cout, g.H_out, g.W_out, B))
    bits = {}
    for forced in ("0", "1", None):
        with ctx.tuning(SPARSEOPS_CONV_COLUMNS=forced):
            dY.upload(np.full(dY.shape, np.nan, np.float32))
            ctx.conv2d(plan, dX, B, dB, dY, "relu")
            assert ctx.last_kernel() == {"0": "gather", "1": "columns", None: kernel}[forced]
            bits[forced] = dY.download().view(np.uint32)
    assert np.array_equal(bits["0"], bits["1"]) and np.array_equal(bits["0"], bits[None])
    ctx.conv_plan_free(plan)
    for a in (dE, dX, dB, dY):
        a.free()
