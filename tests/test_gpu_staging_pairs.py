"""so_stage_out and so_stage_out_transposed on both sides of the 8191 words that come as pairs {value, turn}, large and small in turns; a wait that gave
up in a launch before is reported by the small form too, and nothing is written then."""
import ctypes as ct

import numpy as np
import pytest

import datagen
import hipabi
from conftest import sparse_matrix

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = hipabi.Context(0)
    yield c
    c.close()


def test_sizes(ctx):
    rng = np.random.default_rng(1)
    d = ctx.array(np.zeros(20000, np.float32))
    for words in (1, 255, 256, 257, 20000, 5, 8190, 8191, 8192, 8193, 4097, 1):
        a, out = rng.integers(0, 1 << 32, 20000, dtype=np.uint32), np.zeros(words + 1, np.uint32)
        d.upload(a.view(np.float32))
        ctx._ck(ctx.lib.so_stage_out(ctx.h, out.ctypes.data_as(ct.c_void_p), d.ptr, words * 4))
        assert np.array_equal(out[:words], a[:words]) and out[words] == 0
    d.free()


@pytest.mark.parametrize("rows,cols,stride", [(1, 1, 4), (3, 5, 8), (1, 8191, 8191), (8191, 1, 4), (90, 91, 92), (91, 90, 96), (64, 128, 128), (1000, 8, 8), (1000, 9, 16), (10, 256, 256)])
def test_transposed(ctx, rows, cols, stride):
    a = np.random.default_rng(rows + cols).integers(0, 1 << 32, (rows, stride), dtype=np.uint32)
    d, out, done = ctx.array(a.view(np.float32)), np.zeros((cols, rows), np.uint32), ct.c_int(0)
    for _ in range(2):
        out[:] = 7
        ctx._ck(ctx.lib.so_stage_out_transposed(ctx.h, out.ctypes.data_as(ct.c_void_p), d.ptr, stride, rows, cols, ct.byref(done)))
        assert done.value == 1 and np.array_equal(out, a[:, :cols].T)
    d.free()


def test_reports_waits_that_gave_up(ctx):
    rng = np.random.default_rng(9)
    E = datagen.encode_dense(sparse_matrix(rng, 1024, 1024, .8))
    dE = ctx.upload_ellpack(E.Wd, E.idx, E.nnz, E.m, E.n, E.r, hipabi.LAYOUT_ROW | hipabi.LAYOUT_TILED)
    dX, dY, out = ctx.array(rng.standard_normal((1024, 256)).astype(np.float32)), ctx.empty((1024, 256)), np.full(1000, 7, np.uint32)
    fetch = lambda: ctx.lib.so_stage_out(ctx.h, out.ctypes.data_as(ct.c_void_p), dY.ptr, out.nbytes)    # noqa: E731
    for spins, want in (("0", hipabi.SO_ERR_HIP), (None, hipabi.SO_OK), ("0", hipabi.SO_ERR_HIP), (None, hipabi.SO_OK)):
        out[:] = 7
        with ctx.tuning(SPARSEOPS_MATMUL_TILED="1", SPARSEOPS_WAIT_SPINS=spins):
            ctx.matmul(dE, dX, 256, None, dY, "none")
            assert fetch() == want
        if want == hipabi.SO_OK:
            assert np.array_equal(out, dY.download().view(np.uint32).reshape(-1)[:1000])
        else:
            assert b"gave up" in ctx.lib.so_last_error() and (out == 7).all()
    for a in (dX, dY, dE):
        a.free()
