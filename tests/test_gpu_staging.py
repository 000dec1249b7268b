"""Staged copies (so_stage_in, so_stage_out): every size around the pieces, the pinned areas and the ends by the word,
unaligned places, more calls in a row than the staging memory holds, bytes as they were; a wait that gave up is
reported by so_stage_out as by so_d2h."""
import ctypes as ct

import numpy as np
import pytest

import hipabi

pytestmark = pytest.mark.gpu
PIECE, IN, OUT = 256 << 10, 4 << 20, 1 << 20


def stage_in(ctx, d, a, d2=None, b=None):
    ctx._ck(ctx.lib.so_stage_in(ctx.h, ct.c_void_p(d), a.ctypes.data_as(ct.c_void_p), ct.c_size_t(a.nbytes),
                                ct.c_void_p(d2), b.ctypes.data_as(ct.c_void_p) if b is not None else None, ct.c_size_t(b.nbytes if b is not None else 0)))


def stage_out(ctx, shape, d):
    out = np.full(shape, 7, np.uint32)
    ctx._ck(ctx.lib.so_stage_out(ctx.h, out.ctypes.data_as(ct.c_void_p), ct.c_void_p(d), ct.c_size_t(out.nbytes)))
    return out


@pytest.mark.parametrize("words", [1, 2, 3, 4, 5, 1023, 1025, PIECE // 4 - 1, PIECE // 4, PIECE // 4 + 1, OUT // 4 - 3, OUT // 4, OUT // 4 + 1,
                                   3 * PIECE // 4 + 7, IN // 4 - 64, IN // 4, IN // 4 + 1])
@pytest.mark.parametrize("words2", [0, 1, 6, 5000])
def test_bytes_come_through(ctx, words, words2):
    rng = np.random.default_rng(words + words2)
    d = ctx.array(np.zeros(words + words2 + 16, np.float32))
    at2 = (words + 3) // 4 * 4                                  # the second array right behind the first
    for turn in range(3):
        a, b = (rng.integers(0, 1 << 32, n, dtype=np.uint32) for n in (words, words2))
        stage_in(ctx, d.ptr, a, d.ptr + 4 * at2 if words2 else None, b if words2 else None)
        assert np.array_equal(stage_out(ctx, words, d.ptr), a)
        if words2:
            assert np.array_equal(stage_out(ctx, words2, d.ptr + 4 * at2), b)
    d.free()


def test_unaligned_places_and_many_in_a_row(ctx):
    d = ctx.array(np.zeros(1 << 20, np.float32))
    a = np.arange(1000, dtype=np.uint32)
    stage_in(ctx, d.ptr + 4, a)
    assert np.array_equal(stage_out(ctx, 1000, d.ptr + 4), a)
    parts = [np.random.default_rng(i).integers(0, 1 << 32, 50000, dtype=np.uint32) for i in range(40)]      # 8 MB without a wait
    for i, p in enumerate(parts):
        stage_in(ctx, d.ptr + 4 * 51200 * (i % 20), p)
    for i in range(20):
        assert np.array_equal(stage_out(ctx, 50000, d.ptr + 4 * 51200 * i), parts[20 + i])
    d.free()


def test_errors(ctx):
    lib, a = ctx.lib, np.zeros(4, np.uint32)
    assert lib.so_stage_in(None, None, None, 0, None, None, 0) == hipabi.SO_ERR_INVALID
    assert lib.so_stage_in(ctx.h, None, a.ctypes.data_as(ct.c_void_p), 16, None, None, 0) == hipabi.SO_ERR_INVALID
    assert lib.so_stage_out(None, None, None, 0) == hipabi.SO_ERR_INVALID
    assert lib.so_stage_out(ctx.h, a.ctypes.data_as(ct.c_void_p), None, 16) == hipabi.SO_ERR_INVALID
    assert lib.so_stage_in(ctx.h, None, None, 0, None, None, 0) == hipabi.SO_OK and lib.so_stage_out(ctx.h, None, None, 0) == hipabi.SO_OK


def test_reports_waits_that_gave_up(ctx):
    """Host-forced, as in test_gpu_matmul.py: a tiny poll limit makes the K-tiled kernel's bounded waits give up; the
    launch runs to its end, so_stage_out reports it, and the launch after it is clean."""
    import datagen
    from conftest import sparse_matrix
    rng = np.random.default_rng(9)
    E = datagen.encode_dense(sparse_matrix(rng, 1024, 1024, .8))
    dE = ctx.upload_ellpack(E.Wd, E.idx, E.nnz, E.m, E.n, E.r, hipabi.LAYOUT_ROW | hipabi.LAYOUT_TILED)
    dX, dY = ctx.array(rng.standard_normal((1024, 256)).astype(np.float32)), ctx.empty((1024, 256))
    out = np.zeros(1024 * 256, np.uint32)
    def fetch():
        return ctx.lib.so_stage_out(ctx.h, out.ctypes.data_as(ct.c_void_p), dY.ptr, out.nbytes)
    with ctx.tuning(SPARSEOPS_MATMUL_TILED="1", SPARSEOPS_WAIT_SPINS="0"):
        ctx.matmul(dE, dX, 256, None, dY, "none")
        assert fetch() == hipabi.SO_ERR_HIP and b"gave up" in ctx.lib.so_last_error()
    with ctx.tuning(SPARSEOPS_MATMUL_TILED="1"):
        ctx.matmul(dE, dX, 256, None, dY, "none")
        assert fetch() == hipabi.SO_OK
        assert np.array_equal(out, dY.download().view(np.uint32).ravel())
    for a in (dX, dY, dE):
        a.free()


@pytest.mark.parametrize("rows,cols,stride", [(1, 1, 1), (2, 3, 4), (4, 63, 4), (5, 65, 8), (31, 64, 31), (33, 130, 48), (256, 784, 256), (100, 1000, 112),
                                              (3, 90000, 4), (7, 149000, 8), (16, 65000, 16), (3, 349000, 4)])
def test_transposed_there_and_back(ctx, rows, cols, stride):
    """Pieces of 64 columns and more, tiles of 64 x 32, rows of no multiple of four, padding, sizes around what the staging
    memory holds: the bytes, the zeros behind them and nothing beyond."""
    rng = np.random.default_rng(rows + cols)
    fits_in = ((cols + 3) // 4 * 16 + 1024) * rows <= IN
    d = ctx.array(np.full(cols * stride + 8, 7.0, np.float32))
    done = ct.c_int(-1)
    for turn in range(3):
        a = rng.integers(0, 1 << 32, (rows, cols), dtype=np.uint32)
        ctx._ck(ctx.lib.so_stage_in_transposed(ctx.h, d.ptr, stride, a.ctypes.data_as(ct.c_void_p), rows, cols, ct.byref(done)))
        assert done.value == int(fits_in)
        if not fits_in:
            break
        got = d.download().view(np.uint32)
        assert np.array_equal(got[:cols * stride].reshape(cols, stride)[:, :rows], a.T) and not got[:cols * stride].reshape(cols, stride)[:, rows:].any()
        assert (d.download()[cols * stride:] == 7.0).all()
        out = np.zeros((rows, cols), np.uint32)
        ctx._ck(ctx.lib.so_stage_out_transposed(ctx.h, out.ctypes.data_as(ct.c_void_p), d.ptr, stride, cols, rows, ct.byref(done)))
        assert done.value == int(rows * cols * 4 <= OUT)
        if done.value:
            assert np.array_equal(out, a)
    assert ctx.lib.so_stage_in_transposed(ctx.h, d.ptr, rows - 1, None, rows, cols, ct.byref(done)) == hipabi.SO_ERR_INVALID
    assert ctx.lib.so_stage_out_transposed(ctx.h, None, d.ptr, stride, cols, rows, ct.byref(done)) == hipabi.SO_ERR_INVALID
    d.free()


@pytest.mark.parametrize("rows,cols,taken", [(4000, 64, True), (4096, 252, True), (4096, 253, False), (4097, 64, False), (1024, 1, True), (1025, 1, False),
                                             (3072, 3, True), (3073, 3, False), (4, 262128, True), (4, 262129, False)])
def test_transposed_many_rows(ctx, rows, cols, taken):
    """The rule's edges: 16 bytes per four columns and row, 255 bytes on top, in 4 MB; 1024 rows per column up to 4096."""
    assert taken == ((cols + 3) // 4 * 16 * rows + 255 <= IN and rows <= 1024 * min(cols, 4))
    a = np.random.default_rng(rows + cols).integers(0, 1 << 32, (rows, cols), dtype=np.uint32)
    d, done = ctx.array(np.full(cols * (rows + 4) + 8, 7.0, np.float32)), ct.c_int(-1)
    ctx._ck(ctx.lib.so_stage_in_transposed(ctx.h, d.ptr, rows + 4, a.ctypes.data_as(ct.c_void_p), rows, cols, ct.byref(done)))
    got = d.download()
    assert done.value == int(taken) and (got[cols * (rows + 4):] == 7.0).all()
    if taken:
        got = got[:cols * (rows + 4)].view(np.uint32).reshape(cols, rows + 4)
        assert np.array_equal(got[:, :rows], a.T) and not got[:, rows:].any()
    else:
        assert (got == 7.0).all()
    d.free()
