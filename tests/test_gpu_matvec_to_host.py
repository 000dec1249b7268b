"""so_matvec_to_host: so_matvec's bits in host memory, on every layout; one to 8193 rows (more than 8192 go the general way), rows for every length
class, workgroups of one and of several passes, no columns, and many calls in a row, whose results lie in the same places of the staging memory."""
import ctypes as ct
import time

import numpy as np
import pytest

from conftest import sparse_matrix

import datagen
import hipabi

pytestmark = pytest.mark.gpu


def to_host(ctx, dE, dx, dB, dy, m, layout=0):
    y = np.full(m + 2, 7.0, np.float32)
    ctx._ck(ctx.lib.so_matvec_to_host(ctx.h, dE.h, dx.ptr if dx else None, dB.ptr if dB else None, dy.ptr, ct.c_void_p(y.ctypes.data + 4), layout))
    assert y[0] == 7.0 and y[-1] == 7.0
    return y[1:-1]


def matrix(rng, m, n, kind):
    W = sparse_matrix(rng, m, n, .9)
    if kind == "skewed":                                  # rows for every class: none, a few, a hundred, thousands, more than 4096
        keep = rng.choice([0, 2, 60, 1500], m)
        W = rng.standard_normal((m, n)).astype(np.float32)
        W[rng.random((m, n)) >= (keep / n)[:, None]] = 0
        W[m // 2] = rng.standard_normal(n)
    return datagen.encode_dense(W)


@pytest.mark.parametrize("m,n,kind", [(1, 1, "even"), (15, 40, "even"), (17, 300, "even"), (300, 5000, "skewed"), (1500, 1000, "even"), (4097, 500, "even"), (2000, 4500, "skewed"),
                                      (8192, 130, "even"), (8193, 130, "even"), (8192, 600, "skewed"), (8193, 600, "skewed"), (600, 41000, "even")])
@pytest.mark.parametrize("idx16", [0, hipabi.LAYOUT_IDX16])
def test_bits_of_so_matvec(ctx, m, n, kind, idx16):
    rng = np.random.default_rng(m + n)
    E = matrix(rng, m, n, kind)
    slot = hipabi.LAYOUT_SLOT if E.r <= 1024 else 0
    dE = ctx.upload_ellpack(E.Wd, E.idx, E.nnz, E.m, E.n, E.r, hipabi.LAYOUT_ROW | hipabi.LAYOUT_BINS | slot | idx16)
    dy, dscratch = ctx.empty((m,)), ctx.empty((m,))
    for turn in range(3):
        dx = ctx.array(rng.standard_normal(n).astype(np.float32))
        dB = ctx.array(rng.standard_normal(m).astype(np.float32)) if turn else None
        for layout in (0, hipabi.LAYOUT_ROW, hipabi.LAYOUT_BINS) + ((hipabi.LAYOUT_SLOT,) if slot else ()):
            ctx.matvec(dE, dx, dB, dy, layout)
            assert np.array_equal(to_host(ctx, dE, dx, dB, dscratch, m, layout), dy.download())
        dx.free()
    for a in (dy, dscratch, dE):
        a.free()


@pytest.mark.parametrize("n", [39936, 39937, 40960, 40961])
@pytest.mark.parametrize("layout", [hipabi.LAYOUT_ROW, hipabi.LAYOUT_BINS])
def test_x_keeps_its_place_in_lds(ctx, n, layout):
    """160 KB of LDS hold 40 960 elements of x, 39 936 (less the length classes' 64 bytes) with a workgroup's results beside them: the call is no slower in between than
    the product and so_stage_out on their own (which took half its time there when x gave way)."""
    rng = np.random.default_rng(n)
    m, r = 2048, 6000
    idx = np.sort(rng.integers(0, n - r, (m, r)), axis=1).astype(np.uint32) + np.arange(r, dtype=np.uint32)
    dE = ctx.upload_ellpack(rng.standard_normal((m, r)).astype(np.float32), idx, np.full(m, r, np.uint32), m, n, r, layout | hipabi.LAYOUT_ROW | hipabi.LAYOUT_IDX16)
    dx, dy, dscratch, y = ctx.array(rng.standard_normal(n).astype(np.float32)), ctx.empty((m,)), ctx.empty((m,)), np.empty(m, np.float32)

    def apart():
        ctx.matvec(dE, dx, None, dy, layout)
        ctx._ck(ctx.lib.so_stage_out(ctx.h, y.ctypes.data_as(ct.c_void_p), dy.ptr, 4 * m))

    def us(call):
        best = 1e9
        for _ in range(8):
            t = time.perf_counter()
            for _ in range(20):
                call()
            best = min(best, (time.perf_counter() - t) / 20)
        return best * 1e6

    apart()
    assert np.array_equal(to_host(ctx, dE, dx, None, dscratch, m, layout), y)
    assert us(lambda: to_host(ctx, dE, dx, None, dscratch, m, layout)) < 1.3 * us(apart)
    for a in (dE, dx, dy, dscratch):
        a.free()


def test_lanes_and_no_columns(ctx):
    rng = np.random.default_rng(1)
    E = matrix(rng, 5000, 900, "even")
    dE = ctx.upload_ellpack(E.Wd, E.idx, E.nnz, E.m, E.n, E.r, hipabi.LAYOUT_ROW)
    dx, dy = ctx.array(rng.standard_normal(900).astype(np.float32)), ctx.empty((5000,))
    for lanes in ("8", "16", "32", "64"):
        with ctx.tuning(SPARSEOPS_MATVEC_LANES=lanes):
            ctx.matvec(dE, dx, None, dy)
            assert np.array_equal(to_host(ctx, dE, dx, None, dy, 5000), dy.download())
    for a in (dE, dx):
        a.free()
    E = datagen.encode_dense(np.zeros((300, 0), np.float32))
    dE, dB = ctx.upload_ellpack(E.Wd, E.idx, E.nnz, 300, 0, E.r, hipabi.LAYOUT_ROW | hipabi.LAYOUT_BINS), ctx.array(np.arange(300, dtype=np.float32))
    for layout in (hipabi.LAYOUT_ROW, hipabi.LAYOUT_BINS):
        assert np.array_equal(to_host(ctx, dE, None, dB, dy, 300, layout), np.arange(300))
    for a in (dE, dB, dy):
        a.free()


def test_after_a_launch_whose_waits_may_give_up(ctx):
    """The general way back then, which looks at the word of those waits."""
    rng = np.random.default_rng(9)
    E = datagen.encode_dense(sparse_matrix(rng, 1024, 1024, .8))
    dE = ctx.upload_ellpack(E.Wd, E.idx, E.nnz, E.m, E.n, E.r, hipabi.LAYOUT_ROW | hipabi.LAYOUT_TILED)
    dX, dY, dx, dy = ctx.array(rng.standard_normal((1024, 256)).astype(np.float32)), ctx.empty((1024, 256)), ctx.array(rng.standard_normal(1024).astype(np.float32)), ctx.empty((1024,))
    y = np.zeros(1024, np.float32)
    with ctx.tuning(SPARSEOPS_MATMUL_TILED="1", SPARSEOPS_WAIT_SPINS="0"):
        ctx.matmul(dE, dX, 256, None, dY, "none")
        assert ctx.lib.so_matvec_to_host(ctx.h, dE.h, dx.ptr, None, dy.ptr, y.ctypes.data_as(ct.c_void_p), 0) == hipabi.SO_ERR_HIP
        assert b"gave up" in ctx.lib.so_last_error()
    with ctx.tuning(SPARSEOPS_MATMUL_TILED="1"):
        ctx.matmul(dE, dX, 256, None, dY, "none")
    ctx.matvec(dE, dx, None, dy)
    assert np.array_equal(to_host(ctx, dE, dx, None, dy, 1024), dy.download())
    for a in (dX, dY, dx, dy, dE):
        a.free()


def test_errors(ctx):
    E = datagen.encode_dense(np.eye(4, dtype=np.float32))
    dE, dx = ctx.upload_ellpack(E.Wd, E.idx, E.nnz, 4, 4, E.r, hipabi.LAYOUT_ROW), ctx.array(np.ones(4, np.float32))
    f, y = ctx.lib.so_matvec_to_host, np.zeros(4, np.float32).ctypes.data_as(ct.c_void_p)
    assert f(None, dE.h, dx.ptr, None, dx.ptr, y, 0) == hipabi.SO_ERR_INVALID
    assert f(ctx.h, dE.h, None, None, dx.ptr, y, 0) == hipabi.SO_ERR_INVALID
    assert f(ctx.h, dE.h, dx.ptr, None, dx.ptr, None, 0) == hipabi.SO_ERR_INVALID
    assert f(ctx.h, dE.h, dx.ptr, None, None, y, 0) == hipabi.SO_ERR_INVALID
    assert f(ctx.h, dE.h, dx.ptr, None, dx.ptr, y, hipabi.LAYOUT_BINS) == hipabi.SO_ERR_INVALID
    ctx.graph_begin()
    try:
        assert f(ctx.h, dE.h, dx.ptr, None, dx.ptr, y, 0) == hipabi.SO_ERR_INVALID
    finally:
        ctx.graph_free(ctx.graph_end())
    for a in (dE, dx):
        a.free()
