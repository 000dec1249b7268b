"""The encoder that reads the matrix once, at the edges of its work split: pieces of up to 2048 columns in groups of 256,
rows over workgroups that divide them evenly or not, pieces that the compute units' LDS keeps, that are read again and that
no wave's part of LDS holds; the first sizes it takes (2^22 elements, 768 columns, three quarters of the workgroups' rows).
Bits as numpy's encoder gives them; and the two passes that take over when its workgroups give up waiting for one another."""

import numpy as np
import pytest

import datagen
import hipabi

pytestmark = pytest.mark.gpu


def _check(ctx, W, kernel):
    m, n = W.shape
    E = datagen.encode_dense(W)
    dW = ctx.array(W)
    cap = E.r + 1
    dWd, dIdx, dNnz = ctx.empty((m * cap,)), ctx.empty((m * cap,), np.uint32), ctx.empty((m,), np.uint32)
    dWd.upload(np.full(m * cap, np.float32(7.5)))
    dIdx.upload(np.full(m * cap, 0xDEADBEEF, np.uint32))
    r, total = ctx.encode_dense_noalloc(dW, m, n, cap, dWd, dIdx, dNnz)
    assert ctx.last_kernel() == kernel
    assert (r, total) == (E.r, E.total_nnz)
    assert np.array_equal(dNnz.download(), E.nnz)
    Wd, idx = dWd.download(), dIdx.download()
    assert np.array_equal(Wd[:m * r].view(np.uint32), E.Wd.reshape(-1).view(np.uint32))
    assert np.array_equal(idx[:m * r], E.idx.reshape(-1))
    assert (Wd[m * r:] == 7.5).all() and (idx[m * r:] == 0xDEADBEEF).all()      # nothing past the last slot
    for a in (dW, dWd, dIdx, dNnz):
        a.free()


def _matrix(m, n, keep, seed):
    rng = np.random.default_rng(seed)
    W = datagen.bernoulli_dense(rng, m, n, keep) if keep < 1 else rng.standard_normal((m, n)).astype(np.float32)
    W[m // 2] = 0
    W[m // 3, n // 3:] = 0
    W[m // 4, : n // 2] = np.arange(n // 2) + 1
    W[0, 0], W[-1, -1], W[1, 1], W[2, 2] = -0.0, np.nan, np.inf, 1e-45
    return W


@pytest.mark.parametrize("m,n,keep", [
    (2048, 2048, .1), (2048, 2049, .1), (4095, 2047, .3), (512, 8192, .5), (512, 10241, 1.0), (256, 16384, .2), (200, 20973, .95), (5462, 768, .4),
    (5000, 1023, 1.0), (4097, 1025, .02), (1031, 4099, .6), (770, 6151, .9), (50001, 800, .05)])
def test_encode_once(ctx, m, n, keep):
    _check(ctx, _matrix(m, n, keep, m + n), "encode-once")


@pytest.mark.parametrize("m,n", [(2047, 2048), (8192, 767), (513, 9000)])
def test_other_sizes_take_two_passes(ctx, m, n):
    """Too small, rows too short, rows that divide badly."""
    _check(ctx, _matrix(m, n, .05, m + n), "encode-twice")


def test_a_wait_that_gives_up_is_done_again(ctx):
    W = _matrix(2048, 2100, .2, 5)
    with ctx.tuning(SPARSEOPS_WAIT_SPINS="0"):
        _check(ctx, W, "encode-twice")
    _check(ctx, W, "encode-once")


def test_calls_after_a_wait_that_gave_up_are_spared_it(ctx):
    """2^30 elements in calls that the kernel would take, then it is tried again and, having given up again, left out for
    longer; smaller matrices, which it would not take, do not count; a change of the overrides starts anew."""
    W, small = _matrix(2048, 2100, .2, 5), _matrix(64, 300, .2, 5)
    dW, dWd, dIdx, dNnz = ctx.array(W), ctx.empty((W.size,)), ctx.empty((W.size,), np.uint32), ctx.empty((2048,), np.uint32)
    with ctx.tuning(SPARSEOPS_WAIT_SPINS="0"):
        for spared in (-(-2**30 // W.size), -(-2**31 // W.size)):
            _check(ctx, W, "encode-twice")
            _check(ctx, W, "encode-spared")
            for _ in range(spared - 1):
                ctx.encode_dense_noalloc(dW, 2048, 2100, 2100, dWd, dIdx, dNnz)
                assert ctx.last_kernel() == "encode-spared"
            _check(ctx, small, "encode-twice")
        _check(ctx, W, "encode-twice")
    _check(ctx, W, "encode-once")
    for a in (dW, dWd, dIdx, dNnz):
        a.free()


def test_row_longer_than_the_capacity(ctx):
    W = _matrix(2048, 2100, .2, 6)
    E = datagen.encode_dense(W)
    dW = ctx.array(W)
    cap = E.r - 1
    dWd, dIdx, dNnz = ctx.empty((2048 * cap,)), ctx.empty((2048 * cap,), np.uint32), ctx.empty((2048,), np.uint32)
    dWd.upload(np.full(2048 * cap, np.float32(7.5)))
    with pytest.raises(Exception, match="longest row"):
        ctx.encode_dense_noalloc(dW, 2048, 2100, cap, dWd, dIdx, dNnz)
    assert (dWd.download() == 7.5).all() and np.array_equal(dNnz.download(), E.nnz)
    for a in (dW, dWd, dIdx, dNnz):
        a.free()


@pytest.mark.parametrize("m,n,kernel", [(2048, 2100, "encode-once"), (40, 300, "encode-twice")])
def test_reports_waits_that_gave_up(ctx, m, n, kernel):
    """The encoder's wait for its counts reports, once, a wait on LDS counters that gave up in an earlier launch of the stream."""
    rng = np.random.default_rng(8)
    E = datagen.encode_dense(datagen.bernoulli_dense(rng, 256, 1024, .1))
    dE = ctx.upload_ellpack(E.Wd, E.idx, E.nnz, E.m, E.n, E.r, hipabi.LAYOUT_ROW | hipabi.LAYOUT_TILED)
    dX, dY = ctx.array(rng.standard_normal((1024, 64)).astype(np.float32)), ctx.empty((256, 64))
    W = _matrix(m, n, .2, 9)
    with ctx.tuning(SPARSEOPS_MATMUL_TILED="1", SPARSEOPS_WAIT_SPINS="0"):
        ctx.matmul(dE, dX, 64, None, dY)
    with pytest.raises(hipabi.SoError, match="gave up"):
        _check(ctx, W, kernel)
    _check(ctx, W, kernel)
    for a in (dE, dX, dY):
        a.free()
