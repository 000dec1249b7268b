"""The one-read encoder tells the host from its kernel: what it wrote is there for another context's stream at once, on both sides of the line (6 Mi slots
of the result) beyond which the host waits for the stream's end instead, for one and many rows per workgroup, and call after call."""
import numpy as np
import pytest

import datagen
import hipabi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,keep", [(2048, 2048, .1), (16384, 1024, .2), (2049, 6145, .99), (2048, 6400, .98), (70000, 768, .05)])
def test_seen_from_another_stream(ctx, m, n, keep):
    rng = np.random.default_rng(m + n)
    other = hipabi.Context()
    cap = n
    dWd, dIdx, dNnz = ctx.empty((m * cap,)), ctx.empty((m * cap,), np.uint32), ctx.empty((m,), np.uint32)
    for turn in range(4):
        W = rng.standard_normal((m, n), dtype=np.float32)
        W[rng.random((m, n), dtype=np.float32) >= keep] = 0
        E = datagen.encode_dense(W)
        dW = ctx.array(W)
        copies = [other.empty((m * E.r,)), other.empty((m * E.r,), np.uint32), other.empty((m,), np.uint32)]
        r, total = ctx.encode_dense_noalloc(dW, m, n, cap, dWd, dIdx, dNnz)
        for to, of, size in zip(copies, (dWd, dIdx, dNnz), (m * E.r, m * E.r, m)):
            other._ck(other.lib.so_d2d(other.h, to.ptr, of.ptr, 4 * size))
        assert ctx.last_kernel() == "encode-once" and (r, total) == (E.r, E.total_nnz)
        assert np.array_equal(copies[0].download().view(np.uint32), E.Wd.reshape(-1).view(np.uint32))
        assert np.array_equal(copies[1].download(), E.idx.reshape(-1)) and np.array_equal(copies[2].download(), E.nnz)
        for a in [dW] + copies:
            a.free()
    for a in (dWd, dIdx, dNnz):
        a.free()
    other.close()


@pytest.mark.parametrize("m,n", [(2048, 3072), (2049, 3072), (5000, 1023), (512, 10241)])
def test_the_line_and_pieces_packed_again(ctx, m, n):
    """No zeros: exactly 6 Mi slots and a row more; and, below the line, pieces that LDS does not keep, which are packed again or go straight to memory."""
    test_seen_from_another_stream(ctx, m, n, 2.0)


def test_waits_while_a_launch_holds_part_of_the_chip():
    """Another context's product holds eight compute units for 0.9 ms, in which the encoder's workgroups there cannot start: the others wait for them, which is the faster
    way out up to some 3 ms."""
    mine, other = hipabi.Context(), hipabi.Context()
    m, n = 1024, 40000
    Wd, idx = np.ones((m, n), np.float32), np.tile(np.arange(n, dtype=np.uint32), (m, 1))
    dE = other.upload_ellpack(Wd, idx, np.full(m, n, np.uint32), m, n, n, hipabi.LAYOUT_ROW)
    dx, dy = other.array(np.ones(n, np.float32)), other.empty((m,))
    W = np.zeros((2048, 2048), np.float32)
    W[:, ::7] = 1
    E = datagen.encode_dense(W)
    dW, dWd, dIdx, dNnz = mine.array(W), mine.empty((2048 * 512,)), mine.empty((2048 * 512,), np.uint32), mine.empty((2048,), np.uint32)
    mine.encode_dense_noalloc(dW, 2048, 2048, 512, dWd, dIdx, dNnz)
    assert mine.last_kernel() == "encode-once"
    with other.tuning(SPARSEOPS_MATVEC_LANES="8"):
        for _ in range(2):
            other.timer_begin()
            other.matvec(dE, dx, None, dy, hipabi.LAYOUT_ROW)
            ms = other.timer_end()
        assert 0.6 < ms < 2.0
        for _ in range(3):
            other.matvec(dE, dx, None, dy, hipabi.LAYOUT_ROW)
            r, total = mine.encode_dense_noalloc(dW, 2048, 2048, 512, dWd, dIdx, dNnz)
            assert mine.last_kernel() == "encode-once" and (r, total) == (E.r, E.total_nnz)
            other.sync()
    assert np.array_equal(dWd.download()[:2048 * E.r], E.Wd.reshape(-1))
    for a in (dE, dx, dy, dW, dWd, dIdx, dNnz):
        a.free()
    mine.close()
    other.close()
