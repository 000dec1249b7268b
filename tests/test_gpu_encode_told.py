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
