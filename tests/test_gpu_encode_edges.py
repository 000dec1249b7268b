"""The device encoder and decoder at the edges of their work split: rows shared by four waves or one wave per row
(1024 columns), groups of 4, 256 and 8192 columns, workgroups of 1, 4 or 16 rows (1024, 4096 rows), decode spans of
8192 elements (whole rows or parts of one), more slots per row than a thread holds.  Bits as numpy's encoder gives them."""

import numpy as np
import pytest

import datagen
import hipabi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,keep", [
    (1, 1, 1.0), (3, 5, .5), (7, 255, .3), (1024, 257, .2), (1025, 64, .4), (4096, 33, .3), (4097, 31, .5), (20000, 17, .3), (300, 1023, .1),
    (300, 1024, .1), (33, 1025, .5), (5, 8191, .9), (4, 8192, 1.0), (3, 8193, .6), (2, 16384, .05), (3, 20001, .3), (70, 2047, .99)])
def test_encode_decode_edges(ctx, m, n, keep):
    rng = np.random.default_rng(m * 7 + n)
    W = datagen.bernoulli_dense(rng, m, n, keep) if keep < 1 else rng.standard_normal((m, n)).astype(np.float32)
    W[m // 2] = 0
    W.flat[0] = np.float32(-0.0)
    W.flat[-1] = np.nan if m % 2 else W.flat[-1]
    E = datagen.encode_dense(W)
    dW = ctx.array(W)
    cap = max(1, E.r + 3)
    dWd, dIdx, dNnz = ctx.empty((m * cap,)), ctx.empty((m * cap,), np.uint32), ctx.empty((m,), np.uint32)
    r, total = ctx.encode_dense_noalloc(dW, m, n, cap, dWd, dIdx, dNnz)
    assert (r, total) == (E.r, E.total_nnz)
    assert np.array_equal(dNnz.download(), E.nnz)
    assert np.array_equal(dWd.download()[:m * r], E.Wd.reshape(-1), equal_nan=True)
    assert np.array_equal(dIdx.download()[:m * r], E.idx.reshape(-1))
    dE = ctx.encode_dense(dW, m, n)
    assert dE.r == E.r and np.array_equal(dE.download()[0], E.Wd, equal_nan=True)
    dense = dE.decode()
    assert np.array_equal(dense, np.where(W == 0, np.float32(0), W), equal_nan=True) and not np.signbit(dense[W == 0]).any()
    # rows in any order decode to the same matrix
    for i in range(m):
        c = int(E.nnz[i])
        E.Wd[i, :c], E.idx[i, :c] = E.Wd[i, :c][::-1].copy(), E.idx[i, :c][::-1].copy()
    dR = ctx.upload_ellpack(E.Wd, E.idx, E.nnz, m, n, E.r, hipabi.LAYOUT_ROW)
    assert np.array_equal(dR.decode(), dense, equal_nan=True)
    for a in (dW, dWd, dIdx, dNnz, dE, dR):
        a.free()


@pytest.mark.parametrize("m,n,keep", [
    (3, 8193, 1.0), (5, 20000, .4), (2, 30011, .5), (1300, 8200, .02), (600, 9001, .3), (1, 150000, .9), (9, 65536, .25), (1290, 8192, .3)])
def test_decode_rows_of_several_spans(ctx, m, n, keep):
    """Rows of several decode spans and of more slots than a workgroup holds at a time (2048), ascending and not, shared by
    several workgroups (below two rows per compute unit) and not, empty, full, crowded into one span; more rows than workgroups."""
    rng = np.random.default_rng(m + n)
    W = datagen.bernoulli_dense(rng, m, n, keep) if keep < 1 else rng.standard_normal((m, n)).astype(np.float32)
    W[m // 2, : n // 2] = 0
    W[m // 3, n // 3:] = 0
    W[(m - 1) // 4] = 0 if m > 4 else 1
    W[m - 1] = np.arange(n) + 1 if m > 1 else W[m - 1]
    E = datagen.encode_dense(W)
    dE = ctx.upload_ellpack(E.Wd, E.idx, E.nnz, m, n, E.r, hipabi.LAYOUT_ROW)
    assert np.array_equal(dE.decode(), W)
    for i in range(0, m, max(1, m // 7)):
        p = rng.permutation(int(E.nnz[i]))
        E.Wd[i, :len(p)], E.idx[i, :len(p)] = E.Wd[i, p], E.idx[i, p]
    dR = ctx.upload_ellpack(E.Wd, E.idx, E.nnz, m, n, E.r, hipabi.LAYOUT_ROW)
    assert np.array_equal(dR.decode(), W)
    dE.free()
    dR.free()
