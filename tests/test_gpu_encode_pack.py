"""The encoder's packing pass on both sides of the lines where a workgroup's four waves share a row: 2048 columns with few rows, 4096 with many (1024)."""
import numpy as np
import pytest

import datagen
import hipabi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n", [(1023, 2047), (1023, 2048), (1023, 2049), (1023, 4095), (1024, 2049), (1024, 4095), (1040, 4025), (1000, 4097), (37, 2048), (37, 2049), (2000, 1025)])
@pytest.mark.parametrize("keep", [.03, .8])
def test_pack(ctx, m, n, keep):
    rng = np.random.default_rng(m + n)
    W = datagen.bernoulli_dense(rng, m, n, keep)
    W[m // 2] = 0
    W[m - 1] = np.arange(n) + 1
    E = datagen.encode_dense(W)
    dW, cap = ctx.array(W), n
    dWd, dIdx, dNnz = ctx.empty((m * cap,)), ctx.empty((m * cap,), np.uint32), ctx.empty((m,), np.uint32)
    assert ctx.encode_dense_noalloc(dW, m, n, cap, dWd, dIdx, dNnz) == (E.r, E.total_nnz) and ctx.last_kernel() == "encode-twice"
    assert np.array_equal(dNnz.download(), E.nnz)
    assert np.array_equal(dWd.download()[:m * E.r].view(np.uint32), E.Wd.reshape(-1).view(np.uint32)) and np.array_equal(dIdx.download()[:m * E.r], E.idx.reshape(-1))
    for a in (dW, dWd, dIdx, dNnz):
        a.free()
