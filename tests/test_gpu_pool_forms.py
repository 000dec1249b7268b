"""so_maxpool and so_gap over the forms their kernels take apart: kernels of one, two, three and more columns and rows, batches by lane and by four,
windows that hang over every edge, infinities, NaNs and both zeros; planes of any size beside the groups the average's loads go in.  Bit for bit."""
import numpy as np
import pytest

import hipabi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = hipabi.Context(0)
    yield c
    c.close()


def maxpool(X, k, s, pad):
    """First of the largest in row order, taps outside the image skipped, NaNs never taken: as the reference's loop."""
    C, H, W, B = X.shape
    Ho, Wo = (H + 2 * pad[0] - k[0]) // s[0] + 1, (W + 2 * pad[1] - k[1]) // s[1] + 1
    Y = np.full((C, Ho, Wo, B), -np.inf, np.float32)
    for ho in range(Ho):
        for wo in range(Wo):
            v = Y[:, ho, wo]
            for h in range(ho * s[0] - pad[0], ho * s[0] - pad[0] + k[0]):
                for w in range(wo * s[1] - pad[1], wo * s[1] - pad[1] + k[1]):
                    if 0 <= h < H and 0 <= w < W:
                        np.copyto(v, X[:, h, w], where=X[:, h, w] > v)
    return Y


@pytest.mark.parametrize("B", [1, 3, 4, 8])
@pytest.mark.parametrize("k,s,pad", [((1, 1), (1, 1), (0, 0)), ((1, 1), (2, 3), (0, 0)), ((2, 2), (2, 2), (0, 0)), ((2, 1), (1, 1), (1, 0)), ((3, 3), (2, 2), (1, 1)),
                                     ((3, 3), (1, 1), (2, 2)), ((1, 3), (1, 2), (0, 1)), ((3, 2), (2, 1), (1, 1)), ((7, 3), (2, 1), (3, 1)), ((4, 4), (2, 2), (0, 0)),
                                     ((5, 8), (1, 3), (2, 4)), ((2, 9), (1, 1), (0, 4)), ((17, 17), (1, 1), (8, 8))])
def test_maxpool_forms(ctx, B, k, s, pad):
    rng = np.random.default_rng(B * 100 + k[0] * 10 + k[1])
    C, H, W = 5, 17, 19
    X = rng.integers(-3, 4, (C, H, W, B)).astype(np.float32)             # ties often
    pick = rng.random(X.shape)
    for share, value in ((0.03, np.nan), (0.06, -np.inf), (0.07, np.inf), (0.2, -0.0)):
        X[(pick < share) & (pick >= share - 0.03)] = value
    X[0], X[1] = np.nan, -np.inf
    want = maxpool(X, k, s, pad)
    dX, dY = ctx.array(X), ctx.array(np.full(want.shape, 7, np.float32))
    ctx.maxpool(C, H, W, k, s, pad, dX, B, dY)
    assert np.array_equal(dY.download().view(np.uint32), want.view(np.uint32))
    dX.free()
    dY.free()


@pytest.mark.parametrize("H,W", [(1, 1), (2, 4), (3, 3), (4, 4), (1, 17), (4, 8), (3, 11), (7, 7), (8, 8), (5, 13), (9, 11)])
@pytest.mark.parametrize("C,B", [(1, 1), (67, 1), (70, 3), (33, 4), (5, 129)])
def test_gap_forms(ctx, H, W, C, B):
    rng = np.random.default_rng(H * W + C + B)
    X = rng.standard_normal((C, H, W, B)).astype(np.float32)
    X[0, :, :, 0] = -0.0
    X[-1, H // 2, W // 2, -1] = np.inf
    s = np.zeros((C, B), np.float32)
    for h in range(H):
        for w in range(W):
            s = s + X[:, h, w]
    want = s * (np.float32(1.0) / np.float32(H * W))
    dX, dY = ctx.array(X), ctx.empty((C, B))
    ctx.gap(C, H, W, dX, B, dY)
    assert np.array_equal(dY.download().view(np.uint32), want.view(np.uint32))
    dX.free()
    dY.free()


def test_small_and_flat_kernels_cost_no_more_than_a_square_one(ctx):
    """Only the kernel's own taps are read: at stride 2, 1x2 and 4x1 windows (half of an image of 103 MB) take less time than 3x3 ones, which read all of it.  With
    taps beside the kernel read as well they took 1.04 and 1.4 times as long, and take 0.64 and 0.67 times now; the lines lie half-way."""
    C, H, W, B = 64, 112, 112, 32
    dX, dY = ctx.array(np.zeros((C, H, W, B), np.float32)), ctx.empty((C, H, W, B))

    def us(k, pad):
        times = []
        for _ in range(7):
            ctx.timer_begin()
            for _ in range(30):
                ctx.maxpool(C, H, W, k, (2, 2), pad, dX, B, dY)
            times.append(ctx.timer_end())
        return sorted(times)[3]

    whole = us((3, 3), (1, 1))
    assert us((1, 2), (0, 0)) < 0.84 * whole
    assert us((4, 1), (0, 0)) < 1.03 * whole
    dX.free()
    dY.free()


@pytest.mark.parametrize("B", [1, 4])
@pytest.mark.parametrize("k", [(3, 1), (2, 3), (8, 1), (15, 1), (4, 2), (7, 2), (6, 3), (8, 3), (1, 4), (3, 5), (2, 6), (1, 7), (2, 8), (1, 15), (2, 16)])
def test_maxpool_blocks_and_what_is_left(ctx, B, k):
    rng = np.random.default_rng(k[0] * 20 + k[1])
    X = rng.standard_normal((3, 18, 21, B)).astype(np.float32)
    for s, pad in (((1, 1), (k[0] // 2, k[1] // 2)), ((2, 3), (0, 0))):
        want = maxpool(X, k, s, pad)
        dX, dY = ctx.array(X), ctx.array(np.full(want.shape, 7, np.float32))
        ctx.maxpool(3, 18, 21, k, s, pad, dX, B, dY)
        assert np.array_equal(dY.download().view(np.uint32), want.view(np.uint32))
        dX.free()
        dY.free()
