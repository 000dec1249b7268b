"""so_conv2d_pair: the bits of so_conv2d on each plan, in one launch on the column and the windowed kernel or in two, launched and recorded; a model whose
exporter put a block's projection before, after or behind the main branch."""
import numpy as np
import pytest

import datagen
import hipabi
import onnx_wire as ow

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = hipabi.Context(0)
    yield c
    c.close()


def sparse(rng, m, n, keep):
    W = rng.standard_normal((m, n)).astype(np.float32)
    W[rng.random((m, n)) >= keep] = 0
    return W


class Conv:
    def __init__(self, ctx, rng, Cin, Cout, k, s, H, W, B, keep, bias):
        self.g = hipabi.conv_geom(Cin, Cout, k, k, H, W, (s, s), (k // 2, k // 2))
        E = datagen.encode_dense(sparse(rng, Cout, Cin * k * k, keep))
        self.ctx, self.dE = ctx, ctx.upload_ellpack(E.Wd, E.idx, E.nnz, E.m, E.n, E.r)
        self.plan = ctx.conv_plan(self.dE, self.g)
        ctx.conv_plan_tune(self.plan, B)
        self.dB = ctx.array(rng.standard_normal(Cout).astype(np.float32)) if bias else None
        self.shape = (Cout, self.g.H_out, self.g.W_out, B)
        self.dY = ctx.empty(self.shape)

    def alone(self, dX, B, act):
        self.dY.upload(np.full(self.shape, np.nan, np.float32))
        self.ctx.conv2d(self.plan, dX, B, self.dB, self.dY, act)
        return self.dY.download().view(np.uint32), self.ctx.last_kernel()

    def free(self):
        self.ctx.conv_plan_free(self.plan)
        for a in (self.dE, self.dB, self.dY):
            if a:
                a.free()


#  Cin, H, W, (Cout, k, s, keep) x 2, batches, what runs in one launch: workgroups of one or several sizes, both resident or one behind the other; windows
#  with one and two pixel groups a wave and every number of channels; a last block of channels that is not full; different outputs' sizes
@pytest.mark.parametrize("Cin,H,W,first,second,B,kernel", [
    (16, 14, 14, (32, 3, 2, .3), (32, 1, 2, .6), 1, "columns-pair"), (16, 14, 14, (32, 1, 2, .6), (32, 3, 2, .3), 2, "columns-pair"),
    (37, 13, 9, (61, 3, 1, .2), (7, 5, 2, .3), 3, "columns-pair"), (128, 28, 28, (256, 3, 2, .2), (256, 1, 2, .3), 1, "columns-pair"),
    (256, 14, 14, (512, 3, 2, .2), (512, 1, 2, .2), 8, "columns-pair"), (64, 24, 24, (128, 3, 2, .35), (128, 1, 2, .35), 8, "columns-pair"),
    (64, 56, 56, (128, 3, 2, .2), (128, 1, 2, .2), 32, "window-pair"), (128, 28, 28, (256, 3, 2, .2), (256, 1, 2, .2), 32, "window-pair"),
    (256, 14, 14, (512, 3, 2, .2), (512, 1, 2, .2), 32, "window-pair"), (64, 28, 28, (67, 3, 1, .2), (66, 3, 1, .3), 16, "window-pair"),
    (64, 56, 56, (128, 3, 2, .2), (128, 1, 2, .2), 8, "window-pair"), (32, 16, 16, (64, 3, 2, .2), (64, 1, 2, .4), 4, "window-pair"),
    (16, 14, 14, (32, 3, 2, .3), (32, 1, 2, .6), 5, None), (64, 56, 56, (128, 3, 2, .2), (1, 1, 2, .2), 32, None)])
def test_pair_is_both(ctx, Cin, H, W, first, second, B, kernel):
    rng = np.random.default_rng(Cin + H + B)
    X = rng.standard_normal((Cin, H, W, B)).astype(np.float32)
    X[0, 0, 0, 0], X[-1, -1, -1, -1] = np.inf, np.nan
    dX = ctx.array(X)
    a, b = (Conv(ctx, rng, Cin, o[0], o[1], o[2], H, W, B, o[3], bias) for o, bias in ((first, True), (second, False)))
    for actA, actB in (("relu", "none"), ("none", "relu"), ("tanh", "none")):
        (wantA, _), (wantB, last) = a.alone(dX, B, actA), b.alone(dX, B, actB)
        runs = [lambda: ctx.conv2d_pair(a.plan, b.plan, dX, B, a.dB, a.dY, actA, b.dB, b.dY, actB)]
        ctx.graph_begin()
        runs[0]()
        graph = ctx.graph_end()
        for run in runs + [lambda: ctx.graph_launch(graph)] * 2:
            for c in (a, b):
                c.dY.upload(np.full(c.shape, np.nan, np.float32))
            run()
            assert np.array_equal(a.dY.download().view(np.uint32), wantA) and np.array_equal(b.dY.download().view(np.uint32), wantB)
        runs[0]()
        assert ctx.last_kernel() == (kernel if kernel and actA != "tanh" else last)
        ctx.sync()
        ctx.graph_free(graph)
    for x in (a, b, dX):
        x.free()


def test_pair_refuses(ctx):
    rng = np.random.default_rng(0)
    dX = ctx.array(rng.standard_normal((8, 8, 8, 4)).astype(np.float32))
    a, b, other = Conv(ctx, rng, 8, 8, 3, 1, 8, 8, 4, .5, False), Conv(ctx, rng, 8, 4, 3, 1, 8, 8, 4, .5, False), Conv(ctx, rng, 8, 8, 3, 1, 8, 9, 4, .5, False)
    for plans, outs in (((a, b), (a.dY, a.dY)), ((a, b), (dX, b.dY)), ((a, b), (a.dY, dX)), ((a, other), (a.dY, other.dY))):
        with pytest.raises(hipabi.SoError):
            ctx.conv2d_pair(plans[0].plan, plans[1].plan, dX, 4, None, outs[0], "none", None, outs[1], "none")
    f, p = ctx.lib.so_conv2d_pair, (ctx.h, a.plan, b.plan, dX.ptr, 4, None, a.dY.ptr, 0, None, b.dY.ptr, 0)
    for i, bad in ((1, None), (2, None), (3, None), (6, None), (9, None), (7, 9), (10, -1)):
        assert f(*(p[:i] + (bad,) + p[i + 1:])) != 0
    for x in (a, b, other, dX):
        x.free()


@pytest.mark.parametrize("B", [1, 4, 32])
def test_projection_anywhere(backend, oracle, tmp_path, B):
    """conv1 -> relu -> conv2, projection of the block's input, Add, Relu: the projection first, between and last."""
    from graph_oracle import run_graph
    rng = np.random.default_rng(B)
    t = {"w1": sparse(rng, 32, 16 * 9, .3).reshape(32, 16, 3, 3), "w2": sparse(rng, 32, 32 * 9, .3).reshape(32, 32, 3, 3), "wp": sparse(rng, 32, 16, .5).reshape(32, 16, 1, 1),
         "w0": sparse(rng, 16, 27, .5).reshape(16, 3, 3, 3), "b1": rng.standard_normal(32).astype(np.float32), "bp": rng.standard_normal(32).astype(np.float32)}

    def conv(x, w, y, k, s, b=()):
        return ow.node("Conv", [x, w, *b], [y], kernel_shape=[k, k], pads=[k // 2] * 4, strides=[s, s], dilations=[1, 1], group=1)
    stem = [conv("input", "w0", "x", 3, 1)]
    main = [conv("x", "w1", "c1", 3, 2, ("b1",)), ow.node("Relu", ["c1"], ["r1"]), conv("r1", "w2", "c2", 3, 1)]
    proj = [conv("x", "wp", "p", 1, 2, ("bp",))]
    tail = [ow.node("Add", ["c2", "p"], ["s"]), ow.node("Relu", ["s"], ["y"])]
    X = rng.standard_normal((B, 3, 14, 14)).astype(np.float32)
    seen = set()
    for nodes in (proj + main, main[:2] + proj + main[2:], main + proj):
        payload = ow.model(stem + nodes + tail, [("input", (B, 3, 14, 14))], [("y", (B, 32, 7, 7))], list(t.items()))
        model = backend.SparseOnnxModel(ow.save(str(tmp_path / "m.onnx"), payload))
        desc = model.describe()
        assert len(desc) == 4 and "+residual" in desc[3] and "act=relu" in desc[3] and sum("+residual" in d for d in desc) == 1
        Y = model.run(X)
        assert np.array_equal(Y.reshape(-1), run_graph(oracle, payload, X).reshape(-1))
        seen.add(Y.tobytes())
    assert len(seen) == 1
