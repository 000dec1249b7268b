"""The framework's own work, as its users call it: what is timed and compared when a kernel or a host path changes.

Every case is one pass through a public entry point: the C ABI's ctypes binding (`hipabi.Context`) on operands that
already lie in device memory, or the `sparseops_backend` module (the drop-in for the reference's Python module) on
host arrays.  A case is a dict of plain sizes and options, `kind` says which path it takes:

  matmul   so_matmul, Y = act(E X + b): a pruned layer on a batch.  The sizes run over the reference's published
           table (512 to 2048 square, 50-90 % sparse, 64 dense columns), the large pruned FC layer of the benchmark,
           classifier heads (few rows), ragged sizes, batches from 1 up.
  matvec   so_matvec, y = E x + b: a solver's or a decoder's product with one vector, even rows or Zipf rows.
  hostvec  sparseops_backend.ellpack_matvec on numpy arrays: the reference's own call, host memory to host memory.
  encode   so_ellpack_encode_noalloc: dense weights to ELLPACK, as after every pruning step.
  decode   so_ellpack_decode: back to dense.
  mlp      SparseOnnxModel.run on numpy arrays, fully connected layers: inference on a batch that arrives from the host.
  cnn      SparseOnnxModel.run_device (inputs already on the GPU) or .run (host arrays) on the ResNet-18-shaped
           stack of the benchmark.

Matrices, inputs and models are made from the seed alone, so another seed is another problem of the same shape.
Weights are uploaded and models are loaded in `prepare`, as a program does once; `run` is one call."""
import math
import os
import sys
import tempfile

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "sparse-ops_amd")
for _p in (_PKG, os.path.join(_PKG, "python")):
    if _p not in sys.path:
        sys.path.insert(0, _p)

import datagen  # noqa: E402
import hipabi  # noqa: E402
import onnx_wire  # noqa: E402
import sparseops_backend  # noqa: E402

ACTS = ("none", "relu", "sigmoid", "tanh")

# The copies of a matrix that so_matmul and so_matvec may choose from, as the interface header recommends them: for a
# product with a batch of columns the row-block-merged and the K-tiled copy, for a product with one vector the length
# classes and the 16-bit columns.
MATMUL_LAYOUTS = hipabi.LAYOUT_ROW | hipabi.LAYOUT_TILED | hipabi.LAYOUT_RBM
MATVEC_LAYOUTS = hipabi.LAYOUT_ROW | hipabi.LAYOUT_BINS | hipabi.LAYOUT_IDX16


def listed():
    return [
        # the reference's small published shape: the launch is most of it
        {"name": "matmul_1024_c64", "kind": "matmul", "m": 1024, "n": 1024, "C": 64, "sparsity": 0.9, "rows": "even", "bias": True, "act": "none"},
        # the table's largest shape at 80 %
        {"name": "matmul_2048_c64", "kind": "matmul", "m": 2048, "n": 2048, "C": 64, "sparsity": 0.8, "rows": "even", "bias": False, "act": "none"},
        # the large FC layer of the benchmark: top-10 % of every row, batch 256
        {"name": "matmul_4096_c256", "kind": "matmul", "m": 4096, "n": 4096, "C": 256, "sparsity": 0.9, "rows": "topk", "bias": True, "act": "none"},
        # no size a multiple of anything, moderately pruned, fused ReLU
        {"name": "matmul_ragged", "kind": "matmul", "m": 3001, "n": 2777, "C": 101, "sparsity": 0.7, "rows": "even", "bias": True, "act": "relu"},
        # the reference's call on host arrays, small: latency of copy in, launch, copy out
        {"name": "hostvec_1500", "kind": "hostvec", "m": 1500, "n": 1000, "sparsity": 0.9, "rows": "even", "bias": True},
        # large memory-bound products with one vector: even and skewed rows
        {"name": "matvec_16384", "kind": "matvec", "m": 16384, "n": 16384, "sparsity": 0.95, "rows": "even", "bias": True},
        {"name": "matvec_16384_zipf", "kind": "matvec", "m": 16384, "n": 16384, "sparsity": 0.95, "rows": "zipf", "bias": True},
        # re-encoding a pruned layer, and back
        {"name": "encode_8192", "kind": "encode", "m": 8192, "n": 8192, "sparsity": 0.9, "rows": "even"},
        {"name": "decode_8192", "kind": "decode", "m": 8192, "n": 8192, "sparsity": 0.9, "rows": "even"},
        # the benchmark's MLP, host to host
        {"name": "mlp_b256", "kind": "mlp", "dims": "784-4096-4096-4096-10", "B": 256, "sparsity": 0.9},
        # the benchmark's convolution stack: a throughput batch already on the GPU, one image from the host
        {"name": "cnn_b32", "kind": "cnn", "B": 32, "hw": 224, "width": 64, "sparsity": 0.8, "host": False},
        {"name": "cnn_b1_host", "kind": "cnn", "B": 1, "hw": 224, "width": 64, "sparsity": 0.8, "host": True},
    ]


def _log_size(rng, lo, hi):
    """A whole number of lo..hi, even over the logarithm: odd ones as often as multiples of 16 would be useful to a tile."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("matmul", "matmul", "matmul", "matvec", "hostvec", "encode", "decode", "mlp", "cnn"))
    if kind == "matmul":
        return {"kind": kind, "m": _log_size(rng, 10, 4096), "n": _log_size(rng, 512, 4096), "C": _log_size(rng, 1, 256),
                "sparsity": round(rng.uniform(0.5, 0.95), 3), "rows": rng.choice(("even", "even", "topk")),
                "bias": rng.random() < 0.5, "act": rng.choice(ACTS)}
    if kind in ("matvec", "hostvec"):
        top = 16384 if kind == "matvec" else 4096
        return {"kind": kind, "m": _log_size(rng, 1024, top), "n": _log_size(rng, 1024, top), "sparsity": round(rng.uniform(0.8, 0.98), 3),
                "rows": rng.choice(("even", "zipf")), "bias": rng.random() < 0.5}
    if kind in ("encode", "decode"):
        return {"kind": kind, "m": _log_size(rng, 256, 8192), "n": _log_size(rng, 256, 8192), "sparsity": round(rng.uniform(0.5, 0.98), 3),
                "rows": rng.choice(("even", "zipf"))}
    if kind == "mlp":
        dims = [_log_size(rng, 64, 1024)] + [_log_size(rng, 256, 4096) for _ in range(rng.randint(1, 3))] + [_log_size(rng, 10, 1000)]
        return {"kind": kind, "dims": "-".join(map(str, dims)), "B": _log_size(rng, 1, 256), "sparsity": round(rng.uniform(0.6, 0.95), 3)}
    return {"kind": kind, "B": _log_size(rng, 1, 32), "hw": 32 * rng.randint(2, 7), "width": rng.choice((16, 32, 48, 64)),
            "sparsity": round(rng.uniform(0.6, 0.9), 3), "host": rng.random() < 0.5}


# ---- what a program holds before the call -------------------------------------------------------------------------

_context = None


def context():
    """One context for the process, as a program has it."""
    global _context
    if _context is None:
        _context = hipabi.Context(0)
    return _context


class OnGpu:
    """A torch tensor's memory as the binding's calls take it (they read only `.ptr`)."""

    def __init__(self, tensor):
        self.tensor, self.ptr = tensor, tensor.data_ptr()


class Weights:
    """An uploaded matrix that is freed with the state that holds it."""

    def __init__(self, handle):
        self.handle = handle

    def __del__(self):
        self.handle.free()


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _dense(case, g):
    """The pruned matrix, dense, on the GPU: normal values; `even` keeps each with probability 1 - sparsity, `topk` the
    largest of every row, `zipf` gives row i min(Zipf(1.2), n / 8) entries in random places."""
    m, n, keep = case["m"], case["n"], 1.0 - case["sparsity"]
    W = torch.randn(m, n, device="cuda", generator=g) * (1.0 / math.sqrt(max(1.0, n * keep)))
    if case["rows"] == "topk":
        k = max(1, int(round(n * keep)))
        cut = W.abs().topk(k, dim=1).values[:, -1:]
        return torch.where(W.abs() >= cut, W, torch.zeros((), device="cuda"))
    share = torch.rand(m, n, device="cuda", generator=g)
    if case["rows"] == "even":
        return torch.where(share < keep, W, torch.zeros((), device="cuda"))
    # a Zipf(1.2) length by inverting the tail of the continuous law, cut off at an eighth of the row
    u = torch.rand(m, 1, device="cuda", generator=g).clamp_min(1e-12)
    length = u.pow(-1.0 / 0.2).floor().clamp(1, max(1, n // 8))
    return torch.where(share < length / n, W, torch.zeros((), device="cuda"))


def _host_ellpack(case, g):
    """The matrix as the encoder lays it out, in host arrays."""
    W = _dense(case, g)
    torch.cuda.synchronize()
    E = context().encode_dense(OnGpu(W), case["m"], case["n"])
    Wd, idx, nnz = E.download()
    r = E.r
    E.free()
    return Wd, idx, nnz, r


def _weights(case, g, layouts):
    Wd, idx, nnz, r = _host_ellpack(case, g)
    return Weights(context().upload_ellpack(Wd, idx, nnz, case["m"], case["n"], r, layouts))


def _bias(case, g):
    return torch.randn(case["m"], device="cuda", generator=g) * 0.1 if case["bias"] else None


def _load(payload):
    with tempfile.TemporaryDirectory() as d:
        return sparseops_backend.SparseOnnxModel(onnx_wire.save(os.path.join(d, "model.onnx"), payload))


def _mlp(case, seed):
    dims = [int(d) for d in case["dims"].split("-")]
    rng = np.random.default_rng(seed)
    Ws = [datagen.bernoulli_dense(rng, fout, fin, 1.0 - case["sparsity"], 1.0 / math.sqrt(fin * (1.0 - case["sparsity"])))
          for fin, fout in zip(dims[:-1], dims[1:])]
    acts = ["Relu", "Sigmoid", "Tanh"][:len(Ws) - 1] + [None]
    model = _load(onnx_wire.mlp_model(Ws, acts, case["B"]))
    model.resize_buffers(case["B"])
    return {"model": model, "X": rng.random((case["B"], dims[0]), dtype=np.float32)}


def _cnn(case, seed):
    payload, _ = datagen.resnet18_onnx(seed=seed, batch=case["B"], hw=case["hw"], sparsity=case["sparsity"], width=case["width"])
    model = _load(payload)
    model.resize_buffers(case["B"])
    B, hw = case["B"], case["hw"]
    if case["host"]:
        return {"model": model, "X": np.random.default_rng(seed + 1).standard_normal((B, 3, hw, hw), dtype=np.float32)}
    # [C][H][W][B] in, [classes][B] out: the device entry point's layouts
    return {"model": model, "X": torch.randn(3, hw, hw, B, device="cuda", generator=_generator(seed)),
            "Y": torch.zeros(1000, B, device="cuda")}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "mlp":
        return dict(_mlp(case, seed), kind=kind)
    if kind == "cnn":
        return dict(_cnn(case, seed), kind=kind, host=case["host"], B=case["B"])
    g = _generator(seed)
    m, n = case["m"], case["n"]
    s = {"kind": kind, "m": m, "n": n}
    if kind == "matmul":
        C = case["C"]
        s.update(C=C, act=case["act"], E=_weights(case, g, MATMUL_LAYOUTS), X=torch.randn(n, C, device="cuda", generator=g),
                 Y=torch.zeros(m, C, device="cuda"), bias=_bias(case, g))
        context().matmul_reserve(s["E"].handle, C)
    elif kind == "matvec":
        s.update(E=_weights(case, g, MATVEC_LAYOUTS), X=torch.randn(n, device="cuda", generator=g), Y=torch.zeros(m, device="cuda"),
                 bias=_bias(case, g))
    elif kind == "hostvec":
        W = _dense(case, g).cpu().numpy()
        bias = _bias(case, g)
        s.update(E=sparseops_backend.convert_to_ellpack(W), X=torch.randn(n, device="cuda", generator=g).cpu().numpy(),
                 bias=None if bias is None else bias.cpu().numpy())
    elif kind == "encode":
        W = _dense(case, g)
        # room for rows eight standard deviations longer than expected
        longest = n // 8 if case["rows"] == "zipf" else n * (1.0 - case["sparsity"])
        cap = min(n, int(longest + 8.0 * math.sqrt(longest) + 8.0))
        s.update(W=W, r_cap=cap, Wd=torch.zeros(m * cap, device="cuda"), idx=torch.zeros(m * cap, dtype=torch.int32, device="cuda"),
                 nnz=torch.zeros(m, dtype=torch.int32, device="cuda"))
    else:
        s.update(E=_weights(case, g, hipabi.LAYOUT_ROW), Y=torch.zeros(m, n, device="cuda"))
    torch.cuda.synchronize()   # the framework's calls run on its own stream
    for key in ("W", "X", "Y", "bias", "Wd", "idx", "nnz"):   # the operands as the binding takes them
        s["d" + key] = OnGpu(s[key]) if isinstance(s.get(key), torch.Tensor) else None
    return s


# ---- one pass -----------------------------------------------------------------------------------------------------

def run(s):
    kind = s["kind"]
    if kind == "matmul":
        context().matmul(s["E"].handle, s["dX"], s["C"], s["dbias"], s["dY"], s["act"])
        return s["Y"]
    if kind == "matvec":
        context().matvec(s["E"].handle, s["dX"], s["dbias"], s["dY"])
        return s["Y"]
    if kind == "hostvec":
        return sparseops_backend.ellpack_matvec(s["E"], s["X"], s["bias"])
    if kind == "encode":
        r, total = context().encode_dense_noalloc(s["dW"], s["m"], s["n"], s["r_cap"], s["dWd"], s["didx"], s["dnnz"])
        return {"r": r, "total": total, "nnz": s["nnz"], "Wd": s["Wd"], "idx": s["idx"]}
    if kind == "decode":
        ctx = context()
        ctx._ck(ctx.lib.so_ellpack_decode(ctx.h, s["E"].handle.h, s["dY"].ptr))
        return s["Y"]
    if kind == "cnn" and not s["host"]:
        s["model"].run_device(s["X"].data_ptr(), s["B"], s["Y"].data_ptr())
        return s["Y"]
    return s["model"].run(s["X"])


# ---- what a pass cannot do without, and how close two correct passes are -------------------------------------------

def _kept(case):
    """Stored nonzeros, as expected of the draw."""
    if case["rows"] != "zipf":
        return (1.0 - case["sparsity"]) * case["m"] * case["n"]
    cap = max(1, case["n"] // 8)   # E[min(Zipf, cap)] of the law in _dense: sum over k of P(length >= k)
    return case["m"] * float(np.sum(np.arange(1, cap + 1, dtype=np.float64) ** -0.2))


def _resnet_flops_and_weights(case):
    """(multiply-adds x 2, stored weights) of the stack for one image."""
    w, hw, keep = case["width"], case["hw"] // 2, 1.0 - case["sparsity"]
    flops, weights = 0.0, 0.0

    def conv(cin, cout, k, out_hw):
        nonlocal flops, weights
        nnz = keep * cin * cout * k * k
        weights += nnz
        flops += 2.0 * nnz * out_hw * out_hw

    conv(3, w, 7, hw)
    hw, cin = (hw + 1) // 2, w
    for stage, cout in enumerate((w, 2 * w, 4 * w, 8 * w)):
        for block in range(2):
            down = stage > 0 and block == 0
            hw = (hw + 1) // 2 if down else hw
            conv(cin, cout, 3, hw)
            conv(cout, cout, 3, hw)
            if down:
                conv(cin, cout, 1, hw)
            cin = cout
    return flops + 2.0 * 1000 * cin, weights + 1000.0 * cin


def work(case):
    kind = case["kind"]
    if kind == "mlp":
        dims = [int(d) for d in case["dims"].split("-")]
        nnz = (1.0 - case["sparsity"]) * sum(a * b for a, b in zip(dims[:-1], dims[1:]))
        return {"bytes": 8.0 * nnz + 4.0 * case["B"] * (dims[0] + dims[-1]), "flops": 2.0 * nnz * case["B"]}
    if kind == "cnn":
        flops, weights = _resnet_flops_and_weights(case)
        return {"bytes": 8.0 * weights + 4.0 * case["B"] * (3 * case["hw"] ** 2 + 1000), "flops": flops * case["B"]}
    m, n, nnz = case["m"], case["n"], _kept(case)
    if kind in ("encode", "decode"):
        return {"bytes": 4.0 * m * n + 8.0 * nnz + 4.0 * m, "flops": 0.0}
    C = case.get("C", 1)
    # a weight and its column, row lengths, bias, X, Y; at 65536 columns or fewer a column takes 2 bytes
    return {"bytes": 6.0 * nnz + 4.0 * m + (4.0 * m if case["bias"] else 0.0) + 4.0 * (n + m) * C, "flops": 2.0 * nnz * C}


def tolerance(case):
    """About four times what the 32-bit paths were seen to be away from the same problems in 64 bits, over the listed
    cases and a dozen drawn ones: at most 5.5e-7 in the 2-norm and 3.5e-6 for a single value."""
    if case["kind"] in ("encode", "decode"):
        return "exact"
    return {"rel": 2.5e-6, "max": 1.5e-5}
