"""What is measured: one pass of the work that a program has this framework do.

Seven kinds of call, each through the Python binding's public entry points, over the sizes
of the benchmark configurations, the tests and of ordinary use:

* host_matmul  a product of host arrays through the reference-compatible C ABI: upload,
               multiply, retrieve, release (the Go packages' GPUMatMul call sequence);
* mlp          inference of a small classifier on device tensors: two hidden layers with
               ReLU, an output layer and a row-wise softmax;
* gemm         a product on device tensors: fp32 or fp16 inputs, four layouts, batches;
* linear       a linear layer's forward, from one row (decode) to a full batch (prefill),
               weights stored out x in ("nt") or in x out ("nn"), bias and activation in the
               same call;
* backward     a linear layer's backward: activation gradient, bias, input and weight
               gradients;
* spmm, spmv   CSR times dense matrix, and CSR times vector with a plan kept for the
               structure.

Calls run on a torch stream of their own, as bench.py and a serving loop have it.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "go-nngpu_amd"))
import gonngpu as G  # noqa: E402

_ACT = {"none": G.ACT_NONE, "relu": G.ACT_RELU, "gelu": G.ACT_GELU}


def listed():
    return [
        # One product of host arrays, start to end: the parity configuration's 256 x 256. The
        # smallest call; what it costs is copies, launches and waits.
        {"name": "host_matmul_256", "kind": "host_matmul", "m": 256, "n": 256, "k": 256},
        # A small classifier's inference on a batch of 256 28 x 28 inputs: four short kernels.
        {"name": "mlp_256", "kind": "mlp", "rows": 256, "inputs": 784, "hidden1": 512, "hidden2": 256, "classes": 10},
        # The fp32 product that the benchmark quotes (4096^3), row-major operands.
        {"name": "gemm_f32_4096", "kind": "gemm", "dtype": "f32", "layout": "nn", "batch": 1, "m": 4096, "n": 4096, "k": 4096},
        # An fp32 product of odd sizes, neither operand aligned, A stored transposed.
        {"name": "gemm_f32_odd", "kind": "gemm", "dtype": "f32", "layout": "tn", "batch": 1, "m": 777, "n": 1234, "k": 4099},
        # A batch of 64 middling fp32 products (the batched product's entry point).
        {"name": "gemm_f32_batch", "kind": "gemm", "dtype": "f32", "layout": "nt", "batch": 64, "m": 256, "n": 192, "k": 96},
        # The fp16 headline product, the largest call.
        {"name": "gemm_f16_8192", "kind": "gemm", "dtype": "f16", "layout": "nn", "batch": 1, "m": 8192, "n": 8192, "k": 8192},
        # The fused linear layer of the benchmark: a batch of 512 rows, fp16, GELU.
        {"name": "linear_f16_512", "kind": "linear", "dtype": "f16", "layout": "nt", "act": "gelu", "rows": 512, "inputs": 4096, "outputs": 11008},
        # The same layer in fp32 at a batch of 16: it reads its weights and little else.
        {"name": "linear_f32_16", "kind": "linear", "dtype": "f32", "layout": "nt", "act": "relu", "rows": 16, "inputs": 4096, "outputs": 11008},
        # Decode: four rows through fp16 weights stored in x out (the reference's LinearLayer).
        {"name": "linear_f16_4", "kind": "linear", "dtype": "f16", "layout": "nn", "act": "none", "rows": 4, "inputs": 4096, "outputs": 11008},
        # Training: the fused linear layer's backward in fp32, 512 rows.
        {"name": "backward_f32_512", "kind": "backward", "dtype": "f32", "act": "gelu", "rows": 512, "inputs": 4096, "outputs": 11008},
        # CSR products of the benchmark: 65536 x 65536 with 0.1 % stored, times 256 columns and times a vector.
        {"name": "spmm_65536", "kind": "spmm", "m": 65536, "k": 65536, "mean": 65.5, "n": 256},
        {"name": "spmv_65536", "kind": "spmv", "m": 65536, "k": 65536, "mean": 65.5},
    ]


def _size(rng, lo, hi):
    """A size between lo and hi, spread over its logarithm; half of them multiples of 32."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if v >= 64 and rng.random() < 0.5:
        v = v // 32 * 32
    return max(lo, min(hi, v))


def draw(rng):
    kind = rng.choice(["host_matmul", "mlp", "gemm", "gemm", "gemm", "linear", "linear", "linear", "backward", "spmm", "spmv"])
    if kind == "host_matmul":
        return {"kind": kind, "m": _size(rng, 16, 1024), "n": _size(rng, 16, 1024), "k": _size(rng, 16, 1024)}
    if kind == "mlp":
        return {"kind": kind, "rows": _size(rng, 1, 1024), "inputs": _size(rng, 64, 1024), "hidden1": _size(rng, 64, 1024),
                "hidden2": _size(rng, 32, 512), "classes": _size(rng, 2, 1000)}
    if kind == "gemm":
        dtype = rng.choice(["f32", "f32", "f16"])
        batch = rng.choice([1, 1, 1, _size(rng, 2, 96)])
        most = 512 if batch > 1 else 8192
        while True:
            c = {"kind": kind, "dtype": dtype, "layout": rng.choice(["nn", "nt", "tn", "tt"]), "batch": batch,
                 "m": _size(rng, 32, most), "n": _size(rng, 32, most), "k": _size(rng, 32, most)}
            if work(c)["flops"] <= (2.0 * 8192**3 if dtype == "f16" else 2.0 * 4096**3):
                return c
    if kind == "linear":
        return {"kind": kind, "dtype": rng.choice(["f32", "f16"]), "layout": rng.choice(["nt", "nn"]), "act": rng.choice(["none", "relu", "gelu"]),
                "rows": _size(rng, 1, 1024), "inputs": _size(rng, 256, 8192), "outputs": _size(rng, 256, 11008)}
    if kind == "backward":
        return {"kind": kind, "dtype": rng.choice(["f32", "f16"]), "act": rng.choice(["relu", "gelu"]), "rows": _size(rng, 16, 1024),
                "inputs": _size(rng, 128, 4096), "outputs": _size(rng, 128, 11008)}
    c = {"kind": kind, "m": _size(rng, 1024, 65536), "k": _size(rng, 1024, 65536), "mean": round(rng.uniform(4.0, 65.0), 1)}
    if kind == "spmm":
        c["n"] = _size(rng, 8, 256)
    return c


# ------------------------------------------------------------------ inputs
def _normal(g, shape, std=1.0):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).mul_(std)


def _stored(g, rows, cols, transposed, std, dtype, batch=1):
    """op(X) is rows x cols; the stored array is its transpose where `transposed` says so."""
    shape = (cols, rows) if transposed else (rows, cols)
    x = _normal(g, shape if batch == 1 else (batch,) + shape, std)
    return x.half() if dtype == "f16" else x


def _csr(g, m, k, mean):
    """CSR with row lengths around `mean`, distinct uniform columns sorted per row, values U[-1, 1)."""
    lens = torch.poisson(torch.full((m,), float(mean), device="cuda"), generator=g).long()
    rows = torch.repeat_interleave(torch.arange(m, device="cuda"), lens)
    keys = torch.unique(rows * k + torch.randint(0, k, (rows.numel(),), generator=g, device="cuda"))
    rows, col = keys // k, (keys % k).int()
    ptr = torch.zeros(m + 1, dtype=torch.int64, device="cuda")
    ptr[1:] = torch.cumsum(torch.bincount(rows, minlength=m), 0)
    val = torch.rand(col.numel(), generator=g, device="cuda").mul_(2.0).sub_(1.0)
    return ptr.int(), col, val


def _inputs(c, seed):
    """The inputs of one pass, from the seed alone (host arrays for the host product)."""
    kind = c["kind"]
    if kind == "host_matmul":
        r = np.random.default_rng(seed)
        return {"a": r.standard_normal((c["m"], c["k"]), dtype=np.float32), "b": r.standard_normal((c["k"], c["n"]), dtype=np.float32)}
    g = torch.Generator(device="cuda").manual_seed(seed)
    if kind == "mlp":
        sizes = [c["inputs"], c["hidden1"], c["hidden2"], c["classes"]]
        s = {"x": torch.rand((c["rows"], c["inputs"]), generator=g, device="cuda")}  # pixels in [0, 1)
        for i, (a, b) in enumerate(zip(sizes, sizes[1:])):
            s["w%d" % i] = _normal(g, (a, b), math.sqrt(2.0 / a))
            s["b%d" % i] = _normal(g, (b,), 0.01)
        return s
    if kind == "gemm":
        ta, tb = c["layout"][0] == "t", c["layout"][1] == "t"
        return {"a": _stored(g, c["m"], c["k"], ta, 1.0, c["dtype"], c["batch"]),
                "b": _stored(g, c["k"], c["n"], tb, 0.02 if c["dtype"] == "f16" else 1.0, c["dtype"], c["batch"])}
    if kind == "linear":
        return {"x": _stored(g, c["rows"], c["inputs"], False, 1.0, c["dtype"]),
                "w": _stored(g, c["inputs"], c["outputs"], c["layout"] == "nt", 0.02, c["dtype"]), "b": _normal(g, (c["outputs"],), 0.01)}
    if kind == "backward":
        s = {"x": _stored(g, c["rows"], c["inputs"], False, 1.0, c["dtype"]), "w": _stored(g, c["inputs"], c["outputs"], False, 0.02, c["dtype"]),
             "g": _normal(g, (c["rows"], c["outputs"]), 0.1)}
        s["pre"] = _normal(g, (c["rows"], c["outputs"]), 1.0)  # what the forward kept: X W + b
        return s
    ptr, col, val = _csr(g, c["m"], c["k"], c["mean"])
    dense = _normal(g, (c["k"], c["n"]) if kind == "spmm" else (c["k"],))
    return {"ptr": ptr, "col": col, "val": val, "d": dense}


_stream = None


def _use_stream():
    """Makes a stream of its own torch's current one (the default stream would be waited for around every call)."""
    global _stream
    if torch.cuda.current_stream().cuda_stream == 0:
        if _stream is None:
            _stream = torch.cuda.Stream()
        torch.cuda.synchronize()
        torch.cuda.set_stream(_stream)


def _empty(*shape, dtype=torch.float32):
    return torch.empty(shape, dtype=dtype, device="cuda")


def prepare(case, seed):
    _use_stream()
    c, s = case, _inputs(case, seed)
    s["c"] = dict(c)
    kind = c["kind"]
    if kind == "mlp":
        s["h1"], s["h2"] = _empty(c["rows"], c["hidden1"]), _empty(c["rows"], c["hidden2"])
        s["logits"], s["y"] = _empty(c["rows"], c["classes"]), _empty(c["rows"], c["classes"])
    elif kind == "gemm":
        s["y"] = _empty(c["m"], c["n"]) if c["batch"] == 1 else _empty(c["batch"], c["m"], c["n"])
    elif kind == "linear":
        s["y"] = _empty(c["rows"], c["outputs"])
    elif kind == "backward":
        s["grad"], s["db"] = _empty(c["rows"], c["outputs"]), _empty(c["outputs"])
        s["dx"], s["dw"] = _empty(c["rows"], c["inputs"]), _empty(c["inputs"], c["outputs"])
        if c["dtype"] == "f16":
            s["grad16"] = _empty(c["rows"], c["outputs"], dtype=torch.float16)
    elif kind == "spmm":
        s["y"] = _empty(c["m"], c["n"])
    elif kind == "spmv":
        s["y"] = _empty(c["m"])
        s["plan"] = _Plan(c["m"], c["k"], s["ptr"], s["col"])
    return s


class _Plan:
    """The SpMV plan a program keeps beside its matrix, released with it."""

    def __init__(self, m, k, ptr, col):
        self.plan = G.SpmvPlan(m, k, col.numel(), ptr, col)

    def __del__(self):
        torch.cuda.synchronize()
        self.plan.release()


def run(state):
    s, c = state, state["c"]
    kind = c["kind"]
    if kind == "host_matmul":
        m, n, k = c["m"], c["n"], c["k"]
        a, b, y = G.Buffer(data=s["a"]), G.Buffer(data=s["b"]), G.Buffer(4 * m * n)
        G.call("perform_mps_matrix_multiplication", a.handle, m, k, b.handle, k, n, y.handle, m, n, None)
        out = y.to_array((m, n))
        for buf in (a, b, y):
            buf.release()
        return out
    if kind == "mlp":
        G.gemm(s["x"], s["w0"], s["h1"], bias=s["b0"], act=G.ACT_RELU)
        G.gemm(s["h1"], s["w1"], s["h2"], bias=s["b1"], act=G.ACT_RELU)
        G.gemm(s["h2"], s["w2"], s["logits"], bias=s["b2"])
        G.softmax_rows(s["logits"], s["y"])
        return {"logits": s["logits"], "y": s["y"]}
    if kind == "gemm":
        more = {}
        if c["batch"] > 1:
            more = {"batch": c["batch"], "strideA": c["m"] * c["k"], "strideB": c["k"] * c["n"], "strideC": c["m"] * c["n"]}
        G.gemm(s["a"], s["b"], s["y"], transA=c["layout"][0] == "t", transB=c["layout"][1] == "t", **more)
        return s["y"]
    if kind == "linear":
        G.gemm(s["x"], s["w"], s["y"], transB=c["layout"] == "nt", bias=s["b"], act=_ACT[c["act"]])
        return s["y"]
    if kind == "backward":
        G.activation_backward(s["g"], s["pre"], _ACT[c["act"]], s["grad"], s["db"])
        grad = s["grad"]
        if c["dtype"] == "f16":
            G.cast_f32_f16(grad, s["grad16"])
            grad = s["grad16"]
        G.gemm(grad, s["w"], s["dx"], transB=True)
        G.gemm(s["x"], grad, s["dw"], transA=True)
        return {"grad": s["grad"], "db": s["db"], "dx": s["dx"], "dw": s["dw"]}
    if kind == "spmm":
        G.spmm_csr(c["m"], c["n"], c["k"], s["col"].numel(), s["ptr"], s["col"], s["val"], s["d"], s["y"])
        return s["y"]
    s["plan"].plan.run(s["val"], s["d"], s["y"])
    return s["y"]


def work(case):
    c = case
    kind = c["kind"]
    if kind == "host_matmul":
        m, n, k = c["m"], c["n"], c["k"]
        return {"bytes": 4.0 * (m * k + k * n + m * n), "flops": 2.0 * m * n * k}
    if kind == "mlp":
        sizes = [c["inputs"], c["hidden1"], c["hidden2"], c["classes"]]
        w = float(sum(a * b for a, b in zip(sizes, sizes[1:])))
        return {"bytes": 4.0 * (w + sum(sizes[1:]) + c["rows"] * (c["inputs"] + 2 * c["classes"])), "flops": 2.0 * c["rows"] * w}
    if kind in ("gemm", "linear"):
        e = 2.0 if c["dtype"] == "f16" else 4.0
        m, n, k, b = (c["rows"], c["outputs"], c["inputs"], 1) if kind == "linear" else (c["m"], c["n"], c["k"], c["batch"])
        return {"bytes": b * (e * (m * k + k * n) + 4.0 * m * n), "flops": 2.0 * b * m * n * k}
    if kind == "backward":
        e = 2.0 if c["dtype"] == "f16" else 4.0
        r, i, o = c["rows"], c["inputs"], c["outputs"]
        return {"bytes": e * (r * i + i * o) + 4.0 * (3 * r * o + o + r * i + i * o), "flops": 4.0 * r * i * o}
    nnz, n = c["m"] * c["mean"], c.get("n", 1)
    return {"bytes": 4.0 * (c["m"] + 1) + 8.0 * nnz + 4.0 * n * (c["k"] + c["m"]), "flops": 2.0 * nnz * n}


def tolerance(case):
    # Sums in fp32, of fp32 values or of fp16 values whose products are exact in fp32: the path is
    # 1e-7 to 2.5e-6 off its value in 64 bits over these sizes (longer sums more), and so is any
    # other order of the sums.
    if case["kind"] in ("spmm", "spmv"):
        return {"rel": 1e-6}
    # The gradient is rounded to fp16 between the activation's backward and the products: one
    # unit in the last place of the activation's derivative can move that rounding.
    if case["kind"] == "backward" and case["dtype"] == "f16":
        return {"rel": 1e-4, "max": 1e-2}
    return {"rel": 1e-5}


# ------------------------------------------------------------------ the same in 64 bits
def _act64(x, act):
    if act == "relu":
        return x.clamp_min(0.0)
    if act == "gelu":
        return 0.5 * x * (1.0 + torch.tanh(0.7978845608028654 * (x + 0.044715 * x**3)))
    return x


def _grad64(x, act):
    if act == "relu":
        return (x > 0).double()
    k, a = 0.7978845608028654, 0.044715
    t = torch.tanh(k * (x + a * x**3))
    return 0.5 * (1.0 + t) + 0.5 * x * (1.0 - t * t) * k * (1.0 + 3.0 * a * x * x)


def exact(case, seed):
    _use_stream()
    c, s = case, _inputs(case, seed)
    kind = c["kind"]
    if kind == "host_matmul":
        return s["a"].astype(np.float64) @ s["b"].astype(np.float64)
    s = {k: v.double() if v.is_floating_point() else v for k, v in s.items()}
    if kind == "mlp":
        h = (s["x"] @ s["w0"] + s["b0"]).clamp_min(0.0)
        h = (h @ s["w1"] + s["b1"]).clamp_min(0.0)
        logits = h @ s["w2"] + s["b2"]
        return {"logits": logits, "y": torch.softmax(logits, 1)}
    if kind == "gemm":
        a = s["a"].transpose(-1, -2).contiguous() if c["layout"][0] == "t" else s["a"]
        b = s["b"].transpose(-1, -2).contiguous() if c["layout"][1] == "t" else s["b"]
        return a @ b
    if kind == "linear":
        w = s["w"].t().contiguous() if c["layout"] == "nt" else s["w"]
        return _act64(s["x"] @ w + s["b"], c["act"])
    if kind == "backward":
        grad = s["g"] * _grad64(s["pre"], c["act"])
        return {"grad": grad, "db": grad.sum(0), "dx": grad @ s["w"].t().contiguous(), "dw": s["x"].t().contiguous() @ grad}
    rows = torch.repeat_interleave(torch.arange(c["m"], device="cuda"), (s["ptr"][1:] - s["ptr"][:-1]).long())
    col = s["col"].long()
    d = s["d"] if kind == "spmm" else s["d"][:, None]
    y = torch.zeros((c["m"], d.shape[1]), dtype=torch.float64, device="cuda")
    for j in range(0, d.shape[1], 32):  # 32 columns at a time: the products of all entries with them take about 1 GB
        y[:, j : j + 32].index_add_(0, rows, d[:, j : j + 32][col] * s["val"][:, None])
    return y if kind == "spmm" else y[:, 0]
