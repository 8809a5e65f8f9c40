"""The performance cases of the framework: what its users run, through its
public entry points, on one GPU.

The families and what each stands for in real use:
  step_small   a whole fp32 train step of the reference's MLP classifier
               (Linear, ReLU, Linear, softmax cross-entropy, Adam), replayed
               from a captured graph; small batches, where launches count
  step_large   a whole bf16 train step of the L-layer GELU/MSE MLP with fp32
               master weights and AdamW, replayed from a captured graph
  linear       the forward of one Linear layer with its activation
  linear_bwd   the backward of one Linear layer: input gradient, weight
               gradient and bias gradient
  softmax      row softmax with the row maxima and sums
  xent         softmax cross-entropy of a classifier head, forward and backward
  layernorm    LayerNorm forward and backward (affine)
  batchnorm    BatchNorm (f16, NCHW, affine) training forward and backward
  adamw        one optimizer step over a flat parameter buffer
The single layers are eager calls of `_C.op_call`, as a program without a
plan makes them; their outputs are allocated once, as a program's would be.
"""
import math
import os
import struct
import sys

import torch

_PY = os.path.abspath(os.path.join("ai-compiler-framework_amd", "python"))
if _PY not in sys.path:
    sys.path.insert(0, _PY)

from aicf_cuda import _C  # noqa: E402
from aicf_hip import mlp  # noqa: E402

K = _C.OpKind
DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
EPILOGUE = {"none": 1, "relu": 0, "gelu": 3}  # with a bias


def _schema(tag):
    return int.from_bytes(tag, "little")


GEPI, ADAM, LNEP, BNEP = (_schema(t) for t in (b"GEPI", b"ADAM", b"LNEP", b"BNEP"))
HYPER = {"lr": 1e-3, "beta1": 0.9, "beta2": 0.999, "eps": 1e-8}


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # the reference's own configuration: the smallest whole step
        {"name": "step_small_64x784x256x10", "kind": "step_small", "batch": 64, "din": 784, "hidden": 256,
         "classes": 10},
        # the benchmark's configuration: the largest whole step
        {"name": "step_large_8192x4096x4", "kind": "step_large", "batch": 8192, "width": 4096, "layers": 4},
        # the wide up-projection of the GEMM+epilogue configuration
        {"name": "linear_bf16_8192x4096x11008_gelu", "kind": "linear", "dtype": "bf16", "rows": 8192,
         "fin": 4096, "fout": 11008, "act": "gelu"},
        # an f16 hidden layer over image rows (784 inputs) and a last batch that is not full
        {"name": "linear_f16_3000x784x1000_relu", "kind": "linear", "dtype": "f16", "rows": 3000, "fin": 784,
         "fout": 1000, "act": "relu"},
        # the backward of an ordinary bf16 layer
        {"name": "linear_bwd_bf16_4096x1024x4096", "kind": "linear_bwd", "dtype": "bf16", "rows": 4096,
         "fin": 1024, "fout": 4096},
        # the backward of an fp32 layer with odd sizes
        {"name": "linear_bwd_f32_777x1000x523", "kind": "linear_bwd", "dtype": "f32", "rows": 777, "fin": 1000,
         "fout": 523},
        # the widest common row softmax of the row-kernel configuration
        {"name": "softmax_16384x8192", "kind": "softmax", "rows": 16384, "cols": 8192},
        # a classifier head over an odd number of classes
        {"name": "xent_4096x10007", "kind": "xent", "rows": 4096, "cols": 10007},
        # LayerNorm of fp32 activations of the benchmark's width
        {"name": "layernorm_f32_8192x4096", "kind": "layernorm", "dtype": "f32", "rows": 8192, "cols": 4096},
        # LayerNorm of small f16 activations, a batch that is not full
        {"name": "layernorm_f16_1500x1000", "kind": "layernorm", "dtype": "f16", "rows": 1500, "cols": 1000},
        # BatchNorm of an early convolution's feature maps
        {"name": "batchnorm_32x64x56x56", "kind": "batchnorm", "batch": 32, "channels": 64, "height": 56,
         "width": 56},
        # the optimizer over all parameters of the 4 x 4096^2 MLP, with the bf16 shadow
        {"name": "adamw_67125248", "kind": "adamw", "params": 4 * (4096 * 4096 + 4096), "shadow": True},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    """A size of lo..hi, even over the logarithm: any, or a multiple of 8, of 64 or a power of two."""
    n = _log(rng, lo, hi)
    step = rng.choice((1, 8, 64, 0))
    if step:
        n = -(-n // step) * step
    else:
        n = 1 << max(0, round(math.log2(n)))
    return min(max(n, lo), hi)


def draw(rng):
    kind = rng.choice(("step_small", "step_large", "linear", "linear", "linear_bwd", "linear_bwd", "softmax", "xent",
                       "layernorm", "layernorm", "batchnorm", "batchnorm", "adamw"))
    if kind == "step_small":
        return {"kind": kind, "batch": _size(rng, 16, 256), "din": _size(rng, 32, 1024),
                "hidden": 8 * rng.randint(4, 64), "classes": rng.randint(2, 32)}
    if kind == "step_large":
        return {"kind": kind, "batch": _size(rng, 256, 8192), "width": 64 * rng.randint(4, 64),
                "layers": rng.randint(2, 4)}
    if kind in ("linear", "linear_bwd"):
        c = {"kind": kind, "dtype": rng.choice(("f32", "f16", "bf16", "bf16")), "rows": _size(rng, 16, 8192),
             "fin": _size(rng, 32, 8192), "fout": _size(rng, 10, 8192)}
        most = 2e11 if c["dtype"] != "f32" else 2e10  # multiply-adds
        while c["rows"] * c["fin"] * c["fout"] > most:
            c["rows"] = (c["rows"] + 1) // 2
        if kind == "linear":
            c["act"] = rng.choice(("none", "relu", "gelu"))
        return c
    if kind in ("softmax", "xent", "layernorm"):
        c = {"kind": kind, "rows": _size(rng, 16, 16384), "cols": _size(rng, 16, 32768)}
        if kind == "layernorm":
            c["dtype"] = rng.choice(("f32", "f16"))
            c["cols"] = _size(rng, 64, 8192)
        while c["rows"] * c["cols"] > 16384 * 8192:
            c["rows"] = (c["rows"] + 1) // 2
        return c
    if kind == "batchnorm":
        c = {"kind": kind, "batch": _size(rng, 2, 128), "channels": _size(rng, 3, 1024)}
        c["height"] = c["width"] = rng.choice((1, 4, 7, 8, 14, 16, 28, 32, 56, 64, 112))
        while c["batch"] * c["channels"] * c["height"] * c["width"] > 1 << 26:
            c["channels"] = (c["channels"] + 1) // 2
        return c
    return {"kind": "adamw", "params": _size(rng, 1000, 1 << 27), "shadow": rng.random() < 0.5}


# ------------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) + 1)
    return g


def _randn(g, shape, dtype=torch.float32, scale=1.0, shift=0.0):
    return torch.randn(shape, device="cuda", generator=g).mul_(scale).add_(shift).to(dtype)


def _kaiming(g, fout, fin, dtype):
    b = math.sqrt(6.0 / fin)
    return torch.empty((fout, fin), device="cuda").uniform_(-b, b, generator=g).to(dtype)


class _Step:
    """A captured train step: the executor with its graph, given back with the object."""

    def __init__(self, ex, names):
        self.ex, self.names = ex, names
        self.outputs = {n: ex.value(n) for n in names}

    def __del__(self):
        torch.cuda.synchronize()  # no replay is under way when its graph goes
        self.ex.close()


def _small_inputs(c, seed):
    g = _gen(seed)
    B, din, dh, dout = c["batch"], c["din"], c["hidden"], c["classes"]
    params = {"0.W": _kaiming(g, dh, din, torch.float32), "0.b": _randn(g, (dh,), scale=0.01),
              "2.W": _kaiming(g, dout, dh, torch.float32), "2.b": _randn(g, (dout,), scale=0.01)}
    x = _randn(g, (B, din))
    t = torch.randint(0, dout, (B,), device="cuda", generator=g, dtype=torch.int32)
    # optimizer state of a run that has been going for a while
    s = 1.0 / math.sqrt(B * dh)
    m = {n: _randn(g, p.shape, scale=s) for n, p in params.items()}
    v = {n: (torch.rand(p.shape, device="cuda", generator=g) + 0.5) * s * s for n, p in params.items()}
    return {"x": x, "t": t}, params, m, v


def _large_inputs(c, seed):
    g = _gen(seed)
    B, D, L = c["batch"], c["width"], c["layers"]
    lay = mlp.FlatLayout(D, L)
    P = torch.zeros(lay.total, device="cuda")
    b = math.sqrt(6.0 / D)
    P[:L * D * D].uniform_(-b, b, generator=g)
    P[L * D * D:].uniform_(-0.01, 0.01, generator=g)
    x = _randn(g, (B, D), torch.bfloat16)
    t = _randn(g, (B, D))
    s = 3.0 / (D * math.sqrt(B))  # about a gradient's own size
    m = _randn(g, (lay.total,), scale=s)
    v = (torch.rand(lay.total, device="cuda", generator=g) + 0.5) * (s * s)
    return {"x": x, "t": t}, {"flat.params": P}, m, v


STEP_AT = 100  # steps already taken


def _inputs(c, seed):
    """The tensors of a single layer's case."""
    g = _gen(seed)
    k = c["kind"]
    if k == "linear":
        dt = DTYPES[c["dtype"]]
        return {"x": _randn(g, (c["rows"], c["fin"]), dt), "W": _kaiming(g, c["fout"], c["fin"], dt),
                "b": _randn(g, (c["fout"],), dt, 0.1)}
    if k == "linear_bwd":
        dt = DTYPES[c["dtype"]]
        return {"x": _randn(g, (c["rows"], c["fin"]), dt), "W": _kaiming(g, c["fout"], c["fin"], dt),
                "dy": _randn(g, (c["rows"], c["fout"]), dt, 0.1, 0.02)}
    if k == "softmax":
        return {"x": _randn(g, (c["rows"], c["cols"]), scale=2.0, shift=0.1)}
    if k == "xent":
        return {"x": _randn(g, (c["rows"], c["cols"]), scale=2.0),
                "t": torch.randint(0, c["cols"], (c["rows"],), device="cuda", generator=g, dtype=torch.int32)}
    if k == "layernorm":
        dt, s = DTYPES[c["dtype"]], (c["rows"], c["cols"])
        return {"x": _randn(g, s, dt, 1.5, 0.3), "g": _randn(g, s[1:], dt, 0.2, 1.0), "b": _randn(g, s[1:], dt, 0.2),
                "dy": _randn(g, s, dt, 1.0, 0.1)}
    if k == "batchnorm":
        s, dt = (c["batch"], c["channels"], c["height"], c["width"]), torch.float16
        return {"x": _randn(g, s, dt, 1.5, 0.3), "g": _randn(g, s[1:2], dt, 0.2, 1.0),
                "b": _randn(g, s[1:2], dt, 0.2), "dy": _randn(g, s, dt, 1.0, 0.1)}
    n = (c["params"],)
    return {"P": _randn(g, n, scale=0.02), "G": _randn(g, n, scale=1e-3), "M": _randn(g, n, scale=3e-4),
            "V": (torch.rand(n, device="cuda", generator=g) + 0.5) * 1e-6,
            "step": torch.full((), STEP_AT, device="cuda", dtype=torch.int32)}


def prepare(case, seed):
    c = dict(case)
    k = c["kind"]
    if k == "step_small":
        inputs, params, m, v = _small_inputs(c, seed)
        ir, lowered, plan = mlp.build_mlp_xent(c["batch"], c["din"], c["hidden"], c["classes"], fuse_small=True,
                                               **HYPER)
        ex = mlp.make_executor(ir, lowered, plan, own_graph=True)
        ex.build_env(inputs=inputs, params=params, reuse_static=False)
        for n in params:
            ex.value(f"opt.m.{n}").copy_(m[n])
            ex.value(f"opt.v.{n}").copy_(v[n])
        ex.value("opt.step").fill_(STEP_AT)
        ex.capture(inputs=inputs, params=params, reuse_static=True)
        names = ["logits", "loss", "pred", "row_loss", "d_x"] + [p + n for n in params
                                                                 for p in ("", "opt.m.", "opt.v.")]
        return _Step(ex, names)
    if k == "step_large":
        inputs, params, m, v = _large_inputs(c, seed)
        ir, lowered, plan = mlp.build_mlp_mse(c["batch"], c["width"], c["layers"], fuse_optimizer=True,
                                              fuse_colsum=True, fuse_tail=True, **HYPER)
        ex = mlp.make_executor(ir, lowered, plan, own_graph=True)
        ex.build_env(inputs=inputs, params=params, reuse_static=False)
        ex.value("opt.m.flat").copy_(m)
        ex.value("opt.v.flat").copy_(v)
        ex.value("opt.step").fill_(STEP_AT)
        mlp.refresh_shadow(ex)
        ex.capture(inputs=inputs, params=params, reuse_static=True)
        return _Step(ex, ["y", "loss", "d_x", "flat.params", "opt.m.flat", "opt.v.flat", "wb.flat"])
    s = _inputs(c, seed)
    s["case"] = c
    f32 = torch.float32

    def out(shape, dtype=f32):
        return torch.empty(shape, device="cuda", dtype=dtype)

    if k == "linear":
        s["y"] = out((c["rows"], c["fout"]), s["x"].dtype)
        s["attrs"] = struct.pack("<iii", 0, 1, EPILOGUE[c["act"]])
    elif k == "linear_bwd":
        dt = s["x"].dtype
        s["dx"] = torch.empty_like(s["x"])
        s["dW"] = out(s["W"].shape, torch.float16 if dt == torch.float16 else f32)
        s["db"] = out((c["fout"],))
    elif k == "softmax":
        s["y"], s["rmax"], s["rsum"] = torch.empty_like(s["x"]), out((c["rows"],)), out((c["rows"],))
    elif k == "xent":
        s["loss"], s["dx"] = out(()), torch.empty_like(s["x"])
        s["pred"], s["row"] = out((c["rows"],), torch.int32), out((c["rows"],))
    elif k == "layernorm":
        s["y"], s["dx"] = torch.empty_like(s["x"]), torch.empty_like(s["x"])
        s["mean"], s["rstd"] = out((c["rows"],)), out((c["rows"],))
        s["dg"], s["db"] = out((c["cols"],)), out((c["cols"],))
    elif k == "batchnorm":
        s["y"], s["dx"] = torch.empty_like(s["x"]), torch.empty_like(s["x"])
        for n in ("mean", "rstd", "dg", "db"):
            s[n] = out((c["channels"],))
    elif c["shadow"]:
        s["Wb"] = s["P"].to(torch.bfloat16)
    return s


# ----------------------------------------------------------------- one pass
def run(s):
    if isinstance(s, _Step):
        s.ex.replay(1)
        return s.outputs
    c = s["case"]
    k = c["kind"]
    if k == "linear":
        _C.op_call(K.GemmEpilogue, [s["x"], s["W"], s["b"]], [s["y"]], GEPI, s["attrs"])
        return {"y": s["y"]}
    if k == "linear_bwd":
        _C.op_call(K.Gemm, [s["dy"], s["W"]], [s["dx"]], 0, struct.pack("<ii", 0, 0))
        _C.op_call(K.Gemm, [s["dy"], s["x"]], [s["dW"]], 0, struct.pack("<ii", 1, 0))
        _C.op_call(K.ReduceSum, [s["dy"]], [s["db"]])
        return {n: s[n] for n in ("dx", "dW", "db")}
    if k == "softmax":
        _C.op_call(K.RowSoftmax, [s["x"]], [s["y"], s["rmax"], s["rsum"]])
        return {n: s[n] for n in ("y", "rmax", "rsum")}
    if k == "xent":
        _C.op_call(K.SoftmaxXent, [s["x"], s["t"]], [s["loss"], s["dx"], s["pred"], s["row"]])
        return {n: s[n] for n in ("loss", "dx", "pred", "row")}
    if k == "layernorm":
        _C.op_call(K.LayerNormFwd, [s["x"], s["g"], s["b"]], [s["y"], s["mean"], s["rstd"]], LNEP,
                   struct.pack("<f", 1e-5))
        _C.op_call(K.LayerNormBwd, [s["x"], s["dy"], s["g"], s["mean"], s["rstd"]], [s["dx"], s["dg"], s["db"]])
        return {n: s[n] for n in ("y", "mean", "rstd", "dx", "dg", "db")}
    if k == "batchnorm":
        _C.op_call(K.BatchNormFwd, [s["x"], s["g"], s["b"]], [s["y"], s["mean"], s["rstd"]], BNEP,
                   struct.pack("<fI", 1e-5, 0))
        _C.op_call(K.BatchNormBwd, [s["x"], s["dy"], s["g"], s["mean"], s["rstd"]], [s["dx"], s["dg"], s["db"]])
        return {n: s[n] for n in ("y", "mean", "rstd", "dx", "dg", "db")}
    outs = [s["P"], s["M"], s["V"]] + ([s["Wb"]] if c["shadow"] else [])
    _C.op_call(K.StepInc, [s["step"]], [s["step"]])
    _C.op_call(K.AdamStep, [s["P"], s["G"], s["M"], s["V"], s["step"]], outs, ADAM,
               struct.pack("<fffff", HYPER["lr"], HYPER["beta1"], HYPER["beta2"], HYPER["eps"], 0.01))
    return {n: s[n] for n in ("P", "M", "V", "Wb") if n in s}


# ------------------------------------------------------- what a pass has to do
def work(case):
    c = dict(case)
    k = c["kind"]
    if k == "step_small":
        B, a, h, o = c["batch"], c["din"], c["hidden"], c["classes"]
        n = a * h + h + h * o + o
        return {"bytes": 4.0 * (2 * B * a + 2 * B * o + 3 * B) + 24.0 * n,
                "flops": 6.0 * B * (a * h + h * o) + 12.0 * n}
    if k == "step_large":
        B, D, L = c["batch"], c["width"], c["layers"]
        n = L * (D * D + D)
        # inputs, target, y and d_x once; parameters and moments read and written, the shadow read and written
        return {"bytes": B * D * (2 + 4 + 2 + 2) + 28.0 * n, "flops": 6.0 * B * D * D * L + 12.0 * n}
    if k in ("linear", "linear_bwd"):
        R, a, o = c["rows"], c["fin"], c["fout"]
        e = 4.0 if c["dtype"] == "f32" else 2.0
        if k == "linear":
            return {"bytes": e * (R * a + o * a + o + R * o), "flops": 2.0 * R * a * o}
        w = 2.0 if c["dtype"] == "f16" else 4.0
        return {"bytes": e * (2 * R * a + o * a + R * o) + w * o * a + 4.0 * o, "flops": 4.0 * R * a * o + R * o}
    if k in ("softmax", "xent"):
        R, C = c["rows"], c["cols"]
        return {"bytes": 8.0 * R * C + (8.0 if k == "softmax" else 12.0) * R, "flops": 5.0 * R * C}
    if k == "layernorm":
        R, C = c["rows"], c["cols"]
        e = 4.0 if c["dtype"] == "f32" else 2.0
        return {"bytes": 4 * e * R * C + 8.0 * R + (2 * e + 8) * C, "flops": 17.0 * R * C}
    if k == "batchnorm":
        C = c["channels"]
        n = c["batch"] * C * c["height"] * c["width"]
        return {"bytes": 8.0 * n + 20.0 * C, "flops": 17.0 * n}
    return {"bytes": (30.0 if c["shadow"] else 28.0) * c["params"], "flops": 12.0 * c["params"]}


def tolerance(case):
    """About four times the error of this path against 64 bits."""
    k = case["kind"]
    if k == "step_small":
        return {"rel": 1e-5, "differ": 0.001}
    if k == "step_large":  # every stored activation is rounded to bf16; the input gradient has passed through them all
        return {"rel": 1.6e-2}
    if k in ("linear", "linear_bwd"):
        return {"rel": {"f32": 5e-6, "f16": 1e-3, "bf16": 8e-3}[case["dtype"]]}
    if k == "xent":
        return {"rel": 2e-6, "differ": 0.001}
    if k == "softmax":
        return {"rel": 2e-6}
    if k == "layernorm":
        return {"rel": 5e-6 if case["dtype"] == "f32" else 1e-3}
    if k == "batchnorm":
        return {"rel": 1e-3}
    return {"rel": 8e-3 if case["shadow"] else 2e-6}  # the shadow is a bf16 rounding


# ------------------------------------------------------------- in 64 bits
def _adam64(P, g, m, v, lr=HYPER["lr"], wd=0.0):
    b1, b2, t = HYPER["beta1"], HYPER["beta2"], STEP_AT + 1
    m = b1 * m + (1 - b1) * g
    v = b2 * v + (1 - b2) * g * g
    P = P * (1 - lr * wd) - lr / (1 - b1 ** t) * m / ((v / (1 - b2 ** t)).sqrt() + HYPER["eps"])
    return P, m, v


def _gelu64(x):
    return torch.nn.functional.gelu(x, approximate="tanh")


def _dgelu64(x):
    k0, k1 = math.sqrt(2 / math.pi), 0.044715
    t = torch.tanh(k0 * (x + k1 * x ** 3))
    return 0.5 * (1 + t) + 0.5 * x * (1 - t * t) * k0 * (1 + 3 * k1 * x * x)


def exact(case, seed):
    c = dict(case)
    k = c["kind"]
    if k == "step_small":
        inputs, params, m, v = _small_inputs(c, seed)
        x, t, B = inputs["x"].double(), inputs["t"].long(), c["batch"]
        p = {n: q.double() for n, q in params.items()}
        h = torch.relu(x @ p["0.W"].T + p["0.b"])
        z = h @ p["2.W"].T + p["2.b"]
        row = torch.logsumexp(z, 1) - z.gather(1, t[:, None])[:, 0]
        dz = torch.softmax(z, 1)
        dz[torch.arange(B, device="cuda"), t] -= 1.0
        dz /= B
        dh = (dz @ p["2.W"]) * (h > 0)
        grads = {"0.W": dh.T @ x, "0.b": dh.sum(0), "2.W": dz.T @ h, "2.b": dz.sum(0)}
        r = {"logits": z, "loss": row.mean(), "pred": None, "row_loss": row, "d_x": dh @ p["0.W"]}
        for n in params:
            r[n], r["opt.m." + n], r["opt.v." + n] = _adam64(p[n], grads[n], m[n].double(), v[n].double())
        return r
    if k == "step_large":
        inputs, params, m, v = _large_inputs(c, seed)
        B, D, L = c["batch"], c["width"], c["layers"]
        P = params.pop("flat.params").double()
        W = [P[i * D * D:(i + 1) * D * D].view(D, D) for i in range(L)]
        Wb = [w.float().bfloat16().double() for w in W]  # the products read the bf16 shadow
        b = [P[L * D * D + i * D:L * D * D + (i + 1) * D] for i in range(L)]
        h, z = [inputs["x"].double()], []
        for i in range(L):
            z.append(h[i] @ Wb[i].T + b[i])
            if i < L - 1:
                h.append(_gelu64(z[i]))
        d = z[-1] - inputs["t"].double()
        r = {"y": z[-1], "loss": (d * d).mean(), "wb.flat": None}
        d *= 2.0 / (B * D)
        g = torch.empty_like(P)
        for i in range(L - 1, -1, -1):
            g[i * D * D:(i + 1) * D * D] = (d.T @ h[i]).view(-1)
            g[L * D * D + i * D:L * D * D + (i + 1) * D] = d.sum(0)
            d = d @ Wb[i]
            if i:
                d *= _dgelu64(z[i - 1])
        r["d_x"] = d
        r["flat.params"], r["opt.m.flat"], r["opt.v.flat"] = _adam64(P, g, m.double(), v.double())
        return r
    s = _inputs(c, seed)
    d = {n: t.double() for n, t in s.items() if t.is_floating_point()}
    if k == "linear":
        y = d["x"] @ d["W"].T + d["b"]
        return {"y": torch.relu(y) if c["act"] == "relu" else _gelu64(y) if c["act"] == "gelu" else y}
    if k == "linear_bwd":
        return {"dx": d["dy"] @ d["W"], "dW": d["dy"].T @ d["x"], "db": d["dy"].sum(0)}
    if k == "softmax":
        return {"y": torch.softmax(d["x"], 1), "rmax": d["x"].amax(1), "rsum": d["x"].sum(1)}
    if k == "xent":
        x, t = d["x"], s["t"].long()
        row = torch.logsumexp(x, 1) - x.gather(1, t[:, None])[:, 0]
        p = torch.softmax(x, 1)
        p[torch.arange(c["rows"], device="cuda"), t] -= 1.0
        return {"loss": row.mean(), "dx": p / c["rows"], "pred": None, "row": row}
    if k in ("layernorm", "batchnorm"):
        x, dy = d["x"], d["dy"]
        over, shape = ((1,), (1, -1)) if k == "layernorm" else ((0, 2, 3), (1, -1, 1, 1))
        others = (0,) if k == "layernorm" else (0, 2, 3)
        n = c["cols"] if k == "layernorm" else x.numel() // c["channels"]
        mu = x.mean(over, keepdim=True)
        rs = 1.0 / ((x - mu).square().mean(over, keepdim=True) + 1e-5).sqrt()
        xh = (x - mu) * rs
        g, b = d["g"].view(shape), d["b"].view(shape)
        q = dy * g
        dx = (q - q.sum(over, keepdim=True) / n - xh * (q * xh).sum(over, keepdim=True) / n) * rs
        return {"y": xh * g + b, "mean": mu.reshape(-1), "rstd": rs.reshape(-1), "dx": dx,
                "dg": (dy * xh).sum(others), "db": dy.sum(others)}
    r = dict(zip("PMV", _adam64(d["P"], d["G"], d["M"], d["V"], wd=0.01)))
    if c["shadow"]:
        r["Wb"] = r["P"]
    return r
