"""The work that users of this framework have it do, as timed cases.

Each case is one call (or one training step) through the public Python entry
points, with resident device inputs as a program keeps them between calls.
``listed()`` gives the named cases, ``draw(rng)`` further ones of the same
ranges (odd and ragged sizes among them), ``prepare`` / ``run`` make and take
one pass, ``exact`` computes what the pass returns in 64 bits with torch alone.

The ranges, by kind:

linear      Float32 Linear with a fused activation: rows 1..4096, widths
            16..4096; forward alone, or the training step (forward, then dW,
            db and dx)
tensordot   Float32 batched product with broadcast batch dimensions: 1..64
            matrices of 16..1024
matmul_f64  Float64 matmul and its backward rule (gradients of both
            operands): sizes 16..2048
conv2d      Float32 NCHW Conv2d with bias and ReLU: 1..32 images of 3..128
            channels, 1 x 1 to 5 x 5 kernels, stride 1 or 2
gemm_bf16   bf16 A W^T with bias and activation: 16..4096 each way (K in
            steps of 8)
w8_linear   int8-weight Linear on bf16 rows: 1..2048 rows (decode to
            prefill), widths up to 11008 (K in steps of 16)
w8_mlp      SiLU-gated FFN on int8 weights: 1..512 rows, hidden up to 4096,
            intermediate up to 11008
quant_linear per-tensor W8A8 QuantLinear (the post-training-quantized Linear):
            rows 1..4096, widths 16..4096, any K
"""
import math

import torch

import momijo_amd as mj

ACTIVATIONS = {"none": mj.EPI_NONE, "relu": mj.EPI_RELU, "gelu": mj.EPI_GELU_TANH,
               "silu": mj.EPI_SILU}


def listed():
    return [
        # the smallest call: one hidden layer of a small fp32 MLP
        dict(name="linear_small", kind="linear", rows=256, k=256, n=256, act="relu", train=False),
        # a training step of a wide fp32 layer
        dict(name="linear_train", kind="linear", rows=4096, k=4096, n=4096, act="relu", train=True),
        # attention-like batched products, ragged, one operand broadcast
        dict(name="tensordot_batched", kind="tensordot", outer=4, inner=8, m=300, n=517, k=257),
        # double-precision matmul node of the autograd tape, forward and backward
        dict(name="matmul_f64", kind="matmul_f64", m=2048, n=2048, k=2048),
        # a 3 x 3 layer of a residual network's first stage
        dict(name="conv2d_3x3", kind="conv2d", images=32, c=64, size=56, oc=64, kernel=3, stride=1,
             pad=1),
        # the large dense bf16 product
        dict(name="gemm_bf16_4096", kind="gemm_bf16", m=4096, n=4096, k=4096, act="none",
             bias=False),
        # a ragged projection with its epilogue, as a sequence of 1000 tokens gives it
        dict(name="gemm_bf16_ragged", kind="gemm_bf16", m=1000, n=3000, k=1040, act="gelu",
             bias=True),
        # decode, one token: the up projection of an LLM's FFN
        dict(name="w8_decode", kind="w8_linear", rows=1, n=11008, k=4096, act="none", bias=True),
        # prefill of 2048 tokens through one int8-weight projection
        dict(name="w8_prefill", kind="w8_linear", rows=2048, n=4096, k=4096, act="gelu",
             bias=True),
        # batched decode of a whole FFN
        dict(name="w8_mlp_decode", kind="w8_mlp", rows=16, k=4096, i=11008, h=4096),
        # prefill of 512 tokens through a whole FFN
        dict(name="w8_mlp_prefill", kind="w8_mlp", rows=512, k=4096, i=11008, h=4096),
        # a post-training-quantized fp32 layer
        dict(name="quant_linear", kind="quant_linear", rows=4096, k=4096, n=4096),
    ]


# the largest listed product of each kind, in multiply-adds of one matrix
# product: no drawn case is larger
_MOST = {"linear": 4096 ** 3, "tensordot": 32 * 300 * 517 * 257, "matmul_f64": 2048 ** 3,
         "conv2d": 32 * 64 * 64 * 9 * 56 * 56, "gemm_bf16": 4096 ** 3,
         "w8_linear": 2048 * 4096 * 4096, "w8_mlp": 512 * 4096 * 11008,
         "quant_linear": 4096 ** 3}


def draw(rng):
    def size(lo, hi, step=1):
        """Log-uniform in [lo, hi], a multiple of `step`; half of the draws
        are multiples of 64 as well, as most layer widths are."""
        v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
        if v >= 64 and rng.random() < 0.5:
            step = 64
        return max(lo, min(hi, int(round(v / step)) * step)) // step * step or step

    while True:
        kind = rng.choice(sorted(_MOST))
        act = rng.choice(sorted(ACTIVATIONS))
        if kind == "linear":
            c = dict(kind=kind, rows=size(1, 4096), k=size(16, 4096), n=size(16, 4096), act=act,
                     train=rng.random() < 0.5)
            macs = c["rows"] * c["k"] * c["n"]
        elif kind == "tensordot":
            c = dict(kind=kind, outer=rng.choice([1, 2, 3, 4]), inner=rng.choice([1, 4, 8, 16]),
                     m=size(16, 1024), n=size(16, 1024), k=size(16, 1024))
            macs = c["outer"] * c["inner"] * c["m"] * c["n"] * c["k"]
        elif kind == "matmul_f64":
            c = dict(kind=kind, m=size(16, 2048), n=size(16, 2048), k=size(16, 2048))
            macs = c["m"] * c["n"] * c["k"]
        elif kind == "conv2d":
            kernel = rng.choice([1, 3, 3, 5])
            c = dict(kind=kind, images=rng.choice([1, 2, 4, 8, 16, 32]),
                     c=rng.choice([3, 16, 32, 64, 96, 128]), size=rng.randint(7, 112),
                     oc=rng.choice([16, 32, 64, 96, 128]), kernel=kernel,
                     stride=rng.choice([1, 1, 2]), pad=kernel // 2)
            o = _conv_out(c)
            macs = c["images"] * c["oc"] * c["c"] * kernel * kernel * o * o
        elif kind == "gemm_bf16":
            c = dict(kind=kind, m=size(16, 4096), n=size(16, 4096), k=size(16, 4096, 8), act=act,
                     bias=rng.random() < 0.5)
            macs = c["m"] * c["n"] * c["k"]
        elif kind == "w8_linear":
            c = dict(kind=kind, rows=size(1, 2048), n=size(256, 11008), k=size(256, 11008, 16),
                     act=act, bias=rng.random() < 0.5)
            macs = c["rows"] * c["n"] * c["k"]
        elif kind == "w8_mlp":
            c = dict(kind=kind, rows=size(1, 512), k=size(256, 4096, 16),
                     i=size(256, 11008, 16), h=size(256, 4096, 16))
            macs = c["rows"] * c["i"] * max(c["k"], c["h"])
        else:
            c = dict(kind=kind, rows=size(1, 4096), k=size(16, 4096), n=size(16, 4096))
            macs = c["rows"] * c["k"] * c["n"]
        if macs <= _MOST[kind]:
            return c


def _conv_out(c):
    return (c["size"] + 2 * c["pad"] - c["kernel"]) // c["stride"] + 1


class _Gen:
    """Seeded device tensors: the same seed gives the same sequence."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(1000003 * int(seed) + 17)

    def normal(self, shape, std=1.0, dtype=torch.float32):
        t = torch.randn(shape, generator=self.g, device="cuda",
                        dtype=torch.float64 if dtype == torch.float64 else torch.float32)
        return (t * std).to(dtype) if std != 1.0 else t.to(dtype)

    def bias(self, n):
        return (torch.rand(n, generator=self.g, device="cuda") - 0.5) / 8


def _inputs(case, seed):
    """The plain tensors of a case, in the order that they are drawn."""
    g, kind = _Gen(seed), case["kind"]
    if kind == "linear":
        rows, k, n = case["rows"], case["k"], case["n"]
        t = dict(x=g.normal((rows, k)), w=g.normal((n, k), k ** -0.5), b=g.bias(n))
        if case["train"]:
            t["dy"] = g.normal((rows, n))
        return t
    if kind == "tensordot":
        return dict(a=g.normal((case["outer"], case["inner"], case["m"], case["k"])),
                    b=g.normal((case["inner"], case["k"], case["n"])))
    if kind == "matmul_f64":
        m, n, k = case["m"], case["n"], case["k"]
        return dict(a=g.normal((m, k), dtype=torch.float64), b=g.normal((k, n), dtype=torch.float64),
                    g=g.normal((m, n), dtype=torch.float64))
    if kind == "conv2d":
        c, oc, kk = case["c"], case["oc"], case["kernel"]
        return dict(x=g.normal((case["images"], c, case["size"], case["size"])),
                    w=g.normal((oc, c, kk, kk), (2.0 / (c * kk * kk)) ** 0.5), b=g.bias(oc))
    if kind == "gemm_bf16":
        m, n, k = case["m"], case["n"], case["k"]
        return dict(a=g.normal((m, k), dtype=torch.bfloat16),
                    w=g.normal((n, k), k ** -0.5, dtype=torch.bfloat16),
                    b=g.bias(n) if case["bias"] else None)
    if kind == "w8_linear":
        rows, n, k = case["rows"], case["n"], case["k"]
        return dict(x=g.normal((rows, k), dtype=torch.bfloat16), w=g.normal((n, k), 0.02),
                    b=g.bias(n) if case["bias"] else None)
    if kind == "w8_mlp":
        k, i, h = case["k"], case["i"], case["h"]
        return dict(x=g.normal((case["rows"], k), dtype=torch.bfloat16), wg=g.normal((i, k), 0.02),
                    wu=g.normal((i, k), 0.02), wd=g.normal((h, i), 0.02))
    rows, k, n = case["rows"], case["k"], case["n"]
    return dict(x=g.normal((rows, k)), w=g.normal((n, k), k ** -0.5), b=g.bias(n))


def prepare(case, seed):
    t, kind = _inputs(case, seed), case["kind"]
    if kind == "linear":
        layer = mj.Linear(case["k"], case["n"])
        layer.weight, layer.bias_t = mj.Tensor(t["w"]), mj.Tensor(t["b"])
        return dict(case=case, layer=layer, x=mj.Tensor(t["x"]),
                    dy=mj.Tensor(t["dy"]) if case["train"] else None)
    if kind == "tensordot":
        return dict(case=case, a=mj.Tensor(t["a"]), b=mj.Tensor(t["b"]))
    if kind == "matmul_f64":
        return dict(case=case, **{name: mj.Tensor(v) for name, v in t.items()})
    if kind == "conv2d":
        kk, s, p = case["kernel"], case["stride"], case["pad"]
        layer = mj.Conv2d(case["c"], case["oc"], (kk, kk), (s, s), (p, p))
        layer.weight, layer.bias_t = mj.Tensor(t["w"]), mj.Tensor(t["b"])
        return dict(case=case, layer=layer, x=mj.Tensor(t["x"]))
    if kind == "gemm_bf16":
        return dict(case=case, **t)
    if kind == "w8_linear":
        layer = mj.W8Linear.from_float(t["w"], t["b"], ACTIVATIONS[case["act"]])
        return dict(case=case, layer=layer, x=t["x"])
    if kind == "w8_mlp":
        ffn = mj.W8MLP(*(mj.W8Linear.from_float(t[name]) for name in ("wg", "wu", "wd")))
        return dict(case=case, layer=ffn, x=t["x"])
    s_w, s_x = _tensor_scale(t["w"]), _tensor_scale(t["x"])
    wq = mj.quantize_symmetric_int8(mj.Tensor(t["w"]), s_w)
    layer = mj.QuantLinear(case["k"], case["n"], wq, mj.Tensor(t["b"]), s_w, s_x)
    return dict(case=case, layer=layer, x=mj.Tensor(t["x"]))


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "linear":
        y = state["layer"].forward_act(state["x"], ACTIVATIONS[case["act"]])
        if not case["train"]:
            return y.torch
        dw, db, dx = state["layer"].backward(state["x"], state["dy"])
        return dict(y=y.torch, dw=dw.torch, db=db.torch, dx=dx.torch)
    if kind == "tensordot":
        return mj.tensordot(state["a"], state["b"]).torch
    if kind == "matmul_f64":
        y = mj.matmul(state["a"], state["b"])
        ga, gb = mj.matmul_backward(state["a"], state["b"], state["g"])
        return dict(y=y.torch, ga=ga.torch, gb=gb.torch)
    if kind == "conv2d":
        return state["layer"].forward_act(state["x"], mj.EPI_RELU).torch
    if kind == "gemm_bf16":
        return mj.gemm_bf16_nt(state["a"], state["w"], state["b"], ACTIVATIONS[case["act"]])
    if kind == "w8_linear":
        return state["layer"].forward(state["x"])
    if kind == "w8_mlp":
        y, h = state["layer"].forward(state["x"])
        return dict(y=y, h=h)
    return state["layer"].forward(state["x"]).torch


def work(case):
    kind = case["kind"]
    if kind == "linear":
        rows, k, n = case["rows"], case["k"], case["n"]
        nbytes, flops = 4 * (rows * k + n * k + n + rows * n), 2 * rows * k * n
        if case["train"]:  # dy read; dW, db and dx written
            nbytes += 4 * (rows * n + n * k + n + rows * k)
            flops *= 3
        return dict(bytes=nbytes, flops=flops)
    if kind == "tensordot":
        o, i, m, n, k = (case[name] for name in ("outer", "inner", "m", "n", "k"))
        return dict(bytes=4 * (o * i * m * k + i * k * n + o * i * m * n),
                    flops=2 * o * i * m * n * k)
    if kind == "matmul_f64":  # a, b, g read; y, ga, gb written
        m, n, k = case["m"], case["n"], case["k"]
        return dict(bytes=8 * 2 * (m * k + k * n + m * n), flops=3 * 2 * m * n * k)
    if kind == "conv2d":
        o, kk = _conv_out(case), case["kernel"]
        out = case["images"] * case["oc"] * o * o
        taps = case["c"] * kk * kk
        image = case["images"] * case["c"] * case["size"] ** 2
        return dict(bytes=4 * (image + case["oc"] * (taps + 1) + out), flops=2 * out * taps)
    if kind == "gemm_bf16":
        m, n, k = case["m"], case["n"], case["k"]
        return dict(bytes=2 * (m * k + n * k + m * n) + (4 * n if case["bias"] else 0),
                    flops=2 * m * n * k)
    if kind == "w8_linear":
        rows, n, k = case["rows"], case["n"], case["k"]
        return dict(bytes=n * k + 4 * n + 2 * rows * (k + n) + (4 * n if case["bias"] else 0),
                    flops=2 * rows * n * k)
    if kind == "w8_mlp":
        rows, k, i, h = case["rows"], case["k"], case["i"], case["h"]
        return dict(bytes=2 * i * k + h * i + 4 * (2 * i + h) + 2 * rows * (k + i + h),
                    flops=2 * rows * i * (2 * k + h))
    rows, k, n = case["rows"], case["k"], case["n"]
    return dict(bytes=4 * rows * k + n * k + 4 * n + 4 * rows * n, flops=2 * rows * k * n)


def tolerance(case):
    kind = case["kind"]
    if kind in ("linear", "tensordot", "conv2d"):
        return {"rel": 5e-6}
    if kind == "matmul_f64":
        return {"rel": 5e-15}
    if kind in ("gemm_bf16", "w8_linear"):
        return {"rel": 4e-3}
    if kind == "w8_mlp":  # h is rounded to bf16 before the down projection
        return {"rel": 5e-3}
    return {"rel": 2e-7}  # exact integer sums, two fp32 roundings


def _act(v, act):
    if act == "relu":
        return torch.clamp(v, min=0)
    if act == "gelu":
        return 0.5 * v * (1 + torch.tanh(math.sqrt(2 / math.pi) * (v + 0.044715 * v ** 3)))
    if act == "silu":
        return v * torch.sigmoid(v)
    return v


def _tensor_scale(t):
    """Per-tensor symmetric scale: max|t| / 127 in Float32."""
    return float((t.abs().max() / 127.0).item())


def _w8(w):
    """Per-row symmetric int8 (scale max|row| / 127 in Float32, round half to
    even): the dequantized weight in 64 bits."""
    s = w.abs().amax(1) / 127.0
    s = torch.where(s == 0, torch.ones_like(s), s).double()[:, None]
    return torch.clamp(torch.round(w.double() / s), -127, 127) * s


def exact(case, seed):
    t, kind = _inputs(case, seed), case["kind"]
    d = {name: None if v is None else v.double() for name, v in t.items()}
    if kind == "linear":
        y = _act(d["x"] @ d["w"].T + d["b"], case["act"])
        if not case["train"]:
            return y
        return dict(y=y, dw=d["dy"].T @ d["x"], db=d["dy"].sum(0), dx=d["dy"] @ d["w"])
    if kind == "tensordot":
        return torch.stack([torch.stack([d["a"][o, i] @ d["b"][i] for i in range(case["inner"])])
                            for o in range(case["outer"])])
    if kind == "matmul_f64":
        return dict(y=d["a"] @ d["b"], ga=d["g"] @ d["b"].T, gb=d["a"].T @ d["g"])
    if kind == "conv2d":
        o, w = _conv_out(case), d["w"].reshape(case["oc"], -1)
        out = []
        for x in d["x"]:
            cols = torch.nn.functional.unfold(x[None], case["kernel"], padding=case["pad"],
                                              stride=case["stride"])[0]
            out.append(torch.clamp(w @ cols + d["b"][:, None], min=0).reshape(-1, o, o))
        return torch.stack(out)
    if kind == "gemm_bf16":
        v = d["a"] @ d["w"].T
        return _act(v if d["b"] is None else v + d["b"], case["act"])
    if kind == "w8_linear":
        v = d["x"] @ _w8(t["w"]).T
        return _act(v if d["b"] is None else v + d["b"], case["act"])
    if kind == "w8_mlp":
        h = _act(d["x"] @ _w8(t["wg"]).T, "silu") * (d["x"] @ _w8(t["wu"]).T)
        return dict(y=h @ _w8(t["wd"]).T, h=h)
    # x and w quantized as the layer defines it (Float32 quotient, half away
    # from zero), the product and the dequantize in 64 bits
    s_w, s_x = _tensor_scale(t["w"]), _tensor_scale(t["x"])
    q = []
    for v, s in ((t["x"], s_x), (t["w"], s_w)):
        v = v / torch.tensor(s, dtype=torch.float32, device=v.device)
        v = torch.trunc(v + torch.where(v >= 0, 0.5, -0.5).to(torch.float32))
        q.append(torch.clamp(v, -128, 127).double())
    return (q[0] @ q[1].T) * (s_x * s_w) + d["b"]
