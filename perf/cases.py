"""Performance cases of the ConvRot INT8 linear: the work a program gives this
library through its public entry points, over the sizes it meets in use.

``listed()`` are fixed cases, ``draw()`` gives more of the same ranges;
``prepare()`` makes what the program holds before the call (activations,
prepared weights), ``run()`` is one pass.  ``exact()`` restates each path in
float64 torch from the definitions, without the library.

Inputs follow the benchmark's: activations N(0, 1) with 1% of the channels x30
(the outlier channels of a transformer's residual stream), weights N(0, 0.02),
biases N(0, 0.01), gradients N(0, 1).
"""

import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "oko-xpu-kernels_amd"))

from xpu_kernels import int8, rope  # noqa: E402

DEV = "cuda"
#: the activations of the fused FFN: [hidden | gate] pairs or a single tensor
PAIRED = ("situ", "geglu_erf")


# ------------------------------------------------------------------- the cases
def listed():
    return [
        # a projection for 16 tokens decoded together: two short launches, the
        # 16 MB weight read once
        dict(name="linear_decode", kind="linear", m=16, k=4096, n=4096, bias=True,
             residual=False, dtype="bf16"),
        # an attention projection at 1024 tokens (a 32 x 32 latent), the unit
        # tests' reference shape
        dict(name="linear_1024", kind="linear", m=1024, k=1280, n=1280, bias=True,
             residual=False, dtype="bf16"),
        # the FFN up-projection alone at 4096 tokens, the benchmark's headline shape
        dict(name="linear_up", kind="linear", m=4096, k=1280, n=10240, bias=True,
             residual=False, dtype="bf16"),
        # an attention output projection added to the residual stream with a
        # per-channel gate, a ragged token count
        dict(name="linear_residual", kind="linear", m=3974, k=3072, n=3072, bias=True,
             residual=True, dtype="bf16"),
        # one token through a fused GEGLU FFN: launches and latency
        dict(name="ffn_token", kind="ffn", m=1, k=1280, inner=5120, act="geglu_erf"),
        # the benchmark's fused GEGLU FFN at 4096 tokens
        dict(name="ffn_4096", kind="ffn", m=4096, k=1280, inner=5120, act="geglu_erf"),
        # a wider model's FFN with its own activation, a ragged token count
        dict(name="ffn_situ", kind="ffn", m=3952, k=3072, inner=8192, act="situ"),
        # the front of an attention block: the qkv accumulator, RMSNorm + rope of
        # q and k read from it, v dequantized from it
        dict(name="qkv_rope", kind="qkv", s=4096, h=24, d=128, k=3072),
        # fine-tuning around frozen int8 weights: forward, dx through the int8
        # weight, the bias gradient
        dict(name="train_int8", kind="train", m=4096, k=1280, n=5120, mode="int8"),
        # the same with the default backward (dx through the dequantized
        # weight), on the down-projection
        dict(name="train_dense", kind="train", m=4096, k=5120, n=1280, mode="dense"),
        # quantization-aware training: the weight quantized in every forward,
        # straight-through dx, dW and db
        dict(name="train_ste", kind="ste", m=4096, k=1280, n=5120),
        # loading a model: one weight rotated, quantized and laid out
        dict(name="prepare_weight", kind="prepare", n=10240, k=1280),
    ]


def _log_int(rng, lo, hi, step=1):
    """A multiple of ``step`` in [lo, hi], uniform in its logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


_MOST_FLOPS = 2.0 * 3952 * 3072 * (2 * 8192 + 8192)      # the largest listed case


def draw(rng):
    while True:
        c = _draw(rng)
        if work(c)["flops"] <= _MOST_FLOPS:
            return c


def _draw(rng):
    kind = rng.choice(("linear", "linear", "linear", "ffn", "ffn", "qkv", "train", "train", "ste",
                       "prepare"))
    if kind == "linear":
        # decode batches to a 64 x 64 latent's tokens; fp32 activations are
        # what an fp32 model passes
        return dict(kind=kind, m=_log_int(rng, 1, 4096), k=_log_int(rng, 256, 8192, 256),
                    n=_log_int(rng, 256, 10240, 16), bias=rng.random() < 0.7,
                    residual=rng.random() < 0.25,
                    dtype="fp32" if rng.random() < 0.15 else "bf16")
    if kind == "ffn":
        return dict(kind=kind, m=_log_int(rng, 1, 4096), k=_log_int(rng, 512, 3072, 256),
                    inner=_log_int(rng, 1024, 8192, 256),
                    act=rng.choice(("situ", "geglu_erf", "gelu_erf")))
    if kind == "qkv":
        return dict(kind=kind, s=_log_int(rng, 256, 4096), h=rng.randint(8, 24),
                    d=rng.choice((64, 128)), k=_log_int(rng, 512, 3072, 256))
    if kind == "train":
        return dict(kind=kind, m=_log_int(rng, 256, 4096), k=_log_int(rng, 512, 5120, 256),
                    n=_log_int(rng, 512, 10240, 16), mode=rng.choice(("int8", "dense")))
    if kind == "ste":
        return dict(kind=kind, m=_log_int(rng, 256, 4096), k=_log_int(rng, 512, 5120, 256),
                    n=_log_int(rng, 512, 5120, 16))
    return dict(kind=kind, n=_log_int(rng, 1024, 16384, 16), k=_log_int(rng, 512, 8192, 256))


# ------------------------------------------------------------------ the inputs
class _Rand:
    """Seeded inputs on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(int(seed) % (1 << 62))

    def normal(self, *shape, std=1.0, dtype=torch.bfloat16):
        t = torch.randn(*shape, generator=self.g, device=DEV, dtype=torch.float32)
        return t.mul_(std).to(dtype)

    def activation(self, m, k, dtype=torch.bfloat16):
        t = torch.randn(m, k, generator=self.g, device=DEV, dtype=torch.float32)
        idx = torch.randperm(k, generator=self.g, device=DEV)[: max(1, k // 100)]
        t[:, idx] *= 30.0
        return t.to(dtype)


def _inputs(case, seed):
    """The raw tensors of a case (before any weight preparation)."""
    r, c, kind = _Rand(seed), case, case["kind"]
    if kind == "linear":
        dt = torch.float32 if c["dtype"] == "fp32" else torch.bfloat16
        s = dict(x=r.activation(c["m"], c["k"], dt), w=r.normal(c["n"], c["k"], std=0.02),
                 bias=r.normal(c["n"], std=0.01) if c["bias"] else None, res=None, rscale=None)
        if c["residual"]:
            s.update(res=r.normal(c["m"], c["n"], dtype=dt), rscale=r.normal(c["n"], std=0.5, dtype=dt))
        return s
    if kind == "ffn":
        up = 2 * c["inner"] if c["act"] in PAIRED else c["inner"]
        return dict(x=r.activation(c["m"], c["k"]), up=r.normal(up, c["k"], std=0.02),
                    down=r.normal(c["k"], c["inner"], std=0.02), bias=r.normal(c["k"], std=0.01))
    if kind == "qkv":
        hd = c["h"] * c["d"]
        ang = torch.arange(c["s"], device=DEV, dtype=torch.float32)[:, None] * torch.pow(
            torch.tensor(10000.0, device=DEV),
            -torch.arange(c["d"] // 2, device=DEV, dtype=torch.float32) / (c["d"] // 2))[None]
        f = torch.stack((ang.cos(), -ang.sin(), ang.sin(), ang.cos()), dim=-1)
        return dict(x=r.activation(c["s"], c["k"]), w=r.normal(3 * hd, c["k"], std=0.02),
                    qn=r.normal(c["d"], std=0.1, dtype=torch.float32) + 1.0,
                    kn=r.normal(c["d"], std=0.1, dtype=torch.float32) + 1.0,
                    freqs=f.reshape(1, c["s"], 1, c["d"] // 2, 2, 2))
    if kind == "train":
        return dict(x=r.activation(c["m"], c["k"]), w=r.normal(c["n"], c["k"], std=0.02),
                    bias=r.normal(c["n"], std=0.01, dtype=torch.float32),
                    dy=r.normal(c["m"], c["n"]))
    if kind == "ste":
        return dict(x=r.activation(c["m"], c["k"]), w=r.normal(c["n"], c["k"], std=0.02),
                    bias=r.normal(c["n"], std=0.01), dy=r.normal(c["m"], c["n"]))
    return dict(w=r.normal(c["n"], c["k"], std=0.02))


def prepare(case, seed):
    s = _inputs(case, seed)
    kind = s["kind"] = case["kind"]
    if kind == "linear":
        s["w8"], s["ws"] = int8.prepare_weight(s.pop("w"))
    elif kind == "ffn":
        s["up8"], s["ups"] = int8.prepare_weight(s.pop("up"))
        s["down8"], s["downs"] = int8.prepare_weight(s.pop("down"))
        s["act"] = case["act"]
    elif kind == "qkv":
        s["w8"], s["ws"] = int8.prepare_weight(s.pop("w"))
        s["h"], s["d"] = case["h"], case["d"]
    elif kind == "train":
        s["w8"], s["ws"] = int8.prepare_weight(s.pop("w"))
        s["mode"] = case["mode"]
        s["x"].requires_grad_(True)
        s["bias"].requires_grad_(True)
    elif kind == "ste":
        s["mod"] = int8.TrainableInt8Linear(s.pop("w"), s.pop("bias"))
        s["x"].requires_grad_(True)
    return s


# -------------------------------------------------------------------- one pass
def run(s):
    kind = s["kind"]
    if kind == "linear":
        if s["res"] is None:
            return int8.linear(s["x"], s["w8"], s["ws"], s["bias"])
        return int8.linear(s["x"], s["w8"], s["ws"], s["bias"], residual=s["res"],
                           residual_scale=s["rscale"])
    if kind == "ffn":
        return int8.ffn(s["x"], s["up8"], s["ups"], s["down8"], s["downs"], s["bias"],
                        act=s["act"])
    if kind == "qkv":
        h, d = s["h"], s["d"]
        hd = h * d
        acc, xs, ws = int8.linear(s["x"], s["w8"], s["ws"], return_acc=True)
        qkv = acc.view(1, acc.shape[0], 3, h, d)
        q, k = rope.rms_rope_split_half_dequant(qkv[:, :, 0], qkv[:, :, 1], s["freqs"], ws[:hd],
                                                ws[hd:2 * hd], xs, s["qn"], s["kn"])
        return q, k, int8.dequant_slice(acc[:, 2 * hd:], xs, ws[2 * hd:])
    if kind == "train":
        x, bias = s["x"], s["bias"]
        x.grad = bias.grad = None
        y = int8.int8_linear(x, s["w8"], s["ws"], bias, mode=s["mode"])
        y.backward(s["dy"])
        return y, x.grad, bias.grad
    if kind == "ste":
        x, mod = s["x"], s["mod"]
        x.grad = mod.weight.grad = mod.bias.grad = None
        y = mod(x)
        y.backward(s["dy"])
        return y, x.grad, mod.weight.grad, mod.bias.grad
    return int8.prepare_weight(s["w"])


# --------------------------------------------------------- work and tolerances
def work(case):
    c, kind = case, case["kind"]
    if kind == "linear":
        m, n, k = c["m"], c["n"], c["k"]
        e = 4 if c["dtype"] == "fp32" else 2
        b = e * m * k + n * k + 4 * n + e * m * n + (2 * n if c["bias"] else 0)
        if c["residual"]:
            b += e * m * n + e * n
        return dict(bytes=b, flops=2.0 * m * n * k)
    if kind == "ffn":
        m, k, f = c["m"], c["k"], c["inner"]
        up = 2 * f if c["act"] in PAIRED else f
        return dict(bytes=2 * m * k * 2 + (up + f) * k + 4 * (up + k) + 2 * k,
                    flops=2.0 * m * k * (up + f))
    if kind == "qkv":
        m, n, k = c["s"], 3 * c["h"] * c["d"], c["k"]
        return dict(bytes=2 * m * k + n * k + 4 * n + 2 * m * n + 8 * m * c["d"],
                    flops=2.0 * m * n * k)
    if kind == "train":
        m, n, k = c["m"], c["n"], c["k"]
        # forward: x, w8 -> y; backward: dy, w8 -> dx, dbias
        return dict(bytes=2 * (2 * m * k + n * k + 2 * m * n) + 16 * n, flops=4.0 * m * n * k)
    if kind == "ste":
        m, n, k = c["m"], c["n"], c["k"]
        # x, w -> y; dy, w -> dx; dy, x -> dw, db
        return dict(bytes=2 * (3 * m * k + 3 * n * k + 3 * m * n) + 4 * n, flops=6.0 * m * n * k)
    n, k = c["n"], c["k"]
    return dict(bytes=3 * n * k + 4 * n, flops=8.0 * n * k)


def tolerance(case):
    """The int8 paths are bit for bit defined (exact integer sums, every fp32
    step rounded in a fixed order).  Where sums of bf16 products are formed in
    fp32 (the dense dx, dW) or a row's mean of squares is (RMSNorm), their
    order is free: against float64 these paths measure 1.7e-3 to 3.0e-3
    relative (the bf16 rounding of the results), stated about three times over."""
    kind = case["kind"]
    if kind == "qkv" or kind == "ste" or (kind == "train" and case["mode"] == "dense"):
        return {"rel": 8e-3}
    return "exact"


# --------------------------------------------------------- float64 definitions
def _rot(t):
    """The ConvRot rotation of every 256-group, kron(H4, H4, H4, H4) / 16, in
    float64 (H4 is symmetric, and so is the product)."""
    h4 = torch.tensor(((1, 1, 1, -1), (1, 1, -1, 1), (1, -1, 1, 1), (-1, 1, 1, 1)),
                      dtype=torch.float64, device=t.device) / 2
    h = h4
    for _ in range(3):
        h = torch.kron(h, h4)
    t = t.double()
    return (t.reshape(-1, 256) @ h).reshape(t.shape)


def _quant(v):
    """Row scale and codes of float64 rows (as float64)."""
    s = (v.abs().amax(dim=-1) / 127.0).clamp_min(1e-30)
    return torch.round(v / s[:, None]).clamp_(-127, 127), s


def _prepared(w):
    """prepare_weight's codes (float64) and scales: the rotated rows rounded to bf16."""
    wr = _rot(w).to(torch.bfloat16).double()
    return _quant(wr)


def _lin(x, w8, ws, bias=None):
    q, s = _quant(_rot(x.to(torch.bfloat16)))
    y = (q @ w8.t()) * (s[:, None] * ws[None, :])
    return y if bias is None else y + bias.double()


def _gelu(t):
    return 0.5 * t * (1.0 + torch.erf(t * math.sqrt(0.5)))


def _act(name, t):
    if name == "gelu_erf":
        return _gelu(t)
    h, g = t.chunk(2, dim=-1)
    if name == "geglu_erf":
        return h * _gelu(g)
    return torch.tanh(g / 4.0) * torch.sigmoid(g) * torch.tanh(h / 25.0)


def exact(case, seed):
    s, kind = _inputs(case, seed), case["kind"]
    if kind == "linear":
        y = _lin(s["x"], *_prepared(s["w"]), s["bias"])
        return y if s["res"] is None else s["res"].double() + s["rscale"].double() * y
    if kind == "ffn":
        a = _act(case["act"], _lin(s["x"], *_prepared(s["up"])))
        return _lin(a, *_prepared(s["down"]), s["bias"])
    if kind == "qkv":
        n, h, d = case["s"], case["h"], case["d"]
        qkv = _lin(s["x"], *_prepared(s["w"])).reshape(n, 3, h, d)
        f = s["freqs"].double()[0]                           # [S, 1, D/2, 2, 2]

        def normed(t, w):
            t = t * torch.rsqrt(t.square().mean(dim=-1, keepdim=True) + 1e-6) * w.double()
            a, b = t[..., : d // 2], t[..., d // 2:]
            return torch.cat((f[..., 0, 0] * a + f[..., 0, 1] * b,
                              f[..., 1, 0] * a + f[..., 1, 1] * b), dim=-1)[None]
        return normed(qkv[:, 0], s["qn"]), normed(qkv[:, 1], s["kn"]), qkv[:, 2].reshape(n, h * d)
    if kind == "train":
        w8, ws = _prepared(s["w"])
        dy = s["dy"].double()
        if case["mode"] == "int8":
            ws16 = ws.float().to(torch.bfloat16).double()
            q, a = _quant((dy * ws16).to(torch.bfloat16).double())
            dx = _rot((q @ w8) * a[:, None])
        else:
            dx = dy @ _rot((w8 * ws[:, None]).to(torch.bfloat16))
        return _lin(s["x"], w8, ws, s["bias"]), dx, dy.sum(dim=0)
    if kind == "ste":
        w8, ws = _quant(_rot(s["w"]))
        dy = s["dy"].double()
        return (_lin(s["x"], w8, ws, s["bias"]), dy @ s["w"].double(),
                dy.t().contiguous() @ s["x"].double(), dy.sum(dim=0))
    return None, _prepared(s["w"])[1]
