"""Products of few rows that quantize x in their own launch: the edges of the rule
(64 groups of 256 columns in all, 16 rows) on both sides, each count of waves, ragged
columns and column blocks past the last, more than 512 column blocks, all
epilogues; rows of zeros, of subnormal and of huge values; an output that
overlaps x.  The codes and scales are the library quantizer's (checked against
the oracle elsewhere), the rest the exact integer product and the epilogue's fp32
operations in torch, so every result is equal bit for bit."""

import pytest
import torch

from gpu_util import activation, weight
from xpu_kernels import int8
from xpu_kernels.int8 import _lib as L
from xpu_kernels.int8 import ops

pytestmark = pytest.mark.gpu

# (M, N, K): 1, 16, 17, 32, 33, 64 and (two launches) 65 and 80 groups; 16 and 17 rows
SHAPES = [(1, 16, 256), (1, 1280, 1280), (16, 208, 256), (3, 4096, 1280), (17, 496, 256),
          (1, 1296, 4352), (8, 4112, 1024), (2, 8224, 4096), (16, 8208, 512), (3, 1040, 2816),
          (11, 8240, 768), (16, 2064, 1024), (1, 272, 16384), (13, 528, 1280), (16, 1296, 1280),
          (1, 512, 16640)]


def rows(m, k, seed, dev):
    x = activation(m, k, seed=seed).to(dev)
    if m > 2:
        x[1] = 0
        x[2] = x[2] * 1e-38
    if m > 4:
        x[3] = x[3] * 1e34
        x[4, 5] = 3e38
    return x


def product(x, w8, ws):
    q, xs = int8.quantize(x)
    acc = (q.double() @ w8.double().t()).to(torch.int32)
    return acc, acc.float() * (ws[None, :] * xs[:, None]), xs


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_rowq_exact(dev, m, n, k):
    w8, ws = int8.prepare_weight(weight(n, k, seed=n + k).to(dev))
    assert ops._packed_for(w8) is not None
    x = rows(m, k, m + k, dev)
    b16 = weight(1, n, seed=3, std=0.01)[0].to(dev)
    res = activation(m, n, seed=m, n_out=0).to(dev)
    rscale = weight(1, n, seed=4, std=0.5)[0].to(dev)
    acc, y, xs = product(x, w8, ws)
    got, gxs = int8.linear_acc(x, w8, ws)
    assert torch.equal(got, acc) and torch.equal(gxs, xs)
    assert torch.equal(int8.linear(x, w8, ws), y.to(torch.bfloat16))
    yb = (y + b16.float()).to(torch.bfloat16)
    assert torch.equal(int8.linear(x, w8, ws, b16), yb)
    assert torch.equal(int8.linear(x, w8, ws, b16.float()), yb)
    assert torch.equal(int8.linear(x, w8, ws, b16, residual=res, residual_scale=rscale),
                       torch.addcmul(res, yb, rscale))


# (M, inner, K): 4, 8 and 8 waves of two groups, and (two launches) 65 groups or more
@pytest.mark.parametrize("act", ["situ", "geglu_erf", "gelu_erf"])
@pytest.mark.parametrize("m,f,k", [(1, 256, 256), (3, 1280, 1280), (6, 768, 1280), (16, 512, 1024),
                                   (5, 8192, 768), (13, 1024, 1280)])
def test_rowq_ffn_exact(dev, m, f, k, act):
    up8, ups = int8.prepare_weight(weight((1 if act == "gelu_erf" else 2) * f, k, seed=f).to(dev))
    down8, downs = int8.prepare_weight(weight(k, f, seed=k).to(dev))
    b = weight(1, k, seed=5, std=0.01)[0].to(dev)
    x = activation(m, k, seed=m).to(dev)
    # the same chain from the separate calls: the up-projection's bf16 output, the
    # quantizer with the activation in its load
    h = product(x, up8, ups)[1].to(torch.bfloat16)
    q, s = int8.quantize_act(h, act)
    acc = (q.double() @ down8.double().t()).to(torch.int32)
    want = (acc.float() * (downs[None, :] * s[:, None]) + b.float()).to(torch.bfloat16)
    assert torch.equal(int8.ffn(x, up8, ups, down8, downs, b, act=act), want)


def same(a, b):
    """Equal but for the payload of NaNs."""
    nan = a.isnan()
    return torch.equal(nan, b.isnan()) and torch.equal(a[~nan], b[~nan])


def non_finite_rows(m, k, dev):
    x = activation(m, k, seed=m + k).to(dev)
    x[0, 7] = float("inf")
    if m > 1:
        x[1, 3] = float("nan")
    if m > 2:
        x[2, 0], x[2, k - 1] = float("inf"), -float("inf")
    return x


# 4, 8 and 16 waves, two groups a lane's segment, two weight blocks a block
@pytest.mark.parametrize("m,n,k", [(1, 1280, 1280), (3, 1296, 2560), (16, 208, 1024), (2, 8224, 4096),
                                   (11, 8240, 768)])
def test_rowq_non_finite(dev, m, n, k):
    """Rows with infinities and NaN: what the separate quantizer and product give, in
    those rows and in the others, which share their waves."""
    w8, ws = int8.prepare_weight(weight(n, k, seed=n + k).to(dev))
    x = non_finite_rows(m, k, dev)
    acc, y, xs = product(x, w8, ws)
    got, gxs = int8.linear_acc(x, w8, ws)
    assert torch.equal(got, acc) and same(gxs, xs)
    assert same(int8.linear(x, w8, ws), y.to(torch.bfloat16))
    assert same(int8.linear(x, w8.clone(), ws), y.to(torch.bfloat16))


# the up-projection that quantizes its rows, K split over waves, and the persistent
# kernel with its tables in LDS windows (256x256, 192x256 and GELU's 192x192)
@pytest.mark.parametrize("act", ["situ", "geglu_erf", "gelu_erf"])
@pytest.mark.parametrize("m,f,k", [(6, 768, 1280), (304, 1280, 512), (892, 5376, 512),
                                   (2315, 2560, 256)])
def test_ffn_non_finite(dev, m, f, k, act):
    """The same through an FFN: a row scale that is no number in the epilogues'
    activations, against the unfused chain."""
    up8, ups = int8.prepare_weight(weight((1 if act == "gelu_erf" else 2) * f, k, seed=f).to(dev))
    down8, downs = int8.prepare_weight(weight(k, f, seed=k).to(dev))
    ups[3], ups[f - 1] = float("inf"), float("nan")
    x = non_finite_rows(m, k, dev)
    acc, xs = int8.linear_acc(x, up8, ups)
    q, s = int8.dequant_act_quantize(acc, xs, ups, act)
    want = int8.dequant(int8.int_mm(q, down8.t()), s, downs)
    assert same(int8.ffn(x, up8, ups, down8, downs, act=act), want)


def test_rowq_output_over_x(dev):
    lib = L._lib()
    m, k = 4, 1024
    w8, ws = int8.prepare_weight(weight(k, k, seed=7).to(dev))
    x = activation(m, k, seed=8).to(dev)
    want = int8.linear(x, w8, ws)
    need = lib.xpuint8_linear_workspace_size(m, k, k)
    work = torch.empty(need, device=dev, dtype=torch.uint8)
    rc = lib.xpuint8_linear_packed_stream(L._stream(dev), L._ptr(x), L._ptr(w8),
                                          L._ptr(ops._packed_for(w8)), L._ptr(ws), None, 0,
                                          L._ptr(x), m, k, k, L._ptr(work), need)
    assert rc == 0, lib.xpuint8_last_error()
    assert torch.equal(x, want)
