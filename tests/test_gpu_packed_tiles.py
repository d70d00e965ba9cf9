"""The tiles that products of two block-layout operands take (the packed
weight): each tile of the persistent kernel at its edges -- ragged rows and
columns, the shortest K, one round of tiles and several -- with the dequant,
residual and int32 epilogues.  The reference is the exact integer product in
float64 and the epilogue's fp32 operations one by one in torch, so the results
are equal bit for bit."""

import pytest
import torch

from gpu_util import activation, weight
from xpu_kernels import int8

pytestmark = pytest.mark.gpu


def reference(x, w8, ws, bias, res=None, rscale=None):
    """(int32 product, bf16 output) from the library's own quantizer (checked
    against the oracle elsewhere) and plain torch."""
    q, xs = int8.quantize(x)
    acc = (q.double() @ w8.double().t()).to(torch.int32)
    y = acc.float() * (ws[None, :] * xs[:, None])
    y = (y + bias.float()).to(torch.bfloat16)
    return acc, y if res is None else torch.addcmul(res, y, rscale)


# (M, N, K) and the kernel and tile that the dequant product takes (checked in
# test_kernel_choice.py): the persistent kernel's five tiles in one round and in
# several, split K (a long K), and the tiles of the kernel that splits K over a
# block's waves (one row block and one column block past the batch; fewer K steps
# than waves; a long K at 33 rows), each with ragged rows and columns.  linear_acc takes
# the same, but for split K, which has no int32 form
SHAPES = {
    (4090, 5104, 2048): ("persistent", 256, 320),
    (1050, 10912, 256): ("persistent", 192, 320),
    (3000, 10240, 1280): ("persistent", 192, 320),
    (3974, 3072, 3072): ("persistent", 192, 256),
    (1355, 6160, 256): ("persistent", 192, 256),
    (2060, 9232, 1280): ("persistent", 192, 256),
    (920, 6224, 256): ("persistent", 192, 192),
    (1541, 3856, 5120): ("persistent", 192, 192),
    (2323, 6144, 256): ("persistent", 192, 192),
    (1251, 4752, 3072): ("persistent", 128, 192),
    (2147, 11024, 256): ("persistent", 128, 192),
    (4090, 1264, 6144): ("splitk", 128, 160),
    (65, 16, 256): ("wavek", 16, 16),
    (129, 208, 256): ("wavek", 16, 16),
    (35, 320, 5120): ("wavek", 16, 16),
    (64, 1280, 5120): ("wavek", 16, 32),
    (525, 976, 2048): ("wavek", 16, 32),
    (438, 496, 1024): ("wavek", 32, 32),
    (135, 992, 3840): ("wavek", 32, 32),
    (1000, 1296, 1280): ("wavek", 32, 64),
    (700, 2064, 6144): ("wavek", 32, 64),
    (400, 1936, 2048): ("wavek", 64, 64),
    (1218, 624, 6400): ("wavek", 64, 64),
    (449, 1696, 256): ("wavek", 64, 64),
}


@pytest.mark.parametrize("m,n,k", list(SHAPES))
def test_packed_tiles_exact(dev, m, n, k):
    w8, ws = int8.prepare_weight(weight(n, k, seed=n + k).to(dev))
    x = activation(m, k, seed=m + k).to(dev)
    bias = weight(1, n, seed=3, std=0.01)[0].to(dev)
    res = activation(m, n, seed=m, n_out=0).to(dev)
    rscale = weight(1, n, seed=4, std=0.5)[0].to(dev)
    acc, y = reference(x, w8, ws, bias)
    assert torch.equal(int8.linear(x, w8, ws, bias), y)
    got, xs = int8.linear_acc(x, w8, ws)
    assert torch.equal(got, acc)
    _, yr = reference(x, w8, ws, bias, res, rscale)
    assert torch.equal(int8.linear(x, w8, ws, bias, residual=res, residual_scale=rscale), yr)


# The FFN's up-projection, (M, inner, K): what its product takes for the paired
# activations (a ragged batch in each) and for GELU
FFN_SHAPES = {
    (4090, 5120, 512): (("persistent", 256, 320), ("persistent", 256, 320)),
    (2315, 2560, 256): (("persistent", 256, 256), ("persistent", 192, 192)),
    (892, 5376, 512): (("persistent", 192, 256), ("persistent", 128, 192)),
    (514, 5120, 256): (("persistent", 128, 256), ("persistent", 128, 192)),
    (357, 4608, 256): (("persistent", 128, 192), ("wavek", 64, 64)),
    (304, 1280, 512): (("wavek", 64, 64), ("wavek", 32, 64)),
    (45, 2816, 256): (("wavek", 32, 64), ("skinny", 48, 16)),
    (33, 1536, 256): (("wavek", 32, 32), ("skinny", 48, 16)),
    (19, 512, 256): (("wavek", 16, 32), ("skinny", 32, 16)),
    (16, 1024, 512): (("skinny", 16, 64), ("skinny", 16, 16)),
}


@pytest.mark.parametrize("m,inner,k", list(FFN_SHAPES))
@pytest.mark.parametrize("act", ["situ", "geglu_erf", "gelu_erf"])
def test_ffn_packed_tiles_exact(dev, act, m, inner, k):
    """Against the library's unfused chain (int32 product, the row kernel that
    dequantizes, activates and quantizes it, int32 product, dequant), each
    checked against the oracle elsewhere.  Row magnitudes from 2^-16 to 2^8 put the
    table lookups inside and on both sides of the epilogue's windows."""
    up_rows = inner if act == "gelu_erf" else 2 * inner
    uw8, us = int8.prepare_weight(weight(up_rows, k, seed=inner + k).to(dev))
    dw8, ds = int8.prepare_weight(weight(k, inner, seed=inner + k + 1).to(dev))
    mag = torch.exp2(torch.linspace(-16, 8, m))[torch.randperm(m, generator=torch.Generator().manual_seed(m))]
    x = (activation(m, k, seed=m).float() * mag[:, None]).to(torch.bfloat16).to(dev)
    bias = weight(1, k, seed=6, std=0.01)[0].to(dev)
    acc, xs = int8.linear_acc(x, uw8, us)
    q, s = int8.dequant_act_quantize(acc, xs, us, act)
    want = int8.dequant(int8.int_mm(q, dw8.t()), s, ds, bias)
    got = int8.ffn(x, uw8, us, dw8, ds, bias, act=act)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


# one row group of one 256-group; rows per block that do not divide N; two groups
# per lane (K > 16384); longer than the one-pass kernel takes
@pytest.mark.parametrize("n,k", [(16, 256), (10240, 1280), (48, 5120), (1040, 768), (32, 16896),
                                 (16, 33024)])
def test_prepare_weight_packed_exact(dev, n, k):
    """prepare_weight's one-pass codes, scales and packed copy against the two
    separate passes."""
    from xpu_kernels.int8 import _lib as L, ops
    w = weight(n, k, seed=n + k).to(dev)
    w8, ws = int8.prepare_weight(w)
    w8r, wsr = int8.prepare_weight(w, pack=False)
    assert torch.equal(w8, w8r) and torch.equal(ws, wsr)
    packed = torch.empty(n * k, device=dev, dtype=torch.int8)
    assert L._lib().xpuint8_pack_weight_stream(L._stream(dev), L._ptr(w8r), L._ptr(packed), n,
                                               k) == 0
    assert torch.equal(ops._packed_for(w8), packed)
