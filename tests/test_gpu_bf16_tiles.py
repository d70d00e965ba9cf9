"""The bf16 products of the backward, linear_dx (dy @ w) and linear_dw (dy^T @ x),
on each tile of the persistent kernel at its edges: ragged rows and columns, a
contraction that is not a multiple of 32 or shorter than one step, one round of
tiles and several, and the contraction split across blocks.

The bar is linear_dx's: each element within one bf16 rounding of the float64
value plus the fp32 accumulation error, 2^-8 |ref| + 2^-14 sum |a||b|."""

import pytest
import torch

from xpu_kernels import int8
from xpu_kernels.int8 import _lib as L

pytestmark = pytest.mark.gpu


def check(got, a, b):
    """got = a @ b (a, b already oriented) within the bound, in float64."""
    a, b = a.double(), b.double().contiguous()
    ref, mag = a @ b, a.abs() @ b.abs()
    bound = 2.0 ** -8 * ref.abs() + 2.0 ** -14 * mag
    err = (got.double() - ref).abs()
    assert bool((err <= bound).all()), float((err / bound.clamp_min(1e-300)).max())


def operand(rows, cols, std, seed, dev):
    g = torch.Generator(device=dev).manual_seed(seed)
    return (torch.randn(rows, cols, generator=g, device=dev) * std).to(torch.bfloat16)


# (M, N, K): 256x320 (one round, 1040 % 32 = 16), 192x256 (one; several), 128x256 (two
# slices), 128x192 (one tile row; two, three slices), 128x128 (a single short step;
# one slice; four, six and eight slices with a ragged last one)
@pytest.mark.parametrize("m,n,k", [(3800, 1040, 5120), (3000, 3072, 3072), (2500, 528, 2576),
                                   (3665, 7056, 1024), (1500, 1040, 2000), (40, 16, 272),
                                   (1206, 848, 768), (322, 5648, 2048), (205, 2672, 768),
                                   (1166, 3824, 1024), (129, 80, 16), (300, 4112, 528)])
def test_linear_dx_tiles(dev, m, n, k):
    dy, w = operand(m, n, 1e-3, m, dev), operand(n, k, 0.02, n + k, dev)
    check(int8.linear_dx(dy, w), dy, w)


# (M, N, K), the contraction over M: 256x256, 192x256, 128x256, 128x192 (a batch of
# 1, of 17 and odd ones), 128x128 whole and in slices
@pytest.mark.parametrize("m,n,k", [(267, 3856, 3584), (1001, 5120, 5120), (373, 8544, 2816),
                                   (1585, 2480, 3072), (615, 4896, 1024), (17, 48, 144),
                                   (1, 160, 272), (2893, 544, 768), (2129, 2768, 768),
                                   (3009, 976, 2816), (1971, 672, 512), (33, 16, 16)])
def test_linear_dw_tiles(dev, m, n, k):
    dy, x = operand(m, n, 1e-3, m, dev), operand(m, k, 1.0, n + k, dev)
    check(int8.linear_dw(dy, x), dy.t(), x)


def test_linear_dx_wide_rows(dev):
    """A weight of 2^27 + 16 columns: the lanes' byte offsets past 32 bits."""
    m, n, k = 8, 16, (1 << 27) + 16
    dy = operand(m, n, 1e-2, 1, dev)
    w = torch.empty(n, k, device=dev, dtype=torch.bfloat16)
    for r in range(n):
        w[r] = operand(1, k, 0.02, 100 + r, dev)[0]
    dx = int8.linear_dx(dy, w)
    for cut in (slice(0, 4096), slice(k // 2, k // 2 + 4096), slice(k - 4096, k)):
        check(dx[:, cut], dy, w[:, cut])


@pytest.mark.parametrize("m,n,k", [(205, 2672, 768), (322, 5648, 2048), (1024, 5120, 1280)])
def test_dense_backward_in_less_workspace(dev, m, n, k):
    """xpuint8_linear_backward_dense_stream in the least workspace it takes (a size
    that names no device), nothing written past it: dx as linear_dx_stream gives it
    with that much for its partial sums, bit for bit."""
    lib = L._lib()
    dy = operand(m, n, 1e-3, m, dev)
    w8, ws = int8.prepare_weight(operand(n, k, 0.02, n + k, dev))
    wd = int8.dequant_weight(w8, ws)
    part = lib.xpuint8_linear_dx_workspace_size(m, n, k)
    least = (2 * n * k + 255) // 256 * 256 + (-(-m // 32) * n * 4 + 255) // 256 * 256 + part
    work = torch.full((least + 4096,), 0x55, device=dev, dtype=torch.uint8)
    dx = torch.empty(m, k, device=dev, dtype=torch.bfloat16)
    rc = lib.xpuint8_linear_backward_dense_stream(L._stream(dev), L._ptr(dy), L._ptr(w8), L._ptr(ws),
                                                  L._ptr(dx), None, 0, m, n, k, L._ptr(work), least)
    assert rc == 0, lib.xpuint8_last_error()
    assert bool((work[least:] == 0x55).all())
    want = torch.empty_like(dx)
    w2 = torch.empty(max(part, 16), device=dev, dtype=torch.uint8)
    assert lib.xpuint8_linear_dx_stream(L._stream(dev), L._ptr(dy), L._ptr(wd), L._ptr(want), m, n,
                                        k, L._ptr(w2) if part else None, part) == 0
    assert torch.equal(dx, want)
    check(dx, dy, wd)
