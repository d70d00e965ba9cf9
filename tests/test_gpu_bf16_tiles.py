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


# (M, N, K) and the kernel, tile and contraction slices that it takes (checked in
# test_kernel_choice.py): every tile of the persistent kernel in one round and, where
# a product can have them, in several, whole and in slices, with ragged rows and
# columns, contractions that end inside a 32-row step (1040, 3824) or a slice and one
# of a single short step; and the split-K kernel
DX_SHAPES = {
    (3800, 1040, 5120): ("persistent", 256, 320, 1),    # 240 tiles
    (2500, 1040, 10240): ("persistent", 256, 320, 1),    # 320 tiles
    (3000, 3072, 3072): ("persistent", 192, 256, 1),    # 192 tiles
    (3969, 224, 5280): ("persistent", 192, 256, 1),    # 441 tiles
    (2500, 528, 2576): ("persistent", 128, 256, 1),    # 220 tiles
    (2394, 128, 2512): ("persistent", 128, 256, 1),    # 190 tiles
    (3665, 7056, 1024): ("persistent", 128, 256, 2),    # 232 tiles
    (130, 7168, 3328): ("persistent", 128, 256, 8),    # 208 tiles
    (3798, 128, 1184): ("persistent", 128, 192, 1),    # 210 tiles
    (2346, 288, 4896): ("persistent", 128, 192, 1),    # 494 tiles
    (561, 2080, 3216): ("persistent", 128, 192, 2),    # 170 tiles
    (129, 1936, 5440): ("persistent", 128, 192, 4),    # 232 tiles
    (1500, 1040, 2000): ("persistent", 128, 128, 1),    # 192 tiles
    (40, 16, 272): ("persistent", 128, 128, 1),    # 3 tiles
    (1206, 848, 768): ("persistent", 128, 128, 1),    # 60 tiles
    (129, 80, 16): ("persistent", 128, 128, 1),    # 2 tiles
    (322, 5648, 2048): ("persistent", 128, 128, 5),    # 240 tiles
    (205, 2672, 768): ("persistent", 128, 128, 8),    # 96 tiles
    (1166, 3824, 1024): ("persistent", 128, 128, 3),    # 240 tiles
    (300, 4112, 528): ("persistent", 128, 128, 8),    # 120 tiles
    (390, 2080, 5120): ("splitk", 128, 160, 1),    # 128 tiles
}
# the contraction over M: batches of 1, of 17 and odd ones
DW_SHAPES = {
    (267, 3856, 3584): ("persistent", 256, 256, 1),    # 224 tiles
    (1001, 5120, 5120): ("persistent", 256, 256, 1),    # 400 tiles
    (103, 1648, 4944): ("persistent", 192, 256, 1),    # 180 tiles
    (373, 8544, 2816): ("persistent", 192, 256, 1),    # 495 tiles
    (1585, 2480, 3072): ("persistent", 128, 256, 1),    # 240 tiles
    (105, 3136, 4944): ("persistent", 128, 256, 1),    # 500 tiles
    (2129, 2768, 768): ("persistent", 128, 256, 3),    # 198 tiles
    (3077, 160, 4720): ("persistent", 128, 256, 6),    # 228 tiles
    (615, 4896, 1024): ("persistent", 128, 192, 1),    # 234 tiles
    (105, 3712, 4432): ("persistent", 128, 192, 1),    # 696 tiles
    (3009, 976, 2816): ("persistent", 128, 192, 2),    # 240 tiles
    (1407, 160, 5408): ("persistent", 128, 192, 4),    # 232 tiles
    (17, 48, 144): ("persistent", 128, 128, 1),    # 2 tiles
    (1, 160, 272): ("persistent", 128, 128, 1),    # 6 tiles
    (33, 16, 16): ("persistent", 128, 128, 1),    # 1 tiles
    (2893, 544, 768): ("persistent", 128, 128, 7),    # 210 tiles
    (1971, 672, 512): ("persistent", 128, 128, 7),    # 168 tiles
    (2112, 1680, 2000): ("splitk", 160, 160, 1),    # 143 tiles
}


@pytest.mark.parametrize("m,n,k", list(DX_SHAPES))
def test_linear_dx_tiles(dev, m, n, k):
    dy, w = operand(m, n, 1e-3, m, dev), operand(n, k, 0.02, n + k, dev)
    check(int8.linear_dx(dy, w), dy, w)


@pytest.mark.parametrize("m,n,k", list(DW_SHAPES))
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
