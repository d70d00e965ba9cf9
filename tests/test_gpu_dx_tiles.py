"""linear_dx_int8's kernels by shape: one round of the split-K kernel on the weight
as stored, else the transposed weight in the block layout with the packed
products' tiles (a contraction that ends inside a 64-byte step, whose padded
copy runs into the product's region; one and two row blocks; a batch just large
enough for that region), else, for a few rows of such a contraction or rows of
dy too long to be quantized into the layout, row-major operands.  Bit for bit
the oracle's, twice in a row through one workspace that the first call left full."""

import numpy as np
import pytest
import torch

import oracle as O
from gpu_util import bits, mismatch, npy, weight
from xpu_kernels import int8
from xpu_kernels.int8 import _lib as L
from xpu_kernels.int8 import ops

pytestmark = pytest.mark.gpu


# (M, N, K)
SHAPES = [(2060, 2064, 1280), (2180, 1104, 2560),                # split K; 16 * 16 + 16 tiles more
          (33, 528, 256), (65, 1040, 512), (130, 48, 256), (300, 2608, 768), (1273, 528, 512),
          (24, 16, 256), (23, 16, 256), (1, 16, 512), (7, 1296, 256), (16, 64, 256),
          # N > 32768: whole; in contraction slices through the transposed weight (M <=
          # 256) and on the weight as stored
          (3, 32784, 256), (70, 33024, 256), (300, 33024, 256)]


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_dx_int8_by_shape_exact(dev, m, n, k):
    lib = L._lib()
    w8, ws = int8.prepare_weight(weight(n, k, seed=n + k).to(dev))
    g = torch.Generator().manual_seed(m + n)
    need = lib.xpuint8_linear_dx_int8_workspace_size(m, n, k)
    work = torch.full((need,), 0x55, device=dev, dtype=torch.uint8)
    guard = torch.full((m * k + 4096,), 7.0, device=dev, dtype=torch.bfloat16)
    for _ in range(2):
        dy = (torch.randn(m, n, generator=g) * 1e-3).to(torch.bfloat16)
        dx = dy.to(dev)
        rc = lib.xpuint8_linear_dx_int8_stream(L._stream(dev), L._ptr(dx), L._ptr(ws), L._ptr(w8),
                                               L._ptr(guard), m, n, k, L._ptr(work), need)
        assert rc == 0, lib.xpuint8_last_error()
        got = bits(guard[: m * k].view(m, k))
        want = O.linear_dx_int8(bits(dy), npy(w8), npy(ws))
        assert np.array_equal(got, want), mismatch(got, want)
        assert bool((guard[m * k:] == 7.0).all())


def test_dx_int8_long_rows_unsplit(dev):
    """N > 32768 with enough tiles for the split-K kernel, row-major dy codes and the
    weight as stored: the row quantizer's codes, the exact product in float64 and
    the inverse rotation, each checked elsewhere."""
    m, n, k = 2060, 33024, 1280
    g = torch.Generator(device=dev).manual_seed(5)
    w8 = torch.randint(-127, 128, (n, k), generator=g, device=dev, dtype=torch.int8)
    ws = torch.rand(n, generator=g, device=dev) * 1e-2 + 1e-4
    dy = (torch.randn(m, n, generator=g, device=dev) * 1e-3).to(torch.bfloat16)
    q, a = int8.quantize_row(dy, ws)
    acc = (q.double() @ w8.double()).to(torch.int32)
    want = int8.rotate((acc.float() * a[:, None]).to(torch.bfloat16))
    assert torch.equal(int8.linear_dx_int8(dy, w8, ws), want)


# one round of the split-K kernel (which reads the second packed form); more rounds,
# few tiles, a short contraction (which do not)
@pytest.mark.parametrize("m,n,k,reads", [(2060, 2064, 1280, True), (4096, 1040, 1536, False),
                                         (300, 2608, 768, False), (2060, 528, 1280, False)])
def test_second_packed_form_only_where_read(dev, m, n, k, reads):
    """int8 backwards and linear_dx_int8 make the weight's second packed form, which
    stays with it, only for a product that reads it."""
    w8, ws = int8.prepare_weight(weight(n, k, seed=n + k).to(dev))
    dy = (torch.randn(m, n, generator=torch.Generator().manual_seed(m)) * 1e-3).to(torch.bfloat16)
    want = int8.linear_dx_int8(dy.to(dev), w8.clone(), ws)      # (no packed copy)
    x = torch.zeros(m, k, device=dev, dtype=torch.bfloat16, requires_grad=True)
    for _ in range(2):
        x.grad = None
        int8.int8_linear(x, w8, ws, mode="int8").backward(dy.to(dev))
        assert torch.equal(x.grad, want)
        assert (ops._packed_entry(w8)[4] is not None) == reads
    assert torch.equal(int8.linear_dx_int8(dy.to(dev), w8, ws), want)
    assert (ops._packed_entry(w8)[4] is not None) == reads
