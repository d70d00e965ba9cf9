"""The int8 backward's one launch over dy -- column-scaled row quantizer and the bias
gradient's 32-row chunk sums -- at the edges of both: a last chunk of one row, one
short of a chunk, odd rows, one lane and all 1024 lanes of columns, columns that the
two summing blocks split unevenly, and rows too long for it (two launches).  dx and
dbias bit for bit the oracle's; dbias alone and dx alone agree with the separate calls."""

import numpy as np
import pytest
import torch

import oracle as O
from gpu_util import bits, mismatch, npy, weight
from xpu_kernels import int8
from xpu_kernels.int8 import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [(1, 16, 256), (31, 528, 256), (33, 1040, 512), (65, 2064, 256),
                                   (100, 16384, 256), (257, 5120, 512), (64, 16400, 256),
                                   (1283, 48, 256)])
def test_backward_int8_sums_exact(dev, m, n, k):
    w8, ws = int8.prepare_weight(weight(n, k, seed=n + k).to(dev))
    x = torch.zeros(m, k, device=dev, dtype=torch.bfloat16, requires_grad=True)
    bias = torch.zeros(n, device=dev, dtype=torch.float32, requires_grad=True)
    dy = (torch.randn(m, n, generator=torch.Generator().manual_seed(m + n)) * 1e-3).to(torch.bfloat16)
    int8.int8_linear(x, w8, ws, bias, mode="int8").backward(dy.to(dev))
    assert np.array_equal(bits(bias.grad.to(torch.bfloat16)), O.column_sum(bits(dy)))
    want = O.linear_dx_int8(bits(dy), npy(w8), npy(ws))
    assert np.array_equal(bits(x.grad), want), mismatch(bits(x.grad), want)
    assert np.array_equal(bits(int8.linear_dx_int8(dy.to(dev), w8, ws)), want)


def test_backward_int8_sums_non_finite(dev):
    """Infinities and NaN in dy: dx and dbias as the separate calls give them."""
    m, n, k = 100, 1040, 512
    w8, ws = int8.prepare_weight(weight(n, k, seed=n + k).to(dev))
    x = torch.zeros(m, k, device=dev, dtype=torch.bfloat16, requires_grad=True)
    bias = torch.zeros(n, device=dev, dtype=torch.float32, requires_grad=True)
    dy = (torch.randn(m, n, generator=torch.Generator().manual_seed(3)) * 1e-3).to(torch.bfloat16)
    dy[5, 17], dy[40, 100], dy[41, 101], dy[70, 101] = (float("inf"), float("nan"), float("inf"),
                                                        -float("inf"))
    dy = dy.to(dev)
    int8.int8_linear(x, w8, ws, bias, mode="int8").backward(dy)
    for got, want in ((x.grad, int8.linear_dx_int8(dy, w8, ws)),
                      (bias.grad.to(torch.bfloat16), ops.column_sum(dy))):
        nan = want.isnan()
        assert torch.equal(got.isnan(), nan) and torch.equal(got[~nan], want[~nan])
    assert bool(bias.grad.isnan()[[100, 101]].all()) and bool(bias.grad.isinf()[17])
