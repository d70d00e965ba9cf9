"""The kernel and tile that each shape of the tile tests takes on 256 CUs
(xpuint8_gemm_choice, no device needed), as written beside it there: a refit of the
time models that takes a tile away from those tests fails here.  And what they
leave out: no tile that the models can choose."""

import ctypes

import pytest
import torch

import test_gpu_bf16_tiles as bf16
import test_gpu_packed_tiles as packed
from xpu_kernels.int8 import _lib as L

KERNELS = ["skinny", "wavek", "splitk", "persistent"]
LINEAR, ACC, SITU, GEGLU, GELU, DX, DW = 0, 1, 3, 4, 5, 6, 7


@pytest.fixture(scope="module")
def lib():
    if torch.cuda.is_available():
        props = torch.cuda.get_device_properties(0)
        if props.multi_processor_count != 256:
            pytest.skip("the shapes are chosen for 256 CUs")
    return L.open_library(L.library_path())


def choice(lib, product, m, n, k):
    c = (ctypes.c_int32 * 4)()
    assert lib.xpuint8_gemm_choice(product, m, n, k, c) == 0, lib.xpuint8_last_error()
    return KERNELS[c[0]], c[1], c[2], c[3]


def test_bf16_shapes_take_their_tiles(lib):
    for product, shapes in ((DX, bf16.DX_SHAPES), (DW, bf16.DW_SHAPES)):
        for shape, want in shapes.items():
            assert choice(lib, product, *shape) == want, shape


def test_packed_shapes_take_their_tiles(lib):
    for shape, want in packed.SHAPES.items():
        assert choice(lib, LINEAR, *shape)[:3] == want, shape
        acc = choice(lib, ACC, *shape)[:3]
        assert acc == want or want[0] == "splitk", shape
    for shape, (paired, gelu) in packed.FFN_SHAPES.items():
        assert choice(lib, SITU, *shape)[:3] == choice(lib, GEGLU, *shape)[:3] == paired, shape
        assert choice(lib, GELU, *shape)[:3] == gelu, shape


def test_shapes_cover_every_tile():
    """Each tile of each kernel, the bf16 ones also in slices where they have them."""
    pp = {(256, 320), (192, 320), (192, 256), (192, 192), (128, 192)}
    wavek = {(16, 16), (16, 32), (32, 32), (32, 64), (64, 64)}
    got = set(packed.SHAPES.values())
    assert got == ({("persistent", *t) for t in pp} | {("wavek", *t) for t in wavek}
                   | {("splitk", 128, 160)})
    pair = {(256, 320), (256, 256), (192, 256), (128, 256), (128, 192)}
    pair_wavek = {(16, 32), (32, 32), (32, 64), (64, 64)}
    assert {p for p, _ in packed.FFN_SHAPES.values()} == (
        {("persistent", *t) for t in pair} | {("wavek", *t) for t in pair_wavek}
        | {("skinny", 16, 64)})
    for shapes, large, split_k in ((bf16.DX_SHAPES, (256, 320), 128), (bf16.DW_SHAPES, (256, 256), 160)):
        forms = {(t[0], t[1], t[2], t[3] > 1) for t in shapes.values()}
        assert forms == ({("persistent", *t, False) for t in (large, (192, 256))}
                         | {("persistent", 128, c, s) for c in (256, 192, 128) for s in (False, True)}
                         | {("splitk", split_k, 160, False)})


@pytest.mark.parametrize("args,code", [((2, 64, 256, 256), 6), ((8, 64, 256, 256), 6),
                                       ((-1, 64, 256, 256), 6), ((0, 64, 24, 256), 2),
                                       ((6, 64, 24, 256), 2), ((0, 64, 256, 1 << 20), 4)])
def test_choice_refuses(lib, args, code):
    assert lib.xpuint8_gemm_choice(*args, (ctypes.c_int32 * 4)()) == code
    assert lib.xpuint8_gemm_choice(0, 64, 256, 256, None) == 6
