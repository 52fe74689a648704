"""Row-major 1x1 convolution on both kernels and on either side of the lines between them: pixel
counts around one and two 64-pixel windows, next to images that make the batch small or large."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)
EDGES = [1, 2, 31, 32, 33, 63, 64, 65, 66, 127, 128, 129, 191, 193, 640]


def _route(pixels, c_in, c_out):
    """(wavefronts of the kernel that writes whole lines or 0, wavefronts per window of the other one)."""
    from nestedtensor_amd import _C
    route = (ctypes.c_int * 2)()
    tiles = sum((n + 63) // 64 + 1 for n in pixels)
    _C.check(_C.lib.nt_conv1x1_route(len(pixels), tiles, c_in, c_out, _C.dtype_code(torch.float16), 0, route))
    return tuple(route)


def _check(pixels, c_in, c_out, dtype):
    import nestedtensor_amd as nt
    from nestedtensor_amd import _C
    assert _C.lib.nt_conv1x1_supported(c_in, c_out, _C.dtype_code(dtype))
    g = torch.Generator("cuda").manual_seed(c_in + c_out)
    maps = [torch.randn(c_in, 1, n, device=DEV, generator=g).to(dtype) for n in pixels]
    w = (torch.randn(c_out, c_in, 1, 1, device=DEV, generator=g) * c_in ** -0.5).to(dtype)
    got = torch.conv2d(nt.nested_tensor(maps, dtype=dtype, device=DEV), w)
    # one rounding to the type, and fp32 sums of c_in products
    unit = 2.0 ** (-11 if dtype == torch.float16 else -8)
    a = w.double().reshape(c_out, c_in)
    for m, y in zip(maps, got.unbind()):
        b = m.double().reshape(c_in, -1)
        exact, size = a @ b, a.abs() @ b.abs()
        err = (y.double().reshape(c_out, -1) - exact).abs()
        assert bool((err <= unit * exact.abs() + c_in * 2.0 ** -23 * size + 2.0 ** -24).all())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("c_in,c_out", [(16, 32), (32, 128), (64, 256), (80, 96), (96, 512), (128, 64), (128, 384)])
def test_conv1x1_small_batches(c_in, c_out, dtype):
    _check(EDGES, c_in, c_out, dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("c_in,c_out,pixels", [
    (64, 256, 131072 - 200), (64, 256, 131072 + 200),        # 64 MiB of result
    (48, 128, 270001), (96, 256, 131072 + 200),              # whole lines
    (112, 128, 270001), (96, 64, 540001),                    # too many channels for those
    (128, 256, 1024 * 64 - 2000), (128, 256, 1024 * 64 + 200)])   # two wavefronts per window and one
def test_conv1x1_large_batches(c_in, c_out, pixels, dtype):
    _check(EDGES + [pixels] + EDGES, c_in, c_out, dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("c_in,c_out,pixels,waves", [
    (16, 32, 1100001, 8), (32, 96, 360001, 8), (48, 512, 70001, 8),
    (64, 224, 160001, 7), (64, 384, 90001, 6), (80, 192, 180001, 6), (64, 512, 70001, 4), (96, 256, 140001, 4),
    (80, 480, 75001, 2), (96, 512, 70001, 2)])
def test_conv1x1_whole_lines(c_in, c_out, pixels, waves, dtype):
    """Every number of wavefronts that the LDS leaves room for, and every depth of the loads."""
    pixels = [7, 192, 255, 256, 257, 1001] + EDGES + [pixels] + EDGES
    assert _route(pixels, c_in, c_out) == (waves, 0)
    _check(pixels, c_in, c_out, dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("c_in,c_out", [(128, 384), (128, 512), (112, 448)])
@pytest.mark.parametrize("large", [0, 200001])
def test_conv1x1_weight_fills_the_lds(c_in, c_out, large, dtype):
    """Weights beside which the pixels of the other kernel find no room."""
    pixels = EDGES + [large] * (large > 0)
    assert _route(pixels, c_in, c_out)[0] == 0
    _check(pixels, c_in, c_out, dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("c_in,c_out,pixels,parts", [
    (16, 128, 20001, 4), (128, 512, 20001, 4), (48, 96, 40001, 2), (64, 32, 40001, 2), (128, 32, 190001, 2), (96, 96, 540001, 2),
    (16, 32, 100001, 1), (32, 160, 100001, 1), (128, 512, 100001, 1), (64, 64, 250001, 1), (48, 32, 250001, 1), (112, 32, 600001, 1)])
def test_conv1x1_wavefronts_of_a_window(c_in, c_out, pixels, parts, dtype):
    pixels = EDGES + [pixels] + EDGES
    assert _route(pixels, c_in, c_out) == (0, parts)
    _check(pixels, c_in, c_out, dtype)
