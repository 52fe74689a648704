"""Row-major 1x1 convolution of small batches where its tiles meet the ends of an image: pixel counts
around one, two and three 64-pixel windows.  (The kernel that writes whole lines, for large
results, is run on such images by test_gpu_conv1x1_routes.py.)"""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)
PIXELS = [1, 2, 7, 63, 64, 65, 127, 128, 129, 191, 192, 193, 255, 256, 257, 640, 1001]


@pytest.mark.parametrize("c_in,c_out", [(16, 32), (48, 64), (64, 96), (112, 32)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_conv1x1_window_edges(c_in, c_out, dtype):
    import nestedtensor_amd as nt
    from nestedtensor_amd import _C
    assert _C.lib.nt_conv1x1_supported(c_in, c_out, _C.dtype_code(dtype))
    g = torch.Generator().manual_seed(c_in + c_out)
    maps = [torch.randn(c_in, 1, n, generator=g).to(dtype) for n in PIXELS]
    w = (torch.randn(c_out, c_in, 1, 1, generator=g) * c_in ** -0.5).to(dtype)
    got = torch.conv2d(nt.nested_tensor(maps, dtype=dtype, device=DEV), w.to(DEV))
    # one rounding to the type, and fp32 sums of c_in products
    unit = 2.0 ** (-11 if dtype == torch.float16 else -8)
    for m, y in zip(maps, got.unbind()):
        a, b = w.double().reshape(c_out, c_in), m.double().reshape(c_in, -1)
        exact, size = a @ b, a.abs() @ b.abs()
        err = (y.cpu().double().reshape(c_out, -1) - exact).abs()
        assert bool((err <= unit * exact.abs() + c_in * 2.0 ** -23 * size + 2.0 ** -24).all())
