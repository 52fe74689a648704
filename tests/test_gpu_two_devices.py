"""Kernels that need more dynamic LDS than a launch has by default, first on one device and then on
another of the same process: the allowance is each device's own."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,E,conv", [(torch.float32, 256, None), (torch.float16, 256, (96, 512)), (torch.float16, 64, (16, 32))])
def test_large_lds_on_each_device(dtype, E, conv):
    if torch.cuda.device_count() < 2:
        pytest.skip("needs two devices")
    import nestedtensor_amd as nt
    g = torch.Generator().manual_seed(E)
    tokens = [torch.randn(n, E, generator=g).to(dtype) for n in (300, 7, 600)]
    weights = [(torch.randn(s, generator=g) * 0.05).to(dtype) for s in ((3 * E, E), (3 * E,), (E, E), (E,))]
    maps = [torch.randn(conv[0], 9, n, generator=g).to(dtype) for n in (70, 3)] if conv else []
    kernel = torch.randn(*conv[::-1], 1, 1, generator=g).to(dtype) if conv else None
    results = []
    for dev in ("cuda:0", "cuda:1"):
        x = nt.nested_tensor(tokens, dtype=dtype, device=dev)
        w_in, b_in, w_out, b_out = (w.to(dev) for w in weights)
        y = [torch.ops.nestedtensor.min_mha(E // 64, 64, 0.0, False, x, x, x, w_in, b_in, 0.125, w_out, b_out)]
        if conv:
            y.append(torch.conv2d(nt.nested_tensor(maps, dtype=dtype, device=dev), kernel.to(dev)))
        results.append([t._impl.buffer.cpu() for t in y])
    for a, b in zip(*results):
        assert torch.equal(a, b)
