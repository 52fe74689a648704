"""Which kernel a 1x1 convolution runs on, for 256 compute units: host logic, no GPU."""
import ctypes

import pytest
import torch

from nestedtensor_amd import _C

F16 = _C.dtype_code(torch.float16)


def _route(c_in, c_out, windows, images=8):
    route = (ctypes.c_int * 2)()
    _C.check(_C.lib.nt_conv1x1_route(images, windows + images, c_in, c_out, F16, 256, route))
    return tuple(route)


@pytest.mark.parametrize("c_in", range(16, 129, 16))
def test_every_supported_pair_has_a_kernel_at_every_size(c_in):
    for c_out in range(32, 513, 32):
        assert _C.lib.nt_conv1x1_supported(c_in, c_out, F16)
        for windows in (1, 100, 512, 513, 1024, 1025, 2048, 2049, 5000, 8193, 10 ** 6):
            waves, parts = _route(c_in, c_out, windows)
            assert (waves == 0) != (parts == 0)
            if parts:
                assert c_out * (c_in + 8) * 2 <= 160 * 1024 and c_out // 32 >= parts // 2


@pytest.mark.parametrize("c_in,c_out", [(8, 32), (24, 64), (144, 64), (64, 40), (64, 544)])
def test_other_depths_are_refused(c_in, c_out):
    assert not _C.lib.nt_conv1x1_supported(c_in, c_out, F16)
    assert _C.lib.nt_conv1x1_route(1, 2, c_in, c_out, F16, 256, (ctypes.c_int * 2)()) != 0


@pytest.mark.parametrize("c_in,c_out,windows,route", [
    # one round of 2048 wavefronts: four, two or one to a window
    (64, 256, 512, (0, 4)), (64, 256, 513, (0, 2)), (64, 256, 1024, (0, 2)), (64, 256, 1025, (0, 1)), (64, 96, 512, (0, 2)),
    (64, 64, 2048, (0, 1)), (128, 512, 600, (0, 2)), (128, 512, 2048, (0, 1)),
    # beyond: two in three half rounds, or for many input channels
    (64, 64, 2049, (0, 2)), (64, 64, 3072, (0, 2)), (64, 64, 3073, (0, 1)), (128, 64, 3073, (0, 2)), (128, 64, 20000, (0, 2)),
    # 32 output channels
    (32, 32, 1024, (0, 2)), (32, 32, 1025, (0, 1)), (32, 32, 2049, (0, 1)), (64, 32, 2049, (0, 2)), (64, 32, 3073, (0, 1)),
    (96, 32, 8192, (0, 2)), (96, 32, 8193, (0, 1)), (32, 32, 14000, (0, 1)),
    # few channels go to whole lines before the result is large
    (16, 32, 6144, (0, 1)), (16, 32, 6145, (8, 0)), (16, 64, 4096, (0, 1)), (16, 64, 4097, (8, 0)), (32, 96, 4096, (0, 1)),
    (32, 96, 4097, (8, 0)), (48, 64, 4097, (0, 1)),
    (64, 256, 2048, (0, 1)), (64, 256, 2049, (7, 0))])
def test_wavefronts_of_a_window(c_in, c_out, windows, route):
    assert _route(c_in, c_out, windows) == route
