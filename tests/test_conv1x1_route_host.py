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
