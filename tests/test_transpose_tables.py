"""Host tables of ragged transposes and 1x1 convolutions against the tensor expressions
that define them, over every mode, element size and awkward extent (no GPU needed)."""
import random

import pytest
import torch

from nestedtensor_amd import _C, ops

CPU = torch.device("cpu")


def _expected(rows, cols, elem_bytes):
    B = rows.numel()
    tr, tc = ops._transpose_tile(int(rows.max()) if B else 0, int(cols.max()) if B else 0, elem_bytes)
    if (tr, tc) == (64, 64) and elem_bytes == 2 and bool((rows % 64 != 0).any()):
        tr = tc = 0
        tiles = torch.where((rows > 0) & (cols > 0), ((rows + 63) // 64 + 1) * ((cols + 63) // 64),
                            torch.zeros_like(rows))
    else:
        tiles = ((rows + tr - 1) // tr) * ((cols + tc - 1) // tc)
    table = torch.zeros((4, B + 1), dtype=torch.int64)
    table[0, :B], table[1, :B] = rows, cols
    table[2, 1:], table[3, 1:] = torch.cumsum(tiles, 0), torch.cumsum(rows * cols, 0)
    return table, int(table[2, B]), tr, tc


def _sizes(rng):
    c = rng.choice([0, 1, 3, 16, 17, 64, 65])
    B = rng.choice([0, 1, 2, 5, 12])
    return torch.tensor([[c, rng.choice([0, 1, 8, 33]), rng.choice([1, 2, 8, 64])] for _ in range(B)],
                        dtype=torch.int64).reshape(B, 3)


@pytest.mark.parametrize("strided", [False, True])
def test_transpose_and_conv_tables(strided):
    rng = random.Random(7)
    for _ in range(200):
        chw = _sizes(rng)
        hwc = chw[:, [1, 2, 0]].contiguous()
        spatial = chw[:, 1] * chw[:, 2]
        cases = [(ops._NCHW_TO_NHWC, chw, chw[:, 0], spatial, hwc), (ops._NHWC_TO_NCHW, hwc, spatial, chw[:, 0], chw),
                 (ops._CHANNELS_LAST_TO_ROW_MAJOR, chw, spatial, chw[:, 0], chw)]
        for mode, given, rows, cols, result in cases:
            if strided:
                given = given.t().contiguous().t()
            for elem_bytes in (1, 2, 4, 8):
                table, sizes, tiles, tr, tc = ops._transpose_tables(given, mode, elem_bytes, CPU)
                exp, exp_tiles, exp_tr, exp_tc = _expected(rows, cols, elem_bytes)
                assert torch.equal(table, exp) and torch.equal(sizes, result)
                assert (tiles, tr, tc) == (exp_tiles, exp_tr, exp_tc)
        tile = int(_C.lib.nt_conv1x1_tile_pixels())
        table, tiles, pixels = ops._conv1x1_tables(chw, CPU)
        exp = torch.zeros((2, chw.size(0) + 1), dtype=torch.int64)
        exp[0, 1:] = torch.cumsum(spatial, 0)
        exp[1, 1:] = torch.cumsum(torch.where(spatial > 0, (spatial + tile - 1) // tile + 1, spatial), 0)
        assert torch.equal(table, exp) and (tiles, pixels) == (int(exp[1, -1]), int(exp[0, -1]))
        grown = ops._sizes_with_extent(chw, 1, 9)
        assert grown.is_contiguous() and grown.data_ptr() != chw.data_ptr() or chw.numel() == 0
        assert torch.equal(grown[:, [0, 2]], chw[:, [0, 2]]) and bool((grown[:, 1] == 9).all())
