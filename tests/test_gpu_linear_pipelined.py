"""The pipelined projection kernel: every tile shape its launcher can pick, with row and
column remainders and with fewer, as many and more K tiles than its LDS ring holds."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)


def _bound(x, w, ref, dtype):
    # fp32 accumulation of K products (K roundings of partial sums below sum |x||w|),
    # the bias, and one rounding of the result to the storage type
    unit = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8, torch.float32: 2.0 ** -24}[dtype]
    return (x.abs() @ w.abs().t()) * (x.size(1) * 2.0 ** -24) + ref.abs() * unit + 1e-6


def _tile(M, N, K, dtype, n_split=-1):
    """(rows, columns, K tiles in flight; 0: not the pipelined kernel) that the launcher picks."""
    from nestedtensor_amd import _C
    tile = (ctypes.c_int * 3)()
    _C.check(_C.lib.nt_linear_tile(M, N, K, K, N if n_split < 0 else n_split, n_split, _C.dtype_code(dtype), 0, tile))
    return tuple(tile)


def _case(M, N, K, dtype):
    g = torch.Generator("cuda").manual_seed(M + 3 * N + 7 * K)
    x = torch.randn(M, K, device=DEV, generator=g).to(dtype)
    w = (torch.randn(N, K, device=DEV, generator=g) * 0.25).to(dtype)
    b = torch.randn(N, device=DEV, generator=g).to(dtype)
    ref = x.double() @ w.double().t() + b.double()
    return x, w, b, ref, _bound(x.double(), w.double(), ref, dtype)


@pytest.mark.parametrize("dtype,M,N,K,tile", [
    (torch.float16, 10843, 264, 256, (128, 128, 4)),    # as many K tiles as the ring holds
    (torch.bfloat16, 10843, 264, 448, (128, 128, 4)),   # seven K tiles
    (torch.float16, 10843, 264, 192, (192, 128, 3)),
    (torch.bfloat16, 10940, 264, 320, (192, 128, 3)),
    (torch.float16, 32938, 264, 192, (256, 128, 3)),
    (torch.bfloat16, 18980, 264, 448, (256, 128, 3)),
    (torch.float16, 21971, 264, 128, (320, 128, 2)),
    (torch.bfloat16, 21971, 264, 192, (320, 128, 2)),
    (torch.float16, 3665, 1100, 192, (128, 256, 3)),
    (torch.bfloat16, 3859, 1100, 448, (128, 256, 3)),
    (torch.float16, 7254, 1100, 128, (192, 256, 2)),
    (torch.bfloat16, 7254, 1100, 320, (192, 256, 2)),
    (torch.float16, 6963, 1544, 128, (256, 256, 2)),
    (torch.bfloat16, 27953, 264, 448, (256, 256, 2)),
    (torch.float16, 32938, 264, 128, (320, 256, 2)),
    (torch.bfloat16, 26956, 520, 192, (320, 256, 2)),
    (torch.float16, 10754, 300, 128, (256, 128, 0)),    # rows that end inside a 16-byte piece
    (torch.bfloat16, 24962, 300, 128, (256, 192, 0)),
    (torch.float16, 52878, 200, 128, (256, 256, 0)),    # few columns, two K tiles
    (torch.float32, 300, 520, 160, (128, 128, 4)),
    (torch.float32, 6001, 768, 128, (192, 128, 3)),
    (torch.float32, 6001, 768, 64, (256, 128, 0)),      # two K tiles and one round of tiles
    (torch.float32, 20000, 520, 64, (256, 256, 2)),
    # remainders and depths on whatever is picked
    (torch.float16, 6430, 520, 256, None), (torch.bfloat16, 6430, 520, 448, None), (torch.float16, 6536, 520, 192, None),
    (torch.bfloat16, 6536, 520, 320, None), (torch.float16, 9822, 520, 192, None), (torch.float16, 9822, 520, 320, None),
    (torch.float16, 7172, 1100, 192, None), (torch.bfloat16, 6430, 520, 128, None), (torch.float16, 8073, 768, 192, None),
    (torch.float16, 8073, 768, 448, None), (torch.bfloat16, 8974, 1100, 128, None), (torch.float16, 8974, 1100, 320, None),
    (torch.float16, 9822, 1100, 128, None), (torch.bfloat16, 9822, 1100, 448, None), (torch.float16, 7172, 2304, 128, None),
    (torch.bfloat16, 7172, 2304, 256, None),
])
def test_linear_pipelined_shapes(dtype, M, N, K, tile):
    from nestedtensor_amd import ops
    assert tile is None or _tile(M, N, K, dtype) == tile
    x, w, b, ref, bound = _case(M, N, K, dtype)
    assert bool(((ops.linear(x, w, b).double() - ref).abs() <= bound).all())
    relu = ops.linear(x, w, b, "relu").double()
    assert bool(((relu - ref.clamp_min(0)).abs() <= bound).all())
    # the slope of gelu is at most 1.13, its error 4e-7 in fp32 before the one rounding
    gelu = 0.5 * ref * torch.special.erfc(-ref * 0.5 ** 0.5)
    assert bool(((ops.linear(x, w, b, "gelu").double() - gelu).abs() <= 1.13 * bound + 4e-7).all())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,E,tile", [
    (4121, 640, (320, 128, 2)),
    (2690, 512, (192, 128, 3)),
    (2054, 640, (128, 128, 4)),
    (9845, 384, (256, 256, 2)),
    (4068, 512, (128, 256, 3)),
    (5128, 640, (192, 256, 2)),
    (3273, 640, (256, 128, 3)),
    (8202, 640, (320, 256, 2)),
    (10799, 128, (256, 128, 0)),    # two K tiles, a boundary between K and V at a multiple of 128
    (10781, 128, None), (5423, 256, None), (2561, 512, None), (8073, 512, None), (4045, 512, None), (5479, 512, None),
    (3305, 640, None), (10779, 512, None),
])
def test_linear_qkv_pipelined_shapes(M, E, tile, dtype):
    from nestedtensor_amd import _C
    assert tile is None or _tile(M, 3 * E, E, dtype, 2 * E) == tile
    x, w, b, ref, bound = _case(M, 3 * E, E, dtype)
    ld = (M + 72 + 7) // 8 * 8
    qk = torch.empty(M, 2 * E, dtype=dtype, device=DEV)
    vt = torch.full((E, ld), 7.0, dtype=dtype, device=DEV)
    _C.check(_C.lib.nt_linear_qkv(_C.ptr(x), E, _C.ptr(w), _C.ptr(b), _C.ptr(qk), 2 * E, _C.ptr(vt), ld, M, E, E,
                                  _C.dtype_code(dtype), _C.current_stream(DEV)))
    assert bool(((qk.double() - ref[:, :2 * E]).abs() <= bound[:, :2 * E]).all())
    assert bool(((vt[:, :M].double() - ref[:, 2 * E:].t()).abs() <= bound[:, 2 * E:].t()).all())
    assert bool((vt[:, M:] == 7.0).all())          # nothing is written past the last token


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K,tile", [
    (40001, 64, 128, (128, 64, 0)), (40001, 65, 128, (256, 128, 0)), (33000, 33, 64, (128, 64, 0)),
    (70003, 8, 72, (128, 64, 0)), (16385, 64, 8, (128, 64, 0)),
    (33001, 64, 2048, (128, 64, 0)), (33001, 64, 2112, (192, 128, 3)), (33001, 64, 2056, (128, 64, 0))])
def test_linear_few_columns(M, N, K, tile, dtype):
    from nestedtensor_amd import ops
    assert _tile(M, N, K, dtype) == tile
    x, w, b, ref, bound = _case(M, N, K, dtype)
    assert bool(((ops.linear(x, w, b).double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K,tile", [
    (33000, 200, 72, (256, 256, 0)),     # K of no whole tile
    (33000, 480, 480, (256, 192, 0)),
    (20000, 190, 488, (256, 128, 0)),
    (9000, 300, 104, (128, 128, 0)),
])
def test_linear_ragged_depth(M, N, K, tile, dtype):
    from nestedtensor_amd import ops
    assert _tile(M, N, K, dtype) == tile
    x, w, b, ref, bound = _case(M, N, K, dtype)
    assert bool(((ops.linear(x, w, b).double() - ref).abs() <= bound).all())
