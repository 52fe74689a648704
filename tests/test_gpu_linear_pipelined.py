"""The pipelined projection kernel: every tile shape its launcher can pick, with row and
column remainders and with fewer, as many and more K tiles than its LDS ring holds."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)


def _bound(x, w, ref, dtype):
    # fp32 accumulation of K products (K roundings of partial sums below sum |x||w|),
    # the bias, and one rounding of the result to the storage type
    unit = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8, torch.float32: 2.0 ** -24}[dtype]
    return (x.abs() @ w.abs().t()) * (x.size(1) * 2.0 ** -24) + ref.abs() * unit + 1e-6


def _case(M, N, K, dtype):
    g = torch.Generator("cuda").manual_seed(M + 3 * N + 7 * K)
    x = torch.randn(M, K, device=DEV, generator=g).to(dtype)
    w = (torch.randn(N, K, device=DEV, generator=g) * 0.25).to(dtype)
    b = torch.randn(N, device=DEV, generator=g).to(dtype)
    ref = x.double() @ w.double().t() + b.double()
    return x, w, b, ref, _bound(x.double(), w.double(), ref, dtype)


@pytest.mark.parametrize("dtype,M,N,K", [
    (torch.float16, 6430, 520, 256),    # 128 x 128, ring of four, as many K tiles
    (torch.bfloat16, 6430, 520, 448),   # ... seven K tiles
    (torch.float16, 6536, 520, 192),    # 192 x 128, ring of three
    (torch.bfloat16, 6536, 520, 320),
    (torch.float16, 9822, 520, 192),    # 256 x 128, ring of three
    (torch.float16, 9822, 520, 320),
    (torch.float16, 7172, 1100, 192),   # 320 x 128, ring of two
    (torch.bfloat16, 6430, 520, 128),   # ... two K tiles
    (torch.float16, 8073, 768, 192),    # 128 x 256, ring of three
    (torch.float16, 8073, 768, 448),
    (torch.bfloat16, 8974, 1100, 128),  # 192 x 256, ring of two
    (torch.float16, 8974, 1100, 320),
    (torch.float16, 9822, 1100, 128),   # 256 x 256
    (torch.bfloat16, 9822, 1100, 448),
    (torch.float16, 7172, 2304, 128),   # 320 x 256
    (torch.bfloat16, 7172, 2304, 256),
    (torch.float32, 300, 520, 160),     # fp32: 128 x 128
    (torch.float32, 6001, 768, 128),    # 192 x 128
])
def test_linear_pipelined_shapes(dtype, M, N, K):
    from nestedtensor_amd import ops
    x, w, b, ref, bound = _case(M, N, K, dtype)
    assert bool(((ops.linear(x, w, b).double() - ref).abs() <= bound).all())
    relu = ops.linear(x, w, b, "relu").double()
    assert bool(((relu - ref.clamp_min(0)).abs() <= bound).all())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,E", [
    (10781, 128),   # 320 x 128 tiles, two K tiles
    (5423, 256),    # 192 x 128
    (2561, 512),    # 128 x 128
    (8073, 512),    # 256 x 256
    (4045, 512),    # 128 x 256
    (5479, 512),    # 192 x 256
    (3305, 640),    # 256 x 128, a boundary between K and V at a multiple of 128
    (10779, 512),   # 320 x 256
])
def test_linear_qkv_pipelined_shapes(M, E, dtype):
    from nestedtensor_amd import _C
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
@pytest.mark.parametrize("M,N,K", [(40001, 64, 128), (40001, 65, 128), (33000, 33, 64), (70003, 8, 72), (16385, 64, 8)])
def test_linear_few_columns(M, N, K, dtype):
    from nestedtensor_amd import ops
    x, w, b, ref, bound = _case(M, N, K, dtype)
    assert bool(((ops.linear(x, w, b).double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K", [
    (33000, 200, 72),     # K of no whole tile: 256 x 256
    (20000, 190, 488),    # 256 x 192
    (33000, 480, 480),
    (9000, 300, 104),     # 256 x 128
])
def test_linear_ragged_depth(M, N, K, dtype):
    from nestedtensor_amd import ops
    x, w, b, ref, bound = _case(M, N, K, dtype)
    assert bool(((ops.linear(x, w, b).double() - ref).abs() <= bound).all())
