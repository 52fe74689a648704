"""fp32 projections on the bf16 matrix instruction: every tile shape with row, column and
step remainders, operand rows that lie anywhere, and what the split cannot carry
(infinities, NaN, magnitudes next to the largest and the smallest fp32 numbers)."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)


def _tile(M, N, K):
    from nestedtensor_amd import _C
    tile = (ctypes.c_int * 3)()
    _C.check(_C.lib.nt_linear_tile(M, N, K, K, N, -1, _C.dtype_code(torch.float32), 0, tile))
    return tuple(tile)


def _case(M, N, K, seed=0):
    g = torch.Generator("cuda").manual_seed(M + 3 * N + 7 * K + seed)
    x = torch.randn(M, K, device=DEV, generator=g)
    w = torch.randn(N, K, device=DEV, generator=g) * 0.25
    b = torch.randn(N, device=DEV, generator=g)
    return x, w, b


def _bound(x, w, ref):
    # Were the sums of an instruction cut off, not rounded, after every four k: K / 4 units of
    # 2^-23 of partial sums below sum |x||w| for the first parts, 7 K / 4 of them at 2^-7 of it
    # for the other products (0.53 K roundings of 2^-24 in all), 2^-34 per k for the product left
    # out; the two sums added, the bias and the store; twice half the smallest fp32 number
    return (x.double().abs() @ w.double().abs().t()) * ((0.55 * x.size(1) + 4) * 2.0 ** -24) + ref.abs() * 2.0 ** -24 + 2.0 ** -148


@pytest.mark.parametrize("M,N,K,tile", [
    (1, 1, 192, (64, 128, -1)), (3, 130, 192, (64, 128, -1)), (64, 129, 208, (64, 128, -1)),
    (1000, 300, 224, (64, 128, -1)), (500, 2050, 2064, (128, 64, -1)), (60001, 33, 192, (128, 64, -1)),
    (2000, 1536, 512, (128, 128, -1)), (2001, 1537, 528, (128, 128, -1)), (129, 12000, 208, (128, 128, -1)),
    (8040, 768, 768, (192, 128, -1)), (40000, 128, 208, (192, 128, -1)),
    (20001, 1026, 208, (256, 128, -1)), (16001, 1024, 208, (256, 128, -1)), (16001, 1022, 240, (256, 128, -1)),
    (16001, 1025, 1040, (320, 128, -1)), (8040, 2304, 768, (320, 128, -1)), (8167, 2300, 304, (320, 128, -1)),
])
def test_linear_split_shapes(M, N, K, tile):
    from nestedtensor_amd import ops
    assert _tile(M, N, K)[2] == -1 and (tile is None or _tile(M, N, K) == tile)
    x, w, b = _case(M, N, K)
    ref = x.double() @ w.double().t() + b.double()
    bound = _bound(x, w, ref)
    assert bool(((ops.linear(x, w, b).double() - ref).abs() <= bound).all())
    assert bool(((ops.linear(x, w, b, "relu").double() - ref.clamp_min(0)).abs() <= bound).all())
    gelu = 0.5 * ref * torch.special.erfc(-ref * 0.5 ** 0.5)
    assert bool(((ops.linear(x, w, b, "gelu").double() - gelu).abs() <= 1.13 * bound + 4e-7).all())


def test_linear_split_is_chosen_by_depth():
    assert _tile(8040, 768, 192)[2] == -1 and _tile(8040, 768, 176)[2] != -1 and _tile(8040, 768, 200)[2] != -1


@pytest.mark.parametrize("M,N,K,lda,shift", [(300, 200, 192, 201, 1), (700, 64, 208, 1000, 3), (129, 333, 256, 257, 0)])
def test_linear_split_unaligned_rows(M, N, K, lda, shift):
    from nestedtensor_amd import _C
    x, w, b = _case(M, N, K)
    held = torch.full((M * lda + 4,), float("nan"), device=DEV)
    rows = held[shift:shift + M * lda].view(M, lda)
    rows[:, :K] = x
    out = torch.full((M, N + 3), 7.0, device=DEV)
    _C.check(_C.lib.nt_linear(_C.ptr(rows), lda, _C.ptr(w), _C.ptr(b), _C.ptr(out), N + 3, M, N, K,
                              _C.dtype_code(torch.float32), _C.current_stream(DEV)))
    ref = x.double() @ w.double().t() + b.double()
    assert bool(((out[:, :N].double() - ref).abs() <= _bound(x, w, ref)).all())
    assert bool((out[:, N:] == 7.0).all())


@pytest.mark.parametrize("M,N,K", [(5, 7, 192), (300, 200, 256), (2001, 1537, 224), (8040, 2304, 208)])
def test_linear_split_special_values(M, N, K):
    from nestedtensor_amd import ops
    inf, big = float("inf"), torch.finfo(torch.float32).max
    x, w, b = _case(M, N, K)
    for i, v in enumerate((inf, -inf, float("nan"), big, -big)):
        x[(3 * i) % M, (5 * i) % K] = v
    w[N - 1, 3] = inf
    w[N // 2, :] = 0.0                                   # infinity times zero
    ref = x.double() @ w.double().t() + b.double()
    y = ops.linear(x, w, b)
    assert torch.equal(torch.isnan(y), torch.isnan(ref))
    over = ref.abs() > big                               # infinities and what 32 bits cannot hold
    near = over & (ref.abs() < 2.0 * big)                # a partial sum may or may not have overflowed
    assert torch.equal(y[over & ~near], ref[over & ~near].float())
    fine = ~over & ~torch.isnan(ref) & (ref.abs() < 0.5 * big)
    bound = _bound(torch.nan_to_num(x, 0.0, 0.0, 0.0), torch.nan_to_num(w, 0.0, 0.0, 0.0), ref)
    assert bool(((y.double() - ref).abs()[fine] <= bound[fine]).all())


@pytest.mark.parametrize("M,N,K", [(5, 7, 192), (300, 200, 256), (2001, 1537, 224)])
@pytest.mark.parametrize("ex,ew", [
    (-118, 100), (90, -120), (-60, -40), (-100, 0), (0, -101),
    (-128, 100), (-134, 100), (-140, 105), (-147, 105), (105, -140), (-1, -130),      # denormal operands
    (-66, -64), (-70, -75),                                                            # denormal results
    (60, 50), (107, -10), (113, -20), (-20, 124)])                                     # results or operands too large to split
def test_linear_split_magnitudes(M, N, K, ex, ew):
    from nestedtensor_amd import ops
    x, w, _ = _case(M, N, K)
    xs, ws = torch.ldexp(x, torch.tensor(ex, device=DEV)), torch.ldexp(w, torch.tensor(ew, device=DEV))
    xs, ws = xs.nan_to_num(posinf=0.0, neginf=0.0), ws.nan_to_num(posinf=0.0, neginf=0.0)
    ref = xs.double() @ ws.double().t()
    y = ops.linear(xs, ws, None).double()
    # (a result that fp32 recomputes: one rounding per k of partial sums)
    bound = _bound(xs, ws, ref) if ex + ew < 80 and max(ex, ew) < 108 else \
        xs.double().abs() @ ws.double().abs().t() * ((K + 2) * 2.0 ** -24) + 2.0 ** -148
    assert bool(((y - ref).abs() <= bound).all())


def test_linear_split_mixed_magnitudes():
    """One operand below the smallest bf16 number among ordinary ones is not taken for zero."""
    from nestedtensor_amd import ops
    x, w, _ = _case(300, 200, 256)
    x[17, 9] = 2.0 ** -140
    x[17, 10:] = 0.0
    x[17, :9] = 0.0
    w[:, 9] = torch.ldexp(w[:, 9], torch.tensor(100, device=DEV))
    ref = x.double() @ w.double().t()
    y = ops.linear(x, w, None).double()
    assert bool(((y - ref).abs() <= _bound(x, w, ref)).all())
    assert bool((y[17] != 0).all())


@pytest.mark.parametrize("M,N,K", [(4000, 512, 256), (4000, 768, 768), (2000, 1024, 1024)])
def test_linear_split_precision(M, N, K):
    """No further from 64 bits than a chain of fp32 multiply-adds, one rounding per k."""
    from nestedtensor_amd import ops
    x, w, b = _case(M, N, K)
    ref = x.double() @ w.double().t() + b.double()
    acc = torch.zeros(M, N, device=DEV)
    for k in range(K):
        acc = (acc.double() + x[:, k:k + 1].double() * w[:, k].double()).float()
    chain = ((acc + b).double() - ref).norm()
    assert (ops.linear(x, w, b).double() - ref).norm() <= chain


def _chain(x, w):
    """fp32 multiply-adds, one rounding per product."""
    acc = torch.zeros(x.size(0), w.size(0), device=DEV)
    for k in range(x.size(1)):
        acc = (acc.double() + x[:, k:k + 1].double() * w[:, k].double()).float()
    return acc


@pytest.mark.parametrize("steps", [1, 2, 4, 16, 48])
@pytest.mark.parametrize("positive", [False, True])
@pytest.mark.parametrize("M,N", [(9000, 1030), (200, 100)])
def test_linear_split_one_product_per_step(M, N, steps, positive):
    """Sums of few products, one in 16 k, are no less precise than chains of fp32 multiply-adds.
    (1.01: seven roundings of products below 2^-7 of the largest add sqrt(7) 2^-7 of one
    rounding, in quadrature; the product left out is below 2^-34.)"""
    from nestedtensor_amd import ops
    K = 16 * max(steps, 12)
    g = torch.Generator("cuda").manual_seed(steps)
    at = torch.randint(0, 16, (M, steps), device=DEV, generator=g) + 16 * torch.arange(steps, device=DEV)
    x = torch.zeros(M, K, device=DEV).scatter_(1, at, torch.randn(M, steps, device=DEV, generator=g))
    w = torch.randn(N, K, device=DEV, generator=g)
    if positive:
        x, w = x.abs(), w.abs()
    assert _tile(M, N, K)[2] == -1
    ref = x.double() @ w.double().t()
    err, chain = ((t.double() - ref).norm() for t in (ops.linear(x, w, None), _chain(x, w)))
    assert err <= 1.01 * chain


def test_linear_split_largest_rests():
    """1 + 2^-8 - 2^-17: the second and third parts are as large as they can be."""
    from nestedtensor_amd import ops
    v = 1 + 2.0 ** -8 - 2.0 ** -17
    x, w = torch.zeros(300, 768, device=DEV), torch.full((256, 768), v, device=DEV)
    x[:, 5] = v
    assert torch.equal(ops.linear(x, w, None), (x.double() @ w.double().t()).float())
    x.fill_(v)
    y = ops.linear(x, w, None)
    # 48 steps of exact sums, one rounding each
    assert bool(((y.double() - 768 * v * v).abs() <= 48 * 2.0 ** -24 * 768 * v * v).all())
