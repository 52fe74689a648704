"""fp32 attention on the bf16 matrix instruction: key and query remainders of its 32-key and
32-query blocks for every head_dim, and what the split of an operand cannot carry."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)
F32 = 0


def _run(q_lens, k_lens, H, hd, qkv=None, scale=None, seed=0):
    """Outputs of both entry points, and Q, K, V in 64 bits per sequence and head."""
    from nestedtensor_amd import _C
    B, E = len(q_lens), H * hd
    g = torch.Generator("cuda").manual_seed(seed + hd)
    Tq, Tk = sum(q_lens), sum(k_lens)
    q = torch.randn(Tq, E, device=DEV, generator=g)
    kv = torch.randn(max(Tk, 1), 2 * E + 4, device=DEV, generator=g)     # rows of K and V in one buffer
    k, v = kv[:, :E], kv[:, E:2 * E]
    if qkv is not None:
        qkv(q, k, v)
    scale = hd ** -0.5 if scale is None else scale
    stream = _C.current_stream(DEV)
    ql, kl = (ctypes.c_int64 * B)(*q_lens), (ctypes.c_int64 * B)(*k_lens)
    n = int(_C.lib.nt_attention_schedule_items(ql, B, 128))
    work = torch.empty(8 * n, dtype=torch.int32, device=DEV)
    _C.check(_C.lib.nt_attention_schedule(ql, kl, B, 128, _C.ptr(work), n, stream))
    off = [torch.tensor([0] + list(l)).cumsum(0).to(DEV) for l in (q_lens, k_lens)]
    ld = kv.stride(0)
    listed, padded = torch.full((Tq, E), 7.0, device=DEV), torch.full((Tq, E), 7.0, device=DEV)
    _C.check(_C.lib.nt_varlen_attention_scheduled(_C.ptr(q), E, _C.ptr(k), ld, _C.ptr(v), ld, _C.ptr(listed), E,
                                                  _C.ptr(work), n, H, hd, ctypes.c_float(scale), F32, stream))
    _C.check(_C.lib.nt_varlen_attention(_C.ptr(q), E, _C.ptr(k), ld, _C.ptr(v), ld, _C.ptr(padded), E, _C.ptr(off[0]),
                                        _C.ptr(off[1]), B, H, hd, max(q_lens), ctypes.c_float(scale), F32, stream))
    assert torch.equal(listed.view(torch.int32), padded.view(torch.int32))
    return listed, _reference(q, k, v, off, H, hd, scale)


def _reference(q, k, v, off, H, hd, scale):
    out, mag = torch.zeros_like(q, dtype=torch.float64), torch.zeros_like(q, dtype=torch.float64)
    for b in range(len(off[0]) - 1):
        sq = slice(int(off[0][b]), int(off[0][b + 1]))
        sk = slice(int(off[1][b]), int(off[1][b + 1]))
        if sk.start == sk.stop:
            continue
        qh, kh, vh = (t.double().reshape(-1, H, hd).transpose(0, 1).contiguous() for t in (q[sq], k[sk], v[sk]))
        s = torch.matmul(qh, kh.transpose(1, 2).contiguous()) * scale
        s_abs = torch.matmul(qh.abs(), kh.abs().transpose(1, 2).contiguous()) * abs(scale)
        p = torch.softmax(s, -1)
        out[sq] = torch.matmul(p, vh).transpose(0, 1).reshape(-1, H * hd)
        # relative error of a probability: that of its score, 2 hd roundings of partial sums
        # below sum |q||k|, one of the score times log2 e and an exponential's; of the sum over
        # Lk keys: 2 Lk roundings
        rel = (s_abs.amax(-1, keepdim=True) * (2 * hd + 4) + 2 * kh.size(1) + 8) * 2.0 ** -24 * 2
        mag[sq] = (torch.matmul(p, vh.abs()) * rel).transpose(0, 1).reshape(-1, H * hd)
    return out, mag


@pytest.mark.parametrize("hd", [32, 64, 128])
@pytest.mark.parametrize("q_lens,k_lens", [
    ((1, 31, 32, 33), (1, 31, 32, 33)), ((129, 5, 128, 64), (63, 64, 65, 0)), ((3, 200), (257, 1)),
    ((97,), (1000,)), ((0, 40, 0), (3, 0, 7))])
def test_attention_f32_shapes(hd, q_lens, k_lens):
    y, (ref, bound) = _run(q_lens, k_lens, 3, hd)
    assert bool(((y.double() - ref).abs() <= bound + 1e-30).all())


@pytest.mark.parametrize("hd", [32, 64, 128])
def test_attention_f32_special_values(hd):
    inf, nan = float("inf"), float("nan")
    lens = (70, 150, 40, 33, 20)
    H = 2

    def plant(q, k, v):
        v[3, 1] = inf                   # sequence 0
        v[70 + 100, 5] = nan            # sequence 1
        k[220 + 10, 2] = inf            # sequence 2: infinite scores of either sign
        q[260 + 7, 3] = -inf            # sequence 3: one query row
        v[293 + 2, 0] = torch.finfo(torch.float32).max      # its first part rounds to infinity

    y, (ref, bound) = _run(lens, lens, H, hd, plant)
    assert torch.equal(torch.isnan(y), torch.isnan(ref))
    assert torch.equal(torch.isinf(y), torch.isinf(ref.float()))
    assert torch.equal(y[torch.isinf(y)], ref.float()[torch.isinf(y)])
    fine = torch.isfinite(ref) & torch.isfinite(bound)
    assert bool(fine[:70].any()) and bool(fine[293:].all())
    assert bool(((y.double() - ref).abs()[fine] <= bound[fine] + 1e-30).all())


@pytest.mark.parametrize("hd", [32, 64, 128])
@pytest.mark.parametrize("eq,ek,ev", [
    (-118, 118, 0), (120, -119, 0), (0, 0, -116), (-60, 58, 90),
    (0, 0, -128), (0, 0, -134), (0, 0, -140), (100, -128, 0), (100, -134, 0), (105, -140, 0), (105, -147, 0),   # denormal K, V
    (-105, 106, 0), (60, -59, 110), (113, -112, 0), (-118, 119, 0)])                                           # up to those too large to split
def test_attention_f32_magnitudes(hd, eq, ek, ev):
    def scale(q, k, v):
        for t, e in ((q, eq), (k, ek), (v, ev)):
            t.copy_(torch.ldexp(t, torch.tensor(e, device=DEV)))

    y, (ref, bound) = _run((37, 130), (37, 130), 2, hd, scale)
    assert bool(((y.double() - ref).abs() <= bound + 2.0 ** -148).all())


def _chain(q, k, v, lens, H, hd, scale):
    """The layer in fp32 with one rounding per product: chains of multiply-adds."""
    out, a = torch.zeros_like(q), 0
    scale = (torch.tensor(scale, dtype=torch.float32) * torch.tensor(1.4426950408889634, dtype=torch.float32)).item()
    for L in lens:
        qh, kh, vh = (t[a:a + L].reshape(L, H, hd).transpose(0, 1).contiguous() for t in (q, k, v))
        qh = qh * scale
        s = torch.zeros(H, L, L, device=DEV)
        for d in range(hd):
            s = (s.double() + qh[:, :, d:d + 1].double() * kh[:, None, :, d].double()).float()
        p = torch.exp2(s - s.amax(-1, keepdim=True))
        o = torch.zeros_like(qh)
        for n in range(L):
            o = (o.double() + p[:, :, n:n + 1].double() * vh[:, n:n + 1].double()).float()
        out[a:a + L] = (o * (1.0 / p.sum(-1, keepdim=True))).transpose(0, 1).reshape(L, H * hd)
        a += L
    return out


def _one_key_in(every):
    def scores(q, k, v):
        hd = q.size(1) // 3
        for h in range(3):
            q[:, h * hd] = 2.0 * hd ** 0.5
            k[:, h * hd] = -1000.0               # probabilities of zero
            k[::every, h * hd] = 0.0
    return scores


@pytest.mark.parametrize("hd", [32, 64, 128])
@pytest.mark.parametrize("lens,qkv", [
    ((37, 130, 300), None), ((5, 9, 17, 3, 12), None), ((40, 200), lambda q, k, v: q.mul_(16)),
    ((40, 200), lambda q, k, v: v.abs_()),
    ((64,) * 20, _one_key_in(32)), ((128,) * 10, _one_key_in(32)), ((512,), _one_key_in(32)),
    ((32,) * 20, _one_key_in(16)), ((64,) * 20, _one_key_in(16)), ((256, 256), _one_key_in(16))])
def test_attention_f32_precision(hd, lens, qkv):
    """The 2-norm of the error is no larger than that of fp32 multiply-adds, also where few
    probabilities of a tile are other than zero.  (Two parts and three products are off by
    more than ten times that.)"""
    kept = []

    def inputs(q, k, v):
        if qkv is not None:
            qkv(q, k, v)
        kept.extend((q, k, v))

    y, (ref, _) = _run(lens, lens, 3, hd, inputs)
    err, chain = ((t.double() - ref).norm() for t in (y, _chain(*kept, lens, 3, hd, hd ** -0.5)))
    assert err <= chain, float(err / chain)


@pytest.mark.parametrize("hd", [32, 64, 128])
def test_attention_f32_small_probabilities(hd):
    """A probability of 2^-124 keeps its 24 bits: two keys, the one with all the weight worth 0."""
    # a scale that times log2 e is one in fp32, so that the scores, of at most 24 bits, are exact
    log2e = torch.tensor(1.4426950408889634, dtype=torch.float32)
    scale = torch.tensor(0.6931471805599453, dtype=torch.float32)
    near = [scale]
    for towards in (0.0, 1.0):
        x = scale
        for _ in range(4):
            x = torch.nextafter(x, torch.tensor(towards, dtype=torch.float32))
            near.append(x)
    scale = next(float(x) for x in near if float(x * log2e) == 1.0)
    g = torch.Generator("cuda").manual_seed(hd)
    B = 400
    score = -(104 + 21 * torch.rand(B, device=DEV, generator=g)).mul(2 ** 16).round().div(2 ** 16)
    worth = (1 + torch.rand(B, hd, device=DEV, generator=g)) * 2.0 ** 90

    def plant(q, k, v):
        q.zero_()
        k.zero_()
        q[:, 0] = 1.0
        k[1::2, 0] = score
        v[0::2] = 0.0
        v[1::2] = worth

    y, _ = _run((2,) * B, (2,) * B, 1, hd, plant, scale=scale)
    ref = torch.exp2(score.double())[:, None] * worth.double()       # (the sum is 1 within 2^-104)
    # two units of 2^-23 for the exponential, a rounding each for the sums and the quotient
    assert bool(((y[0::2].double() - ref).abs() <= 6 * 2.0 ** -24 * ref).all())
