"""The attention work list written by nt_attention_schedule, against the list spelled out on
the host: several launches' worth of sequences, empty ones, ties, cross-attention."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)


def _expected(q_lens, k_lens, q_tile):
    q0 = [sum(q_lens[:b]) for b in range(len(q_lens))]
    k0 = [sum(k_lens[:b]) for b in range(len(k_lens))]
    order = sorted(range(len(k_lens)), key=lambda b: -k_lens[b])     # stable: ties in their order
    return [[q0[b], q_lens[b], r, 0, k0[b], k_lens[b], 0, 0] for b in order for r in range(0, q_lens[b], q_tile)]


@pytest.mark.parametrize("B,cross", [(1, False), (4, True), (180, False), (181, True), (400, False)])
@pytest.mark.parametrize("q_tile", [128, 32])
def test_schedule(B, cross, q_tile):
    from nestedtensor_amd import _C
    g = torch.Generator().manual_seed(B + q_tile)
    q = torch.randint(0, 300, (B,), generator=g)
    q[0] = 9000                                  # more tiles than a wavefront has lanes
    k = torch.randint(0, 40, (B,), generator=g) if cross else q
    sizes = [torch.stack([t, torch.full_like(t, 64)], 1) for t in (q, k)]
    got = _C.ops.attention_schedule.default(sizes[0], sizes[1], q_tile, DEV)
    exp = _expected(q.tolist(), k.tolist(), q_tile)
    assert got.dtype == torch.int32 and got.cpu().tolist() == exp


def test_schedule_rejects_token_indices_beyond_int32():
    from nestedtensor_amd import _C
    sizes = torch.tensor([[1 << 30, 64], [1 << 30, 64]])
    with pytest.raises(RuntimeError, match="the work list holds token indices as int32"):
        _C.ops.attention_schedule.default(sizes, sizes, 1 << 20, DEV)


def test_schedule_is_kept_per_stream():
    # a work list that a kernel on one stream wrote is not handed to work on another
    import nestedtensor_amd as nt
    impl = nt.nested_tensor([torch.randn(n, 64) for n in (5, 130)], device=DEV, dtype=torch.float16)._impl
    first = impl.attention_schedule()
    assert impl.attention_schedule() is first
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        other = impl.attention_schedule()
    torch.cuda.synchronize()
    assert other.data_ptr() != first.data_ptr() and torch.equal(other, first)
