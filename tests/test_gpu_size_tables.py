"""Nested sizes and offsets written from launch arguments (nt_upload_sizes), against the host's
prefix sums, at the edges of one and of four launches and past them; which stream may read them."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)


# 896 extents per launch, four launches: 448 and 1792 constituents of two extents
@pytest.mark.parametrize("B,D", [(1, 1), (3, 2), (448, 2), (449, 2), (1792, 2), (1793, 2), (896, 1), (298, 3), (299, 3),
                                 (2, 896), (2, 897), (5, 0)])
def test_upload_sizes(B, D):
    from nestedtensor_amd import _C
    g = torch.Generator().manual_seed(B * 7 + D)
    sizes = torch.randint(0, 60 if D < 4 else 2, (B, D), generator=g)
    sizes_dev, offsets = _C.ops.upload_sizes.default(sizes, DEV)
    assert torch.equal(sizes_dev.cpu(), sizes)
    assert torch.equal(offsets.cpu()[1:], sizes.prod(1).cumsum(0)) and int(offsets[0]) == 0


def test_upload_sizes_beyond_int32():
    from nestedtensor_amd import _C
    sizes = torch.tensor([[1 << 33, 1], [3, 5], [1 << 16, 1 << 18]])        # extents and offsets past 32 bits
    for s in (sizes, sizes[1:]):
        sizes_dev, offsets = _C.ops.upload_sizes.default(s, DEV)
        assert torch.equal(sizes_dev.cpu(), s) and torch.equal(offsets.cpu()[1:], s.prod(1).cumsum(0))


@pytest.mark.parametrize("n", [1, 384, 385, 1536, 1537])
def test_upload_table(n):
    from nestedtensor_amd import _C
    table = torch.arange(2 * n).reshape(2, n)[1] * (1 << 34)
    assert torch.equal(_C.ops.upload_table.default(table, DEV).cpu(), table)


def test_tables_are_kept_per_stream():
    import nestedtensor_amd as nt
    packed = nt.nested_tensor([torch.randn(n, 16) for n in (3, 0, 7)], device=DEV)._impl
    side = torch.cuda.Stream()

    def tables():
        return packed.sizes_dev(), packed.offsets_dev(), packed.row_offsets_dev()

    first = tables()
    assert all(a is b for a, b in zip(first, tables()))
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        second = tables()
    torch.cuda.synchronize()
    for a, b in zip(first, second):
        assert a.data_ptr() != b.data_ptr() and torch.equal(a, b)
    assert second[2].tolist() == [0, 3, 3, 10]


def test_graph_replays_between_calls_on_other_streams():
    # the graph reads the tables and the work list that it was captured with, whatever runs on
    # another stream and is allocated on its own in between
    import nestedtensor_amd as nt
    g = torch.Generator().manual_seed(7)
    rows = nt.nested_tensor([torch.randn(n, 64, generator=g) for n in (5, 130, 64, 1)], device=DEV, dtype=torch.float16)
    maps = nt.nested_tensor([torch.randn(16, h, w, generator=g) for h, w in ((9, 17), (4, 30))], device=DEV, dtype=torch.float16)
    weights = [(torch.randn(s, generator=g) * 0.1).half().to(DEV) for s in ((192, 64), (192,), (64, 64), (64,), (32, 16, 1, 1))]

    def work():
        y = torch.ops.nestedtensor.min_mha(1, 64, 0.0, False, rows, rows, rows, *weights[:2], 0.125, *weights[2:4])
        z = torch.conv2d(maps, weights[4]).contiguous(memory_format=torch.channels_last)
        return y._impl.buffer, rows.to_padded_tensor(0), z._impl.buffer, maps.to_padded_tensor(0)

    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    work()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        work()
        with torch.cuda.graph(graph, stream=side):
            outs = work()
    torch.cuda.synchronize()
    for _ in range(3):
        expect = work()
        with torch.cuda.stream(side):
            junk = [torch.full((n,), -1, dtype=torch.int64, device=DEV) for n in (8, 16, 40, 64, 200, 600) for _ in range(20)]
        torch.cuda.synchronize()
        for t in (rows, maps):
            t._impl.buffer.add_(0.5)
        graph.replay()
        torch.cuda.synchronize()
        expect = work()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(outs, expect))
        del junk
