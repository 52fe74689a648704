"""Pad and un-pad of constituents with two and three ragged dims by flat 16-byte chunks, bit for
bit against slicing: rows shorter than a chunk, rows of one element, chunks over several rows,
constituents that begin anywhere inside a chunk, empty ones, and guards behind both buffers."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)
SHAPES = {
    "images": [(3, 17, 33), (3, 40, 5), (3, 1, 64), (3, 64, 1)],
    "three": [(1, 1, 1), (2, 5, 3), (4, 1, 7), (3, 9, 2)],
    "empty": [(2, 3, 5), (0, 4, 6), (3, 0, 9), (1, 7, 0)],
    "inner": [(5, 9, 3), (11, 2, 3), (1, 31, 3)],          # two ragged dims, a regular last one
    "flat": [(7, 300), (50, 1), (3, 65)],                  # two ragged dims
    "wide": [(2, 3000), (5, 1111)],
}


@pytest.mark.parametrize("dtype", [torch.uint8, torch.float16, torch.float32, torch.float64])
@pytest.mark.parametrize("name", sorted(SHAPES))
@pytest.mark.parametrize("wider", [0, 3])
def test_planes(name, dtype, wider):
    from nestedtensor_amd import _C
    eb = torch.empty(0, dtype=dtype).element_size()
    shapes = SHAPES[name]
    D = len(shapes[0])
    nrag = 2 if name == "inner" or D == 2 else 3
    ext = [max(s[k] for s in shapes) + (wider if k < nrag else 0) for k in range(D)]
    parts = [(torch.rand(s) * 200 + 1).to(dtype) for s in shapes]
    sizes = torch.tensor(shapes)
    sizes_dev, offsets = _C.ops.upload_sizes.default(sizes, DEV)
    total = int(offsets[-1])
    flat = torch.cat([t.reshape(-1) for t in parts])
    # both buffers at the start of an allocation and one element into it, a guard behind them
    for shift in (0, 1):
        packed = torch.full((total + shift + 40,), 99, dtype=dtype, device=DEV)
        packed[shift:shift + total] = flat.to(DEV)
        expect = torch.full([len(shapes)] + ext, 7, dtype=dtype)
        for b, t in enumerate(parts):
            expect[(b,) + tuple(slice(0, n) for n in t.shape)] = t
        n = expect.numel()
        padded = torch.full((n + shift + 40,), 99, dtype=dtype, device=DEV)
        seven = torch.tensor([7], dtype=dtype).view(torch.uint8)
        bits = int.from_bytes(bytes(seven.tolist()), "little")
        stream = _C.current_stream(DEV)
        _C.check(_C.lib.nt_add_padding(_C.ptr(packed[shift:]), _C.ptr(padded[shift:]), _C.ptr(offsets), _C.ptr(sizes_dev),
                                       len(shapes), D, nrag, _C.i64_array(ext), eb, bits, stream))
        assert torch.equal(padded[shift:shift + n].cpu(), expect.reshape(-1))
        assert bool((padded[:shift] == 99).all()) and bool((padded[shift + n:] == 99).all())
        back = torch.full((total + shift + 40,), 99, dtype=dtype, device=DEV)
        _C.check(_C.lib.nt_remove_padding(_C.ptr(padded[shift:]), _C.ptr(back[shift:]), _C.ptr(offsets), _C.ptr(sizes_dev),
                                          len(shapes), D, nrag, _C.i64_array(ext), eb, stream))
        assert torch.equal(back[shift:shift + total].cpu(), flat)
        assert bool((back[:shift] == 99).all()) and bool((back[shift + total:] == 99).all())


@pytest.mark.parametrize("dtype", [torch.uint8, torch.float16, torch.float32, torch.float64])
@pytest.mark.parametrize("name,cut", [("images", (2, 9, 12)), ("three", (2, 4, 3)), ("inner", (4, 6, 3)), ("flat", (7, 70)),
                                      ("flat", (20, 299)), ("wide", (3, 1200))])
def test_planes_cut_off(name, cut, dtype):
    # padded extents below a constituent's: pad cuts off, row by row, whatever chunk the row ends in
    from nestedtensor_amd import _C
    eb = torch.empty(0, dtype=dtype).element_size()
    shapes = SHAPES[name]
    nrag = 2 if name == "inner" or len(cut) == 2 else 3
    parts = [(torch.rand(s) * 200 + 1).to(dtype) for s in shapes]
    sizes_dev, offsets = _C.ops.upload_sizes.default(torch.tensor(shapes), DEV)
    packed = torch.cat([t.reshape(-1) for t in parts]).to(DEV)
    expect = torch.full((len(shapes),) + cut, 7, dtype=dtype)
    for b, t in enumerate(parts):
        inside = tuple(slice(0, min(n, m)) for n, m in zip(t.shape, cut))
        expect[(b,) + inside] = t[inside]
    padded = torch.full((expect.numel() + 40,), 99, dtype=dtype, device=DEV)
    seven = torch.tensor([7], dtype=dtype).view(torch.uint8)
    _C.check(_C.lib.nt_add_padding(_C.ptr(packed), _C.ptr(padded), _C.ptr(offsets), _C.ptr(sizes_dev), len(shapes), len(cut),
                                   nrag, _C.i64_array(cut), eb, int.from_bytes(bytes(seven.tolist()), "little"),
                                   _C.current_stream(DEV)))
    assert torch.equal(padded[:expect.numel()].cpu(), expect.reshape(-1))
    assert bool((padded[expect.numel():] == 99).all())
    # un-pad of that has no result, but writes nothing outside the packed buffer
    back = torch.full((packed.numel() + 40,), 99, dtype=dtype, device=DEV)
    _C.check(_C.lib.nt_remove_padding(_C.ptr(padded), _C.ptr(back), _C.ptr(offsets), _C.ptr(sizes_dev), len(shapes), len(cut),
                                      nrag, _C.i64_array(cut), eb, _C.current_stream(DEV)))
    assert bool((back[packed.numel():] == 99).all())


def test_planes_cut_off_a_constituent_past_32_bits():
    from nestedtensor_amd import _C
    shapes, cut = [(70000, 70000), (3, 60)], (70, 50)
    sizes_dev, offsets = _C.ops.upload_sizes.default(torch.tensor(shapes), DEV)
    packed = torch.empty(int(offsets[-1]), dtype=torch.uint8, device=DEV)
    parts = [packed[:70000 * 70000].view(70000, 70000), packed[70000 * 70000:].view(3, 60)]
    parts[0][:71] = torch.randint(1, 99, (71, 70000), dtype=torch.uint8, device=DEV)
    parts[1].copy_(torch.randint(1, 99, (3, 60), dtype=torch.uint8, device=DEV))
    padded = torch.full((2, 70, 50), 99, dtype=torch.uint8, device=DEV)
    _C.check(_C.lib.nt_add_padding(_C.ptr(packed), _C.ptr(padded), _C.ptr(offsets), _C.ptr(sizes_dev), 2, 2, 2,
                                   _C.i64_array(cut), 1, 7, _C.current_stream(DEV)))
    assert torch.equal(padded[0], parts[0][:70, :50])
    assert torch.equal(padded[1, :3], parts[1][:, :50]) and bool((padded[1, 3:] == 7).all())


# few short rows of many constituents go row by row: un-pad up to five rows of 1 KiB from 4096
# rows on, pad one, two, three .. rows of 1 KiB, 256, 64 .. bytes from 16384 constituents on
@pytest.mark.parametrize("dtype", [torch.uint8, torch.float16, torch.float64])
@pytest.mark.parametrize("B,rows,row_bytes", [
    (4095, 1, 1024), (4096, 1, 1024), (820, 5, 1024), (820, 5, 1040), (700, 6, 48), (1024, 4, 8),
    (16383, 2, 256), (16384, 2, 256), (16384, 2, 272), (16384, 3, 64), (16384, 3, 72), (16384, 1, 1032), (20000, 4, 16)])
@pytest.mark.parametrize("three", [False, True])
def test_many_constituents_of_few_short_rows(B, rows, row_bytes, dtype, three):
    from nestedtensor_amd import _C
    eb = torch.empty(0, dtype=dtype).element_size()
    g = torch.Generator().manual_seed(B + rows)
    ext = [rows, row_bytes // eb]
    sizes = torch.stack([torch.randint(0, n + 1, (B,), generator=g) for n in ext], 1)
    sizes[0], sizes[-1] = torch.tensor(ext), torch.tensor(ext)
    if three:
        ext, sizes = [1] + ext, torch.cat([torch.ones(B, 1, dtype=torch.int64), sizes], 1)
    sizes_dev, offsets = _C.ops.upload_sizes.default(sizes, DEV)
    total = int(offsets[-1])
    packed = torch.randint(1, 100, (total,), generator=g).to(dtype).to(DEV)
    i = torch.arange(rows, device=DEV).view(1, -1, 1)
    j = torch.arange(row_bytes // eb, device=DEV).view(1, 1, -1)
    s0, s1 = (sizes_dev[:, k].view(-1, 1, 1) for k in (-2, -1))
    inside = (i < s0) & (j < s1)
    expect = torch.full(inside.shape, 7, dtype=dtype, device=DEV)
    expect[inside] = packed[(offsets[:-1].view(-1, 1, 1) + i * s1 + j)[inside]]
    n_ragged = len(ext)
    padded = torch.ops.nestedtensor.add_padding(packed, sizes_dev, offsets, ext, n_ragged, 7.0)
    assert torch.equal(padded.view(expect.shape), expect)
    assert torch.equal(torch.ops.nestedtensor.remove_padding(padded, sizes_dev, offsets, total, n_ragged), packed)
