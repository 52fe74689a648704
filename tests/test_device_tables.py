"""Who may read which device table of a nested size, and for how long: launches, streams and
captures are stubbed, so everything here runs on the host."""
import sys

import pytest
import torch

from nestedtensor_amd import impl as impl_module
from nestedtensor_amd.impl import NestedTensorImpl


class Device:
    """The stubbed device: the stream that is current, whether it is capturing, and which
    stream wrote a table (a table's entry of -1 - stream is all that its writer leaves)."""

    def __init__(self, monkeypatch):
        self.stream, self.capturing, self.launches = 1, False, 0
        monkeypatch.setattr(impl_module, "current_stream_id", lambda device: self.stream)
        monkeypatch.setattr(impl_module._C, "require_device", lambda *a: None)
        monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: self.capturing)
        monkeypatch.setattr(impl_module, "_upload_sizes", lambda sizes, device: (self._table(), self._table()))

    def _table(self):
        self.launches += 1
        return torch.tensor([-1 - self.stream])


@pytest.fixture
def device(monkeypatch):
    return Device(monkeypatch)


def nested(lengths=(3, 5)):
    return NestedTensorImpl(torch.zeros(sum(lengths) * 2), torch.tensor([[n, 2] for n in lengths]))


def writer(table):
    return -1 - int(table[0])


def test_first_use_seen_by_another_thread(device):
    # Between any two lines of a thread's first use (stream 1), a thread on stream 2 asks for the
    # same tables: it must get tables that its own stream wrote.
    seen = []

    def look(frame, event, arg):
        if frame.f_code.co_filename != impl_module.__file__:
            return None
        if event == "line":
            sys.settrace(None)
            device.stream = 2
            seen.append((writer(shared.sizes_dev()), writer(shared.offsets_dev())))
            device.stream = 1
            sys.settrace(look)
        return look

    for first in (NestedTensorImpl.sizes_dev, NestedTensorImpl.offsets_dev):
        shared = nested()
        sys.settrace(look)
        try:
            own = first(shared)
        finally:
            sys.settrace(None)
        assert writer(own) == 1
    assert len(seen) > 4 and set(seen) == {(2, 2)}


def test_tables_of_a_conversion_serve_every_stream(device):
    made = nested()
    sizes, offsets = torch.zeros(2, 2, dtype=torch.int64), torch.zeros(3, dtype=torch.int64)
    made.adopt_device_metadata(sizes, offsets)
    same = made.with_buffer(made.buffer + 1)
    for device.stream in (1, 2):
        assert made.sizes_dev() is sizes and made.offsets_dev() is offsets
        assert same.sizes_dev() is sizes and same.offsets_dev() is offsets
    assert device.launches == 0
