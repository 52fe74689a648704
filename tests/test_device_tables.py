"""Who may read which device table of a nested size, and for how long: launches, streams and
captures are stubbed, so everything here runs on the host."""
import sys
import weakref

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
        monkeypatch.setattr(impl_module, "_attention_schedule", lambda *a: self._table())
        monkeypatch.setattr(impl_module, "_attention_plan", lambda *a: self._table())

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


TABLES = {
    "sizes": NestedTensorImpl.sizes_dev,
    "offsets": NestedTensorImpl.offsets_dev,
    "row offsets": NestedTensorImpl.row_offsets_dev,
    "last dim rows": lambda t: t.last_dim_rows()[0],
    "work list": NestedTensorImpl.attention_schedule,
}


@pytest.mark.parametrize("name", sorted(TABLES))
def test_captured_table_outlives_calls_on_other_streams(device, name):
    table, a = TABLES[name], nested()
    shared = a.with_buffer(a.buffer + 1)
    table(a)                                             # warm-up on the default stream and on the side stream
    device.stream = 2
    table(a)
    device.capturing = True
    captured = weakref.ref(table(a))
    also = weakref.ref(table(shared))
    device.capturing = False
    memory = nested((4, 4))
    for device.stream in (1, 3, 1, 2):
        table(a)
        table(shared)
        a.attention_schedule(kv=memory)
    assert captured() is not None and writer(captured()) == 2
    assert also() is not None and writer(also()) == 2
    device.capturing, device.stream = True, 2
    assert table(a) is captured()


@pytest.mark.parametrize("name", sorted(TABLES))
def test_streams_in_turn_write_a_table_once_each(device, name):
    table, a = TABLES[name], nested()
    mine = {}
    for device.stream in (1, 2):
        mine[device.stream] = table(a)
        assert writer(mine[device.stream]) == device.stream
    launches = device.launches
    for device.stream in (1, 2, 1, 2, 2, 1):
        assert table(a) is mine[device.stream]
    assert device.launches == launches


@pytest.mark.parametrize("name", sorted(TABLES))
def test_capture_takes_what_eager_calls_have_made(device, name):
    table, a = TABLES[name], nested()
    device.capturing = True
    own = table(a)                                       # nothing made yet: the graph writes its own ..
    device.capturing = False
    first = table(a)
    assert first is not own                              # .. which eager calls do not see
    device.stream, device.capturing = 2, True
    assert table(a) is first


@pytest.mark.parametrize("table", [lambda q, kv: q.attention_schedule(kv=kv), lambda q, kv: q.attention_plan(8, 64, kv=kv)],
                         ids=["work list", "plan"])
def test_captured_table_outlives_calls_with_other_keys(device, table):
    queries, memory, other = nested(), nested((7, 1)), nested((2, 2))
    table(queries, memory)
    device.capturing = True
    captured = weakref.ref(table(queries, memory))
    device.capturing = False
    assert captured() is table(queries, memory)
    kept = [weakref.ref(table(queries, keys)) for keys in (other, memory, other)]
    assert captured() is not None
    assert kept[0]() is None and kept[1]() is None          # only the last one is kept otherwise
