"""Packed storage of a nested tensor: buffer + nested size + device offsets.

Counterpart of the reference's NestedTensorImpl / EfficientSizeNode
(nestedtensor/csrc/nested_tensor_impl.h:46-173,
nestedtensor/csrc/storage/EfficientSizeNode.h:53-138): one contiguous 1-D
buffer, a host int64 table ``sizes[B, D]`` and the per-dimension "regular or
not" summary ``opt_sizes``.  What is new here is the device side of the
metadata: ``sizes`` mirrored in HBM and int64 element ``offsets[B + 1]`` built
by the device prefix scan (nt_offsets_from_sizes), both cached on the impl and
created on first use on the buffer's stream.  Only nested_dim 1 exists
(EfficientSizeNode.h:86-88).

Two storage layouts exist, as in the reference (Packed.h:100-163): every
constituent row-major contiguous, or, for constituents [C, H, W], every
constituent stored as [H, W, C] ("channels last", the nested stride is then
(1, W * C, C)).  The second is a flag on the impl, not a stride table: these
are the only two layouts the reference's kernels accept, and the constituent
extents, hence the element offsets, are the same in both.
"""

import torch

from . import _C


class NestedTensorImpl:
    __slots__ = ("buffer", "sizes", "_opt_sizes", "_tables", "_summary", "_attn_schedule", "_attn_plan", "_kept",
                 "channels_last")

    def __init__(self, buffer, sizes, channels_last=False):
        """buffer: 1-D contiguous tensor; sizes: CPU int64 [B, D], or 0-d for an
        empty nested tensor (EfficientSizeNode.h:8-12).  channels_last: the
        buffer holds each [C, H, W] constituent as [H, W, C]."""
        if buffer.dim() != 1:
            raise RuntimeError("Given buffer must be vector, i.e. dim 1 Tensor.")
        if not buffer.is_contiguous():
            raise RuntimeError("Given buffer must be contiguous.")
        assert sizes.dtype == torch.int64 and sizes.device.type == "cpu"
        if channels_last and not (sizes.dim() == 2 and sizes.size(1) == 3):
            raise RuntimeError("ChannelsLast memory format requires 4 dim input.")
        self.channels_last = bool(channels_last)
        self.buffer = buffer
        self.sizes = sizes
        self._opt_sizes = None
        self._tables = None
        self._summary = None
        self._attn_schedule = None
        self._attn_plan = None
        self._kept = None

    # ---- host metadata ----------------------------------------------------
    @property
    def B(self):
        return self.sizes.size(0) if self.sizes.dim() > 0 else 0

    @property
    def D(self):
        return self.sizes.size(1) if self.sizes.dim() > 0 else 0

    def dim(self):
        # EfficientSizeNode::dim (EfficientSizeNode.h:94-96)
        return 1 + self.sizes.size(1) if self.sizes.dim() > 0 else 1

    def nested_dim(self):
        return 1

    def _summarize(self):
        """(regular extents with -1 where they differ, largest, smallest, numel) of a nested
        size with at least one extent, taken once (the nested size never changes)."""
        if self._summary is None:
            self._summary = _size_summary(self.sizes)
        return self._summary

    def numel(self):
        # EfficientSizeNode::numel (EfficientSizeNode.h:113-131)
        if self.sizes.dim() == 0 or self.sizes.numel() == 0:
            return 0
        return self._summarize()[3]

    def opt_sizes(self):
        # construct_efficient_size (EfficientSizeNode.h:27-49)
        if self._opt_sizes is None:
            res = [self.B]
            if self.B > 0 and self.D > 0:
                res += [None if v < 0 else v for v in self._summarize()[0]]
            self._opt_sizes = res
        return list(self._opt_sizes)

    def max_sizes(self):
        # get_max_size_from_efficient_size (masking.cpp:83-103)
        return list(self._summarize()[1]) if self.B > 0 and self.D > 0 else []

    def min_sizes(self):
        return list(self._summarize()[2]) if self.B > 0 and self.D > 0 else []

    def has_empty_constituent(self):
        return self.B > 0 and self.D > 0 and min(self._summarize()[2]) == 0

    def shapes(self):
        return [tuple(int(v) for v in row) for row in self.sizes] if self.sizes.dim() > 0 else []

    def strides(self):
        """Per-constituent element strides: row-major (Packed.h:10-19), or
        (1, W * C, C) for the channels-last layout (nested_tensor_impl.cpp:188-192)."""
        out = []
        for s in self.shapes():
            if self.channels_last:
                out.append((1, s[2] * s[0], s[0]))
                continue
            st, acc = [], 1
            for v in reversed(s):
                st.append(acc)
                acc *= v
            out.append(tuple(reversed(st)))
        return out

    # ---- device metadata ---------------------------------------------------
    def _table(self, which):
        """Entry `which` of _tables = (stream, sizes, offsets): the stream that wrote the two
        device tables (None: they are ordered like the buffer itself, any stream may read
        them) and the tables, either None where only the other is known.  The three are
        one attribute, assigned and read once: another thread sees all of them or none."""
        tables = self._tables
        if tables is not None and tables[which] is not None and (
                tables[0] is None or usable_on(tables[0], current_stream_id(self.buffer.device))):
            return tables[which]
        _C.require_device(self.buffer, "device metadata")
        if self.sizes.dim() != 2:
            return (None, self.sizes.to(self.buffer.device), None)[which]
        # written by one launch (nt_upload_sizes) on first use
        stream = current_stream_id(self.buffer.device)
        tables = (stream,) + tuple(_upload_sizes(self.sizes, self.buffer.device))
        if not torch.cuda.is_current_stream_capturing():
            self._tables = tables
        return tables[which]

    def sizes_dev(self):
        """int64 [B, D] mirror of the nested size."""
        return self._table(1)

    def offsets_dev(self):
        """int64 [B + 1] element offsets, scanned on the device."""
        return self._table(2)

    def share_offsets(self, other):
        """Take over the device offsets of `other`, whose constituents hold as many elements."""
        tables = other._tables
        if tables is not None:
            self._tables = (tables[0], None, tables[2])

    def kept(self, name, build):
        """What build() returns, kept under `name` with this nested size for later calls on
        the same device and stream.  For device metadata that kernels wrote: work on
        another stream gets its own (see usable_on)."""
        device = self.buffer.device
        stream = current_stream_id(device)
        if self._kept is None:
            self._kept = {}
        entry = self._kept.get(name)
        if entry is None or entry[0] != device or not usable_on(entry[1], stream):
            entry = (device, stream, build())
            if not torch.cuda.is_current_stream_capturing():
                self._kept[name] = entry
        return entry[2]

    def row_offsets_dev(self):
        """int64 [B + 1] offsets counted in rows of the first constituent dim
        (token offsets for a [B, L_i, E] nested tensor)."""
        _C.require_device(self.buffer, "device metadata")
        return self.kept("rows", lambda: _upload_sizes(self.sizes[:, :1], self.buffer.device)[1])

    def last_dim_rows(self):
        """(row_offsets, total_rows): int64 [B + 1] on the device, the number of
        rows along the last dim (product of all other constituent dims) of the
        constituents before b, and their total."""
        def build():
            rows = self.sizes[:, :-1].prod(1)
            return _upload_sizes(rows.reshape(-1, 1), self.buffer.device)[1], int(rows.sum())
        _C.require_device(self.buffer, "device metadata")
        return self.kept("last_dim_rows", build)

    def attention_schedule(self, kv=None, q_tile=128):
        """Work list of the attention kernel (nt_attention_schedule), built from the
        host copies of the nested sizes and cached on the device: int32 [n_work, 8] rows {first query
        token, query length, first query row of the tile, 0, first key token, key
        length, 0, 0}, one per q_tile query rows of every sequence, longest key
        sequences first (they take the most key tiles, so they should start
        first).  Tiles that do not exist are never listed, hence never launched.
        kv: the nested tensor of the keys (None: self-attention)."""
        if kv is None or kv.sizes is self.sizes:
            kv = self
        cached = self._attn_schedule
        stream = current_stream_id(self.buffer.device)
        if cached is not None and cached[0] is kv.sizes and usable_on(cached[2], stream):
            return cached[1]
        sched = _attention_schedule(self.sizes, kv.sizes, q_tile, self.buffer.device)
        if not torch.cuda.is_current_stream_capturing():
            self._attn_schedule = (kv.sizes, sched, stream)      # holds kv.sizes, so the identity test stays valid
        return sched

    def attention_plan(self, num_heads, head_dim, kv=None):
        """Plan of the planned attention kernel (nt_attention_plan) for this nested
        size, `num_heads` heads and the compute units of the buffer's device: an
        int32 vector on the device, cached like the work list.
        kv: the nested tensor of the keys (None: self-attention)."""
        if kv is None or kv.sizes is self.sizes:
            kv = self
        cached = self._attn_plan
        if cached is not None and cached[0] is kv.sizes and cached[1] == (num_heads, head_dim):
            return cached[2]
        plan = _C.ops.attention_plan.default(self.sizes[:, 0].contiguous(), kv.sizes[:, 0].contiguous(),
                                             num_heads, head_dim, self.buffer.device)
        self._attn_plan = (kv.sizes, (num_heads, head_dim), plan)
        return plan

    def adopt_device_metadata(self, sizes_dev, offsets_dev):
        """Take over device copies of the nested size and of the element offsets
        that a conversion has already built for this nested size."""
        if sizes_dev.device == self.buffer.device and tuple(sizes_dev.shape) == tuple(self.sizes.shape):
            self._tables = (None, sizes_dev, offsets_dev if offsets_dev.numel() == self.B + 1 else None)

    def with_buffer(self, buffer, channels_last=None):
        """Same nested size over another buffer (in the same layout unless
        channels_last says otherwise); shares the cached metadata when the
        device matches."""
        out = NestedTensorImpl(buffer, self.sizes,
                               self.channels_last if channels_last is None else channels_last)
        out._opt_sizes = self._opt_sizes
        out._summary = self._summary
        if buffer.device == self.buffer.device:
            out._tables = self._tables
            out._attn_schedule = self._attn_schedule
            out._attn_plan = self._attn_plan
            if self._kept is None:
                self._kept = {}
            out._kept = self._kept
        return out


def current_stream_id(device):
    """Identity of torch's current stream on `device` (0: the default stream)."""
    return torch._C._cuda_getCurrentRawStream(device.index)


def usable_on(made_on, stream):
    """Whether metadata that a kernel wrote on stream `made_on` may be read by work on
    `stream`.  On another stream nothing orders the reader behind the writer, and the
    block could be handed out again while the reader still runs, so such a caller writes
    its own copy (a launch).  A capture keeps what its eager warm-up has made."""
    return made_on == stream or torch.cuda.is_current_stream_capturing()


_attention_schedule = _C.ops.attention_schedule.default
_size_summary = _C.ops.size_summary.default
_upload_sizes = _C.ops.upload_sizes.default
_offsets_from_sizes = _C.ops.offsets_from_sizes.default


def device_offsets(sizes_dev, B, D):
    """offsets[b] = sum_{c<b} prod_k sizes[c, k] on the device (nt_offsets_from_sizes)."""
    return _offsets_from_sizes(sizes_dev.reshape(B, D))
