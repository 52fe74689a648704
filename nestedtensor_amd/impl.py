"""Packed storage of a nested tensor: buffer + nested size + device offsets.

Counterpart of the reference's NestedTensorImpl / EfficientSizeNode
(nestedtensor/csrc/nested_tensor_impl.h:46-173,
nestedtensor/csrc/storage/EfficientSizeNode.h:53-138): one contiguous 1-D
buffer, a host int64 table ``sizes[B, D]`` and the per-dimension "regular or
not" summary ``opt_sizes``.  What is new here is the device side of the
metadata: ``sizes`` mirrored in HBM and int64 element ``offsets[B + 1]``, written
by one launch (nt_upload_sizes) on first use and kept on the impl for the stream
that asked.  Only nested_dim 1 exists
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
    __slots__ = ("buffer", "sizes", "_opt_sizes", "_given", "_summary", "_attn_plan", "_kept", "_ragged", "channels_last")

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
        self._given = None
        self._summary = None
        self._attn_plan = None
        self._kept = {}
        self._ragged = None

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

    def _extents(self, which):
        """The regular (0), largest (1) or smallest (2) extents, [] where there are none.  Asked
        on every call of most operators, so the summary is looked at before the table is."""
        summary = self._summary
        if summary is None:
            if self.B == 0 or self.D == 0:
                return []
            summary = self._summarize()
        return list(summary[which])

    def max_sizes(self):
        # get_max_size_from_efficient_size (masking.cpp:83-103)
        return self._extents(1)

    def min_sizes(self):
        return self._extents(2)

    def ragged_dims(self):
        """(number of leading constituent dims up to and including the last irregular one, at
        least 1; whether a constituent is empty): what every padding call asks, answered once."""
        if self._ragged is None:
            n = 1
            for k, v in enumerate(self._extents(0)):
                if v < 0:
                    n = k + 1
            self._ragged = n, 0 in self._extents(2)
        return self._ragged

    def has_empty_constituent(self):
        return self.ragged_dims()[1]

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
    def kept(self, name, build, keys=None):
        """What build() returns, kept under `name` with this nested size for later calls.

        One entry per stream that asked, and none is replaced or dropped while the nested
        size lives.  Per stream, because nothing orders work on one stream behind the
        kernel that wrote another's table.  For good, because a captured graph reads the
        table it was given on every replay, whatever other streams do in between.  A
        capture takes what eager calls on its stream have made, or else on any stream;
        what it has to write itself is part of the graph and not kept.

        keys: the other nested size that the table depends on.  Only the last one's table
        is kept per stream (with that nested size itself, so the identity test stays valid),
        and what a capture was given."""
        device = self.buffer.device
        if device.index is None:                                 # a host tensor
            _C.require_device(self.buffer, "device metadata")
        key = (name, current_stream_id(device))                  # _kept is for one device (with_buffer)
        entry = self._kept.get(key)
        if entry is not None and entry[0] is keys:
            return entry[1] if keys is None else self._given_out(entry[1])
        if torch.cuda.is_current_stream_capturing():
            made = [e[1] for k, e in list(self._kept.items()) if k[0] == name and e[0] is keys]
            return self._given_out(made[0]) if made else build()
        entry = (keys, build())
        if keys is not None:
            self._kept[key] = entry
            return entry[1]
        return self._kept.setdefault(key, entry)[1]      # the first of two threads on one stream wins

    def _given_out(self, table):
        """`table`, kept with this nested size from now on if a capture is under way."""
        if torch.cuda.is_current_stream_capturing():
            self._kept["captured", id(table)] = (None, table)
        return table

    def device_tables(self):
        """(int64 [B, D] mirror of the nested size, int64 [B + 1] element offsets) on the device."""
        given = self._given
        if given is not None and given[0] is not None and given[1] is not None:
            return given
        return self.kept("sizes", self._write_tables)

    def _write_tables(self):
        # one launch (nt_upload_sizes) on first use
        if self.sizes.dim() != 2:
            return self.sizes.to(self.buffer.device), None
        return _upload_sizes(self.sizes, self.buffer.device)

    def sizes_dev(self):
        given = self._given
        return given[0] if given is not None and given[0] is not None else self.kept("sizes", self._write_tables)[0]

    def offsets_dev(self):
        given = self._given
        return given[1] if given is not None and given[1] is not None else self.kept("sizes", self._write_tables)[1]

    def row_offsets_dev(self):
        """int64 [B + 1] offsets counted in rows of the first constituent dim
        (token offsets for a [B, L_i, E] nested tensor)."""
        return self.kept("rows", lambda: _upload_sizes(self.sizes[:, :1], self.buffer.device)[1])

    def last_dim_rows(self):
        """(row_offsets, total_rows): int64 [B + 1] on the device, the number of
        rows along the last dim (product of all other constituent dims) of the
        constituents before b, and their total."""
        def build():
            rows = self.sizes[:, :-1].prod(1)
            return _upload_sizes(rows.reshape(-1, 1), self.buffer.device)[1], int(rows.sum())
        return self.kept("last_dim_rows", build)

    def attention_schedule(self, kv=None, q_tile=128):
        """Work list of the attention kernel (nt_attention_schedule), built from the
        host copies of the nested sizes and kept per stream (see kept): int32 [n_work, 8]
        rows {first query token, query length, first query row of the tile, 0, first key
        token, key length, 0, 0}, one per q_tile query rows of every sequence, longest key
        sequences first (they take the most key tiles, so they should start
        first).  Tiles that do not exist are never listed, hence never launched.
        kv: the nested tensor of the keys (None: self-attention)."""
        if kv is None or kv.sizes is self.sizes:
            return self.kept("work list", lambda: _attention_schedule(self.sizes, self.sizes, q_tile, self.buffer.device))
        return self.kept("work list of keys",
                         lambda: _attention_schedule(self.sizes, kv.sizes, q_tile, self.buffer.device), kv.sizes)

    @property
    def _attn_schedule(self):
        """The work lists written for this nested size, None before the first."""
        return [e[1] for k, e in list(self._kept.items()) if k[0] in ("work list", "work list of keys")] or None

    def attention_plan(self, num_heads, head_dim, kv=None):
        """Plan of the planned attention kernel (nt_attention_plan) for this nested
        size, `num_heads` heads and the compute units of the buffer's device: an
        int32 vector on the device, cached like the work list.
        kv: the nested tensor of the keys (None: self-attention)."""
        if kv is None or kv.sizes is self.sizes:
            kv = self
        cached = self._attn_plan
        if cached is not None and cached[0] is kv.sizes and cached[1] == (num_heads, head_dim):
            return self._given_out(cached[2])
        plan = _attention_plan(self.sizes[:, 0].contiguous(), kv.sizes[:, 0].contiguous(), num_heads, head_dim,
                               self.buffer.device)
        self._attn_plan = (kv.sizes, (num_heads, head_dim), plan)
        return plan

    def adopt_device_metadata(self, sizes_dev, offsets_dev):
        """Take over device copies of the nested size and of the element offsets
        that a conversion has already built for this nested size.  They are ordered like
        the buffer that was written with them, so every stream may read them."""
        if sizes_dev.device == self.buffer.device and tuple(sizes_dev.shape) == tuple(self.sizes.shape):
            self._given = (sizes_dev, offsets_dev if offsets_dev.numel() == self.B + 1 else None)

    def share_offsets(self, other):
        """Take over the offsets that a conversion has built for `other`, whose
        constituents hold as many elements."""
        if other._given is not None:
            self._given = (None, other._given[1])

    def with_buffer(self, buffer, channels_last=None):
        """Same nested size over another buffer (in the same layout unless
        channels_last says otherwise); shares the cached metadata when the
        device matches."""
        out = NestedTensorImpl(buffer, self.sizes,
                               self.channels_last if channels_last is None else channels_last)
        out._opt_sizes = self._opt_sizes
        out._summary = self._summary
        out._ragged = self._ragged
        if buffer.device == self.buffer.device:
            out._given = self._given
            out._attn_plan = self._attn_plan
            out._kept = self._kept
        return out


def current_stream_id(device):
    """Identity of torch's current stream on `device` (0: the default stream)."""
    return torch._C._cuda_getCurrentRawStream(device.index)


_attention_plan = _C.ops.attention_plan.default
_attention_schedule = _C.ops.attention_schedule.default
_size_summary = _C.ops.size_summary.default
_upload_sizes = _C.ops.upload_sizes.default
_offsets_from_sizes = _C.ops.offsets_from_sizes.default


def device_offsets(sizes_dev, B, D):
    """offsets[b] = sum_{c<b} prod_k sizes[c, k] on the device (nt_offsets_from_sizes)."""
    return _offsets_from_sizes(sizes_dev.reshape(B, D))
