"""Bit-packed HQMQ cache containers (device memory owned by torch).

PackedTensor holds one tensor (K or V) of one layer: the code planes, the
per-token scales, the Med3x flag plane and outlier sideband, and the joint
codebook the codes index.  PackedKV pairs a K and a V PackedTensor.
Plane layout: include/hqmq_amd.h.
"""
from __future__ import annotations

import threading
from dataclasses import dataclass
from typing import Optional

import torch

from . import _lib as L

TILE = 16          # tokens per sideband tile
T_ALIGN = 64       # plane capacity is rounded up to whole attention super-tiles


def _round_up(x: int, m: int) -> int:
    return (x + m - 1) // m * m


class RangeWatch:
    """The largest finite scales the quantize kernels have written, as fp32 bits, one slot per tensor that shares the watch,
    and their way to the host: a copy into pinned memory behind every append that may have changed them, waited for only when
    the value is looked at.  Every copy has a buffer and an event of its own, recorded on the stream of the append, so that
    appends on several streams or threads, and on another device than the current one, are all waited for."""

    _SPARE_MOST, _PENDING_MOST = 4, 64      # buffers kept for the next copies; copies nobody has looked at

    def __init__(self, device, slots: int = 1):
        self.device_values = torch.zeros(slots, dtype=torch.int32, device=device)
        self.issued = 0                     # copies sent so far
        self._most = [0.0] * slots          # largest values seen on the host; 0: nothing written yet
        self._pending, self._spare = {}, []          # by number: (buffer, event)
        self._lock = threading.Lock()

    def __getstate__(self):
        """Copies and pickles take the values along, waited for; buffers, events and the lock are this object's own."""
        self.read(0, wait=not (self.device_values.is_cuda and torch.cuda.is_current_stream_capturing()))
        return {"device_values": self.device_values, "issued": self.issued, "_most": list(self._most)}

    def __setstate__(self, state):
        self.__dict__.update(state, _pending={}, _spare=[], _lock=threading.Lock())

    def fetch(self) -> None:
        """Sends the values to the host behind the work of the current stream of their device."""
        with self._lock:
            host, event = self._spare.pop() if self._spare else (None, None)
        if host is None:
            host = torch.zeros(self.device_values.numel(), dtype=torch.int32, pin_memory=self.device_values.is_cuda)
            event = torch.cuda.Event()
        host.copy_(self.device_values, non_blocking=True)            # on that stream, whichever device is current
        event.record(torch.cuda.current_stream(self.device_values.device))
        with self._lock:
            self.issued += 1
            self._pending[self.issued] = host, event
            oldest = next(iter(self._pending)) if len(self._pending) > self._PENDING_MOST else None
        if oldest is not None:
            self._take(oldest, wait=True)

    def read(self, slot: int, wait: bool):
        """The largest value of a slot over all copies sent so far, waiting for them or as they stand, and their number."""
        with self._lock:
            issued, pending = self.issued, tuple(self._pending)
        for number in pending:
            self._take(number, wait)
        return self._most[slot], issued

    def _take(self, number: int, wait: bool) -> None:
        entry = self._pending.get(number)
        if entry is None:                                            # another thread has looked at it
            return
        if wait:
            entry[1].synchronize()
        with self._lock:
            self._most = [max(m, v) for m, v in zip(self._most, entry[0].view(torch.float32).tolist())]
            if wait and self._pending.pop(number, None) is not None and len(self._spare) < self._SPARE_MOST:
                self._spare.append(entry)


class PackedTensor:
    """Packed codes of a (B, H, T, d_h) tensor; rows [0, length) are valid."""

    def __init__(self, B: int, H: int, t_cap: int, d_head: int, secondary_size: int, radius_bits: int,
                 dtype: torch.dtype, device, joint: Optional[torch.Tensor] = None, outliers: bool = False,
                 sideband_frac: float = 0.125, layout: Optional[tuple] = None, watch: Optional[tuple] = None):
        if d_head % 4:
            raise ValueError(f"d_head={d_head} not divisible by 4")
        self._attn_plans = {}
        self.B, self.H, self.d_head, self.n = B, H, d_head, d_head // 4
        self.d_head_orig = d_head            # smaller for zero-padded heads (PaddedHQMQ): what Q and O carry
        self.t_cap = _round_up(max(t_cap, 1), T_ALIGN)
        self.secondary_size, self.radius_bits = secondary_size, radius_bits
        self.qmax = (1 << radius_bits) - 1
        self.dtype, self.device = dtype, torch.device(device)
        # (idx_bits, main_bits, aux_bits); the default is the tight layout of include/hqmq_amd.h
        self.idx_bits, self.main_bits, self.aux_bits = layout or L.layout_bits(secondary_size, radius_bits)
        n = self.n
        z = dict(dtype=torch.uint8, device=self.device)
        self.main = torch.zeros(B, H, self.t_cap, (n * self.main_bits + 7) // 8, **z)
        self.aux = torch.zeros(B, H, self.t_cap, (n * self.aux_bits + 7) // 8, **z) if self.aux_bits else None
        self.scale = torch.zeros(B, H, self.t_cap, dtype=dtype, device=self.device)
        self.joint = joint
        # the largest finite scale written so far as fp32 bits (the quantize kernel keeps it up to date): the attention
        # kernels' range guard for bf16 / fp32 caches; fp16 scales cannot leave the range
        # (watch: a RangeWatch and this tensor's slot in it, for tensors that are appended together)
        self._watch, self._slot = (None, 0) if dtype == torch.float16 else watch or (RangeWatch(self.device), 0)
        self.scale_max = self._watch_view = None if self._watch is None else self._watch.device_values[self._slot:self._slot + 1]
        # host-side copy of "scale_max lies outside [2^-8, 2^15)": such a cache takes the layout-generic attention kernel, which
        # guards the fp16 range (refresh_range reads the device value; due after bulk appends and every
        # RANGE_CHECK_EVERY small ones, done when the flag is next looked at)
        self._wide = self._huge = False
        self._range_seen = 0                 # copies of the watch that the flag takes account of
        self._appends_since_range_check = 0
        self.length = 0                      # rows written when all sequences advance together
        self.lengths: Optional[torch.Tensor] = None  # per-sequence rows (int32, device) for ragged batches
        self.flags = self.sideband = self.sb_tile_off = self.sb_count = self.sb_overflow = self.sb_coord = None
        self.sb_cap = 0
        if outliers:
            self.flags = torch.zeros(B, H, self.t_cap, (n + 7) // 8, **z)
            self.sb_cap = max(64, int(self.t_cap * n * sideband_frac))
            self.sideband = torch.zeros(B, H, self.sb_cap, 4, dtype=dtype, device=self.device)
            # tiles not yet written read as "no entries"
            self.sb_tile_off = torch.full((B, H, self.t_cap // TILE), 0x7fffffff, dtype=torch.int32, device=self.device)
            self.sb_coord = torch.zeros(B, H, self.sb_cap, dtype=torch.int16, device=self.device)
            self.sb_count = torch.zeros(B, H, dtype=torch.int32, device=self.device)
            self.sb_overflow = torch.zeros(1, dtype=torch.int32, device=self.device)

    @property
    def has_outliers(self) -> bool:
        return self.flags is not None

    def row_bytes(self) -> float:
        """Stored bytes per (token, head), excluding sideband entries."""
        b = self.main.shape[-1] + self.scale.element_size()
        if self.aux is not None:
            b += self.aux.shape[-1]
        if self.flags is not None:
            b += self.flags.shape[-1]
        return b

    def nbytes(self, length: Optional[int] = None) -> int:
        """Algorithmic bytes of the first `length` rows of every (b, h) stream, sideband included."""
        t = self.length if length is None else length
        total = self.B * self.H * t * self.row_bytes()
        if self.sb_count is not None:
            total += int(self.sb_count.sum().item()) * 4 * self.scale.element_size()
        return int(total)

    # arguments of the library's calls that are kept while the attributes they are made of stay what they are
    _STRUCT_FIELDS = frozenset(("main", "aux", "flags", "scale", "sideband", "sb_tile_off", "sb_coord", "sb_count", "sb_overflow", "sb_cap", "joint",
                                "scale_max", "B", "H", "n", "d_head", "t_cap", "dtype", "qmax", "idx_bits", "main_bits", "aux_bits"))

    def __setattr__(self, name, value):
        object.__setattr__(self, name, value)
        if name in self._STRUCT_FIELDS:
            d = self.__dict__
            d["_struct"] = d["_append_template"] = None
            d["_attn_plans"] = {}

    def __getstate__(self):
        """What a copy or a pickle takes along: the tensors and the state, no argument blocks (they hold addresses)."""
        state = dict(self.__dict__)
        for name in ("_struct", "_append_template", "_attn_plans", "_fp8_view"):
            state.pop(name, None)
        if state.pop("_watch_view") is self.scale_max:          # a part of the watch's tensor, there as here
            del state["scale_max"]
        return state

    def __setstate__(self, state):
        d = self.__dict__
        d.update(state, _struct=None, _append_template=None, _attn_plans={})
        d["_watch_view"] = None if self._watch is None else self._watch.device_values[self._slot:self._slot + 1]
        d.setdefault("scale_max", d["_watch_view"])

    @property
    def wide_range(self) -> bool:
        """V scales of a bf16 / fp32 cache outside [2^-8, 2^15).  Waits for the bulk appends whose values have not been
        looked at yet (under stream capture, which begins with everything done, it is read as it stands)."""
        watch = self._watch
        if watch is not None and self._range_seen != watch.issued:
            capturing = torch.cuda.is_current_stream_capturing()
            value, issued = watch.read(self._slot, wait=not capturing)
            self._take_range(value)
            if not capturing:                          # looked at without waiting: due again afterwards
                self._range_seen = issued
        return self._wide

    @wide_range.setter
    def wide_range(self, value: bool) -> None:
        self._wide = bool(value)
        if self._watch is not None:
            self._range_seen = self._watch.issued

    def c_struct(self) -> L.Packed:
        """The tensors as the library takes them; the same object until one of them is replaced."""
        s = self._struct
        if s is not None and s.main_plane == self.main.data_ptr():
            return s
        s = self._make_struct()
        object.__setattr__(self, "_struct", s)
        return s

    def _make_struct(self) -> L.Packed:
        s = L.Packed()
        s.main_plane, s.aux_plane, s.flag_plane = L.ptr(self.main), L.ptr(self.aux), L.ptr(self.flags)
        s.scale_plane = L.ptr(self.scale)
        s.scale_sb, s.scale_sh, s.scale_st = self.scale.stride(0), self.scale.stride(1), self.scale.stride(2)
        s.sideband, s.sb_tile_off, s.sb_cap = L.ptr(self.sideband), L.ptr(self.sb_tile_off), self.sb_cap
        s.sb_coord, s.sb_count = L.ptr(self.sb_coord), L.ptr(self.sb_count)
        s.joint, s.joint_sh, s.K = L.ptr(self.joint), self.joint.stride(0), self.joint.shape[1]
        s.scale_max_bits = L.ptr(self.scale_max)
        return s

    RANGE_CHECK_EVERY = 256     # small appends between two reads of the largest scale; set it to 1 (per cache or on the
                                # class) to read after every append: one device read each, and no window in which a bf16
                                # scale that left [2^-8, 2^15) still meets the unguarded kernels

    def refresh_range(self) -> bool:
        """Reads the largest scale written so far (one device read) and records whether it lies outside [2^-8, 2^15),
        the range inside which the specialised attention kernels keep P * (V scale) and the verbatim chunks in fp16's
        normal range.  The largest scale only grows: a cache of tiny values leaves the flag again when larger ones
        arrive; a cache beyond 2^15 keeps it."""
        if self.scale_max is not None and not self._huge:
            v = float(self.scale_max.view(torch.float32).item())
            if self.scale_max is self._watch_view:          # and what appends on other streams have sent
                v = max(v, self._watch.read(self._slot, wait=True)[0])
            self._take_range(v)
        self._appends_since_range_check = 0
        return self._wide

    def _take_range(self, v: float) -> None:
        self._huge = self._huge or v >= 32768.0
        self._wide = self._huge or 0.0 < v < 2.0 ** -8

    def note_append(self, rows: int, fetch: bool = True) -> bool:
        """Called by the quantizer after an append of `rows` rows per sequence: after bulk appends (a prefill) and every
        RANGE_CHECK_EVERY-th small one the range is due to be read again, never while the stream is being captured.  The
        value sets out for the host at once (fetch=False: the caller fetches the shared watch) and is waited for when the
        flag is next used.  Returns whether it is due."""
        if self.scale_max is None or self._huge:
            return False
        self._appends_since_range_check += 1
        if (rows < 64 and self._appends_since_range_check < self.RANGE_CHECK_EVERY) or torch.cuda.is_current_stream_capturing():
            return False
        if self.scale_max is not self._watch_view:         # somebody else's tensor
            self.refresh_range()
            return False
        self._appends_since_range_check = 0
        if fetch:
            self._watch.fetch()
        return True

    def crop_(self, lengths) -> None:
        """Forgets the rows from `lengths` on (an int for all sequences or an int tensor of B entries): the outlier list and
        its tile offsets go back to the state after the last kept row, so that the rows can be appended again.
        The planes themselves are left as they are (later appends overwrite them)."""
        _crop([self], lengths)

    def with_fp8_table(self) -> "PackedTensor":
        """A view of the same planes whose joint table is rounded to float8_e4m3fn (kept in the table's dtype:
        every e4m3 number is exact there).  The rounded table is computed once per table."""
        import copy
        cached = getattr(self, "_fp8_view", None)
        if cached is None or cached[0] is not self.joint:
            view = copy.copy(self)
            view.joint = self.joint.to(torch.float8_e4m3fn).to(self.joint.dtype)
            cached = (self.joint, view)
            self._fp8_view = cached
        view = cached[1]
        view.length, view.lengths = self.length, self.lengths
        view.wide_range, view._huge = self.wide_range, self._huge
        return view

    def overflowed(self) -> bool:
        """True if an append found the sideband full (reads one int from the device).  The chunks that found no room
        were kept as plain HQMQ chunks (flag cleared, radius code written): nothing decodes to zero, the price is the
        accuracy of those chunks."""
        return self.sb_overflow is not None and bool(int(self.sb_overflow.item()))

    def check_overflow(self) -> None:
        """Raises if an append ran out of sideband room (see overflowed)."""
        if self.overflowed():
            raise L.HqmqError(f"outlier sideband overflow: more than {self.sb_cap} flagged chunks in one (b, h) stream "
                              "(the chunks beyond it were stored as plain HQMQ chunks); allocate the cache with a larger "
                              "sideband_frac")


def _crop_outliers_torch(t, lengths) -> None:
    """What ops.crop does, in torch: for caches whose tensors are not on the GPU (bookkeeping without kernels)."""
    B, H, tiles = t.B, t.H, t.t_cap // TILE
    lens = torch.full((B,), lengths, dtype=torch.int64, device=t.device) if isinstance(lengths, int) else lengths.to(torch.int64)
    tile, r = lens // TILE, lens % TILE
    tc = tile.clamp(max=tiles - 1)
    off = t.sb_tile_off.gather(2, tc.view(B, 1, 1).expand(B, H, 1)).squeeze(2).to(torch.int64)
    # flagged chunks of the kept rows of the tile the cut falls into
    rows = tc.view(B, 1, 1) * TILE + torch.arange(TILE, device=t.device).view(1, 1, TILE)
    fl = t.flags.gather(2, rows.view(B, 1, TILE, 1).expand(B, H, TILE, t.flags.shape[-1]))
    bits = sum((fl >> i) & 1 for i in range(8)).to(torch.int64).sum(-1)                          # (B, H, TILE)
    kept = torch.arange(TILE, device=t.device).view(1, 1, TILE) < r.view(B, 1, 1)
    count = t.sb_count.to(torch.int64)
    new = torch.where((tile >= tiles).view(B, 1) | (off > count), count, off + (bits * kept).sum(-1))
    t.sb_count.copy_(torch.minimum(new, count).to(torch.int32))
    first_free = (lens + TILE - 1) // TILE             # tiles from here on hold no kept row: unwritten again
    gone = torch.arange(tiles, device=t.device).view(1, 1, tiles) >= first_free.view(B, 1, 1)
    t.sb_tile_off.masked_fill_(gone.expand(B, H, tiles), 0x7fffffff)
    dropped = torch.arange(t.t_cap, device=t.device).view(1, 1, t.t_cap, 1) >= lens.view(B, 1, 1, 1)
    t.flags.masked_fill_(dropped, 0)                   # no flag without an entry behind it


def _crop(tensors, lengths) -> None:
    """Crops PackedTensors of one cache; those that carry outliers share a launch where their shapes agree."""
    if isinstance(lengths, int):
        for t in tensors:
            t.length = min(t.length, lengths)
    else:
        for t in tensors:
            if lengths.numel() != t.B:
                raise L.HqmqError(f"crop_ needs one length per sequence ({t.B}), got {tuple(lengths.shape)}")
        lengths = lengths.reshape(-1).to(device=tensors[0].main.device).clamp(min=0).to(torch.int32).contiguous()
        for t in tensors:
            t.lengths = lengths.to(t.main.device)
    flagged = [t for t in tensors if t.flags is not None]
    if not flagged:
        return
    if not flagged[0].flags.is_cuda:
        for t in flagged:
            _crop_outliers_torch(t, lengths)
        return
    from . import ops
    shared = len({(t.B, t.H, t.t_cap, t.n, t.flags.device) for t in flagged}) == 1
    for group in [flagged] if shared else [[t] for t in flagged]:
        ops.crop(group, lengths if isinstance(lengths, int) else group[0].lengths)


@dataclass
class PackedKV:
    """The compressed K and V of one layer."""
    K: PackedTensor
    V: PackedTensor

    @property
    def length(self) -> int:
        return self.K.length

    def nbytes(self, length: Optional[int] = None) -> int:
        return self.K.nbytes(length) + self.V.nbytes(length)

    def crop_(self, lengths) -> None:
        """Forgets the rows from `lengths` on in K and V (see PackedTensor.crop_)."""
        _crop([self.K, self.V], lengths)
