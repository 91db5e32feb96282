"""Persistent, capacity-growing page storage on the HIP device.

Mirrors ``PolarKBlockStorage`` and ``QuantVBlockStorage``
(rfsn_v11/generation/storage.py:17-169): structure-of-arrays buffers
``[B, H, capacity, ...]``, lazy allocation at capacity 4, capacity doubling,
``[:block_count]`` views, and the same growth telemetry
(``reallocation_count``, ``bytes_copied_during_growth``).  The HIP encoder
writes pages straight into the slots; a bulk reservation performs the
reference's sequence of doublings as one reallocation and one copy while
reporting the counters the doubling sequence would produce.
"""

from __future__ import annotations

from dataclasses import dataclass, field
from math import prod
from typing import Optional, Tuple

import torch

from . import _lib
from .payload import PolarKeyBlock, QuantizedVBlock


def _doublings(capacity: int, needed: int):
    """Capacities at which the reference would call ``_grow`` to reach ``needed``."""
    caps = []
    while needed > capacity:
        caps.append(capacity)
        capacity *= 2
    return caps, capacity


def _regrow(t: Optional[torch.Tensor], new_cap: int) -> Optional[torch.Tensor]:
    if t is None:
        return None
    shape = list(t.shape)
    shape[2] = new_cap
    out = torch.zeros(shape, dtype=t.dtype, device=t.device)
    out[:, :, : t.shape[2]] = t
    return out


# The storages' buffers; their forms are the encoder's at the first reservation, then their own.
_KEY_BUFFERS = dict.fromkeys(("radii", "angle_codes_l1", "angle_codes_deep", "radii_scales"))
_VALUE_BUFFERS = dict.fromkeys(("codes", "scales"))


class Growth:
    """Larger buffers of one or two storages, not yet theirs: ``commit`` hands
    them over, so a caller whose append is rejected afterwards leaves the
    storages as they were.

    Slots [0, block_count) are copied from the present buffers, the ``fresh``
    slots after them are left to the caller, who writes them next, and the
    slots past those are zero.  On a HIP device that is one tp_grow_rows launch
    for every buffer (none when there is nothing to copy or clear) instead of a
    fill and a copy each, twice over for a first reservation above the initial
    capacity (measured: a 32,773-token prompt into a new cache of 8 heads 198 ->
    122 us, 6,100 float32 tokens 189 -> 95, four chunks of 2,048 with their
    history read back 494 -> 274)."""

    def __init__(self, fresh: int = 0):
        self.fresh = fresh
        self._sets: list = []  # (storage, {attribute: new buffer}, capacity, reallocations, bytes grown)
        # (old buffer or None, its capacity, new buffer, its capacity, pages kept, page bytes, (batch, head) rows)
        self._rows: list = []

    def add(self, storage, shapes: dict, needed: int, initial_capacity: int, device) -> None:
        """Room for ``needed`` pages in ``storage``; ``shapes`` maps its buffer
        attributes to ((B, H), page shape, dtype), or None for a buffer that the
        layout does not have: the forms of a first reservation.  A buffer that is
        there grows in its own form, on its own device, whatever ``shapes`` says
        (its pages may be ``append``'s, of another length).  The counters move as
        the reference's sequence of doublings from the initial capacity moves them
        (storage.py:34-73)."""
        held = getattr(storage, next(iter(shapes)))
        first = held is None
        cap = initial_capacity if first else storage.capacity
        caps, new_cap = _doublings(cap, needed)
        if not caps and not first:
            return
        if not first:
            device = held.device
        make = torch.empty if device.type == "cuda" else torch.zeros
        made, per_slot = {}, 0
        for name, spec in shapes.items():
            old, old_cap = None if first else getattr(storage, name), 0
            if old is not None:
                shape, dtype = list(old.shape), old.dtype
                old_cap, shape[2] = shape[2], new_cap
            elif first and spec is not None:
                (B, H), page, dtype = spec
                shape = [B, H, new_cap, *page]
            else:
                made[name] = None
                continue
            page_bytes, rows = prod(shape[3:]) * dtype.itemsize, shape[0] * shape[1]
            new = made[name] = make(shape, dtype=dtype, device=device)
            per_slot += rows * page_bytes
            if page_bytes:
                self._rows.append((old, old_cap, new, new_cap, storage.block_count, page_bytes, rows))
        self._sets.append((storage, made, new_cap, len(caps), per_slot * sum(caps)))

    def fill(self) -> None:
        """Copies the kept pages and clears the spare ones."""
        held, launches, dev, heads = [], [], None, 0  # one launch for a cache's two storages
        for old, old_cap, new, cap, keep, page, rows in self._rows:
            if not new.is_cuda:
                if keep:
                    new[:, :, :keep] = old[:, :, :keep]
                continue
            used = min(cap, keep + self.fresh)
            if keep or used < cap:
                if keep and not old.is_contiguous():
                    old = old.contiguous()
                held.append(old)
                if rows != heads or new.device != dev:
                    dev, heads, bufs = new.device, rows, []
                    launches.append((dev, heads, bufs))
                bufs.append(_lib.TPGrow(old.data_ptr() if keep else None, new.data_ptr(),
                                        old_cap * page if keep else 0, cap * page, keep * page, used * page))
        for dev, heads, bufs in launches:
            st = _lib.call_on(dev, _lib.lib().tp_grow_rows, (_lib.TPGrow * len(bufs))(*bufs), len(bufs), heads,
                              _lib.stream_handle(dev))
            _lib.check(st, "tp_grow_rows")

    def buffers(self, storage) -> dict:
        """``storage``'s buffers by name as they will be after ``commit``."""
        for s, made, _, _, _ in self._sets:
            if s is storage:
                return made
        return vars(storage)

    def commit(self) -> None:
        for storage, made, cap, reallocs, grown in self._sets:
            for name, new in made.items():
                setattr(storage, name, new)
            storage.capacity = cap
            storage.reallocation_count += reallocs
            storage.bytes_copied_during_growth += grown


@dataclass
class PolarKBlockStorage:
    radii: Optional[torch.Tensor] = None
    angle_codes_l1: Optional[torch.Tensor] = None
    angle_codes_deep: Optional[torch.Tensor] = None
    radii_scales: Optional[torch.Tensor] = None
    block_count: int = 0
    capacity: int = 0
    metadata: dict = field(default_factory=dict)
    reallocation_count: int = 0
    bytes_copied_during_growth: int = 0

    def _buffers(self):
        return [t for t in (self.radii, self.angle_codes_l1, self.angle_codes_deep, self.radii_scales) if t is not None]

    def plan(self, growth: Growth, needed: int, encoder, B: int, H: int, device, initial_capacity: int = 4) -> None:
        """Adds what ``needed`` pages take to ``growth`` (storage.py:34-73 growth rule)."""
        growth.add(self, encoder.page_shapes(B, H) if self.radii is None else _KEY_BUFFERS, needed, initial_capacity,
                   device)

    def reserve(self, needed: int, encoder, B: int, H: int, device, initial_capacity: int = 4) -> None:
        """Make room for ``needed`` pages."""
        if self.radii is None:
            self.metadata = encoder.metadata
        growth = Growth()
        self.plan(growth, needed, encoder, B, H, torch.device(device), initial_capacity)
        growth.fill()
        growth.commit()

    def append(self, block: PolarKeyBlock, initial_capacity: int = 4) -> None:
        """Copy one 4-D page into the next slot (storage.py:75-87)."""
        B, H = block.radii.shape[:2]
        if self.radii is None:
            self.radii = torch.zeros((B, H, initial_capacity) + tuple(block.radii.shape[2:]), dtype=block.radii.dtype, device=block.radii.device)
            self.angle_codes_l1 = torch.zeros((B, H, initial_capacity) + tuple(block.angle_codes_l1.shape[2:]), dtype=torch.uint8, device=block.radii.device)
            self.angle_codes_deep = torch.zeros((B, H, initial_capacity) + tuple(block.angle_codes_deep.shape[2:]), dtype=torch.uint8, device=block.radii.device)
            self.radii_scales = (
                torch.zeros((B, H, initial_capacity, 1, 1), dtype=torch.float16, device=block.radii.device)
                if block.radii_scales is not None else None
            )
            self.metadata = block.metadata
            self.capacity = initial_capacity
        elif self.block_count >= self.capacity:
            self.bytes_copied_during_growth += sum(t.numel() * t.element_size() for t in self._buffers())
            self.reallocation_count += 1
            new_cap = self.capacity * 2
            self.radii = _regrow(self.radii, new_cap)
            self.angle_codes_l1 = _regrow(self.angle_codes_l1, new_cap)
            self.angle_codes_deep = _regrow(self.angle_codes_deep, new_cap)
            self.radii_scales = _regrow(self.radii_scales, new_cap)
            self.capacity = new_cap
        idx = self.block_count
        self.radii[:, :, idx] = block.radii
        self.angle_codes_l1[:, :, idx] = block.angle_codes_l1
        self.angle_codes_deep[:, :, idx] = block.angle_codes_deep
        if self.radii_scales is not None and block.radii_scales is not None:
            self.radii_scales[:, :, idx] = block.radii_scales.reshape(B, H, 1, 1)
        self.block_count += 1

    def to_unified_block(self, shape: Tuple[int, ...]) -> PolarKeyBlock:
        """5-D view of the valid pages (storage.py:89-102)."""
        if self.radii is None or self.block_count == 0:
            raise ValueError("No compressed blocks to materialize")
        n = self.block_count
        return PolarKeyBlock(
            radii=self.radii[:, :, :n],
            angle_codes_l1=self.angle_codes_l1[:, :, :n],
            angle_codes_deep=self.angle_codes_deep[:, :, :n],
            radii_scales=self.radii_scales[:, :, :n] if self.radii_scales is not None else None,
            shape=shape,
            block_size=self.metadata.get("block_size", shape[-1]),
            head_dim=shape[-1],
            metadata=self.metadata,
        )


@dataclass
class QuantVBlockStorage:
    codes: Optional[torch.Tensor] = None
    scales: Optional[torch.Tensor] = None
    group_size: int = 32
    block_count: int = 0
    capacity: int = 0
    reallocation_count: int = 0
    bytes_copied_during_growth: int = 0

    def plan(self, growth: Growth, needed: int, B: int, H: int, device, initial_capacity: int = 4) -> None:
        # Stored 6-D [B, H, cap, 1, 64, 128] like storage.py:121-131.
        growth.add(self, {"codes": ((B, H), (1, 64, 128), torch.int8), "scales": ((B, H), (1, 64, 4), torch.float16)}
                   if self.codes is None else _VALUE_BUFFERS, needed, initial_capacity, device)

    def reserve(self, needed: int, B: int, H: int, device, initial_capacity: int = 4) -> None:
        growth = Growth()
        self.plan(growth, needed, B, H, torch.device(device), initial_capacity)
        growth.fill()
        growth.commit()

    def append(self, block: QuantizedVBlock, initial_capacity: int = 4) -> None:
        """Copy one page ``codes [B,H,1,64,128]`` into the next slot (storage.py:149-158)."""
        B, H = block.codes.shape[:2]
        if self.codes is None:
            self.reserve(1, B, H, block.codes.device, initial_capacity)
        elif self.block_count >= self.capacity:
            self.bytes_copied_during_growth += self.codes.numel() + self.scales.numel() * 2
            self.reallocation_count += 1
            self.codes = _regrow(self.codes, self.capacity * 2)
            self.scales = _regrow(self.scales, self.capacity * 2)
            self.capacity *= 2
        idx = self.block_count
        self.codes[:, :, idx] = block.codes.reshape(B, H, 1, 64, 128)
        self.scales[:, :, idx] = block.scales.reshape(B, H, 1, 64, 4)
        self.group_size = block.group_size
        self.block_count += 1

    def to_quantized_block(self) -> QuantizedVBlock:
        """5-D view ``[B, H, S, 64, .]`` of the valid pages (storage.py:160-169)."""
        if self.codes is None or self.block_count == 0:
            raise ValueError("No quantized V blocks to materialize")
        n = self.block_count
        return QuantizedVBlock(
            codes=self.codes[:, :, :n].squeeze(3),
            scales=self.scales[:, :, :n].squeeze(3),
            group_size=self.group_size,
        )


def pages_of(k_storage: PolarKBlockStorage, v_storage: QuantVBlockStorage, growth: Optional[Growth] = None) -> _lib.TPPages:
    """``tp_pages`` over the whole capacity of a pair of storages (as they will
    be after ``growth`` is committed, if given)."""
    if growth is None:
        k, v, capacity = vars(k_storage), vars(v_storage), k_storage.capacity
    else:
        k, v = growth.buffers(k_storage), growth.buffers(v_storage)
        capacity = k["radii"].shape[2]
    return _lib.TPPages(
        _lib.ptr(k["radii"]),
        _lib.ptr(k["radii_scales"]),
        _lib.ptr(k["angle_codes_l1"]),
        _lib.ptr(k["angle_codes_deep"]),
        _lib.ptr(v["codes"]),
        _lib.ptr(v["scales"]),
        int(capacity),
    )
