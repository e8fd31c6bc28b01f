"""Planned multi-LoRA op: build the adapter-grouped work tiles once per batch, then apply
shrink + expand for every (layer, target) of the step.

The reference rebuilds its segment tensors once per forward
(valora/server/router/model_infer/model_rpc.py:381) and then issues 8 op launches per layer with
the same per-token ids (valora/models/peft/lora_unordered_batch_infer.py:946-988,1611-1622);
``LoraPlan`` is that once-per-forward object for the gfx950 kernels.  The intermediate
``v = x @ A.T`` never becomes a caller-visible tensor: it lives in the plan's scratch buffer
between the two launches, rounded to the operand dtype exactly once -- where the reference stores
its ``delta`` tensor.
"""
from __future__ import annotations

from typing import Optional

import torch

from . import _lib
from ._ext import binding as _b


class LoraPlan:
    def __init__(self, ids: torch.Tensor, a_start: torch.Tensor, a_len: torch.Tensor, max_rank: int,
                 n_slots: int = 4, hidden: int = 4096, bm_shrink: Optional[int] = None,
                 bm_expand: Optional[int] = None, ksplit: Optional[int] = None,
                 reduce_in_expand: Optional[bool] = None, one_launch: Optional[bool] = None,
                 one_launch_no_wait: bool = False, shrink_recompute: bool = False, expand_column_loop: bool = False,
                 one_launch_never_ready: bool = False, _merged: int = -1, _cut: bool = True):
        """``ids``: int64 per-token adapter index (negative = no adapter); ``a_start`` / ``a_len``:
        the pool index (``a_len = n_slots * rank``); ``max_rank``: widest rank among the resident
        adapters (the reference's ``max_lora_dim``, lora_unordered_batch_infer.py:181-182).
        ``one_launch``: asks for shrink and expand as work items of one grid (decode-like batches; forces
        16-token tiles and at most 16 K chunks of all targets together, needs ``max_rank <= 64``; ``runs_in_one_launch`` says
        which calls get it); ``None`` takes the tile table's choice.
        ``one_launch_no_wait`` makes every expand item take its give-up path at once, ``one_launch_never_ready`` after
        waiting out its bound, ``shrink_recompute`` makes a shrink that sums its K chunks inside the launch compute them all
        in one workgroup (all for tests); ``expand_column_loop`` is accepted and without effect."""
        if not ids.is_cuda:
            raise RuntimeError("ids must be a CUDA tensor")
        if ids.dtype != torch.long or a_start.dtype != torch.long or a_len.dtype != torch.long:
            raise RuntimeError("expected scalar type Long")
        self.device = ids.device
        self.T = int(ids.numel())
        self.n_adapters = int(a_start.numel())
        self.n_slots = n_slots
        self.max_rank = int(max_rank)
        # A compensation plan works on the tokens the merged adapter leaves over.  How many those are is known on the
        # device only; the merged adapter is the dominant one, so its tiles are those of a batch half the size.
        # Measured over 64 to 7177 tokens, 4 to 30 adapters of ranks 8 to 128, 2048 to 5120 wide: 0.74 to 1.02 of the
        # time with the whole batch's tiles (918 tokens, ranks 16-64, 8 layers: 630 -> 512 us).
        t_bm_shrink, t_ksplit, t_bm_expand, t_flags = _b.tile_lookup(self.T if _merged < 0 else (self.T + 1) // 2, self.max_rank,
                                                                     hidden, self.n_adapters)
        self.bm_shrink = t_bm_shrink if bm_shrink is None else bm_shrink
        self.bm_expand = t_bm_expand if bm_expand is None else bm_expand
        self.ksplit = max(1, t_ksplit if ksplit is None else ksplit)
        rie = bool(t_flags & _lib.REDUCE_IN_EXPAND) if reduce_in_expand is None else reduce_in_expand
        self.flags = _lib.REDUCE_IN_EXPAND if rie else 0
        self.one_launch = bool(t_flags & _lib.ONE_LAUNCH if one_launch is None else one_launch)
        if self.one_launch and (self.max_rank > 64 or bm_shrink not in (None, 16) or bm_expand not in (None, 16)):
            if one_launch:
                raise RuntimeError("No suitable kernel. the one-launch op needs 16-token tiles and max_rank <= 64")
            self.one_launch = False
        if self.one_launch:
            self.bm_shrink = self.bm_expand = 16
            self.ksplit = max(2, self.ksplit)
            self.flags = (_lib.REDUCE_IN_EXPAND | _lib.ONE_LAUNCH | (_lib.ONE_LAUNCH_NO_WAIT if one_launch_no_wait else 0) |
                          (_lib.ONE_LAUNCH_NEVER_READY if one_launch_never_ready else 0))
        if shrink_recompute:
            self.flags |= _lib.SHRINK_RECOMPUTE
        if expand_column_loop:
            self.flags |= _lib.EXPAND_COLUMN_LOOP
        # plan, scratch and the calls themselves live on the native side (csrc/binding.cpp)
        if _cut:
            self._native = _b.NativePlan(ids, a_start, a_len, self.max_rank, n_slots, self.bm_shrink, self.bm_expand,
                                         self.ksplit, self.flags, int(_merged))

    @classmethod
    def of_widths(cls, ids: torch.Tensor, a_start: torch.Tensor, a_len: torch.Tensor, max_rank: int, widths,
                  n_slots: int = 4) -> list:
        """One plan per input width, of the same batch: what ``LoraPlan(..., hidden=w)`` makes for each ``w`` of
        ``widths`` (at most four), with the tiles of all of them cut in one launch."""
        plans = [cls(ids, a_start, a_len, max_rank, n_slots=n_slots, hidden=w, _cut=False) for w in widths]
        shapes = [[p.bm_shrink, p.bm_expand, p.ksplit, p.flags] for p in plans]
        for p, native in zip(plans, _b.NativePlan.several(ids, a_start, a_len, int(max_rank), n_slots, shapes)):
            p._native = native
        return plans

    @property
    def buf(self) -> torch.Tensor:
        return self._native.buf

    @property
    def scratch(self) -> torch.Tensor:
        return self._native.scratch

    @property
    def scratch_per_target(self) -> int:
        return self._native.scratch_per_target

    @property
    def handle(self):
        """The plan as the C ABI takes it (``mlora_plan``)."""
        buf = self._native.buf
        return _lib.Plan(_lib.ptr(buf), buf.numel(), self.T, self.n_adapters, self.bm_shrink, self.bm_expand, self.n_slots)

    def runs_in_one_launch(self, h_out: int, n_targets: int = 1) -> bool:
        """Whether a call of this plan on ``n_targets`` targets of ``h_out`` columns is one launch."""
        return self.one_launch and bool(_lib.lib().mlora_runs_in_one_launch(self.T, self.n_adapters, self.max_rank, int(h_out),
                                                                            self.ksplit, int(n_targets)))

    def rebuild(self, ids: Optional[torch.Tensor] = None) -> None:
        """Cut the tiles again, in place, for the next batch of the same size (``ids`` of the same length; None
        re-reads the tensor the plan was made from, whose contents may have changed).  One launch on the current
        stream, no allocation: a serving loop that replays one HIP graph per step captures this call at the
        head of the step and refills its ids tensor before each replay (the reference rebuilds its segment
        tensors once per forward, valora/server/router/model_infer/model_rpc.py:381)."""
        self._native.rebuild(ids)

    # -- introspection (synchronises; for tests and diagnostics) --------------------------------
    def header(self) -> dict:
        h = self.buf[:128].view(torch.int32).cpu().tolist()
        names = ["magic", "T", "n_adapters", "n_tiles_shrink", "n_tiles_expand", "n_groups", "max_rank",
                 "reserved", "bm_shrink", "bm_expand", "n_active"]
        return dict(zip(names, h))

    def perm(self) -> torch.Tensor:
        n = self.header()["n_active"]
        return self.buf.view(torch.int32)[32:32 + n].clone()

    def _section(self, index: int) -> torch.Tensor:
        # layout mirrors plan_layout() in csrc/mlora_internal.h
        T, A = self.T, self.n_adapters
        up8 = lambda v: (v + 7) // 8 * 8
        max_tiles = (T + 15) // 16 + min(A, T)
        off_perm = 32
        off_pad = up8(off_perm + T)
        off_prank = up8(off_pad + T)
        off_ts = up8(off_prank + T)
        off_te = off_ts + max_tiles * 8
        words = self.buf.view(torch.int32)
        h = self.header()
        if index == 0:
            return words[off_pad:off_pad + h["n_active"]].clone()
        if index == 1:
            return words[off_prank:off_prank + h["n_active"]].clone()
        if index == 2:
            return words[off_ts:off_ts + h["n_tiles_shrink"] * 8].view(-1, 8).clone()
        return words[off_te:off_te + h["n_tiles_expand"] * 8].view(-1, 8).clone()

    def position_adapters(self): return self._section(0)
    def position_ranks(self): return self._section(1)
    def tiles_shrink(self): return self._section(2)
    def tiles_expand(self): return self._section(3)

    # -- the op -------------------------------------------------------------------------------------
    def _check(self, x, y, key_buffer, value_buffer):
        for t, w in ((x, key_buffer), (y, value_buffer)):
            if t is None:
                continue
            if t.dim() != 2 or t.size(0) != self.T or not t.is_contiguous():
                raise RuntimeError(f"x and y must be contiguous [T={self.T}, H] matrices")
            if _lib.dtype_code(t.dtype) < 0 or w.dtype != t.dtype:
                raise RuntimeError(f"No suitable kernel. h_in={t.size(1)} h_out={t.size(1)} dtype={t.dtype}")

    def shrink(self, x: torch.Tensor, key_buffer: torch.Tensor, a_start, a_len, a_loc, slot: int) -> None:
        """First launch of the op alone: ``v = x @ A_a.T`` into ``self.scratch``."""
        self._check(x, None, key_buffer, None)
        pa = _lib.make_pool(key_buffer, a_start, a_len, a_loc, x.size(1), self.n_slots)
        _lib.check(_lib.lib().mlora_shrink(
            _lib.current_stream(self.device), self.handle, _lib.ptr(self.scratch), self.scratch.numel(),
            _lib.ptr(x), self.T, x.size(1), self.max_rank, pa, int(slot), int(self.ksplit), None, 0, 0, 0,
            self.flags, _lib.dtype_code(x.dtype)))

    def expand(self, y: torch.Tensor, value_buffer: torch.Tensor, a_start, a_len, a_loc, slot: int,
               scales: torch.Tensor) -> None:
        """Second launch alone: ``y += scale_a * v @ B_a`` with v taken from ``self.scratch``."""
        self._check(None, y, None, value_buffer)
        if scales.dtype != y.dtype:
            scales = scales.to(y.dtype)
        pb = _lib.make_pool(value_buffer, a_start, a_len, a_loc, y.size(1), self.n_slots)
        _lib.check(_lib.lib().mlora_expand(
            _lib.current_stream(self.device), self.handle, _lib.ptr(y), self.T, y.size(1), _lib.ptr(self.scratch),
            None, 0, self.max_rank, pb, int(slot), _lib.ptr(scales), int(self.ksplit), self.flags,
            _lib.dtype_code(y.dtype)))

    def apply_multi(self, ys, x: torch.Tensor, key_buffer: torch.Tensor, value_buffers, a_start: torch.Tensor,
                    a_len: torch.Tensor, a_loc: torch.Tensor, slots, scales: torch.Tensor) -> None:
        """Several targets that read the same ``x`` (q, k, v of a layer; gate and up) in two launches:
        ``ys[i] += scale_a * (x @ A_a[slots[i]].T) @ B_a[slots[i]]``.  ``value_buffers`` is one pool tensor or
        one per target.  Same results as ``apply`` called once per target."""
        # (a call that two launches are faster for -- gate+up, ranks above 32, more than four K chunks -- is run as two
        # by the library whatever the flag says: same tiles, same split, same bits)
        self._native.apply_multi(ys, x, key_buffer, value_buffers, a_start, a_len, a_loc, slots, scales)

    def apply(self, y: torch.Tensor, x: torch.Tensor, key_buffer: torch.Tensor, value_buffer: torch.Tensor,
              a_start: torch.Tensor, a_len: torch.Tensor, a_loc: torch.Tensor, slot: int,
              scales: torch.Tensor) -> None:
        """``y[t] += scale_a * (x[t] @ A_a.T) @ B_a`` in place for every token with an adapter."""
        self._native.apply(y, x, key_buffer, value_buffer, a_start, a_len, a_loc, slot, scales)
