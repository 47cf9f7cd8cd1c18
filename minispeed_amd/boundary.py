"""The fused boundary step: K1 (+ its tile fold) -> K2 -> K3 on the current
HIP stream with one device->host read-back.

Replaces the unfused sequence of minispeed's
``DeepSpeedEngine._take_optimizer_step`` (engine.py:268-322):

    flatten_grads            flat.py:196-213       \\
    has_overflow             precision.py:79-87     > K1 per group
    unscale_grads            flat.py:243-247       /   (+ sumsq per 2048-element tile, folded)
    reduce_gradients         stage_1_and_2.py:86-102   identity at world 1
    clip_gradients           stage_1_and_2.py:105-128  K2 (norm, coef, skip)
    FlatAdam.step            optim/adam.py:59-93   \\
    sync_parameters          stage_1_and_2.py:79-83 > K3 per group
    (stage 3) free_parameters  stage_3.py:88-110   /
    DynamicLossScaler.update precision.py:50-62        K2 (checked on host)

K3 is gated on the device overflow flag, so no launch waits for the host: the
only synchronisation is the wait for the ``ms_step_scalars_t`` that K2 also
writes to pinned host memory.
"""

from __future__ import annotations

import collections
import ctypes
import time
import weakref
from dataclasses import dataclass
from typing import List, Optional, Sequence, Tuple

import numpy as np
import torch

from . import _native
from .flat import FlatParamGroup, record_streams


def adamw_params(
    lr: float, betas: Sequence[float], eps: float, weight_decay: float, step: int,
    grad_scale: float = 1.0, unscale: bool = False,
) -> _native.AdamWParams:
    """Round this step's AdamW scalars the way the torch op sequence of
    optim/adam.py:72-91 does: every Python double becomes fp32 at the op that
    consumes it.  The doubles are computed here and stored into the
    ``c_float`` fields of the struct, a C double -> float conversion that
    rounds to nearest even, as ``np.float32`` does."""
    lr = float(lr)
    beta1, beta2 = (float(b) for b in betas)
    wd = float(weight_decay)
    return _native.AdamWParams(
        neg_lr=-lr,
        decay_alpha=-lr * wd,
        beta1=beta1,
        one_minus_beta1=1.0 - beta1,
        beta2=beta2,
        one_minus_beta2=1.0 - beta2,
        bias_c1=1.0 - beta1 ** step,
        bias_c2=1.0 - beta2 ** step,
        eps=float(eps),
        grad_scale=float(grad_scale),
        decay=1 if wd != 0.0 else 0,
        unscale=_native.SCALE_DIVIDE if unscale else _native.SCALE_NONE,
    )


class _PinnedSlots:
    """64-byte slots of pinned host memory for :class:`HostReadback`, cut from
    4 KB slabs: pinning memory of its own took a new optimizer's first step
    30-40 us (3.3M params 217 -> 188 us, 124M 843 -> 804).  Only
    the newest slab's free slots are kept; an older slab goes back to torch
    with its last user.  The deques are the only shared state and their
    appends and pops are atomic, so a slot may come back from a finalizer at
    any point of any thread."""

    SLOT, SLAB = 64, 4096

    def __init__(self):
        self._free = {}       # device -> slots (slab, offset)
        self._newest = {}     # device -> slab

    def take(self):
        dev = torch.cuda.current_device()
        free = self._free.setdefault(dev, collections.deque())
        try:
            slab, off = free.popleft()
        except IndexError:
            slab, off = torch.empty(self.SLAB, dtype=torch.uint8, pin_memory=True), 0
            self._newest[dev] = slab
            free.extend((slab, k) for k in range(self.SLOT, self.SLAB, self.SLOT))
        return dev, slab, off

    def give(self, dev, slab, off, ready) -> None:
        # a slot whose kernel may still write is not handed out again
        if ready[0] == 1 and self._newest.get(dev) is slab:
            self._free[dev].append((slab, off))


_SLOTS = _PinnedSlots()


class HostReadback:
    """K2's result in pinned host memory, read without a copy and without
    anything between K2 and K3 in the stream.

    ``arm()`` clears the struct's ``ready`` word before K2 is launched with
    ``ptr`` as its host output; K2 writes the struct, makes it visible
    system-wide and then sets ``ready``; ``wait()`` polls that word (K3, queued
    behind K2, keeps running) and returns the struct.  An event recorded
    after K2 for the host to wait on put a 4-5.5 us gap between K2 and K3.
    If the word does not turn within ``patience`` seconds (a deep queue of
    earlier work), the stream is synchronised instead, which also reports a
    device error."""

    _READY = _native.StepScalars.ready.offset

    def __init__(self, patience: float = 5.0):
        dev, slab, off = _SLOTS.take()
        self.host = slab[off:off + _native.SCALARS_BYTES]
        self._bytes = self.host.numpy()
        self._ready = self._bytes[self._READY:self._READY + 4].view(np.uint32)
        self._ready[0] = 1
        weakref.finalize(self, _SLOTS.give, dev, slab, off, self._ready).atexit = False
        self.patience = patience

    @property
    def ptr(self) -> int:
        return self.host.data_ptr()

    def arm(self) -> None:
        self._ready[0] = 0

    @property
    def _pending(self) -> np.ndarray:
        """One truth value: armed, and K2's result not there yet."""
        return self._ready != 1

    def wait(self, stream: int) -> _native.StepScalars:
        ready = self._ready
        spins = 0
        deadline = None
        while ready[0] != 1:
            spins += 1
            if spins & 0x3FF == 0:
                now = time.perf_counter()
                if deadline is None:
                    deadline = now + self.patience
                elif now > deadline:
                    _native.hip_check(_native.hip_runtime().hipStreamSynchronize(stream),
                                      "hipStreamSynchronize")
                    if self._pending[0]:
                        raise RuntimeError("the norm/clip kernel's host result did not arrive")
                    break
        return _native.StepScalars.from_buffer_copy(self._bytes.tobytes())


class Workspace:
    """Device scratch of the boundary step (no allocation per step)."""

    def __init__(self, device: torch.device, ngroups: int):
        self.device = device
        self.nblk = _native.stats_blocks()
        self.ngroups = ngroups
        n = max(1, ngroups) * self.nblk
        self.partials = torch.empty(n, dtype=torch.float64, device=device)
        self.flags = torch.empty(n, dtype=torch.int32, device=device)
        self.scalars = torch.empty(_native.SCALARS_BYTES, dtype=torch.uint8, device=device)
        # K1's tile slots, the groups of a boundary one after another; grown
        # on demand, with every stream that used them recorded
        self.tile_sums: Optional[torch.Tensor] = None
        self.tile_flags: Optional[torch.Tensor] = None
        self._tile_streams: set = set()
        # the boundary call's arguments, filled in for each one
        self.tile_stats = (_native.TileStats * max(1, ngroups))()
        self.groups = (_native.BoundaryGroup * max(1, ngroups))()
        self.norm = _native.NormArgs(
            block_sumsq=self.partials.data_ptr(), block_flag=self.flags.data_ptr(),
            nblk=self.nblk, out=self.scalars.data_ptr())
        # K2 also writes its result to pinned host memory, which the host
        # polls (HostReadback): no copy, and K3, queued behind K2, keeps
        # running while the host does its bookkeeping
        self.readback = HostReadback()
        self.norm.out_host = self.readback.ptr
        self._stream: Optional[torch.cuda.Stream] = None   # stream of the last boundary

    def tile_ptrs(self, ntiles: int, cur: torch.cuda.Stream):
        """Addresses (sums, flags) of at least ``ntiles`` K1 tile slots for
        kernels on the current stream ``cur``."""
        if self.tile_sums is None or self.tile_sums.numel() < ntiles:
            # the replaced buffers' memory stays with the streams recorded on
            # them until those have run what was queued there
            self.tile_sums = torch.empty(max(1, ntiles), dtype=torch.float64, device=self.device)
            self.tile_flags = torch.empty(max(1, ntiles), dtype=torch.int32, device=self.device)
            self._tile_streams = set()
        if cur.cuda_stream not in self._tile_streams:
            self.tile_sums.record_stream(cur)
            self.tile_flags.record_stream(cur)
            self._tile_streams.add(cur.cuda_stream)
        return self.tile_sums.data_ptr(), self.tile_flags.data_ptr()

    def enter(self) -> torch.cuda.Stream:
        """Called at the start of a boundary; returns the current stream,
        which the boundary's kernels run on.  Kernels of the previous
        boundary (K3 reading the scalars and segment tables this boundary
        overwrites) may still run on its stream; if the current stream is
        another one, it first waits for everything queued there."""
        cur = torch.cuda.current_stream(self.device)
        if self._stream is not None and self._stream != cur:
            cur.wait_stream(self._stream)
        self._stream = cur
        return cur

    def finish_readback(self) -> _native.StepScalars:
        """Wait for K2's scalars in pinned host memory (later kernels on the
        stream keep running)."""
        return self.readback.wait(self._stream.cuda_stream)


class LaunchTimer:
    """Optional HIP-event timing of the boundary kernels.

    When attached to an optimizer (``optimizer.launch_timer``), every K1 /
    K2 / K3 launch is bracketed by events recorded on the current stream,
    the stream the kernels run on.  The events are created with
    ``hipEventDisableSystemFence``: a default event performs a system-scope
    release when it is recorded (a cache write-back between the kernels it
    brackets, 10-15 us per event between the boundary kernels), which the
    timing-only events do without, so the timed kernels run back to back as
    in an untimed step.  ``durations_ms(name)`` is valid after the device
    has been synchronised.  ``reserve(n)`` creates n events up front, so
    that a timed region pays only for recording them.
    """

    def __init__(self, reserve: int = 0):
        self._hip = _native.hip_runtime()
        self._events = {}
        self._pool: List[int] = []
        self._owned: List[int] = []
        self.reserve(reserve)

    def _create(self) -> int:
        ev = ctypes.c_void_p()
        _native.hip_check(self._hip.hipEventCreateWithFlags(
            ctypes.byref(ev), _native.HIP_EVENT_DISABLE_SYSTEM_FENCE), "hipEventCreateWithFlags")
        self._owned.append(ev.value)
        return ev.value

    def reserve(self, n: int) -> None:
        self._pool.extend(self._create() for _ in range(n))

    def _record(self) -> int:
        ev = self._pool.pop() if self._pool else self._create()
        stream = torch.cuda.current_stream().cuda_stream
        _native.hip_check(self._hip.hipEventRecord(ev, stream), "hipEventRecord")
        return ev

    def start(self, name: str):
        return (name, self._record())

    def stop(self, token) -> None:
        name, start = token
        self._events.setdefault(name, []).append((start, self._record()))

    def pairs(self, names: Sequence[str]):
        """An event pair for every name, in order, as the array that
        ms_boundary_scan and ms_boundary_update record."""
        events = (ctypes.c_void_p * (2 * len(names)))()
        for k, name in enumerate(names):
            a, b = (self._pool.pop() if self._pool else self._create() for _ in range(2))
            events[2 * k], events[2 * k + 1] = a, b
            self._events.setdefault(name, []).append((a, b))
        return events

    def durations_ms(self, name: str) -> List[float]:
        out = []
        for a, b in self._events.get(name, []):
            ms = ctypes.c_float()
            _native.hip_check(self._hip.hipEventElapsedTime(ctypes.byref(ms), a, b),
                              "hipEventElapsedTime")
            out.append(float(ms.value))
        return out

    def reset(self) -> None:
        """Forget the recorded pairs (their events go back to the pool)."""
        for pairs in self._events.values():
            for a, b in pairs:
                self._pool.extend((a, b))
        self._events.clear()

    def __del__(self):
        hip = getattr(self, "_hip", None)
        for ev in getattr(self, "_owned", ()):
            hip.hipEventDestroy(ev)


@dataclass
class GroupLaunch:
    """What K1/K3 need for one group at one boundary."""

    group: FlatParamGroup
    lr: float
    betas: Sequence[float]
    eps: float
    weight_decay: float
    step: int                     # Adam step number this update would use
    exp_avg: torch.Tensor         # owned-range moments (optim/adam.py:58-65)
    exp_avg_sq: torch.Tensor
    rows: Optional[object]        # the group's BoundaryRows with its gradients, or
    grads: Optional[Sequence[int]]   # (a shard) the address per parameter (0: none)
    grad_dtype: Optional[int] = None   # MS_DTYPE_* of the gradients (default: the params')
    # (sum-of-squares slots, flag slots, count) K5 left for the gradients
    # (contiguous mode): K2's input in the place of what a K1 scan writes
    tile_stats: Optional[Tuple[int, int, int]] = None
    table: Optional[Tuple[int, int]] = None   # _whole_table's


# flat indices that K1 scans for longer than the host takes to upload a table
# (25 us; 64M fp16 gradients at 5 TB/s)
_LONG_SCAN = 1 << 26


def _whole_table(gl: GroupLaunch, write_model: bool, cur: torch.cuda.Stream) -> Tuple[int, int]:
    """(address, rows) of the one table of a group with
    :meth:`FlatParamGroup.boundary_rows`, its model column filled in."""
    g = gl.group
    if gl.table is not None:
        return gl.table
    if write_model and g._partitioned:
        # K3 writes the shard's buffer, whatever the gathered parameters view
        # by now; they become its placeholders once K3 is queued
        gl.rows.set_models(g.shard_pointers())
    elif gl.rows.models(write_model) >= 0:
        g.model_pointers()     # says what is wrong with it
        raise RuntimeError("a parameter changed during the boundary")
    gl.table = g.table("k1").upload(gl.rows.table, cur)
    return gl.table


def _scan_table(gl: GroupLaunch, write_model: bool, gbytes: int, cur: torch.cuda.Stream):
    """K1's (table address, rows).  K1 looks at no model address, so the
    table with the last boundary's model column serves it before the models
    are walked: where it is cached, and where K1 runs longer than another
    upload for K3 takes, should the models have moved (_LONG_SCAN)."""
    g = gl.group
    table = g.table("k1")
    if gl.rows is None:
        return table.upload(g.boundary_table(0, g.numel_padded, gl.grads, None, gbytes), cur)
    if g.numel_padded >= _LONG_SCAN:
        return table.upload(gl.rows.table, cur)
    return table.find(gl.rows.table, cur) or _whole_table(gl, write_model, cur)


def _update_table(gl: GroupLaunch, write_model: bool, gbytes: int, cur: torch.cuda.Stream):
    """K3's (table address, rows): K1's, or its own for a shard."""
    g = gl.group
    if gl.rows is not None:
        return _whole_table(gl, write_model, cur)
    lo, hi = g.own_range
    if hi <= lo:
        return None, 0
    mptrs = g.model_pointers() if write_model else None
    return g.table("k3").upload(g.boundary_table(lo, hi, gl.grads, mptrs, gbytes), cur)


def _inside(ptrs: np.ndarray, buf: torch.Tensor) -> bool:
    """Whether any of the addresses lies in ``buf``'s memory."""
    begin = buf.data_ptr()
    return bool(((ptrs >= begin) & (ptrs < begin + buf.numel() * buf.element_size())).any())


def launch_boundary(
    launches: List[GroupLaunch],
    ws: Workspace,
    cur: torch.cuda.Stream,
    *,
    scaler,
    max_norm: Optional[float],
    materialize_flat_grad: bool,
    write_model: bool,
    timer: Optional[LaunchTimer] = None,
    keep: Sequence[Optional[torch.Tensor]] = (),
) -> None:
    """Launch the whole boundary on ``cur`` (the stream ``ws.enter()``
    returned); ``ws.finish_readback()`` then waits for K2's scalars.

    K1 and K2 of all groups go out in one call (ms_boundary_scan) as soon as
    the gradients' addresses are known; K3's table and arguments are made
    ready behind them, and one call launches every K3 (ms_boundary_update).
    On an idle GPU the step waits for what comes before K1: with all of it
    first, K1 of 124M params started 35 us into the step, of 1.3B 50; it
    starts after 23 and 30 so.  ``write_model``: K3 casts the updated masters
    into the parameters' storage.  Where this raises (a check, device memory
    for a table, the tile slots or the flat gradient), the gradients and
    parameters are as they were: the caller releases them after it.  ``keep``
    holds the tensors behind ``GroupLaunch.grads``; ``cur`` is recorded on
    each, so the caller may drop them once this returns, whichever stream
    allocated them (``GroupLaunch.rows`` records it on its own).
    """
    lib = _native.load()
    scale = float(scaler.loss_scale_factor)
    unscale = scale != 1.0

    # a group whose accumulation pass already scanned the sums has its tile
    # statistics (no second read of the sums); the others' tile slots lie one
    # region after another, K2 reads them all
    scanned = [gl.tile_stats is not None and not materialize_flat_grad
               and gl.group.own_range == (0, gl.group.numel_padded) for gl in launches]
    ntiles = [0 if done else _native.scan_tiles(gl.group.numel_padded)
              for gl, done in zip(launches, scanned)]
    tsum, tflag = ws.tile_ptrs(sum(ntiles), cur)
    scale32 = ctypes.c_float(scale).value
    gbytes = []
    for b, st, gl, done, nt in zip(ws.groups, ws.tile_stats, launches, scanned, ntiles):
        g = gl.group
        b.numel, (b.own_begin, b.own_end) = g.numel_padded, g.own_range
        dtype = _native.ms_dtype(g.params[0].dtype)
        b.model_dtype = _native.ms_dtype(g.model_shard.dtype) if g._partitioned else dtype
        b.grad_dtype = dtype if gl.grad_dtype is None else gl.grad_dtype
        gbytes.append(4 if b.grad_dtype == _native.DTYPE_F32 else 2)
        b.scanned = done
        b.flat_grad = g.flat_grad_for_overwrite().data_ptr() if materialize_flat_grad else None
        b.hp.unscale, b.hp.grad_scale = unscale, scale32
        if done:
            st.sumsq, st.flag, st.ntiles = gl.tile_stats
        else:
            b.segs, b.nseg = _scan_table(gl, write_model, gbytes[-1], cur)
            st.sumsq, st.flag, st.ntiles = tsum, tflag, nt
            tsum += 8 * nt
            tflag += 4 * nt
    norm = ws.norm
    norm.has_clip, norm.max_norm = (0, 0.0) if max_norm is None else (1, float(max_norm))
    norm.scaler_enabled, norm.scale = bool(scaler.enabled), float(scaler.scale)
    norm.good_steps, norm.skipped_steps = int(scaler.good_steps), int(scaler.skipped_steps)
    norm.window = int(scaler.scale_window)
    norm.min_scale, norm.max_scale = float(scaler.min_scale), float(scaler.max_scale)
    events = None if timer is None else timer.pairs(["k1"] * len(launches) + ["k2"])
    ws.readback.arm()
    rc = lib.ms_boundary_scan(ws.groups, ws.tile_stats, len(launches), ctypes.byref(norm), events,
                              cur.cuda_stream)
    _native.check(rc, "ms_boundary_scan")
    try:
        for b, gl, size in zip(ws.groups, launches, gbytes):
            g = gl.group
            master, n = g.shard, b.own_end - b.own_begin
            if n > 0 and not (master.numel() == gl.exp_avg.numel() == gl.exp_avg_sq.numel() == n):
                raise RuntimeError(
                    f"grad/shard shape mismatch: owned range {n} vs master {master.numel()}, "
                    f"moments {gl.exp_avg.numel()}/{gl.exp_avg_sq.numel()}"
                )
            b.own_segs, b.own_nseg = _update_table(gl, write_model, size, cur)
            # K3 reads the gradients themselves also when K1 writes the flat
            # gradient: its unscale rounds exactly as K1's, and 2-byte
            # gradients are 2 B/param less to read than the flat copy (350M
            # fp16 params: K3 1.77 -> 1.54 ms).  Not where a gradient is a
            # view of the flat buffer: K1 unscales it in place
            b.update_from_flat = materialize_flat_grad and _inside(
                gl.grads if gl.rows is None else gl.rows.table[:, 2], g.flat_grad_for_overwrite())
            b.master, b.exp_avg, b.exp_avg_sq = (
                master.data_ptr(), gl.exp_avg.data_ptr(), gl.exp_avg_sq.data_ptr())
            b.hp = adamw_params(gl.lr, gl.betas, gl.eps, gl.weight_decay, gl.step,
                                grad_scale=scale, unscale=unscale)
        if timer is not None:
            events = timer.pairs(["k3"] * sum(gl.group.own_range[1] > gl.group.own_range[0]
                                              for gl in launches))
        rc = lib.ms_boundary_update(ws.groups, len(launches), norm.out, events, cur.cuda_stream)
        _native.check(rc, "ms_boundary_update")
    except BaseException:
        ws.finish_readback()    # K2's result must not land in the next boundary's
        raise
    # Gradients may come from another stream (the one backward ran on): once
    # the caller drops them, the caching allocator could hand their memory to
    # that stream while K1 / K3 still read it here.  Recording this stream on
    # them defers the reuse until everything queued here by then has run.
    if keep:
        record_streams(keep, cur)


# ------------------------------------------------------------------ utility
def scale_in_place(buf: torch.Tensor, mode: int, factor: float) -> None:
    """``buf.div_(factor)`` (mode SCALE_DIVIDE, flat.py:243-247) or
    ``buf.mul_(factor)`` (mode SCALE_MULTIPLY, flat.py:249-257) of a
    contiguous fp32 device buffer, in place by K1, with ``factor`` rounded to
    fp32 first as torch does with a Python scalar."""
    _native.require_hip_tensor(buf, "scaled buffer")
    if buf.dtype != torch.float32 or not buf.is_contiguous():
        raise TypeError("scale_in_place needs a contiguous float32 buffer")
    if buf.numel() == 0:
        return
    _native.check(_native.load().ms_buffer_scale(
        buf.data_ptr(), buf.numel(), mode, float(np.float32(factor)),
        _native.stream_handle(buf.device)), "ms_buffer_scale")


def _scan_buffers(bufs: Sequence[torch.Tensor], readback: Optional[HostReadback] = None) -> torch.Tensor:
    """K1 over each buffer, then K2 over all of them (in order, one group
    each): the ``ms_step_scalars_t`` as device bytes, and through
    ``readback`` on the host.  The scratch is one allocation on the current
    stream, which orders its reuse after the kernels."""
    lib = _native.load()
    device = bufs[0].device
    stream = _native.stream_handle(device)
    nblk = _native.stats_blocks()
    tiles = [_native.scan_tiles(b.numel()) for b in bufs]
    n, slots = len(bufs), len(bufs) * nblk + sum(tiles)
    scratch = torch.empty(12 * slots, dtype=torch.uint8, device=device)
    scalars = torch.empty(_native.SCALARS_BYTES, dtype=torch.uint8, device=device)
    sums = scratch.data_ptr()                 # fp64 slots, then the uint32 ones
    flags = sums + 8 * slots
    stats = (_native.TileStats * n)()
    tsum, tflag = sums + 8 * n * nblk, flags + 4 * n * nblk
    for st, b, nt in zip(stats, bufs, tiles):
        _native.check(lib.ms_buffer_tile_stats(b.data_ptr(), _native.ms_dtype(b.dtype), b.numel(),
                                               tsum, tflag, nt, stream), "ms_buffer_tile_stats")
        st.sumsq, st.flag, st.ntiles = tsum, tflag, nt
        tsum += 8 * nt
        tflag += 4 * nt
    if readback is not None:
        readback.arm()
    _native.check(lib.ms_norm_clip_tiles(stats, n, sums, flags, nblk, 0, 0.0, 0, 1.0, 0, 0, 1, 1.0,
                                         1.0, scalars.data_ptr(),
                                         None if readback is None else readback.ptr, stream),
                  "ms_norm_clip_tiles")
    return scalars


def _scan_to_host(bufs: Sequence[torch.Tensor]) -> _native.StepScalars:
    if torch.cuda.is_current_stream_capturing():
        raise RuntimeError("a scan whose result the host waits for cannot run under graph capture")
    readback = HostReadback()
    _scan_buffers(bufs, readback)
    return readback.wait(_native.stream_handle(bufs[0].device))


def _flat_view(buf: torch.Tensor) -> torch.Tensor:
    return buf.detach().reshape(-1).contiguous()


def sumsq_device(buf: torch.Tensor) -> torch.Tensor:
    """``buf.pow(2).sum()`` as a 0-dim fp32 device tensor (flat.py:232-234):
    K1's fp64 tile partials, summed by K2 and rounded to fp32 once."""
    _native.require_hip_tensor(buf, "sum-of-squares buffer")
    if buf.numel() == 0:
        return torch.zeros((), dtype=torch.float32, device=buf.device)
    scalars = _scan_buffers([_flat_view(buf)])
    off = _native.StepScalars.sumsq.offset
    return scalars[off:off + 4].view(torch.float32).reshape(())


def norm_of(bufs: Sequence[torch.Tensor]) -> float:
    """The global L2 norm of the buffers (stage_1_and_2.py:114-121): every
    buffer's sum of squares as :func:`sumsq_device` gives it, added in order
    in fp32, fp32 square root; one wait for the host's copy."""
    for buf in bufs:
        _native.require_hip_tensor(buf, "sum-of-squares buffer")
    return float(_scan_to_host([_flat_view(b) for b in bufs]).norm)


def scan_nonfinite(buf: torch.Tensor) -> bool:
    """inf/nan test of one device buffer with K1 + K2 (used by
    precision.has_overflow)."""
    _native.require_hip_tensor(buf, "has_overflow buffer")
    _native.ms_dtype(buf.dtype)
    return bool(_scan_to_host([_flat_view(buf)]).overflow)
