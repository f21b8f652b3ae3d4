"""Per-device backward workspaces placed in another HBM region than the
weight gradient they are written beside.

The convolution backwards write the weight gradient and their per-edge gx
messages at the same time.  Device memory on MI355X falls into regions of
about 96 GB, and two buffers written together move about 25 % more bytes per
second when they lie in different regions (config-2 backward 9.7 -> 8.7 ms
with the message workspace away from the gradient; 1 GB write probes at
up to four windows of each buffer tell the cases apart, since a buffer of
several GB may straddle two regions).  A workspace of at least ``PLACE_MIN_BYTES`` is
therefore held per device: ``luna_placed_alloc`` allocates it outside the
region of the gradient buffer of the call that needs it, and every later
call that fits in it reuses it.  A later call whose gradient buffer is new
probes it once against the held workspace (``luna_region_overlap``; the
probe overwrites parts of the gradient buffer before the kernels fill it)
and, if more than half of their write pairs would meet in one region, places
the workspace again, at most
``MAX_REPLACEMENTS`` times per device.  Smaller workspaces, calls under HIP
graph capture, fp64 backwards and ``LUNAEQ_AMD_PLACE=0`` use an ordinary
stream-ordered torch allocation.  (fp64, config 3: the backward is bound by
its FP64 issue and gained nothing, while the relocated workspace tended to
land beside gx, whose pass then took 3.34-3.38 instead of 2.92 ms.)

The held buffer is ordered across streams by one event per device: a call
waits for the previous call's work before it writes the buffer, and records
its own.

Costs the caller sees: the held workspace (``held_info()``) is device memory
outside torch's caching allocator until ``release_all()``; the search
synchronises the stream and may hold spacer allocations of up to
``spacer_budget()`` for the time of one probe sequence (at most
``SPACER_WORKSPACES`` workspaces, half of the free device memory, and
``LUNAEQ_AMD_PLACE_SPACER_GB``); the probe writes into the gradient buffer,
which the backward's kernels then overwrite in full.  When torch runs out of
device memory the held workspaces are released (an out-of-memory observer),
so that a retried allocation can use their memory.
"""

from __future__ import annotations

import ctypes
import os
import threading

import torch

from . import _native

PLACE_MIN_BYTES = 1 << 30
PROBE_BYTES = 2 << 30    # least gradient size the probe places against
MAX_REPLACEMENTS = 3
SHARED_OVERLAP = 0.5    # re-place when more write pairs than this share a region


def _enabled() -> bool:
    return os.environ.get("LUNAEQ_AMD_PLACE", "1") != "0"


SPACER_WORKSPACES = 12      # spacers per search, in workspaces
SPACER_CAP_GB = 128.0


def spacer_budget(nbytes: int, free_bytes: int) -> int:
    """Bytes of spacer allocations one placement search may hold: at most
    ``SPACER_WORKSPACES`` workspaces of ``nbytes``, half of ``free_bytes`` (the
    device's free memory before the search) and ``LUNAEQ_AMD_PLACE_SPACER_GB``
    (default 128 GB); 0 means allocate without searching."""
    cap = float(os.environ.get("LUNAEQ_AMD_PLACE_SPACER_GB", str(SPACER_CAP_GB))) * (1 << 30)
    budget = min(int(cap), SPACER_WORKSPACES * int(nbytes), max(int(free_bytes), 0) // 2)
    return max(budget, 0)


def _free_bytes(device: torch.device) -> int:
    free, _total = torch.cuda.mem_get_info(device)
    return int(free)


def _nbytes(tensor) -> int:
    return tensor.numel() * tensor.element_size()


class _Held:
    """The placed buffer of a device, its last-use event and probe verdicts
    ({gradient buffer address: shares the region})."""

    def __init__(self, device: torch.device, nbytes: int, avoid, stream: int, replacements: int):
        pointer, moved = ctypes.c_void_p(), ctypes.c_int()
        avoid_ptr, avoid_bytes = (avoid.data_ptr(), _nbytes(avoid)) if avoid is not None else (None, 0)
        with torch.cuda.device(device):
            budget = spacer_budget(nbytes, _free_bytes(device))
            _native.check(_native.lib().luna_placed_alloc(nbytes, avoid_ptr, avoid_bytes, budget,
                                                          stream, ctypes.byref(pointer), ctypes.byref(moved)),
                          "luna_placed_alloc")
        self.device, self.pointer, self.nbytes = device, pointer.value, nbytes
        self.moved = bool(moved.value)
        self.replacements = replacements
        # Whatever the search found is the best placement for this gradient.
        self.verdicts = {avoid_ptr: False} if avoid_ptr else {}
        self.event = None

    def shares_region(self, avoid, stream: int) -> bool:
        key = avoid.data_ptr()
        if key not in self.verdicts:
            overlap = ctypes.c_double()
            _native.check(_native.lib().luna_region_overlap(key, _nbytes(avoid), self.pointer, self.nbytes,
                                                            stream, ctypes.byref(overlap)), "luna_region_overlap")
            self.verdicts[key] = overlap.value > SHARED_OVERLAP
        return self.verdicts[key]

    def release(self) -> None:
        if self.event is not None:
            self.event.synchronize()
        if self.pointer:
            _native.check(_native.lib().luna_placed_free(self.pointer), "luna_placed_free")
        self.pointer = None


_lock = threading.Lock()
_held: dict[int, _Held] = {}
_observer = {"attached": False}


def _on_out_of_memory(device, *_args) -> None:
    """torch's out-of-memory observer: free the held workspaces so that the
    caller's retry (or torch's next allocation) can use their memory."""
    if _lock.acquire(blocking=False):
        try:
            for held in _held.values():
                held.release()
            _held.clear()
        finally:
            _lock.release()


def _attach_observer() -> None:
    if _observer["attached"]:
        return
    attach = getattr(torch._C, "_cuda_attach_out_of_memory_observer", None)
    if attach is not None:
        attach(_on_out_of_memory)
    _observer["attached"] = True


def run_with_workspace(device: torch.device, nbytes: int, avoid, launch, place: bool = True) -> None:
    """Call ``launch(pointer)`` with a device workspace of ``nbytes``.

    ``avoid`` is the gradient the launch writes beside the workspace (a probe
    may overwrite parts of it before ``launch`` fills it) or None; ``place``
    False takes an ordinary allocation.
    """
    if (not place or nbytes < PLACE_MIN_BYTES or not _enabled()
            or torch.cuda.is_current_stream_capturing()):
        scratch = torch.empty(nbytes, device=device, dtype=torch.uint8)
        launch(scratch.data_ptr())
        return
    stream = torch.cuda.current_stream(device)
    if avoid is not None and (not avoid.is_contiguous() or _nbytes(avoid) < PROBE_BYTES):
        avoid = None
    index = device.index if device.index is not None else torch.cuda.current_device()
    with _lock:
        held = _held.get(index)
        if held is not None and held.event is not None:
            stream.wait_event(held.event)
        replace = held is None or held.nbytes < nbytes
        if not replace and avoid is not None and held.replacements < MAX_REPLACEMENTS:
            replace = held.shares_region(avoid, stream.cuda_stream)
        if replace:
            count, size = 0, nbytes
            if held is not None:
                count = held.replacements + (held.nbytes >= nbytes)
                size = max(nbytes, held.nbytes)
                held.release()
                del _held[index]
            try:
                held = _Held(torch.device("cuda", index), size, avoid, stream.cuda_stream, count)
            except RuntimeError:
                # No device memory outside torch's cache: an ordinary
                # allocation (torch may free cached blocks for it).
                scratch = torch.empty(nbytes, device=device, dtype=torch.uint8)
                launch(scratch.data_ptr())
                return
            _held[index] = held
            _attach_observer()
        launch(held.pointer)
        held.event = torch.cuda.Event()
        held.event.record(stream)


def held_info() -> dict[int, dict]:
    """Per device: bytes of the held workspace, whether its last placement
    found another region, and how often it was placed again."""
    with _lock:
        return {index: {"bytes": h.nbytes, "other_region": h.moved, "replacements": h.replacements}
                for index, h in _held.items()}


def release_all() -> None:
    """Free every held workspace (waits for its last use)."""
    with _lock:
        for held in _held.values():
            held.release()
        _held.clear()


__all__ = ["run_with_workspace", "held_info", "release_all", "spacer_budget", "PLACE_MIN_BYTES"]
