"""The thin seam between the engine and HIP streams / events.

The engine and the schedulers order device work with exactly three things:
events (``record`` / ``wait``), streams (made current for a ``with`` block) and
profiler ranges.  On an MI355X these are ``torch.cuda`` objects, which are HIP
events, HIP streams and roctx ranges on ROCm.  On a host without a GPU the same
protocol is served by recording objects, so that the host logic (issue order,
event chains, FIFO checks) can be exercised by CPU tests.  The recording
objects never compute anything: tensors that reach them are CPU tensors run by
PyTorch eagerly, which is only ever done by tests.

All streams are created at the default priority.
"""
from __future__ import annotations

import contextlib
import itertools
import threading
from typing import Any

import torch


class HostEvent:
    """Event stand-in that logs ``record`` / ``wait`` with the stream in use."""

    _counter = 0

    def __init__(self, log: list) -> None:
        HostEvent._counter += 1
        self.uid = HostEvent._counter
        self._log = log
        self.recorded_on: str | None = None

    def record(self, stream: Any = None) -> None:
        self.recorded_on = (stream or _host_state.current).name
        self._log.append(("record", self.uid, self.recorded_on))

    def wait(self, stream: Any = None) -> None:
        self._log.append(("wait", self.uid, (stream or _host_state.current).name))

    def synchronize(self) -> None:
        pass


class HostStream:
    """Stream stand-in; only its name matters."""

    def __init__(self, name: str) -> None:
        self.name = name

    def wait_stream(self, other: "HostStream") -> None:
        pass

    def synchronize(self) -> None:
        pass


class _HostState(threading.local):
    def __init__(self) -> None:
        self.current = HostStream("default")


_host_state = _HostState()


class HostDevice:
    """Recording implementation of the seam (no GPU involved)."""

    is_gpu = False

    def __init__(self) -> None:
        self.log: list = []
        self._stream_count = 0

    def new_event(self) -> HostEvent:
        return HostEvent(self.log)

    def starts(self, lanes: int) -> list[HostEvent]:
        events = [self.new_event() for _ in range(lanes)]
        for event in events:
            event.record()
        return events

    def tails(self, events: list) -> list:
        return events

    def new_stream(self, name: str | None = None, cu_mask: "list[int] | None" = None) -> HostStream:
        self._stream_count += 1
        stream = HostStream(name or f"stream{self._stream_count}")
        stream.cu_mask = cu_mask
        return stream

    def current_stream(self) -> HostStream:
        return _host_state.current

    @contextlib.contextmanager
    def stream(self, stream: HostStream):
        previous = _host_state.current
        _host_state.current = stream
        try:
            yield
        finally:
            _host_state.current = previous

    @contextlib.contextmanager
    def range(self, name: str):
        self.log.append(("range", name, _host_state.current.name))
        yield


def stream_key(stream: "torch.cuda.Stream") -> tuple[int, int]:
    """What identifies a HIP stream in the event log: (device index, stream handle)."""
    return (stream.device_index, stream.cuda_stream)


def current_stream_key() -> tuple[int, int]:
    """``stream_key(torch.cuda.current_stream())`` without making a stream object (a launch asks several times)."""
    index = torch._C._cuda_getDevice()
    return (index, torch._C._cuda_getCurrentRawStream(index))


#: one stream object per stream that has been current here; the object only names the stream
_stream_objects: dict[tuple[int, int], "torch.cuda.Stream"] = {}


def current_stream() -> "torch.cuda.Stream":
    key = current_stream_key()
    stream = _stream_objects.get(key)
    if stream is None:
        stream = _stream_objects[key] = torch.cuda.current_stream()
    return stream


def _make_current(stream: "torch.cuda.Stream") -> None:
    """``torch.cuda.set_stream`` for a stream that is one."""
    torch._C._cuda_setStream(stream_id=stream.stream_id, device_index=stream.device_index, device_type=stream.device_type)


class _CurrentStream:
    """``torch.cuda.stream`` for a stream of the current device."""

    __slots__ = ("_stream", "_previous")

    def __init__(self, stream: "torch.cuda.Stream") -> None:
        self._stream = stream

    def __enter__(self) -> "torch.cuda.Stream":
        self._previous = current_stream()
        _make_current(self._stream)
        return self._stream

    def __exit__(self, *exc) -> None:
        _make_current(self._previous)


class _Range:
    __slots__ = ("_name",)

    def __init__(self, name: str) -> None:
        self._name = name

    def __enter__(self) -> None:
        torch.cuda.nvtx.range_push(self._name)

    def __exit__(self, *exc) -> None:
        torch.cuda.nvtx.range_pop()


class HipEvent:
    """A HIP event that knows the stream it was recorded on.

    ``wait`` on that very stream issues nothing: stream order already gives the edge, and under stream capture
    such a wait would make the stream its own child in the runtime's books (see ``capture_plan``).  Nor does a second
    wait of one stream (a wait for work that is still running costs the host 8 us).  While the
    device's ``trace`` is a list, every ``record`` / ``wait`` is logged there in the recording seam's format.
    """

    __slots__ = ("_owner", "_event", "_recorded_on", "_order", "_waited", "uid")
    _counter = 0
    _records = itertools.count(1)

    def __init__(self, owner: "HipDevice") -> None:
        HipEvent._counter += 1
        self.uid = HipEvent._counter
        self._owner = owner
        self._event = torch.cuda.Event()
        self._recorded_on: tuple[int, int] | None = None
        self._order = 0                                         # of the last record among those of all events
        self._waited: tuple[tuple[int, int], ...] = ()          # streams that wait for it already

    def record(self, stream: "torch.cuda.Stream | None" = None) -> None:
        if stream is None:
            stream = current_stream()
        self._recorded_on = key = (stream.device_index, stream.cuda_stream)
        if self._owner.trace is not None:
            self._owner.note(("record", self.uid, key), stream)
        self._event.record(stream)
        self._order, self._waited = next(HipEvent._records), ()

    def wait(self, stream: "torch.cuda.Stream | None" = None) -> None:
        key = (stream.device_index, stream.cuda_stream) if stream is not None else current_stream_key()
        if self._owner.trace is not None:
            self._owner.note(("wait", self.uid, key), stream if stream is not None else current_stream())
        if self._recorded_on is None or key == self._recorded_on or key in self._waited:
            return
        self._event.wait(stream if stream is not None else current_stream())
        self._waited += (key,)

    def synchronize(self) -> None:
        self._event.synchronize()

    def query(self) -> bool:
        return self._event.query()


def cu_mask_words(first: int, count: int, total: int) -> list[int]:
    """Mask words for compute units ``first .. first + count - 1`` of ``total``."""
    if not (0 <= first and count >= 1 and first + count <= total):
        raise ValueError(f"compute units {first}..{first + count - 1} of {total}")
    bits = ((1 << count) - 1) << first
    return [(bits >> (32 * i)) & 0xFFFFFFFF for i in range((total + 31) // 32)]


def _loaded_hip_runtime() -> str:
    """Path of the HIP runtime that this process has already mapped (the one torch uses): a second copy loaded by
    its bare name would be another runtime with streams and contexts of its own."""
    with open("/proc/self/maps") as maps:
        for line in maps:
            path = line.rsplit(" ", 1)[-1].strip()
            if "libamdhip64.so" in path:
                return path
    raise RuntimeError("no HIP runtime is loaded in this process")


def _masked_stream(cu_mask: list[int]) -> int:
    """hipExtStreamCreateWithCUMask through the HIP runtime that torch has loaded; returns the stream handle."""
    import ctypes

    hip = ctypes.CDLL(_loaded_hip_runtime())
    words = (ctypes.c_uint32 * len(cu_mask))(*cu_mask)
    stream = ctypes.c_void_p()
    torch.cuda.current_stream()   # the device's context exists before the raw call
    rc = hip.hipExtStreamCreateWithCUMask(ctypes.byref(stream), ctypes.c_uint32(len(cu_mask)), words)
    if rc != 0 or not stream.value:
        raise RuntimeError(f"hipExtStreamCreateWithCUMask failed with {rc}")
    return stream.value


class HipDevice:
    """The real thing: HIP events, streams and roctx ranges through torch."""

    is_gpu = True

    def __init__(self) -> None:
        #: while a list: the (kind, event id, stream key) log of every event operation
        self.trace: list | None = None
        self.streams_seen: dict[tuple[int, int], "torch.cuda.Stream"] = {}

    def note(self, entry: tuple, stream: "torch.cuda.Stream") -> None:
        if self.trace is not None:
            self.trace.append(entry)
            self.streams_seen[entry[2]] = stream

    def new_event(self) -> HipEvent:
        return HipEvent(self)

    def starts(self, lanes: int) -> "list[HipEvent]":
        """The event, recorded now, that each of ``lanes`` nano-batches starts behind."""
        start = self.new_event()
        start.record()
        return [start] * lanes

    def tails(self, events: "list[HipEvent]") -> "list[HipEvent]":
        """Those of ``events``, recorded by the forward that asks, behind which lies the work of all of them: the last on
        each stream."""
        last = {}
        for event in events:
            other = last.get(event._recorded_on)
            if other is None or other._order < event._order:
                last[event._recorded_on] = event
        return list(last.values())

    def new_stream(self, name: str | None = None, cu_mask: "list[int] | None" = None) -> "torch.cuda.Stream":
        """A stream at the default priority.  ``cu_mask`` (32-bit words, bit i = compute unit i may run this
        stream's work) makes it a stream restricted to those compute units - what the reference does with green
        contexts (examples/ae/up-silu-overlap.cu:236-264).  Such a stream lives until the process ends."""
        if cu_mask is None:
            return torch.cuda.Stream()
        return torch.cuda.ExternalStream(_masked_stream(cu_mask))

    def current_stream(self) -> "torch.cuda.Stream":
        return current_stream()

    def stream(self, stream: "torch.cuda.Stream"):
        if stream is None or stream.device_index != torch._C._cuda_getDevice():
            return torch.cuda.stream(stream)
        return _CurrentStream(stream)

    def range(self, name: str):
        return _Range(name)


_device: HostDevice | HipDevice | None = None


def get_device() -> HostDevice | HipDevice:
    """The process-wide seam; picks HIP when a GPU is visible."""
    global _device
    if _device is None:
        _device = HipDevice() if torch.cuda.is_available() else HostDevice()
    return _device


def set_device(device: HostDevice | HipDevice | None) -> None:
    """Install a seam explicitly (tests install a fresh ``HostDevice``)."""
    global _device
    _device = device
