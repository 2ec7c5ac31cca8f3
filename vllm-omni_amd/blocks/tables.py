"""Tables that forwards share: built once per key (image shapes, device) and handed to calls on any stream or thread."""

from __future__ import annotations

import threading
from collections import OrderedDict
from collections.abc import Callable
from typing import Any

import torch


def _tensors(value) -> tuple[torch.Tensor, ...]:
    if isinstance(value, torch.Tensor):
        return (value,)
    return value.tensors() if hasattr(value, "tensors") else tuple(value)


class TableCache:
    """``build(*key)``, kept for the last ``maxsize`` keys. The value is a tensor, a tuple of tensors, or an object whose
    ``tensors()`` are its tensors.

    Tensors on a GPU are made by work on the stream of the call that builds them, and their memory goes back to that stream
    when an entry is dropped. So the host waits for that work, once per key, before the entry is kept (a later call may be on
    a stream that is not ordered behind it, and inside a graph capture it could not wait for an event from outside), and a
    call on another stream is recorded with the allocator. What is built inside a capture exists only when the graph is
    replayed: it is handed to that call and not kept."""

    def __init__(self, build: Callable[..., Any], maxsize: int):
        self._build, self._maxsize = build, maxsize
        # key -> value, the GPU it is on (None: host memory) and the stream it was made on
        self._entries: OrderedDict[tuple, tuple[Any, torch.device | None, int]] = OrderedDict()
        self._lock = threading.Lock()

    def __reduce__(self):  # a copy of a module starts with an empty cache around its own ``build``
        return TableCache, (self._build, self._maxsize)

    def __call__(self, *key):
        with self._lock:
            entry = self._entries.get(key)
            if entry is not None:
                self._entries.move_to_end(key)
        if entry is None:
            entry = self._make(key)
        value, device, made_on = entry
        if device is not None:
            stream = torch.cuda.current_stream(device)
            if stream.cuda_stream != made_on:
                for t in _tensors(value):
                    t.record_stream(stream)
        return value

    def _make(self, key: tuple) -> tuple[Any, torch.device | None, int]:
        value = self._build(*key)
        entry = (value, None, 0)
        device = _tensors(value)[0].device
        if device.type == "cuda":
            if torch.cuda.is_current_stream_capturing():
                return entry
            stream = torch.cuda.current_stream(device)
            done = torch.cuda.Event()
            done.record(stream)
            done.synchronize()
            entry = (value, device, stream.cuda_stream)
        with self._lock:
            self._entries[key] = entry
            while len(self._entries) > self._maxsize:
                self._entries.popitem(last=False)
        return entry
