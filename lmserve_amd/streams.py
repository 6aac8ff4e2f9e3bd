"""Streams that nothing outside this package is handed.

`torch.cuda.Stream()` deals out the 32 streams of a pool in rotation, and `torch.cuda.graph` records on one of the
same pool: any two owners can hold one stream without knowing. What a thread launches on a stream that another thread
records is recorded with it, and a query of an event recorded there ends the recording with an error. So the streams
that a KV worker's threads use, and the one a step is recorded on, are made by the library.

They are never destroyed (the caching allocator may still hold an event for one) but given back and used again: there
are as many as were in use at once at the busiest moment.
"""
from __future__ import annotations

import threading
from collections import deque
from contextlib import contextmanager
from typing import Deque, Dict, Iterable

import torch

from . import _lib

_free: Dict[int, Deque[torch.cuda.Stream]] = {}   # in rotation: a stream given back is the last to be taken
_lock = threading.Lock()


def take(device: torch.device) -> torch.cuda.Stream:
    """A stream of `device` that no one else holds, until it is given back."""
    index = torch.cuda.current_device() if device.index is None else device.index
    with _lock:
        free = _free.get(index)
        if free:
            return free.popleft()
    with torch.cuda.device(index):
        return torch.cuda.ExternalStream(_lib.stream_create(), device=torch.device("cuda", index))


def give_back(streams: Iterable[torch.cuda.Stream]) -> None:
    """Work that is still queued on them goes before the next holder's."""
    with _lock:
        for s in streams:
            _free.setdefault(s.device.index, deque()).append(s)


@contextmanager
def recording_stream(device: torch.device):
    """A stream to record on. Not used again when the recording failed: it may still be recording."""
    stream = take(device)
    yield stream
    give_back([stream])
