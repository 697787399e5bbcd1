"""The device guard and the current stream of a launch, at the cost of a
lookup: ``torch.cuda.device`` and ``torch.cuda.current_stream`` build an object
per call (1.4 and 1.9 us of host time), and a decode step of short sequences is
bound by its host time.  And the device buffers that calls on a stream share."""
from __future__ import annotations

import threading
from contextlib import nullcontext
from typing import Dict, Optional, Tuple

import torch

_CURRENT = nullcontext()
# torch's own accessor behind its stream object; not part of its documented
# interface, so the object stands in where it is missing
_torch_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def device_guard(device: torch.device):
    """Makes the GPU ``device`` current inside the ``with`` (nothing to do when
    it is); ValueError for a device that is no GPU, also ``cpu:0``."""
    if device.type == "cuda" and device.index is not None \
            and device.index == torch.cuda.current_device():
        return _CURRENT
    return torch.cuda.device(device)


def raw_stream(device: torch.device) -> int:
    """The ``hipStream_t`` of torch's current stream on ``device``."""
    if _torch_raw_stream is None:
        return torch.cuda.current_stream(device).cuda_stream
    index = device.index
    return _torch_raw_stream(torch.cuda.current_device() if index is None else index)


class StreamBuffer:
    """Device memory of the calls on one stream that bring none.  Such a call
    enqueues work that fills it and work that reads it, and a second host
    thread on the stream (torch's default stream is every thread's) must not
    come between them: ``lock`` is held while a call enqueues."""

    def __init__(self):
        self.lock = threading.Lock()
        self.buffer: Optional[torch.Tensor] = None

    def at_least(self, nbytes: int, device: torch.device) -> torch.Tensor:
        """The buffer, grown to ``nbytes`` (lock held)."""
        if self.buffer is None or self.buffer.numel() < nbytes:
            self.buffer = torch.empty(nbytes, dtype=torch.uint8, device=device)
        return self.buffer


def stream_buffer(buffers: Dict[Tuple[int, int], StreamBuffer], device: torch.device,
                  stream: int) -> StreamBuffer:
    """The entry of (``device``, ``stream``) in ``buffers``."""
    key = (device.index if device.index is not None else torch.cuda.current_device(), stream)
    b = buffers.get(key)
    # setdefault: of threads that come here together one's entry is everyone's
    return b if b is not None else buffers.setdefault(key, StreamBuffer())
