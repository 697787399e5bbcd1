"""The device guard and the current stream of a launch, at the cost of a
lookup: ``torch.cuda.device`` and ``torch.cuda.current_stream`` build an object
per call (1.4 and 1.9 us of host time), and a decode step of short sequences is
bound by its host time."""
from __future__ import annotations

from contextlib import nullcontext

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
