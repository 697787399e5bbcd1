"""The host side of a launch without a GPU (the device queries are stood in
for)."""
from contextlib import nullcontext

import numpy as np
import pytest
import torch

from aegaeon_amd import _gpu, inputs
from aegaeon_amd._lib import AegkvError


@pytest.mark.parametrize("device", ["cpu", "cpu:0", "meta", "meta:0"])
def test_guard_refuses_what_is_no_gpu(monkeypatch, device):
    """A CPU device that carries the current GPU's index is refused like one
    that carries none: its addresses must not reach a kernel."""
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    with pytest.raises(ValueError):
        with _gpu.device_guard(torch.device(device)):
            pass
    with pytest.raises(ValueError):
        inputs.prepare_model_inputs([(0, [1], 2, 1)], [[3]], device)


def test_guard_of_the_current_gpu_switches_nothing(monkeypatch):
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 1)
    switched = []
    monkeypatch.setattr(torch.cuda, "device", lambda d: switched.append(d))
    assert _gpu.device_guard(torch.device("cuda", 1)) is _gpu._CURRENT and not switched
    _gpu.device_guard(torch.device("cuda", 0))
    _gpu.device_guard(torch.device("cuda"))
    assert switched == [torch.device("cuda", 0), torch.device("cuda")]


@pytest.mark.parametrize("offsets", [[0, -1], [0, -2], [0, -40], [0, 3, 2], [0, 4, 1, 0]])
def test_decreasing_table_offsets_are_refused_by_the_call(monkeypatch, offsets):
    """Offsets that make every decode table's length negative, or some: the
    library's argument error, whatever the width they lead to."""
    monkeypatch.setattr(inputs, "device_guard", lambda d: nullcontext())
    monkeypatch.setattr(inputs, "raw_stream", lambda d: 0)
    n = len(offsets) - 1
    with pytest.raises(AegkvError):
        inputs.prepare_inputs_from_arrays(np.zeros(8, dtype=np.int32), np.asarray(offsets),
                                          np.full(n, 2), np.ones(n, dtype=np.int32),
                                          np.zeros(n, dtype=np.int64), "cpu")
