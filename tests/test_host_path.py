"""The host side of a launch without a GPU (the device queries are stood in
for)."""
import pytest
import torch

from aegaeon_amd import _gpu, inputs


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
