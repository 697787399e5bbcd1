"""The host side of a launch without a GPU (the device queries, and the
library where a call would enqueue, are stood in for)."""
import threading
import time
from contextlib import nullcontext
from types import SimpleNamespace

import numpy as np
import pytest
import torch

from aegaeon_amd import _gpu, inputs, ops
from aegaeon_amd import attention as A
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


def test_raw_stream_with_and_without_torchs_accessor(monkeypatch):
    streams = {0: 70, 1: 71}
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 1)
    monkeypatch.setattr(_gpu, "_torch_raw_stream", lambda i: streams[i])
    devices = [torch.device("cuda", 0), torch.device("cuda", 1), torch.device("cuda")]
    assert [_gpu.raw_stream(d) for d in devices] == [70, 71, 71]
    monkeypatch.setattr(_gpu, "_torch_raw_stream", None)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda d: SimpleNamespace(
        cuda_stream=streams[1 if d.index is None else d.index]))
    assert [_gpu.raw_stream(d) for d in devices] == [70, 71, 71]


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


class _OnGpu:
    """A CPU tensor that says it is on the first GPU."""

    is_cuda = True
    device = torch.device("cuda", 0)

    def __init__(self, t):
        self._t = t

    def __getattr__(self, name):
        return getattr(self._t, name)


class _Library:
    """Stands in for the two parts of a call that shares its stream's buffer:
    notes who fills the buffer first and who reads it later."""

    def __init__(self):
        self.writer = {}
        self.mixed = 0

    def aegkv_paged_decode_attention_workspace_size(self, batch, *_):
        return 1024 * batch

    def aegkv_paged_decode_attention(self, *args):
        assert args[-2] == 1024 * args[11]
        return self._two_parts(*args[-3:])

    def aegkv_swap_blocks(self, *args):
        assert args[-2] >= args[-4]
        return self._two_parts(*args[-3:])

    def _two_parts(self, ws, nbytes, stream):
        me = threading.get_ident()
        assert ws and nbytes
        self.writer[stream, ws] = me
        time.sleep(0.002)  # the interpreter runs other threads, as it does in a foreign call
        self.mixed += self.writer[stream, ws] != me
        return 0


@pytest.mark.parametrize("streams", [[7, 7], [7, 8], [7, 7, 8, 7]])
def test_threads_share_a_streams_workspace_in_turn(monkeypatch, streams):
    """Two threads' calls on one stream both write the stream's workspace and
    merge from it: a call's two kernels are enqueued with no other's between,
    whatever the batch (the workspace grows); on two streams each has its
    own."""
    lib = _Library()
    local = threading.local()
    monkeypatch.setattr(A._lib, "load", lambda: lib)
    monkeypatch.setattr(A, "device_guard", lambda d: nullcontext())
    monkeypatch.setattr(A, "raw_stream", lambda d: local.stream)
    empty = torch.empty
    monkeypatch.setattr(_gpu.torch, "empty", lambda *a, **k: _OnGpu(empty(*a, dtype=k["dtype"])))
    monkeypatch.setattr(A, "_workspaces", {})
    errors = []

    def work(stream, batch):
        local.stream = stream
        try:
            q = _OnGpu(torch.zeros(batch, 4, 64, dtype=torch.float16))
            cache = _OnGpu(torch.zeros(2, 16, 1, 64, dtype=torch.float16))
            bt = _OnGpu(torch.zeros(batch, 1, dtype=torch.int32))
            sl = _OnGpu(torch.ones(batch, dtype=torch.int32))
            for _ in range(20):
                A.paged_decode_attention(q, cache, cache, bt, sl, 0.1, 16, out=q)
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=work, args=(s, 1 + i)) for i, s in enumerate(streams)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    assert lib.mixed == 0
    assert len(A._workspaces) == len(set(streams))


@pytest.mark.parametrize("staging", ["auto", None])
def test_threads_share_a_streams_swap_staging_in_turn(monkeypatch, staging):
    """The same for a swap's pack and its copy to the host (without staging
    nothing is shared, and nothing is passed on)."""
    lib = _Library()
    if staging is None:
        lib._two_parts = lambda ws, nbytes, stream: int(ws is not None or nbytes != 0)
        lib.aegkv_swap_blocks = lambda *args: lib._two_parts(*args[-3:])
    monkeypatch.setattr(ops._lib, "load", lambda: lib)
    monkeypatch.setattr(torch.cuda, "device", lambda d: nullcontext())
    monkeypatch.setattr(ops, "_stream", lambda d: 7)
    monkeypatch.setattr(ops, "STAGING_BYTES", 1 << 12)
    empty = torch.empty
    monkeypatch.setattr(torch, "empty", lambda *a, **k: _OnGpu(empty(*a, dtype=k["dtype"])))
    monkeypatch.setattr(ops, "_staging", {})
    errors = []

    def work(width):
        try:
            cache = _OnGpu(torch.zeros(4, width, dtype=torch.float16))
            host = torch.zeros(4, width, dtype=torch.float16)
            host.is_pinned = lambda: True
            for _ in range(20):
                ops.swap([0, 2], [1, 3], False, cache, host, staging=staging)
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=work, args=(w,)) for w in (64, 1 << 13)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    assert lib.mixed == 0
    assert len(ops._staging) == (0 if staging is None else 1)
