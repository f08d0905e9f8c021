"""The Python wrapper's current stream (busfill._stream), with torch's GPU state
played by stand-ins: the fast lookup only where torch's own would serve it."""
import types

import pytest
import torch

import busfill as bf


@pytest.fixture
def gpu_state(monkeypatch):
    """torch.cuda with an initialised GPU whose current stream changes with `state`."""
    state = types.SimpleNamespace(up=True, device=0, streams={0: 0, 1: 0x70})

    def current_stream():
        if not state.up:
            raise RuntimeError("Cannot re-initialize CUDA in forked subprocess")
        return types.SimpleNamespace(cuda_stream=state.streams[state.device])

    monkeypatch.setattr(torch.cuda, "is_initialized", lambda: state.up)
    monkeypatch.setattr(torch.cuda, "current_stream", current_stream)
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: state.device, raising=False)
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda d: state.streams[d], raising=False)
    return state


def test_current_stream_follows_device_and_stream(gpu_state):
    assert bf._stream(None) == 0
    gpu_state.device = 1
    assert bf._stream(None) == 0x70
    gpu_state.streams[1] = 0x80
    assert bf._stream(None) == 0x80
    assert bf._stream(5) == 5 and bf._stream(types.SimpleNamespace(cuda_stream=6)) == 6


def test_forked_child_is_refused_as_torch_refuses_it(gpu_state):
    assert bf._stream(None) == 0                       # the parent has used the GPU
    gpu_state.up = False                               # ... a forked child of it may not
    with pytest.raises(RuntimeError, match="forked"):
        bf._stream(None)


def test_without_the_raw_calls(gpu_state, monkeypatch):
    monkeypatch.delattr(torch._C, "_cuda_getCurrentRawStream")
    gpu_state.device = 1
    assert bf._stream(None) == 0x70
