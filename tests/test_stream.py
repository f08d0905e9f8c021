"""The Python wrapper's current stream (busfill._stream), with torch's GPU state
played by stand-ins: the fast lookup only where torch's own would serve it."""
import types

import pytest
import torch

import busfill as bf


@pytest.fixture
def gpu_state(monkeypatch):
    """torch with an initialised GPU whose current stream changes with `state`; nothing looked up yet."""
    state = types.SimpleNamespace(forked=False, device=0, streams={0: 0, 1: 0x70}, objects=0)

    def current_stream():
        if state.forked:
            raise RuntimeError("Cannot re-initialize CUDA in forked subprocess")
        state.objects += 1
        return types.SimpleNamespace(cuda_stream=state.streams[state.device])

    monkeypatch.setattr(torch.cuda, "current_stream", current_stream)
    monkeypatch.setattr(torch._C, "_cuda_isInBadFork", lambda: state.forked, raising=False)
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: state.device, raising=False)
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda d: state.streams[d], raising=False)
    monkeypatch.setattr(bf, "_current_stream", bf._first_current_stream)
    return state


def test_current_stream_follows_device_and_stream(gpu_state):
    assert bf._stream(None) == 0
    gpu_state.device = 1
    assert bf._stream(None) == 0x70
    gpu_state.streams[1] = 0x80
    assert bf._stream(None) == 0x80
    assert gpu_state.objects == 1                      # a Stream object for the first lookup only
    assert bf._stream(5) == 5 and bf._stream(types.SimpleNamespace(cuda_stream=6)) == 6


def test_forked_child_is_refused_as_torch_refuses_it(gpu_state):
    assert bf._stream(None) == 0                       # the parent has used the GPU
    gpu_state.forked = True                            # ... a forked child of it may not
    with pytest.raises(RuntimeError, match="forked"):
        bf._stream(None)


@pytest.mark.parametrize("name", ["_cuda_getCurrentRawStream", "_cuda_getDevice", "_cuda_isInBadFork"])
def test_without_torchs_own_calls(gpu_state, monkeypatch, name):
    monkeypatch.delattr(torch._C, name)
    for _ in range(2):
        gpu_state.device = 1
        assert bf._stream(None) == 0x70
    assert gpu_state.objects == 2
