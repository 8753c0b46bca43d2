"""The Python binding's own host code, without a GPU."""
import types

import torch

import gonngpu as G


def test_current_stream_with_and_without_torchs_raw_handle(monkeypatch):
    """The raw handle comes from a function that torch does not promise to keep: where it is gone, the
    handle is the public Stream object's."""
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 3)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: types.SimpleNamespace(cuda_stream=77))
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda device: 1000 + device, raising=False)
    assert G._current_stream() == 1003
    monkeypatch.delattr(torch._C, "_cuda_getCurrentRawStream")
    assert G._current_stream() == 77
