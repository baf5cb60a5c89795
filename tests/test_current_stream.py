"""plffi's handle of the current stream, with and without torch's private
shortcut to it."""
import types

import plffi
import pytest
import torch


def test_without_the_private_function(monkeypatch):
    monkeypatch.delattr(torch._C, "_cuda_getCurrentRawStream", raising=False)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: types.SimpleNamespace(cuda_stream=0x1230))
    assert plffi._stream(None).value == 0x1230


def test_given_stream():
    assert plffi._stream(types.SimpleNamespace(cuda_stream=0x4560)).value == 0x4560


@pytest.mark.gpu
def test_matches_torch():
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    s = torch.cuda.Stream()
    assert (plffi._stream(None).value or 0) == torch.cuda.current_stream().cuda_stream
    with torch.cuda.stream(s):
        assert plffi._stream(None).value == s.cuda_stream
