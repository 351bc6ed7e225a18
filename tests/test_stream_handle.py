"""Launches go to the stream the caller made current, whichever of torch's calls tells its handle."""

from types import SimpleNamespace

import pytest
import torch


def test_handle_without_the_private_call(monkeypatch):
    from async_llm_amd import native

    asked = []
    monkeypatch.delattr(torch._C, "_cuda_getCurrentRawStream", raising=False)
    monkeypatch.setattr(native, "_raw_stream", None, raising=False)  # as the module finds it on such a build
    monkeypatch.setattr(torch.cuda, "current_stream", lambda d: asked.append(d) or SimpleNamespace(cuda_stream=0x5eed))
    for device in (torch.device("cuda", 3), torch.device("cuda")):
        assert native.current_stream_ptr(device) == 0x5eed
    assert asked == [torch.device("cuda", 3), torch.device("cuda")]


@pytest.mark.gpu
def test_handle_is_the_current_streams():
    from async_llm_amd import native

    def same():
        for device in (torch.device("cuda"), torch.device("cuda", torch.cuda.current_device())):
            assert native.current_stream_ptr(device) == torch.cuda.current_stream(device).cuda_stream

    same()
    with torch.cuda.stream(torch.cuda.Stream()):
        same()
    same()
