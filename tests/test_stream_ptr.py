"""The raw stream getter and the Stream object it stands in for."""
import pytest
import torch

from locks import _lib


def test_torch_without_the_raw_getter(monkeypatch):
    class Stream:
        cuda_stream = 0x7F00

    seen = []
    monkeypatch.delattr(torch._C, "_cuda_getCurrentRawStream", raising=False)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: seen.append(device) or Stream)
    assert _lib.stream_ptr() == 0x7F00 and _lib.stream_ptr("cuda:3") == 0x7F00
    assert seen == [None, "cuda:3"]


def test_refuses_other_devices(monkeypatch):
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda index: index, raising=False)
    assert _lib.stream_ptr("cuda:2") == 2
    with pytest.raises(ValueError, match="cuda device"):
        _lib.stream_ptr("cpu")


@pytest.mark.gpu
def test_follows_the_current_stream():
    side = torch.cuda.Stream()
    for device in (None, "cuda", 0, torch.device("cuda:0")):
        assert _lib.stream_ptr(device) == torch.cuda.current_stream(device).cuda_stream
        with torch.cuda.stream(side):
            assert _lib.stream_ptr(device) == side.cuda_stream
