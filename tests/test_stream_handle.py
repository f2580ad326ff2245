"""The handle of the current stream, with and without the functions of torch that give it directly."""
import types

import pytest
import torch

from nvmai_amd import ops

@pytest.mark.parametrize("absent", [(), ("_raw_stream",), ("_raw_device",), ("_raw_stream", "_raw_device")])
def test_a_torch_without_the_direct_functions(monkeypatch, absent):
    for name, function in (("_raw_stream", lambda device: 100 + device), ("_raw_device", lambda: 3)):
        monkeypatch.setattr(ops, name, None if name in absent else function)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: types.SimpleNamespace(cuda_stream=7))
    monkeypatch.setattr(torch.cuda, "is_initialized", lambda: True)
    assert ops._stream() == (7 if absent else 103)
    monkeypatch.setattr(torch.cuda, "is_initialized", lambda: False)
    assert ops._stream() == 7


@pytest.mark.gpu
def test_the_stream_that_is_current():
    side = torch.cuda.Stream()
    assert ops._stream() == torch.cuda.current_stream().cuda_stream
    with torch.cuda.stream(side):
        assert ops._stream() == side.cuda_stream
