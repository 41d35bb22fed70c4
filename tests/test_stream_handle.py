"""stream_handle: the current stream, also with a torch that lacks the functions
that give its handle directly."""
import importlib.util
import types

import pytest
import torch

from rngd_pd_amd.kernels import handoff


def test_without_the_direct_functions(monkeypatch):
    for name in ("_cuda_getCurrentRawStream", "_cuda_getDevice"):
        monkeypatch.delattr(torch._C, name, raising=False)
    spec = importlib.util.spec_from_file_location("rngd_pd_amd.kernels.handoff_plain",
                                                  handoff.__file__)
    plain = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(plain)
    monkeypatch.setattr(torch.cuda, "is_initialized", lambda: True)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: types.SimpleNamespace(cuda_stream=7))
    assert plain.stream_handle() == 7
    assert plain.stream_handle(5) == 5


@pytest.mark.gpu
def test_is_the_current_stream(cuda):
    torch.zeros(1, device=cuda)
    assert handoff.stream_handle() == torch.cuda.current_stream().cuda_stream
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        assert handoff.stream_handle() == side.cuda_stream
    assert handoff.stream_handle(side) == side.cuda_stream
