"""The current stream's handle, with and without PyTorch's own readers of it."""
import types

import torch

from torchlet_amd.kernels import ops


def test_handle_without_pytorchs_own_readers(monkeypatch):
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: types.SimpleNamespace(cuda_stream=77))
    for name in ("_cuda_getCurrentRawStream", "_cuda_getDevice"):
        with monkeypatch.context() as m:
            m.delattr(torch._C, name, raising=False)
            assert ops._stream_reader()() == 77
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda device: 1000 + device, raising=False)
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: 5, raising=False)
    assert ops._stream_reader()() == 1005
