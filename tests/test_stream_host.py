"""The current stream's handle, without a GPU: from torch's own binding where this torch has it, else from the public stream object."""
import importlib.util

import torch


def _runtime():
    """The module again, beside the imported one."""
    from n2d2_amd import runtime
    spec = importlib.util.spec_from_file_location("n2d2_amd._runtime_again", runtime.__file__)
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    return module


def test_stream_handle_without_the_private_binding(monkeypatch):
    class Stream:
        cuda_stream = 0x1234

    asked = []
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 3)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: asked.append(device) or Stream())
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda device: 0x5000 + device, raising=False)
    assert _runtime().stream_ptr().value == 0x5003 and not asked
    monkeypatch.delattr(torch._C, "_cuda_getCurrentRawStream")
    assert _runtime().stream_ptr().value == 0x1234 and asked == [3]
