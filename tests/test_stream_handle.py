"""The stream handle passed to the library, with and without torch's undocumented shortcut."""
import types

import torch


def test_handle_of_the_current_stream(shtk, monkeypatch):
    from shtnskit_jl_amd import transforms

    device = torch.device("cuda", 1)
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda index: 40 + index, raising=False)
    assert transforms._stream(device).value == 41
    monkeypatch.delattr(torch._C, "_cuda_getCurrentRawStream")
    monkeypatch.setattr(torch.cuda, "current_stream", lambda d: types.SimpleNamespace(cuda_stream=70 + d.index))
    assert transforms._stream(device).value == 71
