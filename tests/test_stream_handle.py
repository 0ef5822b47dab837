"""ops passes the raw handle of torch's current stream; where torch has no direct query for it, the Stream object's."""
import types

import pytest
import torch

import qwengine_amd.ops as ops


@pytest.mark.parametrize("missing", ["_cuda_getCurrentRawStream", "_cuda_getDevice"])
def test_without_the_raw_query(monkeypatch, missing):
    monkeypatch.setattr(torch.cuda, "is_initialized", lambda: True)
    monkeypatch.setattr(torch.cuda, "is_available", lambda: True)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: types.SimpleNamespace(cuda_stream=1234))
    monkeypatch.delattr(torch._C, missing, raising=False)
    assert ops._stream(None) == 1234
