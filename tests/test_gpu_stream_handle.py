"""GPU: the handle of the current stream, with and without torch's private call for it."""
import importlib

import pytest
import torch

operators = importlib.import_module("tigre_amd.operators")


@pytest.mark.gpu
def test_missing_raw_stream(cuda, monkeypatch):
    torch.zeros(1, device=cuda)
    with torch.cuda.stream(torch.cuda.Stream()):
        want = operators._stream_handle().value
        monkeypatch.delattr(torch._C, "_cuda_getCurrentRawStream")
        assert operators._stream_handle().value == want == torch.cuda.current_stream().cuda_stream
