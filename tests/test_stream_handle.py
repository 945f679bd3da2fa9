"""The library's stream is torch's current one, by torch's raw handle or, where a release lacks that private name,
by the public Stream object."""
from types import SimpleNamespace

import pytest
import torch

from duct_amd import solver


@pytest.mark.parametrize("private", [True, False])
def test_current_stream_handle(monkeypatch, private):
    got = []
    monkeypatch.setattr(solver, "set_stream", got.append)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 3)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: SimpleNamespace(cuda_stream=4321))
    if private:
        monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda device: 1000 + device, raising=False)
    else:
        monkeypatch.delattr(torch._C, "_cuda_getCurrentRawStream", raising=False)
    solver._use_current_stream()
    assert got == [1003 if private else 4321]
