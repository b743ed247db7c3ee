"""Forms of a device that the current stream's handle is asked for."""

import pytest
import torch

from taomate_hd_amd import _native


@pytest.mark.parametrize(
    "device,index",
    [
        (torch.device("cuda:1"), 1), ("cuda:1", 1), (1, 1), ("cuda:0", 0),
        (torch.device("cuda"), 3), ("cuda", 3), (None, 3),  # the current device
    ],
)
def test_stream_ptr_takes_every_form_of_a_device(monkeypatch, device, index):
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda i: 1000 + i, raising=False)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 3)
    assert _native.stream_ptr(torch, device) == 1000 + index
    # asked again: of the same device, or of what is the current one by then
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 2)
    assert _native.stream_ptr(torch, device) == 1000 + (2 if index == 3 else index)


@pytest.mark.parametrize("device", [torch.device("cpu"), "cpu", "cpu:0", torch.device("cpu:0")])
def test_stream_ptr_refuses_other_devices(monkeypatch, device):
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda i: 1000 + i, raising=False)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 3)
    with pytest.raises(ValueError):
        _native.stream_ptr(torch, device)
