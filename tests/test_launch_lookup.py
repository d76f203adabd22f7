"""The device and stream lookups of a launch (w4_hip.on_device, raw_stream) against torch's own."""

import pytest
import torch

from tandem_amd.layers import norm, w4_hip


@pytest.mark.gpu
def test_launches_follow_the_current_stream():
    dev = torch.device("cuda", torch.cuda.current_device())
    side = torch.cuda.Stream(dev)
    assert w4_hip.raw_stream(dev.index) == torch.cuda.current_stream(dev).cuda_stream
    x, w = torch.randn(3, 1024, device=dev).half(), torch.ones(1024, device=dev).half()
    want = norm.rms_norm(x, w, 1e-6)
    side.wait_stream(torch.cuda.current_stream(dev))
    with torch.cuda.stream(side), w4_hip.on_device(dev.index):
        assert w4_hip.raw_stream(dev.index) == side.cuda_stream != 0
        got = norm.rms_norm(x, w, 1e-6)
    side.synchronize()
    assert torch.equal(got, want) and torch.cuda.current_device() == dev.index


def test_on_device_switches_only_where_it_must(monkeypatch):
    seen = []
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch.cuda, "device", lambda i: seen.append(i) or w4_hip._HERE)
    for i in (0, 1, 0):
        with w4_hip.on_device(i):
            pass
    assert seen == [1]
