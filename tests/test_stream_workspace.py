"""Who gets which split-K workspace, on the host: the buffers and the streams are stand-ins."""

from __future__ import annotations

import collections
import types

import pytest
import torch

from tandem_amd import decode_graph
from tandem_amd.layers import awq, w4_hip

DEV = torch.device("cuda", 0)


@pytest.fixture
def gpu(monkeypatch):
    """A device whose current stream and capture are set by the test; .made counts new workspaces."""
    state = types.SimpleNamespace(stream=0, capture=0, made=0)

    def new(index):
        state.made += 1
        return (object(), object())

    monkeypatch.setattr(w4_hip, "_new_workspace", new)
    monkeypatch.setattr(w4_hip, "_stream_workspaces", collections.OrderedDict())
    monkeypatch.setattr(w4_hip, "_workspaces", {})
    monkeypatch.setattr(w4_hip, "raw_stream", lambda index: state.stream)
    monkeypatch.setattr(w4_hip, "library", lambda: types.SimpleNamespace(tw4_capture_id=lambda s: state.capture))

    def take(stream, capture=0):
        state.stream, state.capture = stream, capture
        return w4_hip.stream_workspace(DEV)

    state.take = take
    return state


def test_the_least_recently_used_one_goes(gpu):
    main = gpu.take(0)
    for s in range(1, 3 * w4_hip.STREAM_WORKSPACES):
        gpu.take(s)
        assert gpu.take(0) is main  # in use all along
        assert len(w4_hip._stream_workspaces) <= w4_hip.STREAM_WORKSPACES
    assert gpu.made == 3 * w4_hip.STREAM_WORKSPACES


def test_streams_forked_in_one_capture_keep_theirs(gpu):
    first, second = gpu.take(7, 100), gpu.take(8, 100)
    assert first is not second
    for _ in range(3):
        assert gpu.take(7, 100) is first and gpu.take(8, 100) is second
    eager = gpu.take(7)
    gpu.take(7, 101)  # the next capture gives the last one's back, and nothing of a plain stream's
    assert [k[2] for k in w4_hip._stream_workspaces] == [0, 101] and gpu.take(7) is eager


def test_release(gpu):
    gpu.take(0), gpu.take(7), gpu.take(9, 100)
    w4_hip.release_stream_workspace(types.SimpleNamespace(device_index=0, cuda_stream=7))
    assert list(w4_hip._stream_workspaces) == [(0, 0, 0)]


@pytest.mark.parametrize("m,cfg,own", [(300, ("tiled", 8, 2, 2, 1, 2, 4, 1), False), (300, ("tiled", 8, 2, 2, 1, 2, 4, 2), True),
                                       (300, (2, 1, 4, 2, 2, 1), False), (300, (2, 1, 4, 2, 2, 0), True),
                                       (300, (2, 1, 4, 2, 2, 4), True), (16, (2, 1, 4, 2, 2, 4), False)])
def test_only_calls_that_may_split_take_a_streams_own(gpu, m, cfg, own):
    """A layer that splits nothing holds the one workspace it was finalized with, and a capture of it clears no counters."""
    device = w4_hip.workspace(DEV)
    seen = []
    ext = types.SimpleNamespace(w4_gemm=lambda x, w, s, z, *ws: seen.append(ws[:2]), w4_gemm_tiled=lambda x, w, s, z, *ws: seen.append(ws[:2]))
    layer = awq.W4Linear(256, 64, 128)
    layer.packed = layer.zeros = None
    layer._gemm(ext, types.SimpleNamespace(device=DEV, shape=(m, 256)), cfg)
    assert len(w4_hip._stream_workspaces) == int(own)
    assert (seen[0] == device) != own


@pytest.mark.gpu
def test_a_graph_runner_keeps_none():
    """Buckets past 16 whose projections split K: the warm-up's and the captures' workspaces are back when the runner is
    built, and every replay, an eager split call between them, gives the eager result."""
    k, n = 4096, 1024
    layer = awq.W4Linear(k, n, 128).cuda()
    g = torch.Generator(device="cuda").manual_seed(3)
    for t in (layer.qweight, layer.qzeros):
        t.copy_(torch.randint(-2**31, 2**31 - 1, t.shape, device="cuda", dtype=torch.int32, generator=g))
    layer.scales.copy_((torch.rand(layer.scales.shape, device="cuda", generator=g) * 0.01).half())
    layer.finalize(torch.cuda.get_device_name())
    assert layer.gemm_entry(40)[-1] != 1 and layer.gemm_entry(48)[-1] != 1
    emb = torch.randn(100, k, device="cuda", generator=g).half()
    w4_hip._stream_workspaces.clear()
    runner = decode_graph.DecodeGraphRunner(lambda ids: layer(emb[ids]), 48, torch.device("cuda", 0), logits=False)
    assert not w4_hip._stream_workspaces
    for b in (48, 40, 33, 3, 47):
        ids = torch.randint(0, 100, (b,), generator=torch.Generator().manual_seed(b))
        bucket = runner.bucket(b)
        padded = torch.zeros(bucket, dtype=torch.long)
        padded[:b] = ids
        with torch.inference_mode():
            want = layer(emb[padded.cuda()])[:b]
        assert torch.equal(runner.run(ids), want)
