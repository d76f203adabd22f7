"""tw4_gemm_tiled and the rule that picks the M > 16 kernel: on the CPU every choice is compiled and inside the limits of
its entry point; on the GPU every configuration at the edges of its tiles, and the layer's choices against 64 bits.

Bounds: an fp32 sum of K products in any order is within K 2^-23 sum |x w| of the exact one (the matrix core may
truncate), the fp16 result adds half a unit in the last place, 2^-11 |y| (2^-25 where subnormal)."""

from __future__ import annotations

import ctypes
import random

import numpy as np
import pytest
import torch

from oracle import awq_oracle as o
from tandem_amd.layers import awq, w4_hip, w4_plan

CONFIGS = w4_hip.gemm_tiled_configs()


def test_every_choice_is_compiled_and_within_limits():
    rng = random.Random(5)
    sizes = [(m, n, k) for m in (17, 18, 48, 49, 64, 65, 256, 257, 1 << 20) for n in (8, 16, 1032, 151936) for k in (128, 1152, 4096)]
    sizes += [(rng.randint(17, 8192), 8 * rng.randint(1, 4400), 128 * rng.randint(1, 136)) for _ in range(400)]
    for m, n, k in sizes:
        for act in (False, True) if n % 16 == 0 else (False,):
            for cus in (256, 32):
                e = w4_plan.choose(m, n, k, act, cus)
                if e is None:
                    continue
                if e[0] == "mma":
                    assert e[1:] in w4_hip.mma_configs() and m <= 64
                    continue
                if e[0] == "tiled":
                    _, mt, nt, wn, wm, wk, ring, sp = e
                    assert (mt, nt, wn, wm, wk, ring) in CONFIGS and n * k < 1 << 33
                    limit = 2 * (k // 128)
                else:
                    mt, nt, wn, wk, stages, sp = e
                    wm = 1
                    assert (mt, nt, wn, wk, stages) in w4_hip.gemm_configs()
                    limit = -(-(k // 128) // wk)
                tiles = -(-m // (16 * mt * wm)) * -(-n // (16 * nt * wn))
                assert 1 <= sp <= min(16, limit)
                if sp > 1:
                    assert tiles * sp * 256 * mt * wm * nt * wn <= w4_hip.WORKSPACE_FLOATS and tiles <= w4_hip.WORKSPACE_LOCKS


def test_argument_errors_return_before_launch():
    lib, p, odd = w4_hip.library(), ctypes.c_void_p(4096), ctypes.c_void_p(4098)
    cfg = CONFIGS[-1]

    def call(x=p, s=p, ws=p, m=32, n=64, k=256, cfg=cfg, splits=1, act=0):
        return lib.tw4_gemm_tiled(x, p, s, p, p, ws, ws, 1 << 23, 1 << 15, m, n, k, *cfg, splits, act, None)

    for kw, needle in (({"x": None}, "null"), ({"x": odd}, "aligned"), ({"k": 100}, "K % 128"), ({"n": 60}, "N % 8"),
                       ({"n": 24, "act": 1}, "SwiGLU"), ({"splits": 17}, "splits"), ({"splits": 2, "ws": None}, "workspace")):
        assert call(**kw) == w4_hip.TW4_EINVAL
        assert needle in lib.tw4_last_error().decode(), (kw, lib.tw4_last_error())
    # the packed weights end at a whole row tile: N = 8 mod 16 just under 2^33 / K passes 2^32 bytes with its padding rows
    n, k = 1677720, 5120
    assert n * k < 1 << 33 <= (n + 8) * k
    assert call(n=n, k=k) == w4_hip.TW4_EINVAL and "2^33" in lib.tw4_last_error().decode()
    assert all((w4_plan.choose(m, n, k) or ("",))[0] != "tiled" for m in (17, 300, 4096))
    assert call(m=0) == w4_hip.TW4_OK
    assert lib.tw4_capture_id(None) == 0


def _reference(x: np.ndarray, w: np.ndarray, silu: bool):
    """y in 64 bits of x [M, K] and the dense fp16 w [N, K] (gate rows, then up rows), and its bound."""
    x64, w64 = x.astype(np.float64), w.astype(np.float64)
    y = x64 @ w64.T
    err = x.shape[1] * 2.0**-23 * (np.abs(x64) @ np.abs(w64).T)
    if silu:
        (g, u), (eg, eu) = np.split(y, 2, axis=1), np.split(err + 2.0**-11 * np.abs(y) + 2.0**-25, 2, axis=1)
        a = g / (1.0 + np.exp(-g))
        y, err = a * u, 1.1 * eg * (np.abs(u) + eu) + np.abs(a) * eu + 2.0**-18 * np.abs(a * u)  # |silu'| < 1.1
    return y, err + 2.0**-11 * (np.abs(y) + err) + 2.0**-24


def _check(y: torch.Tensor, ref, what) -> None:
    diff = np.abs(y.double().cpu().numpy() - ref[0])
    assert (diff <= ref[1]).all(), (what, float((diff / ref[1]).max()))


class _Case:
    def __init__(self, k, n, seed, interleave=False):
        raw = o.random_awq(k, n, seed=seed)[:3]
        self.w = o.dequant(*raw)
        self.raw = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in raw]
        self.tile = w4_hip.repack(*self.raw, interleave=interleave)
        self.k = k

    def x(self, m, seed):
        return np.random.default_rng(seed).standard_normal((m, self.k)).astype(np.float16)


@pytest.mark.gpu
@pytest.mark.parametrize("cfg", CONFIGS, ids=str)
def test_every_config_at_its_tile_edges(cfg):
    ext = w4_hip.load()
    ws, locks = w4_hip.stream_workspace(torch.device("cuda"))
    mt, nt, wn, wm, _, _ = cfg
    bm, bn = 16 * mt * wm, 16 * nt * wn
    for k, n, ms in ((128, 8, (1, bm)), (128, bn + 8, (bm + 1,)), (384, 2 * bn, (17, 2 * bm - 1)), (1152, bn - 16, (bm - 1,))):
        for silu in (False, True) if n % 16 == 0 else (False,):
            c = _Case(k, n, seed=k + n, interleave=silu)
            for m in ms:
                x = c.x(m, m)
                ref = _reference(x, c.w, silu)
                for splits in (0, 1, 2, 3, 2 * (k // 128)):
                    if splits <= min(16, 2 * (k // 128)):
                        y = ext.w4_gemm_tiled(torch.from_numpy(x).cuda(), *c.tile, ws, locks, *cfg, splits, int(silu))
                        _check(y, ref, (k, n, m, silu, splits))
    assert int(locks.abs().sum()) == 0


def _layer(k, n, silu):
    layer = awq.W4Linear(k, n, 128).cuda()
    c = _Case(k, n, seed=n, interleave=silu)
    for name, t in zip(("qweight", "qzeros", "scales"), c.raw):
        getattr(layer, name).copy_(t)
    if silu:
        layer.enable_silu_mul()
    layer.finalize(torch.cuda.get_device_name())
    return layer, c


@pytest.mark.gpu
@pytest.mark.parametrize("k,n,silu", [(128, 8, False), (1152, 1032, False), (2560, 2560, False), (1024, 4112, True)])
def test_layer_past_the_table(k, n, silu):
    """Shapes no table names, at every kind of kernel the rule chooses, and under autograd (dequantize + matmul)."""
    layer, c = _layer(k, n, silu)
    for m in (17, 33, 48, 49, 64, 65, 130, 257, 1100):
        x = c.x(m, m)
        _check(layer(torch.from_numpy(x).cuda()), _reference(x, c.w, silu), (m, layer.kernel_for(m)))
    x = torch.from_numpy(c.x(1100, 1)).cuda().requires_grad_()
    layer(x).float().sum().backward()
    assert x.grad.shape == x.shape and bool(x.grad.abs().sum() > 0)


@pytest.mark.gpu
def test_graphs_and_streams_share_no_partial_sums():
    """K splits on two streams at once and in two graphs replayed at once, the first graph's workspace dropped by the
    second capture: every result is the eager one."""
    layer, c = _layer(4096, 1024, False)
    assert layer.gemm_entry(40)[-1] > 1
    xs = [torch.from_numpy(c.x(40, i)).cuda() for i in range(2)]
    want = [layer(x) for x in xs]
    streams = [torch.cuda.Stream() for _ in xs]
    graphs, outs, ids = [], [], []
    for x, s in zip(xs, streams):
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            ids.append(w4_hip.library().tw4_capture_id(torch.cuda.current_stream().cuda_stream))
            outs.append(layer(x))
            assert ids[-1] == w4_hip.library().tw4_capture_id(torch.cuda.current_stream().cuda_stream)
        graphs.append(g)
    assert ids[0] != ids[1] and 0 not in ids
    torch.cuda.synchronize()
    for _ in range(3):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                graphs[i].replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(outs, want))
        eager = []
        for x, s in zip(xs, streams):
            with torch.cuda.stream(s):
                eager.append(layer(x))
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(eager, want))
    assert len(w4_hip._stream_workspaces) <= w4_hip.STREAM_WORKSPACES
