"""tw4_gemm_f16 (the fp16 logits product by streaming w) at the edges of its tiles against 64 bits, and which calls of
gemv16.linear take it. Bound: an fp32 sum of K products in any order is within K 2^-23 sum |x w| of the exact one (the
matrix core may truncate), the fp16 result adds half a unit in the last place, 2^-11 |y| (2^-25 where subnormal)."""

from __future__ import annotations

import ctypes

import pytest
import torch
import torch.nn.functional as F

from tandem_amd.layers import gemv16, w4_hip


def test_argument_errors_return_before_launch():
    lib, p, odd = w4_hip.library(), ctypes.c_void_p(4096), ctypes.c_void_p(4104)
    for args, needle in (((None, p, p, 8, 64, 128), "null"), ((p, odd, p, 8, 64, 128), "aligned"),
                         ((p, p, p, 33, 64, 128), "M <= 32"), ((p, p, p, 8, 64, 96), "K % 64"),
                         ((p, p, p, 8, 1 << 20, 4096), "2^31")):
        assert lib.tw4_gemm_f16(*args, None) == w4_hip.TW4_EINVAL
        assert needle in lib.tw4_last_error().decode(), (args, lib.tw4_last_error())
    with pytest.raises(RuntimeError):  # CPU tensors never reach the library
        gemv16.gemm(torch.zeros(8, 128, dtype=torch.float16), torch.zeros(64, 128, dtype=torch.float16))


def _pair(m: int, n: int, k: int):
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    return (torch.randn(m, k, device="cuda", dtype=torch.float16, generator=g),
            torch.randn(n, k, device="cuda", dtype=torch.float16, generator=g) * 0.05)


def _check(y: torch.Tensor, x: torch.Tensor, w: torch.Tensor) -> None:
    x, w = x.double(), w.double()
    ref = x @ w.t().contiguous()
    err = x.shape[1] * 2.0**-23 * (x.abs() @ w.abs().t().contiguous())
    assert bool(((y.double() - ref).abs() <= err + 2.0**-11 * (ref.abs() + err) + 2.0**-25).all())


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 5, 15, 16, 17, 31, 32])
@pytest.mark.parametrize("n,k", [(1, 64), (15, 128), (64, 448), (127, 512), (257, 1088), (4099, 4096)])
def test_gemm_tile_edges(m, n, k):
    x, w = _pair(m, n, k)
    _check(gemv16.gemm(x, w), x, w)


def test_few_columns_stay_with_the_library():
    """Where the kernel's 64-row passes leave most CUs idle or x outgrows L2, F.linear is the faster one (up to 2x)."""
    for n, k in ((1024, 65536), (2048, 32768), (4736, 14336), (8192, 8192), (12288, 8192), (16384, 8192), (8192, 28672)):
        assert 2 * n * k >= gemv16.GEMM_MIN_BYTES and not any(gemv16.streams(m, n, k) for m in (1, 5, 17, 32))
    for n, k in ((131080, 512), (65536, 1024), (32776, 2048), (16384, 4096), (32000, 5120), (128256, 8192), (151936, 2560)):
        assert all(gemv16.streams(m, n, k) for m in (1, 5, 17, 32)) and not gemv16.streams(33, n, k)
    assert gemv16.streams(24, 49152, 12288) and not gemv16.streams(32, 49152, 12288)
    assert not gemv16.streams(8, 32768, 4000) and not gemv16.streams(8, 1 << 20, 2048) and not gemv16.streams(0, 32776, 2048)


@pytest.mark.gpu
def test_linear_takes_it_where_streaming_w_bounds(monkeypatch):
    table = gemv16.table_for(torch.device("cuda"), torch.nn.Module())
    calls = []
    for name in ("gemm", "gemv"):
        real = getattr(gemv16, name)
        monkeypatch.setattr(gemv16, name, lambda *a, real=real, name=name: (calls.append(name), real(*a))[1])
    x, w = _pair(32, 32776, 2048)  # 134 MB of weights
    assert 2 * w.numel() >= gemv16.GEMM_MIN_BYTES
    for m, want in ((1, "gemv"), (4, "gemv"), (5, "gemm"), (32, "gemm")):
        calls.clear()
        _check(gemv16.linear(x[:m], w, table), x[:m], w)
        assert calls == [want] and gemv16.route(x[:m], w, table).startswith(f"tw4_{want}_f16"), m
    calls.clear()
    short, wide = w[:4096], torch.cat([x, x])
    strided = torch.cat([x, x], dim=1)[:, :2048]
    for xx, ww, t in ((x, short, table), (wide, w, table), (strided, w, table), (x, w, {}), (x[:0], w, table)):
        assert torch.equal(gemv16.linear(xx, ww, t), F.linear(xx, ww)) and gemv16.route(xx, ww, t) == "F.linear"
    xg = x.clone().requires_grad_()
    gemv16.linear(xg, w, table).sum().backward()
    assert xg.grad is not None and not calls
