"""Which kernel W4Linear.forward takes past 16 rows: the ladders, a caller's own among them, and the rule on sizes."""

from __future__ import annotations

import contextlib
import copy
import ctypes
import pickle
import types

import numpy as np
import pytest
import torch
import torch.nn.functional as F
from torch.overrides import TorchFunctionMode

from oracle import awq_oracle as o
from tandem_amd.layers import awq, gemv16, w4_hip, w4_plan
from tandem_amd.layers.w4_tables import GFX950_GEMM, OTHERS, RuleLadder

FIXED = ((64, ("mma", 8, 1, 1)), (1024, (4, 2, 4, 1, 2, 0)), (1 << 30, None))


def _layer(k=4096, n=6144, table=GFX950_GEMM):
    layer = awq.W4Linear(k, n, 128)
    layer.awq_layout = False
    layer.gemm_kernels = table
    return layer


def test_layers_without_a_table_take_the_fixed_ladder():
    """finalize(None): every shape takes the defaults."""
    assert awq.DEFAULT_GEMM == FIXED
    for k, n in ((4096, 6144), (256, 64)):
        layer = _layer(k, n, {})
        for m in (17, 64, 65, 1024, 1025, 1 << 18):
            assert layer.gemm_entry(m) == awq.pick_gemm(FIXED, m), m


def test_built_in_ladders_are_continued_by_the_rule():
    for ladder in GFX950_GEMM.values():
        assert isinstance(ladder, RuleLadder)
    layer, other = _layer(), _layer(2304, 4112)
    ladder = GFX950_GEMM[6144, 4096]
    assert layer.gemm_entry(17) == ladder[0][1] and layer.gemm_entry(ladder[-1][0]) == ladder[-1][1]
    for m in (ladder[-1][0] + 1, 700, 5000):
        assert layer.gemm_entry(m) == w4_plan.choose(m, 6144, 4096)
    assert not GFX950_GEMM[OTHERS]
    for m in (17, 700, 5000):
        assert other.gemm_entry(m) == w4_plan.choose(m, 4112, 2304)


@pytest.mark.parametrize("table", [{}, GFX950_GEMM])
def test_a_callers_ladder_is_continued_by_its_last_entry(table):
    cfg = (2, 1, 4, 2, 2, 4)
    layer = _layer(table={**table, (6144, 4096): ((64, cfg), (1024, None))})
    assert layer.gemm_entry(64) == cfg and layer.gemm_entry(65) is None and layer.gemm_entry(5000) is None
    assert layer.kernel_for(5000) == "dequant+matmul"
    layer.gemm_kernels = {**table, (6144, 4096): ((64, None), (128, cfg))}
    assert layer.gemm_entry(5000) == cfg and layer.kernel_for(5000) == f"gemm{cfg}"


def test_ladders_survive_a_copy_of_the_layer():
    for other in (copy.deepcopy(_layer()), pickle.loads(pickle.dumps(_layer()))):
        assert other.gemm_kernels == GFX950_GEMM
        for m in (17, 700, 5000):
            assert other.gemm_entry(m) == _layer().gemm_entry(m)
        assert all(a.fused_rows == b.fused_rows for a, b in zip(other.gemm_kernels.values(), GFX950_GEMM.values()))


def test_a_layer_pickled_before_the_rules_runs():
    layer = _layer(table={(6144, 4096): FIXED})
    assert "cus" not in vars(layer) and "decode_rule" not in vars(layer)  # what such a pickle holds
    assert layer.decode_entry(3) == awq.DEFAULT_KERNEL and layer.gemm_entry(300) == FIXED[1][1]


@contextlib.contextmanager
def _autocast(dtype):
    """torch.autocast("cuda", dtype) without the check for a GPU."""
    was = torch.is_autocast_enabled("cuda"), torch.get_autocast_dtype("cuda")
    torch.set_autocast_enabled("cuda", True)
    torch.set_autocast_dtype("cuda", dtype)
    try:
        yield
    finally:
        torch.set_autocast_enabled("cuda", was[0])
        torch.set_autocast_dtype("cuda", was[1])


class _Counting(TorchFunctionMode):
    seen = 0

    def __torch_function__(self, func, types, args=(), kwargs=None):
        self.seen += func is F.linear
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("follow", [lambda: _autocast(torch.bfloat16), _Counting])
def test_followed_calls_keep_their_side_of_f_linear(follow):
    """Autocast decides the dtype of F.linear's result and a function mode sees the call: past fused_rows, where the layer
    dequantized for F.linear before it had a rule, it does so there still, and below it stays a kernel of its own."""
    for (k, n), rows in (((4096, 6144), 1 << 18), ((12288, 4096), 2048), ((2048, 2048), 1024), ((2304, 4112), 1024)):
        layer = _layer(k, n)
        for m in (17, 300, 1024, 1025, 2048, 2049, 5000):
            x = torch.empty(m, k, dtype=torch.float16)
            assert layer.gemm_entry(m, x) == layer.gemm_entry(m)
            with follow():
                e = layer.gemm_entry(m, x)
                assert (e is None) == (m > rows), (k, n, m, e)
    with _autocast(torch.float16), torch.device("cpu"):  # neither changes a product of float16 tensors
        assert not w4_hip.intercepted() and layer.gemm_entry(5000, x) == layer.gemm_entry(5000)


def test_compiled_layers_run_the_kernels(monkeypatch):
    """Under torch.compile the launch is a graph break; the route is the eager one (dequantize + F.linear past fused_rows)."""
    calls = []
    native = ctypes.CDLL(None).labs  # as a launch: nothing a compiler can trace

    def kernel(name):
        def run(x, *args):
            native(ctypes.c_long(x.data_ptr()))
            calls.append(name)
            return x[:, :64] * 1
        return run

    ext = types.SimpleNamespace(w4_mma=kernel("kernel"), w4_gemm=kernel("kernel"), w4_gemm_tiled=kernel("kernel"))
    monkeypatch.setattr(awq, "_gemm_ok", lambda x: x.shape[0] > 16)
    monkeypatch.setattr(awq, "_hip_ok", lambda x: x.shape[0] <= 16)
    monkeypatch.setattr(w4_hip, "load", lambda: ext)
    for name in ("workspace", "stream_workspace"):
        monkeypatch.setattr(w4_hip, name, lambda device: (None, None))
    monkeypatch.setattr(awq.W4Linear, "_dense", lambda self, x: (calls.append("dense"), x[:, :64] * 1)[1])
    layer = _layer(256, 64)
    layer.packed = layer.zeros = None
    torch._dynamo.reset()
    compiled = torch.compile(layer, backend="eager")
    for m, want in ((17, "kernel"), (100, "kernel"), (1024, "kernel"), (1025, "dense")):
        calls.clear()
        compiled(torch.zeros(m, 256, dtype=torch.float16))
        assert calls == [want], (m, calls)
    torch._dynamo.reset()


@pytest.mark.gpu
def test_autocast_and_modes_on_the_gpu():
    raw = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in o.random_awq(1152, 1032, seed=3)[:3]]
    layer = awq.W4Linear(1152, 1032, 128).cuda()
    for name, t in zip(("qweight", "qzeros", "scales"), raw):
        getattr(layer, name).copy_(t)
    layer.finalize(torch.cuda.get_device_name())
    w = torch.randn(32776, 2048, device="cuda", dtype=torch.float16) * 0.02
    table = gemv16.table_for(torch.device("cuda"), torch.nn.Module())
    x, xh = torch.randn(1100, 1152, device="cuda").half(), torch.randn(32, 2048, device="cuda").half()
    plain, head = layer(x), gemv16.linear(xh, w, table)
    dense, torch_head = F.linear(x, awq.w4_dequant(layer.packed, layer.scales, layer.zeros)), F.linear(xh, w)
    for a, b in ((plain, dense), (head, torch_head)):
        assert a.dtype == torch.float16
        torch.testing.assert_close(a, b, rtol=2e-3, atol=2e-3)  # two roundings to fp16, sums in two orders
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert layer(x).dtype == gemv16.linear(xh, w, table).dtype == torch.bfloat16
        assert layer(x[:300]).dtype == torch.float16
    with _Counting() as mode:
        assert torch.equal(layer(x), dense) and torch.equal(gemv16.linear(xh, w, table), torch_head)
        assert mode.seen == 2
        layer(x[:300])
        assert mode.seen == 2


@pytest.mark.parametrize("k,n", [(4096, 6144), (2304, 4112)])
def test_an_x_that_autograd_follows_takes_no_kernel(k, n):
    """Below a ladder's last m_max as past it."""
    layer = _layer(k, n)
    for m in (17, 24, 64, 65, 300, 5000):
        x = torch.empty(m, k, dtype=torch.float16, requires_grad=True)
        assert layer.gemm_entry(m, x) is None
        with torch.no_grad():
            assert layer.gemm_entry(m, x) == layer.gemm_entry(m)


@pytest.mark.gpu
def test_gradients_are_kept_at_every_size():
    k, n = 4096, 6144  # a shape with a ladder
    raw = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in o.random_awq(k, n, seed=5)[:3]]
    layer = awq.W4Linear(k, n, 128).cuda()
    for name, t in zip(("qweight", "qzeros", "scales"), raw):
        getattr(layer, name).copy_(t)
    layer.finalize(torch.cuda.get_device_name())
    w = awq.w4_dequant(layer.packed, layer.scales, layer.zeros)
    for m in (24, 100):
        x = torch.randn(m, k, device="cuda").half().requires_grad_()
        layer(x).sum().backward()
        assert torch.equal(x.grad, torch.autograd.grad(F.linear(x, w).sum(), x)[0])
    head = torch.randn(151936, 2048, device="cuda", dtype=torch.float16) * 0.02
    table = gemv16.table_for(torch.device("cuda"), torch.nn.Module())
    assert (151936, 2048, 1) in table
    for m in (1, 4, 8):
        x = torch.randn(m, 2048, device="cuda").half().requires_grad_()
        gemv16.linear(x, head, table).sum().backward()
        assert torch.equal(x.grad, torch.autograd.grad(F.linear(x, head).sum(), x)[0])
        assert gemv16.linear(x.detach(), head.requires_grad_(), table).requires_grad
        head.requires_grad_(False)
