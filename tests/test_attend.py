"""One-token attention (tw4_attend_one behind Attention.attend): the value row of each query head's KV head, bit for bit
against the plain torch expression on the CPU, over the layouts the kernel takes and those it leaves to torch."""

from __future__ import annotations

import ctypes

import pytest
import torch

from tandem_amd import model as tmodel
from tandem_amd.layers import w4_hip


def test_argument_errors_return_before_launch():
    lib, p, odd = w4_hip.library(), ctypes.c_void_p(4096), ctypes.c_void_p(4104)
    for args, needle in (((None, p, 1, 8, 2, 128), "null"), ((odd, p, 1, 8, 2, 128), "aligned"),
                         ((p, p, 1, 8, 3, 128), "multiple"), ((p, p, 1, 8, 2, 12), "head_dim"),
                         ((p, p, 1 << 24, 32, 8, 128), "too many")):
        assert lib.tw4_attend_one(*args, None) == w4_hip.TW4_EINVAL
        assert needle in lib.tw4_last_error().decode(), (args, lib.tw4_last_error())
    assert lib.tw4_attend_one(p, p, 0, 8, 2, 128, None) == w4_hip.TW4_OK


@pytest.mark.gpu
@pytest.mark.parametrize("heads,kv,dim", [(1, 1, 8), (3, 3, 64), (4, 2, 12), (5, 1, 40), (16, 8, 128), (40, 8, 128)])
@pytest.mark.parametrize("m", [0, 1, 5, 129])
def test_attend_matches_torch(m, heads, kv, dim):
    attn = tmodel.Attention(tmodel.DecoderConfig(64, 64, heads, kv, dim, 1, 64))
    qkv = torch.randn(m, (heads + 2 * kv) * dim, generator=torch.Generator().manual_seed(m)).half()
    want = attn.attend(qkv)  # CPU: torch
    flat = torch.empty(qkv.numel() + 1, dtype=torch.float16, device="cuda")
    flat[1:] = qkv.flatten().cuda()
    wide = torch.cat([qkv, qkv], dim=1).cuda()
    for x in (qkv.cuda(), flat[1:].view(qkv.shape), wide[:, :qkv.shape[1]], qkv.float().cuda()):
        y = attn.attend(x)
        assert y.is_contiguous() and y.dtype == x.dtype and torch.equal(y.half().cpu(), want)
    x = qkv.cuda()
    copies = attn.attend(x).untyped_storage().data_ptr() != x.untyped_storage().data_ptr()
    assert m == 0 or copies == (m > 1 or heads > kv)  # one row of as many KV heads: a view
    x.requires_grad_()
    attn.attend(x).float().sum().backward()
    assert float(x.grad.double().sum()) == m * heads * dim


def test_plain_is_false_where_torch_follows_the_call():
    """A kernel behind a data pointer is invisible to gradients, tangents, transforms, tracers and dispatch modes."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.fx.experimental.proxy_tensor import make_fx

    x, seen = torch.randn(2, 8), []

    def look(t):
        seen.append(w4_hip.plain(t))
        return t * 2

    assert w4_hip.plain(x) and w4_hip.plain(torch.nn.Parameter(x, requires_grad=False))
    look(x.clone().requires_grad_())
    torch.func.vmap(look)(x)
    torch.func.jvp(look, (x,), (x,))
    with torch.autograd.forward_ad.dual_level():
        look(torch.autograd.forward_ad.make_dual(x, x))
        assert w4_hip.plain(x)
    torch.jit.trace(look, x, check_trace=False)
    make_fx(look)(x)
    with FakeTensorMode() as mode:
        look(mode.from_tensor(x))
    assert len(seen) >= 6 and not any(seen), seen
    with torch.no_grad():
        assert w4_hip.plain(x.clone().requires_grad_())
