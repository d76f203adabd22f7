"""The norm kernels over every compiled width and every form (short and tall batches, four rows per workgroup): a row's result is the same bits
whatever the batch, and within rounding of 64 bits (fp32 arithmetic: K 2^-23 relative for the sum of squares, a few units of
2^-24 behind it, and half a unit in the last place of fp16, 2^-11; the residual is x + r rounded once)."""

from __future__ import annotations

import pytest
import torch

from tandem_amd.layers import norm

EPS = 1e-6


@pytest.mark.gpu
@pytest.mark.parametrize("k", [512 * i for i in (1, 2, 3, 4, 5, 6, 7, 8, 10, 12, 14, 16)])
def test_rows_do_not_depend_on_the_batch(k):
    g = torch.Generator(device="cuda").manual_seed(k)
    rows = 1025
    x0, r0 = (torch.randn(rows, k, device="cuda", dtype=torch.float16, generator=g) for _ in range(2))
    w = (0.5 + torch.rand(k, device="cuda", generator=g)).half()
    want_y = norm.rms_norm(x0, w, EPS)
    want_x, want_r = norm.fused_add_rms_norm(x0.clone(), r0.clone(), w, EPS)
    for m in (1, 3, 639, 640, 641, 642, 643, 1023, 1024):
        x, r = norm.fused_add_rms_norm(x0[-m:].clone(), r0[-m:].clone(), w, EPS)
        assert torch.equal(x, want_x[-m:]) and torch.equal(r, want_r[-m:])
        assert torch.equal(norm.rms_norm(x0[-m:].clone(), w, EPS), want_y[-m:])
    assert torch.equal(want_r, (x0.float() + r0.float()).half())
    for y, s in ((want_y, x0.double()), (want_x, x0.double() + r0.double())):
        ref = s * torch.rsqrt((s * s).mean(-1, keepdim=True) + EPS) * w.double()
        assert bool(((y.double() - ref).abs() <= (2.0**-11 + (k + 8) * 2.0**-23) * ref.abs() + 2.0**-25).all())
