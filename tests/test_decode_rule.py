"""w4_plan.decode, the rule for M <= 16 rows of a shape no table names: on the CPU every choice is a compiled
configuration its entry point takes; on the GPU the layer's choices against the oracle at the sizes where the rule turns.

Bound: K fp32 products of the fp16 weights summed in some order, within K 2^-23 sum |x w|, and one rounding to fp16, 2^-11 |y|."""

from __future__ import annotations

import random

import numpy as np
import pytest
import torch

from oracle import awq_oracle as o
from tandem_amd.layers import awq, w4_hip, w4_plan


def test_every_choice_is_compiled():
    rng = random.Random(11)
    sizes = [(m, n, k) for m in range(1, 17) for n in (8, 4096, 4104, 8192, 8200, 16376, 16384, 151936)
             for k in (128, 2048, 2304, 2432, 4096, 4224, 13312, 13440, 17408, 17536)]
    sizes += [(rng.randint(1, 16), 8 * rng.randint(1, 4400), 128 * rng.randint(1, 140)) for _ in range(400)]
    mma = w4_hip.mma_configs()
    for m, n, k in sizes:
        for cus in (256, 32):
            e = w4_plan.decode(m, n, k, cus)
            assert e is None or (e[0] == "mma" and e[1:] in mma and k <= 17408), (m, n, k, e)


def test_eight_and_sixteen_wavefronts_only_where_they_pay():
    """Sizes where they take 1.1 to 1.4 of the fixed choice's time: many row tiles with a short K, and x past what leaves room
    beside it."""
    for m, n, k in ((1, 20000, 768), (10, 20000, 768), (9, 17000, 1024), (5, 20000, 2048), (6, 8960, 1536), (5, 12800, 1792),
                    (12, 10240, 2048), (12, 3000, 5120), (3, 3000, 5120), (12, 3000, 2304), (4, 4864, 896), (10, 4096, 1024)):
        e = w4_plan.decode(m, n, k)
        assert e is None or e[1] == 4 or e == ("mma", 8, 2, 1), (m, n, k, e)
    assert w4_plan.decode(3, 8960, 1536) == w4_plan.decode(8, 1032, 1152) == ("mma", 8, 1, 1)
    assert w4_plan.decode(2, 1536, 17408) == ("mma", 8, 2, 1)


def test_layers_without_a_table_keep_the_default():
    layer = awq.W4Linear(4096, 9000, 128)
    assert layer.decode_entry(16) == layer.norm_entry(1) == awq.DEFAULT_KERNEL
    layer.decode_rule = True
    assert layer.decode_entry(16) == ("mma", 4, 2, 3) and layer.norm_entry(16) == awq.DEFAULT_KERNEL
    layer.kernels = {(9000, 4096, 16): ("mma", 8, 1, 1)}
    assert layer.decode_entry(16) == layer.norm_entry(16) == ("mma", 8, 1, 1)


@pytest.mark.gpu
@pytest.mark.parametrize("k,n,silu", [(128, 8, False), (1152, 4112, True), (2432, 1032, False), (4224, 4120, False),
                                      (2176, 8208, True), (4224, 8200, False), (1024, 12000, False), (1152, 16392, False),
                                      (2304, 16400, True), (17408, 264, False)])
def test_layer_against_the_oracle(k, n, silu):
    raw = o.random_awq(k, n, seed=k + n)[:3]
    layer = awq.W4Linear(k, n, 128).cuda()
    for name, t in zip(("qweight", "qzeros", "scales"), raw):
        getattr(layer, name).copy_(torch.from_numpy(np.ascontiguousarray(t)).cuda())
    if silu:
        layer.enable_silu_mul()
    layer.finalize(torch.cuda.get_device_name())
    w = torch.from_numpy(o.dequant(*raw)).cuda().double()
    for m in (1, 2, 3, 4, 5, 8, 9, 13, 16):
        x = torch.randn(m, k, generator=torch.Generator().manual_seed(m)).half().cuda()
        y = layer(x).double()
        ref = x.double() @ w.T
        err = k * 2.0**-23 * (x.double().abs() @ w.abs().T)
        if silu:
            (g, u), (eg, eu) = ref.chunk(2, 1), (err + 2.0**-11 * ref.abs() + 2.0**-25).chunk(2, 1)
            a = g * torch.sigmoid(g)
            ref, err = a * u, 1.1 * eg * (u.abs() + eu) + a.abs() * eu + 2.0**-18 * (a * u).abs()  # |silu'| < 1.1
        bound = err + 2.0**-11 * (ref.abs() + err) + 2.0**-24
        assert bool(((y - ref).abs() <= bound).all()), (m, layer.kernel_for(m), float(((y - ref).abs() / bound).max()))
