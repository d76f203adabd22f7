"""The load-time kernels at the edges of their tiles: the repack takes 256 columns x 128 k per workgroup and writes the
padding rows itself, the dequantization 16 rows x 512 k. Every word and every weight is compared with the host layout
utilities and the oracle, bit for bit, over the ways the kernels can be handed their memory (bases that are only
4-byte aligned take the narrow loads and stores)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import awq_oracle as o
from tandem_amd.layers import awq, w4_hip

pytestmark = pytest.mark.gpu

# one half tile; short of, at and past a workgroup's columns; 1, 2, 3, 4, 5, 9 groups; N / 8 even, odd and a multiple of 4
SIZES = [(128, 8), (128, 16), (256, 248), (384, 256), (512, 264), (640, 520), (1152, 288), (128, 4104)]


def _shifted(t: torch.Tensor) -> torch.Tensor:
    """t on the GPU at a base 4 bytes past a 16-byte boundary."""
    words = t.contiguous().view(torch.int32).reshape(-1)
    buf = torch.empty(words.numel() + 4, dtype=torch.int32, device="cuda")
    buf[1:1 + words.numel()] = words.cuda()
    return buf[1:1 + words.numel()].view(t.dtype).reshape(t.shape)


@pytest.mark.parametrize("shift", [False, True])
@pytest.mark.parametrize("k,n", SIZES)
def test_repack_and_dequant_tile_edges(k, n, shift):
    qweight, qzeros, scales, q, z = o.random_awq(k, n, seed=k + n)
    raw = [torch.from_numpy(np.ascontiguousarray(a)) for a in (qweight, qzeros, scales)]
    raw = [_shifted(t) if shift else t.cuda() for t in raw]
    q, z, s = (torch.from_numpy(np.ascontiguousarray(a.T)) for a in (q, z.astype(np.float16), scales))
    for interleave in (False, True) if n % 16 == 0 else (False,):
        order = awq.interleave_gate_up if interleave else lambda t: t
        words = w4_hip.padded_rows(n) * k // 8
        store = torch.full((words + 4,), -1, dtype=torch.int32, device="cuda")  # the kernel writes every word
        packed = store[int(shift):words + int(shift)]
        s_out = torch.empty((n, k // 128), dtype=torch.float16, device="cuda")
        z_out = torch.empty_like(s_out)
        w4_hip.check(w4_hip.library().tw4_repack_awq(
            *(t.data_ptr() for t in raw), packed.data_ptr(), s_out.data_ptr(), z_out.data_ptr(), k, n, int(interleave),
            torch.cuda.current_stream().cuda_stream))
        assert torch.equal(packed.cpu().view(-1, k // 8), awq.pack_rows(order(q)))
        assert (store.cpu()[:int(shift)] == -1).all() and (store.cpu()[words + int(shift):] == -1).all()
        assert torch.equal(s_out.cpu(), awq.tile_major_params(order(s)))
        assert torch.equal(z_out.cpu(), awq.tile_major_params(order(z)))
        for near in (False, True):
            w = w4_hip.dequant(packed.clone().view(-1, k // 8), s_out, z_out, deinterleave=interleave, near=near)
            assert np.array_equal(w.cpu().numpy().view(np.uint16), o.dequant(qweight, qzeros, scales).view(np.uint16))
