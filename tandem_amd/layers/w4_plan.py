"""Which kernel W4Linear runs where no measured table or ladder names one: rules on sizes, `decode` up to 16 rows and
`choose` past them."""

from __future__ import annotations

import ctypes
import functools

from tandem_amd.layers import w4_hip

_KINDS = {1: ("mma",), 2: (), 3: ("tiled",)}


def _cdiv(a: int, b: int) -> int:
    return -(-a // b)


@functools.lru_cache(maxsize=1 << 14)
def choose(m: int, n: int, k: int, act: bool = False, cus: int = 256) -> tuple | None:
    """The kernel for y[m, n] = x[m, k] W^T, m > 16, on a device of `cus` CUs, by the cost model of tw4_gemm_plan
    (csrc/tw4_plan.hip): ("tiled", mt, nt, warps_n, warps_m, warps_k, ring, splits), ("mma", warps_k, unroll, ntile), w4_gemm's
    (mt, nt, warps_n, warps_k, stages, splits), or None: dequantize + torch.matmul, where the fused kernels do not reach
    hipBLASLt's rate by more than the dequantization costs (long, plain calls)."""
    out = (ctypes.c_int * 8)()
    ints = w4_hip.library().tw4_gemm_plan(m, n, k, act, cus, out)
    if ints < 0:
        w4_hip.check(-ints)
    return (*_KINDS[out[0]], *out[1:ints]) if out[0] else None


DECODE_MAX_K = 17408  # the largest K the rule was timed at


def decode(m: int, n: int, k: int, cus: int = 256) -> tuple | None:
    """The decode kernel for 1 <= m <= 16 rows of a shape without table entries, None where the fixed
    choice mma (4, 2, 1) is as good. From 12 shapes (K 1024 .. 16384, N 1032 .. 24000) x M = 1, 2, 4, 8, 16 x every
    compiled matrix-core configuration on MI355X, 256 CUs, weights streamed from HBM; up to 2.2 times faster than the fixed
    choice (one of the 60 points is slower, by 1 %).
    us, fixed -> this choice:

    Row tiles for two and more workgroups per CU (tiles > 2 CUs): reading x again for every 16 rows is what costs, so
      several row tiles share a workgroup from M = 5 on: six from four tiles per CU (8192 x 20000 at M = 16 42.9 -> 22.6),
      three below, where six leave CUs without a workgroup (4096 x 9000 14.3 -> 8.7); a short K (to 2048) is launch and
      x staging instead and keeps one tile, 8 wavefronts, up to M = 12. M = 3, 4: two tiles (8192 x 20000 at M = 4
      22.3 -> 19.3), three from K 4096 on between (13056 x 10240 22.9 -> 18.5).
    One to two tiles per CU: two tiles per workgroup fill each CU once (8192 x 5000 at M = 16 18.0 -> 11.3).
    At most one tile per CU: wavefronts, not x, are short: 16 of them while x fits LDS beside (m k <= 2^16; 16384 x 1536 at M = 4
      10.4 -> 8.1), 8 for a short K.

    Timed and left out: the vector-ALU GEMV at M = 1 (4096 x 9000 6.3 -> 5.4). It takes the 1024 of its magic halves off a sum
    with x in it, so an infinite x gives NaN where the matrix cores give infinities; an eager call is bound by the host there."""
    if k > DECODE_MAX_K:
        return None
    tiles = _cdiv(n, 16)
    if tiles <= cus:
        if k <= 2304:
            return ("mma", 8, 1, 1)
        return ("mma", 16, 2, 1) if m * k <= 1 << 16 else None
    if tiles <= 2 * cus:
        if m < 4:
            return None
        return ("mma", 8, 1, 2) if m <= 8 else ("mma", 4, 2, 2)
    if k <= 2048:
        return ("mma", 8, 1, 1) if m <= 12 else ("mma", 4, 1, 3)
    if m < 3:
        return None
    if tiles >= 4 * cus:
        return ("mma", 4, 1, 6) if m >= 5 else ("mma", 4, 1, 2)
    return ("mma", 4, 2, 3) if m >= 5 or k > 4096 else None
