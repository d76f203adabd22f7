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
    choice mma (4, 2, 1) is as good. From 28 shapes (K 768 .. 17408, N 1032 .. 24000) x 12 M x 11 matrix-core configurations on
    MI355X, 256 CUs, weights streamed from HBM (profiles/decode_rule_sweep.jsonl); at most 1.4 % slower than
    the fixed choice anywhere, 0.91 of its time on average. Against it:

    Row tiles for two and more workgroups per CU (tiles > 2 CUs): reading x again for every 16 rows is what costs, so
      several row tiles share a workgroup: with a long K from M = 5 on six from four tiles per CU (8192 x 20000 at M = 16
      43.2 -> 21.3 us), three below, where six leave CUs without a workgroup (4096 x 9000 14.4 -> 8.7), two at M = 3, 4. A short K
      (to 2048) is launch and x staging instead: 8 wavefronts up to M = 4 (1536 x 8960 at M = 3 4.73 -> 4.07) where the
      workgroups are few, two tiles up to M = 8 (1792 x 12800 at M = 5 5.63 -> 5.41), three from M = 9 on (2048 x 10240 at M = 16
      7.51 -> 5.85).
    One to two tiles per CU: two tiles per workgroup fill each CU once (17408 x 5120 at M = 16 36.1 -> 22.4).
    At most one tile per CU: wavefronts, not x, are short: 8 of them, for a long K while x fits LDS beside (m k <= 2^16; 17408 x 1536
      at M = 2 11.0 -> 9.2).

    Timed and left out: 16 wavefronts at most one tile per CU (5120 x 3000 at M = 12 6.2 -> 7.4) and 8 of them for a short K at M = 5 .. 8
    (2048 x 20000 at M = 5 7.0 -> 9.1), which an earlier form of the rule took from twelve shapes; and the vector-ALU GEMV at M = 1
    (4096 x 9000 6.3 -> 5.4): it takes the 1024 of its magic halves off a sum with x in it, so an infinite x gives NaN where the
    matrix cores give infinities."""
    if k > DECODE_MAX_K:
        return None
    tiles = _cdiv(n, 16)
    if tiles <= cus:
        if k <= 1536:
            return ("mma", 8, 1, 1) if m <= 8 else None
        return ("mma", 8, 2, 1) if k > 2304 and m * k <= 1 << 16 else None
    if tiles <= 2 * cus:
        if m < 4 or (m == 4 and k < 2048):
            return None
        return ("mma", 8, 1, 2) if m <= 8 else ("mma", 4, 2, 2)
    if k <= 2048:
        if m <= 4:
            return ("mma", 8, 1, 1) if tiles < 4 * cus else None
        if m <= 8:
            return ("mma", 4, 1, 2) if k < 2048 else None
        return ("mma", 4, 1, 3)
    if m < 3:
        return None
    if tiles >= 4 * cus:
        return ("mma", 4, 1, 6) if m >= 5 else ("mma", 4, 1, 2)
    return ("mma", 4, 2, 3) if m >= 5 or k > 4096 else None
