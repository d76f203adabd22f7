"""Which kernel W4Linear runs where no measured table or ladder names one: rules on sizes, `decode` up to 16 rows and
`choose` past them.

choose: every candidate's time is predicted from the sizes alone and the fastest is taken. The terms follow the kernels'
structure, so one set of numbers per configuration covers every shape:

    U units (output tiles x K splits) are dealt to the CUs, so the busiest runs ceil(U / CUs) of them, `occ` at a time;
    a unit costs (its stages along K) x (time of a stage, alone on its CU or with a neighbour);
    a K split adds the wait for the last arriver and the traffic of its fp32 partial tiles;
    every launch has a fixed cost, every further unit of a CU a prologue and an epilogue.

The coefficients are microseconds on MI355X, fitted (non-negative least squares on relative errors) to 60,000 timed
calls: 24 (K, N) from 1024 x 4096 to 5120 x 34816 (N = 1032 and 7288 among them) x M = 17 .. 2048 x K splits, weights
streamed from HBM. The choice is within 1.5 % of the fastest candidate on average over those shapes (12 % at worst
past M = 32). For comparison, the fixed choice these shapes had before (8 wavefronts of the decode kernel up to M = 64,
the x-ring GEMM to 1024, dequantize + hipBLASLt above) is 1.1 to 6 times slower: Qwen3-14B gate_up at M = 40 133 us
against 37, Qwen3-8B-sized qkv (K 4096, N 6144) at M = 512 48 against 32.
"""

from __future__ import annotations

import functools

# tw4_gemm_tiled configurations (mt, nt, warps_n, warps_m, warps_k, ring): workgroups per CU, then launch, stage with
# `occ` workgroups on the CU, stage alone (occ 2), split, split traffic per 10^4 partial sums, further unit
TILED: dict[tuple[int, ...], tuple[int, float, float, float, float, float, float]] = {
    (2, 2, 2, 1, 2, 4): (2, 4.443, 0.240, 0.220, 0.694, 1.977, 0.0),      # 32 x 64
    (2, 3, 2, 1, 2, 4): (2, 4.701, 0.322, 0.251, 0.822, 1.471, 0.0),      # 32 x 96
    (3, 2, 2, 1, 2, 4): (2, 4.478, 0.293, 0.212, 0.886, 1.673, 0.039),    # 48 x 64
    (3, 3, 2, 1, 2, 4): (2, 4.819, 0.370, 0.256, 1.030, 0.945, 0.736),    # 48 x 96
    (4, 2, 2, 1, 2, 4): (2, 4.312, 0.332, 0.229, 1.108, 1.282, 0.635),    # 64 x 64
    (4, 3, 2, 1, 2, 4): (2, 5.099, 0.412, 0.275, 1.017, 0.814, 1.157),    # 64 x 96
    (5, 2, 2, 1, 2, 4): (2, 4.358, 0.365, 0.245, 1.420, 0.997, 1.050),    # 80 x 64
    (5, 3, 2, 1, 2, 4): (2, 4.837, 0.459, 0.315, 1.772, 0.842, 2.364),    # 80 x 96
    (5, 4, 2, 1, 2, 4): (2, 5.364, 0.573, 0.369, 2.035, 1.113, 2.748),    # 80 x 128
    (8, 2, 2, 1, 2, 4): (2, 4.618, 0.509, 0.302, 2.035, 0.871, 2.880),    # 128 x 64
    (8, 3, 2, 1, 2, 4): (2, 6.483, 0.793, 0.359, 2.624, 0.382, 4.447),    # 128 x 96
    (8, 4, 2, 1, 2, 4): (1, 6.902, 0.443, 0.0, 2.717, 0.523, 7.899),      # 128 x 128
    (8, 4, 4, 1, 1, 3): (2, 7.850, 1.384, 0.717, 2.187, 1.335, 6.444),    # 128 x 256
    (8, 6, 2, 1, 2, 4): (1, 9.730, 0.600, 0.0, 2.914, 1.666, 8.513),      # 128 x 192
    (8, 6, 2, 2, 1, 3): (1, 10.683, 1.024, 0.0, 3.676, 0.856, 19.989),    # 256 x 192
}
# tw4_gemm's x-ring configurations (mt, nt, warps_n, warps_k, stages), 2 workgroups per CU: a step is warps_k groups.
# Short K ranges and small N: its weights skip LDS, so it starts sooner.
RING: dict[tuple[int, ...], tuple[float, float, float, float, float, float]] = {
    (2, 1, 4, 2, 2): (3.377, 0.872, 0.660, 1.357, 1.714, 0.813),          # 32 x 64
    (4, 2, 4, 2, 2): (4.324, 2.511, 1.242, 1.426, 0.704, 4.418),          # 64 x 128
}
# The matrix-core decode kernel (warps_k, unroll, ntile), M <= 48, 2 workgroups per CU: launch, group per wavefront with two
# workgroups on the CU, alone, the same per 16-token batch tile, further unit, batch tile
MMA: dict[tuple[int, ...], tuple[float, float, float, float, float, float, float]] = {
    (4, 1, 1): (2.950, 0.016, 0.017, 0.733, 0.361, 0.0, 0.009),
    (4, 1, 2): (3.007, 0.167, 0.171, 0.723, 0.337, 0.0, 0.051),
    (4, 1, 3): (2.962, 0.491, 0.267, 0.705, 0.339, 0.0, 0.185),
    (4, 1, 6): (3.715, 1.056, 0.479, 0.814, 0.328, 0.0, 0.750),
}
SPLITS = (1, 2, 3, 4, 6, 8, 12, 16)
PARTIAL_FLOATS, PARTIAL_COUNTERS = 1 << 23, 1 << 15  # the split-K workspace (w4_hip.WORKSPACE_FLOATS / _LOCKS)
# Long calls run at the clock the card's power allows: PFLOP/s of the tiled GEMM and of hipBLASLt's fp16 product there,
# and the dequantization in front of the latter (bytes per us, launches) with the separate activation behind it.
TILED_PFLOPS, DENSE_PFLOPS = 1.24, 1.38
DENSE_BYTES_PER_US, DENSE_LAUNCH_US = 4.4e6, 8.0


def _cdiv(a: int, b: int) -> int:
    return -(-a // b)


def _units(units: int, cus: int, occ: int) -> tuple[int, int, int]:
    """Rounds of `occ` units, units left for a last round, further units, on the busiest CU."""
    n = _cdiv(units, cus)
    return n // occ, n % occ, n - 1


def dense_us(m: int, n: int, k: int, act: bool) -> float:
    """Dequantize + hipBLASLt (+ the separate SwiGLU: two elementwise kernels, 4 reads and 2 writes of M x N / 2)."""
    t = 2.0 * m * n * k / (DENSE_PFLOPS * 1e9)
    t += 2.53 * n * k / DENSE_BYTES_PER_US + DENSE_LAUNCH_US
    return t + (6.0 * m * n / DENSE_BYTES_PER_US + 8.0 if act else 0.0)


@functools.lru_cache(maxsize=4096)
def choose(m: int, n: int, k: int, act: bool = False, cus: int = 256) -> tuple | None:
    """The kernel for y[m, n] = x[m, k] W^T, m > 16, on a device of `cus` CUs: ("tiled", mt, nt, warps_n, warps_m,
    warps_k, ring, splits), ("mma", warps_k, unroll, ntile), w4_gemm's (mt, nt, warps_n, warps_k, stages, splits), or None:
    dequantize + torch.matmul, where the fused kernels do not reach hipBLASLt's rate by more than the dequantization
    costs (long, plain calls)."""
    best, entry = dense_us(m, n, k, act), None
    groups = k // 128

    def offer(t: float, e: tuple) -> None:
        nonlocal best, entry
        if t < best:
            best, entry = t, e

    def split_ok(tiles: int, splits: int, tile_floats: int) -> bool:
        if splits == 1:
            return True
        return splits <= groups and tiles <= PARTIAL_COUNTERS and tiles * splits * tile_floats <= PARTIAL_FLOATS

    if 16 * _cdiv(n, 16) * k < 1 << 33:  # the tiled kernel's 32-bit weight offsets, over whole row tiles
        floor = 2.0 * m * n * k / (TILED_PFLOPS * 1e9)
        for c, (occ, t0, s_full, s_one, d0, d1, u1) in TILED.items():
            bm, bn = 16 * c[0] * c[3], 16 * c[1] * c[2]
            tiles = _cdiv(m, bm) * _cdiv(n, bn)
            for sp in SPLITS:
                if not split_ok(tiles, sp, bm * bn) or (sp > 1 and tiles >= 2 * cus):
                    continue
                full, left, more = _units(tiles * sp, cus, occ)
                stages = 2 * _cdiv(groups, sp)
                t = t0 + stages * (full * s_full + (s_one if left else 0.0)) + u1 * more
                if sp > 1:
                    t += d0 + d1 * sp * bm * bn / 1e4
                offer(max(t, floor), ("tiled", *c, sp))
    if m <= 256:
        for c, (t0, s_full, s_one, d0, d1, u1) in RING.items():
            bm, bn = 16 * c[0], 16 * c[1] * c[2]
            tiles, steps = _cdiv(m, bm) * _cdiv(n, bn), _cdiv(groups, c[3])
            for sp in SPLITS:
                if not split_ok(tiles, sp, bm * bn) or sp > steps:
                    continue
                full, left, more = _units(tiles * sp, cus, 2)
                t = t0 + _cdiv(steps, sp) * (full * s_full + left * s_one) + u1 * more
                if sp > 1:
                    t += d0 + d1 * sp * bm * bn / 1e4
                offer(t, (*c, sp))
    if m <= 48:
        mt = 2 if m <= 32 else 4
        for c, (t0, s_full, s_one, x_full, x_one, u1, t1) in MMA.items():
            full, left, more = _units(_cdiv(_cdiv(n, 16), c[2]), cus, 2)
            per = _cdiv(groups, c[0])
            t = t0 + per * (full * (s_full + x_full * mt) + left * (s_one + x_one * mt)) + u1 * more + t1 * mt
            offer(t, ("mma", *c))
    return entry


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
