"""tw4_gemm_plan, the cost model behind w4_plan.choose: its choice against the same model evaluated in Python from the rows of
csrc/tw4_plan.hip and the terms that bench.fit_terms fits them with, its errors, and what a plan costs the call that makes it."""

from __future__ import annotations

import ctypes
import os
import random
import re
import time

import bench
from tandem_amd.layers import w4_hip, w4_plan

SOURCE = os.path.join(os.path.dirname(w4_hip.__file__), "..", "csrc", "tw4_plan.hip")
SPLITS = (1, 2, 3, 4, 6, 8, 12, 16)


def _rows() -> dict[tuple, list[float]]:
    text, rows = open(SOURCE, encoding="utf-8").read(), {}
    for kind, array, ints in (("tiled", "kPlanTiled", 7), ("gemm", "kPlanRing", 6), ("mma", "kPlanMma", 4)):
        body = re.search(array + r"\[\] = \{\n(.*?)\n\};", text, re.S).group(1)
        for line in body.splitlines():
            v = [float(t) for t in re.findall(r"[\d.]+(?:e-?\d+)?", line.split("//")[0])]
            head = [int(t) for t in v[:ints]]
            cfg = (kind, *(head[:-1]))
            rows[cfg] = v[ints:]
            assert bench.FIT_OCC[cfg] == (head[-1] if kind != "mma" else 2)
            if kind == "mma":
                rows[cfg, "max_m"] = head[-1]
    rows["dense",] = [float(t) for t in re.search(r"kPlanDense\[6\] = \{(.*?)\}", text).group(1).split(",")]
    return rows


ROWS = _rows()


def _cheapest(m: int, n: int, k: int, act: int, cus: int) -> dict[tuple | None, float]:
    up = lambda a, b: -(-a // b)  # noqa: E731
    scale = 256.0 / cus
    costs: dict[tuple | None, float] = {}
    for cfg in bench.FIT_OCC:
        groups = k // 128
        if cfg[0] == "mma":
            if m > ROWS[cfg, "max_m"]:
                continue
            t = bench.fit_terms(cfg, m, n, k, act, 1, cus)
            t[7:] = [v * scale for v in t[7:]]
            costs[cfg] = sum(a * b for a, b in zip(ROWS[cfg], t))
            continue
        bm, bn = (16 * cfg[1] * cfg[4], 16 * cfg[2] * cfg[3]) if cfg[0] == "tiled" else (16 * cfg[1], 16 * cfg[2] * cfg[3])
        if cfg[0] == "gemm" and m > 256 or cfg[0] == "tiled" and 16 * up(n, 16) * k >= 1 << 33:
            continue
        tiles = up(m, bm) * up(n, bn)
        for s in SPLITS:
            if s > 1 and (s > groups or tiles >= 2 * cus or tiles > 1 << 15 or tiles * s * bm * bn > 1 << 23):
                continue
            if cfg[0] == "gemm" and s > up(groups, cfg[4]):
                continue
            t = bench.fit_terms(cfg, m, n, k, act, s, cus)
            t[6:] = [v * scale for v in t[6:]]
            us = sum(a * b for a, b in zip(ROWS[cfg], t))
            if cfg[0] == "tiled":
                us = max(us, 2.0 * m * n * k / 1.24e9 * scale) + 1e-3 * us
            costs[(*cfg, s) if cfg[0] == "tiled" else (*cfg[1:], s)] = us
    if m >= bench.FIT_DENSE_ROWS:
        t = bench.fit_terms(("dense",), m, n, k, act, 1, cus)
        t[1:] = [v * scale if i != 2 else v for i, v in enumerate(t[1:])]
        costs[None] = sum(a * b for a, b in zip(ROWS["dense",], t)) * (1.03 if m % 256 else 1.0)
    return costs


def test_the_choice_is_the_models_cheapest():
    rng = random.Random(3)
    sizes = [(m, n, k) for m in (17, 48, 49, 64, 65, 256, 257, 1535, 1536, 8192) for n in (8, 1032, 24576) for k in (128, 4096)]
    sizes += [(rng.randint(17, 5000), 8 * rng.randint(1, 4400), 128 * rng.randint(1, 136)) for _ in range(150)]
    for m, n, k in sizes:
        for act in (0, 1) if n % 16 == 0 else (0,):
            for cus in (256, 32):
                costs = _cheapest(m, n, k, act, cus)
                e = w4_plan.choose(m, n, k, bool(act), cus)
                assert costs[e] <= min(costs.values()) * (1 + 1e-12), (m, n, k, act, cus, e)


def test_errors():
    lib, out = w4_hip.library(), (ctypes.c_int * 8)()
    for args, needle in (((32, 60, 256, 0, 256), "N % 8"), ((32, 64, 100, 0, 256), "K % 128"), ((0, 64, 256, 0, 256), "M >= 1"),
                         ((32, 64, 256, 0, 0), "CUs")):
        assert lib.tw4_gemm_plan(*args, out) == -w4_hip.TW4_EINVAL and needle in lib.tw4_last_error().decode()
    assert lib.tw4_gemm_plan(32, 64, 256, 0, 256, None) == -w4_hip.TW4_EINVAL


def test_a_plan_costs_less_than_a_launch():
    """The first call at every new prompt length makes one per projection shape (a search in Python took 80-340 us; the bound
    leaves room for a loaded host)."""
    best = 1.0
    for attempt in range(5):
        t = time.perf_counter()
        for m in range(100 + 50 * attempt, 150 + 50 * attempt):
            w4_plan.choose(m, 24576, 4224, False)
        best = min(best, (time.perf_counter() - t) / 50)
    assert best < 40e-6
