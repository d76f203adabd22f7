"""Small-batch fp16 products for decode on MI355X: y[M, N] = x[M, K] @ w[N, K]^T, M <= 32.

Drop-in for python/tandem/layers/triton_gemv.py (12vivi/tandem) on the path of a W4A16 model's
fp16 lm_head: the same ``gemv`` / ``linear`` / ``install`` / ``table_for`` / ``default_table``
functions, the same per-GPU ``CONFIGS`` keyed by (N, K, M bucket) and the same fallback to
``F.linear`` (hipBLASLt here). Two kernels of libtandem_w4.so (hand-written HIP for gfx950, no
Triton), both bound by streaming w once: tw4_gemv_f16 (``gemv``, M <= 8, a config from the table) with
coalesced 16-byte loads and v_dot2_f32_f16, and tw4_gemm_f16 (``gemm``, M <= 32) on the matrix cores with
both operands through LDS, which ``linear`` takes by a rule on sizes (``streams``) for the shapes and batches
the table does not name. A matrix-core form of tw4_gemv_f16 (rows_inflight 16 or 32) stays as a
configuration a caller's table can name; no built-in entry does (tw4_gemm_f16 is faster).

The reference's fused norm / activation prologue (triton_gemv.py:92-178, 330-415) is not part of
this build: it enabled no shape there (triton_gemv.py:316-329).
"""

from __future__ import annotations

import os

import torch
import torch.nn.functional as F
from torch import nn

from tandem_amd.layers import w4_hip

# Config per GPU and (N, K, M bucket): (rows_inflight, rows_per_wave) of tw4_gemv_f16 (rows_inflight
# 16 / 32: the matrix-core form with one / two 128-k chunks per step in flight, rows_per_wave a
# multiple of 16), the fastest of
# `python bench.py tune --projs lm_head --kinds dense16,torch16` on the GPU. Shapes without
# an entry take ``streams``' rule, else F.linear (python/tandem/layers/triton_gemv.py:221-268). Keyed by device name and by
# gfx architecture.
Config = tuple[int, int]
GFX950_DENSE: dict[tuple[int, int, int], Config] = {
    # Qwen3-8B lm_head: 190 / 185 / 188 us at M = 1 / 2 / 4 (82-84 % of 8 TB/s) vs F.linear 243-251 us
    # (M = 5 .. 8: no entry, tw4_gemm_f16 by its rule, 196-197 us where the matrix-core form (32, 16) took 231)
    (151936, 4096, 1): (4, 32),
    (151936, 4096, 2): (2, 32),
    (151936, 4096, 4): (2, 32),
    # Qwen3-1.7B lm_head: 96-99 us at M = 1 .. 4 vs F.linear 203 us (M = 5 .. 8: tw4_gemm_f16 107, (16, 16) 116-119)
    (151936, 2048, 1): (2, 16),
    (151936, 2048, 2): (2, 16),
    (151936, 2048, 4): (2, 16),
}
CONFIGS: dict[str, dict[tuple[int, int, int], Config]] = {
    "AMD Instinct MI355X": GFX950_DENSE,
    "gfx950": GFX950_DENSE,
}

# The decoder projections a step runs through the kernel when the table has their shape (the names
# python/tandem/layers/triton_gemv.py:270 routes), and the K the kernel is compiled for.
PROJECTIONS = ("qkv_proj", "o_proj", "gate_up_proj", "down_proj")
KS = (512, 1024, 2048, 4096)
# Batch buckets of the decode graphs: a table entry for bucket b serves every M up to b.
BUCKETS = (1, 2, 4, 8)
# What ``default_table`` gives every shape: two rows in flight, 32 rows per wavefront (the v_dot2 form).
DEFAULT_CONFIG: Config = (2, 32)


def m_bucket(m: int) -> int:
    """The bucket whose entry serves a batch of m rows: the smallest of BUCKETS that holds m (M past
    the last bucket maps to it; the caller sends those to F.linear)."""
    return next((b for b in BUCKETS if m <= b), BUCKETS[-1])


def _device_keys(device: torch.device) -> list[str]:
    """Table keys of a GPU, most specific first: its marketing name, then its gfx architecture (a
    HIP runtime can report a generic name, or none under rocprofv3)."""
    arch = getattr(torch.cuda.get_device_properties(device), "gcnArchName", "").split(":")[0]
    return [torch.cuda.get_device_name(device), arch]


def table_for(device: torch.device, model: nn.Module) -> dict[tuple[int, int, int], Config]:
    """The measured table of ``device``, or {} (every call then takes F.linear). With
    ``TANDEM_GEMV_FORCE`` set to 1 or 2 (the reference's test switch) every projection of ``model``
    the kernel can run gets ``DEFAULT_CONFIG`` instead (python/tandem/layers/triton_gemv.py:277-282)."""
    if os.environ.get("TANDEM_GEMV_FORCE") in ("1", "2"):
        return default_table(model)
    return next((CONFIGS[k] for k in _device_keys(device) if k in CONFIGS), {})


def gemv(x: torch.Tensor, w: torch.Tensor, rows_inflight: int = 2, rows_per_wave: int = 32,
         out: torch.Tensor | None = None) -> torch.Tensor:
    """y [M, N] = x [M, K] @ w [N, K]^T by tw4_gemv_f16, 1 <= M <= 8, float16 GPU tensors, on the
    current stream (python/tandem/layers/triton_gemv.py:180-218). Shapes the kernel does not take
    raise ValueError; placement, dtype and alignment problems RuntimeError, before any launch.
    ``out``: a float16 [M, N] contiguous 16-byte aligned tensor on x's GPU to write into."""
    if x.dim() != 2 or w.dim() != 2 or x.shape[1] != w.shape[1]:
        raise ValueError(f"gemv: x [M, K] and w [N, K] expected (x {tuple(x.shape)}, w {tuple(w.shape)})")
    (m, k), n = x.shape, w.shape[0]
    if not 1 <= m <= BUCKETS[-1] or k not in KS:
        raise ValueError(f"gemv: 1 <= M <= {BUCKETS[-1]} and K in {KS} (x {tuple(x.shape)}, w {tuple(w.shape)})")
    for name, t in (("x", x), ("w", w)):
        if not (t.is_cuda and t.dtype == torch.float16):
            raise RuntimeError(f"gemv: {name} must be a float16 GPU tensor")
        if not t.is_contiguous() or t.data_ptr() % 16:
            raise RuntimeError(f"gemv: {name} must be contiguous and 16-byte aligned")
    if w.device != x.device:
        raise RuntimeError("gemv: x and w must be on one GPU")
    if out is None:
        out = torch.empty((m, n), dtype=torch.float16, device=x.device)
    elif (tuple(out.shape) != (m, n) or out.dtype != torch.float16 or out.device != x.device
          or not out.is_contiguous() or out.data_ptr() % 16):
        raise RuntimeError(f"gemv: out must be a contiguous 16-byte aligned float16 [{m}, {n}] tensor on x's GPU")
    w4_hip.check(w4_hip.library().tw4_gemv_f16(x.data_ptr(), w.data_ptr(), out.data_ptr(), m, n, k, rows_inflight,
                                               rows_per_wave, w4_hip.raw_stream(x.get_device())))
    return out


def entry(x: torch.Tensor, w: torch.Tensor, table: dict[tuple[int, int, int], Config],
          eager: bool = True) -> Config | None:
    """The table's configuration for F.linear(x, w) if the kernel may run it, else None: a float16
    x of 1 .. 8 contiguous 16-byte aligned rows and a float16 w, and (``eager=False``) only while a
    HIP graph is being captured, which is how the decoder projections run in a decode step."""
    if x.dim() != 2 or not 1 <= x.shape[0] <= BUCKETS[-1]:
        return None
    if x.dtype != torch.float16 or w.dtype != torch.float16 or not x.is_contiguous() or x.data_ptr() % 16:
        return None
    if not eager and not torch.cuda.is_current_stream_capturing():
        return None
    return table.get((w.shape[0], w.shape[1], m_bucket(x.shape[0])))


def gemm(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """y [M, N] = x [M, K] @ w [N, K]^T by tw4_gemm_f16, 1 <= M <= 32, K a multiple of 64, contiguous 16-byte aligned
    float16 tensors on one GPU, on the current stream."""
    if x.dim() != 2 or w.dim() != 2 or x.shape[1] != w.shape[1]:
        raise ValueError(f"gemm: x [M, K] and w [N, K] expected (x {tuple(x.shape)}, w {tuple(w.shape)})")
    for name, t in (("x", x), ("w", w)):
        if not (t.is_cuda and t.dtype == torch.float16 and t.is_contiguous() and t.data_ptr() % 16 == 0):
            raise RuntimeError(f"gemm: {name} must be a contiguous 16-byte aligned float16 GPU tensor")
    if w.device != x.device:
        raise RuntimeError("gemm: x and w must be on one GPU")
    (m, k), n = x.shape, w.shape[0]
    out = torch.empty((m, n), dtype=torch.float16, device=x.device)
    with w4_hip.on_device(x.get_device()):
        w4_hip.check(w4_hip.library().tw4_gemm_f16(x.data_ptr(), w.data_ptr(), out.data_ptr(), m, n, k,
                                                   w4_hip.raw_stream(x.get_device())))
    return out


# Where tw4_gemm_f16 (and tw4_gemv_f16 up to M = 4) takes a product no table entry names: at most 32 rows, at least
# this many bytes of weights, and enough output columns. Against F.linear (hipBLASLt) on MI355X, us: 1.24 GB (4096 x
# 151936) 197 / 212 / 221 at M = 8 / 24 / 32 against 248 / 260 / 265, 0.78 GB (2560 wide) 120 / 136 / 148 against 244 / 166 / 168,
# 134 MB (4096 x 16384) 28.6-29.5 against 32; at 67 MB (4096 x 8192, 2048 x 16384) launch and first loads decide and hipBLASLt is
# ahead (22 against 15, 16.3 against 15.0), and at 48 rows x from L2 makes it level (250 against 252).
# Columns: the kernel deals 16-row tiles of w to two workgroups per CU and never splits K. Below about two passes of 64 rows
# per CU most of the GPU idles: 8192 x 8192 40 us against 30, 16384 x 4096 45 against 30, 5120 x 16384 1.00-1.11 of hipBLASLt's
# time at M = 16-32. Over 14 K from 1024 to 28672 x 11 N x 10 M: from N = 20480 on 0.30-1.03 of it, at N = 16384 up to
# K = 4160 0.62-0.92; the rows of x, read from L2 for every 64 of w, pass it at M > 24 and K = 12288 (49152 columns 1.05).
GEMM_MIN_BYTES = 128 << 20
GEMM_MAX_ROWS = 32
GEMM = ("gemm",)  # the choice of tw4_gemm_f16


def streams(m: int, n: int, k: int) -> bool:
    """Whether tw4_gemm_f16 is the faster kernel for m rows and n x k weights (see above), and takes the sizes."""
    return (1 <= m <= GEMM_MAX_ROWS and k % 64 == 0 and GEMM_MIN_BYTES <= 2 * n * k < 1 << 32
            and (n >= 20480 or (n >= 16384 and k <= 4160)) and (m <= 24 or k <= 8192))


def _streams(x: torch.Tensor, w: torch.Tensor) -> bool:
    """Whether F.linear(x, w) is a product bound by streaming w that tw4_gemm_f16 takes: sizes that ``streams``, plain
    contiguous aligned float16 GPU tensors that no gradient or transform follows."""
    if x.dim() != 2 or w.dim() != 2 or x.shape[1] != w.shape[1] or not streams(x.shape[0], *w.shape):
        return False
    if x.dtype != torch.float16 or w.dtype != torch.float16 or not x.is_cuda or w.device != x.device:
        return False
    if not (w4_hip.plain(x) and w4_hip.plain(w) and x.is_contiguous() and w.is_contiguous()):
        return False
    return x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0


def linear(x: torch.Tensor, w: torch.Tensor, table: dict[tuple[int, int, int], Config],
           eager: bool = True) -> torch.Tensor:
    """F.linear(x, w) (no bias) through tw4_gemv_f16 where ``entry`` finds a configuration, on a GPU with a table through
    tw4_gemm_f16 where streaming w bounds it (the logits head at every other batch up to 32 and every other size; up to
    M = 4, whose x the vector form keeps in LDS whole, tw4_gemv_f16 where it takes K: 184 us against 197 on the Qwen3-8B
    head at M = 1), through F.linear (hipBLASLt) otherwise (python/tandem/layers/triton_gemv.py:285-297)."""
    cfg = _choice(x, w, table, eager)
    if cfg is None:
        return F.linear(x, w)
    return gemm(x, w) if cfg == GEMM else gemv(x, w, *cfg)


def _choice(x: torch.Tensor, w: torch.Tensor, table: dict[tuple[int, int, int], Config], eager: bool) -> tuple | None:
    """What ``linear`` runs: a configuration of gemv, GEMM, or None for F.linear."""
    cfg = entry(x, w, table, eager)
    if cfg is not None:  # unless a gradient or a transform follows the call
        return cfg if w4_hip.plain(x) and w4_hip.plain(w) else None
    if not (eager and table and _streams(x, w)):
        return None
    # F.linear's own result where autocast, a mode or a compiler would change it; a shape the table names stays a kernel up to
    # its last bucket
    m, (n, k) = x.shape[0], w.shape
    if w4_hip.intercepted() and not (m <= BUCKETS[-1] and (n, k, 4) in table):
        return None
    if m > 4 or k not in KS:
        return GEMM
    # rows per wavefront: 32 for the long rows of K = 4096 (20480 columns 0.49 against 0.59 of F.linear's time at M = 1),
    # 16 for shorter ones and few columns, where they leave wavefronts short (1024 x 102400 at M = 4 1.06 against 0.92)
    return (2, 32) if k > 2048 and n >= 20480 else (2, 16)


def route(x: torch.Tensor, w: torch.Tensor, table: dict[tuple[int, int, int], Config], eager: bool = True) -> str:
    """The kernel ``linear`` runs for these tensors, by the same lookups."""
    cfg = _choice(x, w, table, eager)
    return "F.linear" if cfg is None else "tw4_gemm_f16" if cfg == GEMM else f"tw4_gemv_f16{cfg}"


class TabledLinear(nn.Linear):
    """An nn.Linear whose forward goes through ``linear`` with the table it carries, in graph
    capture only (eager calls, e.g. prefill, keep F.linear). ``install`` turns a model's bias-free
    projections into this class in place, so their names, parameters and state dicts stay those of
    nn.Linear."""

    gemv_table: dict

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        return linear(x, self.weight, self.gemv_table, eager=False)


def install(model: nn.Module, table: dict[tuple[int, int, int], Config]) -> int:
    """Route the bias-free decoder projections (PROJECTIONS) of ``model`` through the kernel by
    ``table``, and keep the table on the model for its logits head. Returns how many projections;
    an empty table changes nothing (python/tandem/layers/triton_gemv.py:304-315)."""
    if not table:
        return 0
    chosen = [mod for name, mod in model.named_modules()
              if isinstance(mod, nn.Linear) and mod.bias is None and name.rsplit(".", 1)[-1] in PROJECTIONS]
    for mod in chosen:
        mod.gemv_table = table
        mod.__class__ = TabledLinear
    model.gemv_table = table
    return len(chosen)


def default_table(model: nn.Module) -> dict[tuple[int, int, int], Config]:
    """DEFAULT_CONFIG for every (N, K, bucket) of ``model``'s projections whose K the kernel takes:
    a table that sends them all through it, for tests (python/tandem/layers/triton_gemv.py:418-428)."""
    shapes = {tuple(mod.weight.shape) for name, mod in model.named_modules()
              if isinstance(mod, nn.Linear) and name.rsplit(".", 1)[-1] in PROJECTIONS}
    return {(n, k, b): DEFAULT_CONFIG for n, k in shapes if k in KS for b in BUCKETS}
