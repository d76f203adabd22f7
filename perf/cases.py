"""Performance cases of the W4A16 path: what a user of this package has it do, through its public entry points.

    listed()          the cases, smallest to largest kinds of use
    draw(rng)         one more case of the same ranges
    prepare(case, s)  what a program holds before the call (weights repacked, graphs captured, inputs), from the seed
    run(state)        one pass
    work(case)        bytes and operations the pass cannot do without
    tolerance(case)   largest error another correct implementation at the same precision shows
    exact(case, s)    the same outputs in 64 bits by plain torch, from the checkpoint's tensors

Kinds of case:
    step     a whole decode step (embedding, all layers, logits) replayed by DecodeGraphRunner
    layers   a few decoder layers of a model replayed by DecodeGraphRunner (hidden states): a pipeline stage
    prefill  a few decoder layers run eagerly on the tokens of a prompt chunk
    mlp      one GatedMLP (SwiGLU gate_up + down), eager
    linear   one W4Linear, eager
    head     the fp16 logits head (gemv16.linear with the device's table)
    repack   load time: AutoAWQ tensors -> tile layout (repack_awq)
    dequant  the dense fp16 weight of a repacked layer (w4_dequant), for programs that need it whole

Model sizes are those of the kernel tables: Qwen3-0.6B / 1.7B / 4B / 8B / 14B and Llama-3-8B projections.
Weights: uniform 4-bit q, zero points 4..11, scales that give weights of a trained layer's size (standard
deviation about 1 / sqrt(K)); activations N(0, 1) as a norm leaves them; embeddings N(0, 1).
"""

from __future__ import annotations

import math

import torch

from tandem_amd import decode_graph
from tandem_amd import model as tmodel
from tandem_amd.layers import awq, gemv16
from tandem_amd.loader import QuantConfig

QUANT = QuantConfig("awq", 4, 128)
VOCAB = 151936
# name: hidden, intermediate, query heads, KV heads, layers (head_dim 128)
MODELS = {
    "qwen3-1.7b": (2048, 6144, 16, 8, 28),
    "qwen3-4b": (2560, 9728, 32, 8, 36),
    "qwen3-8b": (4096, 12288, 32, 8, 36),
    "qwen3-14b": (5120, 17408, 40, 8, 40),
    "llama-3-8b": (4096, 14336, 32, 8, 32),
}
TIED = ("qwen3-1.7b", "qwen3-4b")
EPS = 1e-6
NIBBLE = (0, 4, 1, 5, 2, 6, 3, 7)  # nibble of an AutoAWQ word that holds feature j


def listed() -> list[dict]:
    return [
        # the smallest call: one projection of the smallest model for one token, launched eagerly
        {"name": "linear_0.6b_qkv_m1", "kind": "linear", "k": 1024, "n": 4096, "m": 1, "silu": False},
        # interactive decode of the 8B model, one sequence: the whole step
        {"name": "step_8b_b1", "kind": "step", "model": "qwen3-8b", "layers": 36, "batch": 1},
        # a small model serving a few sequences (tied embeddings)
        {"name": "step_1.7b_b5", "kind": "step", "model": "qwen3-1.7b", "layers": 28, "batch": 5},
        # decode layers at the small serving batch
        {"name": "layers_8b_b8", "kind": "layers", "model": "qwen3-8b", "layers": 4, "batch": 8},
        # a larger model at a full serving batch
        {"name": "layers_14b_b40", "kind": "layers", "model": "qwen3-14b", "layers": 3, "batch": 40},
        # a short prompt of an odd length
        {"name": "prefill_llama_m77", "kind": "prefill", "model": "llama-3-8b", "layers": 2, "m": 77},
        # a usual prompt chunk
        {"name": "prefill_8b_m512", "kind": "prefill", "model": "qwen3-8b", "layers": 2, "m": 512},
        # a long prompt chunk through the MLP of the largest model
        {"name": "mlp_14b_m2048", "kind": "mlp", "model": "qwen3-14b", "m": 2048},
        # the largest single projection, a packed batch of prompts
        {"name": "linear_8b_gate_up_m4096", "kind": "linear", "k": 4096, "n": 24576, "m": 4096, "silu": False},
        # logits of a serving batch
        {"name": "head_8b_m24", "kind": "head", "k": 4096, "n": VOCAB, "m": 24},
        # loading: the largest projection of the 8B model, rows interleaved for SwiGLU
        {"name": "repack_8b_gate_up", "kind": "repack", "k": 4096, "n": 24576, "interleave": True},
        # the dense weight of a projection
        {"name": "dequant_8b_down", "kind": "dequant", "k": 12288, "n": 4096},
    ]


def _log(rng, lo: float, hi: float) -> float:
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng) -> dict:
    kind = rng.choice(("linear", "linear", "linear", "mlp", "mlp", "prefill", "prefill", "layers", "layers", "step", "head",
                       "repack", "dequant"))
    if kind == "step":
        name = rng.choice(("qwen3-1.7b", "qwen3-8b"))
        return {"kind": kind, "model": name, "layers": MODELS[name][4], "batch": round(_log(rng, 1, 32))}
    name = rng.choice(tuple(MODELS))
    if kind == "layers":
        return {"kind": kind, "model": name, "layers": rng.randint(2, 4), "batch": round(_log(rng, 1, 64))}
    if kind == "prefill":
        return {"kind": kind, "model": name, "layers": rng.randint(1, 2), "m": round(_log(rng, 17, 2048))}
    if kind == "mlp":
        return {"kind": kind, "model": name, "m": round(_log(rng, 1, 2048))}
    if kind == "head":
        return {"kind": kind, "k": rng.choice((1024, 2048, 4096)), "n": rng.randint(32000, VOCAB), "m": round(_log(rng, 1, 64))}
    k, n = 128 * round(_log(rng, 8, 136)), 8 * round(_log(rng, 128, 4352))
    if kind == "repack":
        return {"kind": kind, "k": k, "n": n, "interleave": n % 16 == 0 and rng.random() < 0.5}
    if kind == "dequant":
        return {"kind": kind, "k": k, "n": n}
    m = round(_log(rng, 1, 4096))
    while m * k * n > 4096 * 4096 * 24576:
        m = max(1, m // 2)
    return {"kind": "linear", "k": k, "n": n, "m": m, "silu": n % 16 == 0 and rng.random() < 0.3}


# ---------------------------------------------------------------------------------------- inputs
def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(seed)


def _raw(k: int, n: int, g: torch.Generator) -> tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """AutoAWQ tensors of a K x N projection: qweight [K, N/8], qzeros [K/128, N/8], scales [K/128, N]."""
    qweight = torch.randint(-2**31, 2**31, (k, n // 8), device="cuda", dtype=torch.int32, generator=g)
    z = torch.randint(4, 12, (k // 128, n // 8, 8), device="cuda", dtype=torch.int32, generator=g)
    qzeros = torch.zeros((k // 128, n // 8), device="cuda", dtype=torch.int32)
    for i in range(8):
        qzeros |= z[:, :, i] << (4 * i)
    s = 0.22 / math.sqrt(k)
    scales = (s * (0.5 + torch.rand((k // 128, n), device="cuda", generator=g))).half()
    return qweight, qzeros, scales


def _randn(g: torch.Generator, *shape: int) -> torch.Tensor:
    return torch.randn(shape, device="cuda", dtype=torch.float16, generator=g)


def _linear(k: int, n: int, raw, silu: bool) -> awq.W4Linear:
    with torch.device("cuda"):
        layer = awq.W4Linear(k, n, 128)
    _fill(layer, raw)
    if silu:
        layer.enable_silu_mul()
    layer.finalize(torch.cuda.get_device_name())
    return layer


def _fill(layer, raw) -> None:
    for name, t in zip(("qweight", "qzeros", "scales"), raw):
        getattr(layer, name).copy_(t)


def _shapes(hidden: int, inter: int, heads: int, kv: int) -> tuple[tuple[str, int, int], ...]:
    return (("qkv", hidden, 128 * (heads + 2 * kv)), ("o", 128 * heads, hidden), ("gate_up", hidden, 2 * inter),
            ("down", inter, hidden))


def _model_raw(name: str, layers: int, head: bool, seed: int):
    """Every tensor of a cut model from the seed, in one order: layer by layer, then the final norm,
    embedding and (untied, when asked for) head."""
    hidden, inter, heads, kv, _ = MODELS[name]
    g = _gen(seed)
    for _ in range(layers):
        for proj, k, n in _shapes(hidden, inter, heads, kv):
            yield proj, _raw(k, n, g)
        for norm in ("n1", "n2"):
            yield norm, (1.0 + 0.2 * (torch.rand(hidden, device="cuda", generator=g) - 0.5)).half()
    yield "norm", (1.0 + 0.2 * (torch.rand(hidden, device="cuda", generator=g) - 0.5)).half()
    yield "embed", _randn(g, VOCAB, hidden)
    if head and name not in TIED:
        yield "head", _randn(g, VOCAB, hidden) * 0.02


def _ids(seed: int, m: int) -> torch.Tensor:
    return torch.randint(0, VOCAB, (m,), device="cuda", generator=_gen(seed + 7919))


@torch.no_grad()
def _model(name: str, layers: int, head: bool, seed: int) -> tmodel.DecoderModel:
    hidden, inter, heads, kv, _ = MODELS[name]
    cfg = tmodel.DecoderConfig(hidden, inter, heads, kv, 128, layers, VOCAB, EPS,
                               tie_word_embeddings=not head or name in TIED)
    default = torch.get_default_dtype()
    torch.set_default_dtype(torch.float16)
    try:
        with torch.device("cuda"):
            m = tmodel.DecoderModel(cfg, QUANT)
    finally:
        torch.set_default_dtype(default)
    i = -1
    for what, t in _model_raw(name, layers, head, seed):
        i += what == "qkv"
        layer = m.model.layers[i]
        if what in ("qkv", "o", "gate_up", "down"):
            lin = {"qkv": layer.self_attn.qkv_proj, "o": layer.self_attn.o_proj, "gate_up": layer.mlp.gate_up_proj,
                   "down": layer.mlp.down_proj}[what]
            _fill(lin, t)
        else:
            {"n1": layer.input_layernorm.weight, "n2": layer.post_attention_layernorm.weight, "norm": m.model.norm.weight,
             "embed": m.model.embed_tokens.weight, "head": m.lm_head.weight if m.lm_head is not None else None}[what].copy_(t)
    return tmodel.prepare(m, torch.device("cuda", torch.cuda.current_device()), torch.cuda.get_device_name())


@torch.no_grad()
def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    if kind in ("step", "layers"):
        m = _model(case["model"], case["layers"], kind == "step", seed)
        runner = decode_graph.DecodeGraphRunner(m, case["batch"], torch.device("cuda", torch.cuda.current_device()),
                                                logits=kind == "step")
        return {"kind": kind, "runner": runner, "ids": _ids(seed, case["batch"]).tolist()}
    if kind == "prefill":
        return {"kind": kind, "model": _model(case["model"], case["layers"], False, seed), "ids": _ids(seed, case["m"])}
    g = _gen(seed)
    if kind == "mlp":
        hidden, inter, heads, kv, _ = MODELS[case["model"]]
        with torch.device("cuda"):
            mlp = tmodel.GatedMLP(hidden, inter, QUANT)
        _fill(mlp.gate_up_proj, _raw(hidden, 2 * inter, g))
        _fill(mlp.down_proj, _raw(inter, hidden, g))
        for lin in (mlp.gate_up_proj, mlp.down_proj):
            lin.finalize(torch.cuda.get_device_name())
        return {"kind": kind, "mlp": mlp, "x": _randn(g, case["m"], hidden)}
    if kind == "head":
        w = _randn(g, case["n"], case["k"]) * 0.02
        table = gemv16.table_for(torch.device("cuda", torch.cuda.current_device()), torch.nn.Module())
        return {"kind": kind, "w": w, "table": table, "x": _randn(g, case["m"], case["k"])}
    raw = _raw(case["k"], case["n"], g)
    if kind == "linear":
        return {"kind": kind, "lin": _linear(case["k"], case["n"], raw, case["silu"]), "x": _randn(g, case["m"], case["k"])}
    if kind == "repack":
        return {"kind": kind, "raw": raw, "interleave": case["interleave"]}
    return {"kind": kind, "packed": awq.repack_awq(*raw, 128)}


@torch.no_grad()
def run(state: dict):
    kind = state["kind"]
    if kind in ("step", "layers"):
        return state["runner"].run(state["ids"])
    if kind == "prefill":
        return state["model"](state["ids"])
    if kind == "mlp":
        return state["mlp"](state["x"])
    if kind == "linear":
        return state["lin"](state["x"])
    if kind == "head":
        return gemv16.linear(state["x"], state["w"], state["table"])
    if kind == "repack":
        return awq.repack_awq(*state["raw"], 128, interleave=state["interleave"])
    return awq.w4_dequant(*state["packed"])


# ------------------------------------------------------------------------------ work, tolerance
def _w4_bytes(k: int, n: int) -> float:
    return n * k / 2 + n * k / 128 * 2.5  # 4-bit weights, a 2-byte scale and a 4-bit zero per group


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind in ("step", "layers", "prefill"):
        hidden, inter, heads, kv, _ = MODELS[case["model"]]
        m = case["m"] if kind == "prefill" else case["batch"]
        nbytes = sum(_w4_bytes(k, n) for _, k, n in _shapes(hidden, inter, heads, kv)) * case["layers"]
        flops = sum(2.0 * m * k * n for _, k, n in _shapes(hidden, inter, heads, kv)) * case["layers"]
        nbytes += 2 * m * hidden + 2 * hidden * (2 * case["layers"] + 1)  # embedding rows, norm weights
        if kind == "step":
            nbytes += 2 * VOCAB * hidden + 2 * m * VOCAB
            flops += 2.0 * m * VOCAB * hidden
        else:
            nbytes += 2 * m * hidden
        return {"bytes": nbytes, "flops": flops}
    if kind == "mlp":
        hidden, inter = MODELS[case["model"]][:2]
        m = case["m"]
        return {"bytes": _w4_bytes(hidden, 2 * inter) + _w4_bytes(inter, hidden) + 4 * m * hidden, "flops": 6.0 * m * hidden * inter}
    k, n = case["k"], case["n"]
    if kind == "head":
        return {"bytes": 2 * k * n + 2 * case["m"] * (k + n), "flops": 2.0 * case["m"] * k * n}
    if kind == "linear":
        m = case["m"]
        return {"bytes": _w4_bytes(k, n) + 2 * m * k + (m * n if case["silu"] else 2 * m * n), "flops": 2.0 * m * k * n}
    if kind == "repack":  # checkpoint tensors in; packed words, fp16 scales and fp16 zeros out
        return {"bytes": _w4_bytes(k, n) + (n + 15) // 16 * 16 * k / 2 + n * k / 128 * 4, "flops": 0}
    return {"bytes": n * k / 2 + n * k / 128 * 4 + 2 * n * k, "flops": 0}


def tolerance(case: dict):
    kind = case["kind"]
    # about four times the relative error against 64 bits that fp16 weights, activations and results with
    # 32-bit sums show: 2-3e-4 for one projection, 4-6e-4 behind SwiGLU or over two projections, 0.8-1e-3 over
    # two to four decoder layers, 2.4e-3 over a whole model
    if kind in ("repack", "dequant"):
        return "exact"
    if kind == "step":
        return {"rel": 1e-2}
    if kind in ("layers", "prefill"):
        return {"rel": 4e-3}
    if kind == "mlp" or kind == "linear" and case["silu"]:
        return {"rel": 2.4e-3}
    return {"rel": 1e-3}


# -------------------------------------------------------------------------------- 64-bit results
def _dense64(raw) -> torch.Tensor:
    """[K, N] float64 weights (q - z) s of AutoAWQ tensors."""
    qweight, qzeros, scales = raw
    shifts = torch.tensor([4 * i for i in NIBBLE], device="cuda", dtype=torch.int32)
    k, n = qweight.shape[0], 8 * qweight.shape[1]
    w = ((qweight[:, :, None] >> shifts) & 15).reshape(k, n).double()
    z = ((qzeros[:, :, None] >> shifts) & 15).reshape(k // 128, n).double()
    w = w.view(k // 128, 128, n)
    w -= z[:, None]
    w *= scales.double()[:, None]
    return w.view(k, n)


def _silu_mul64(y: torch.Tensor) -> torch.Tensor:
    gate, up = y.chunk(2, dim=-1)
    return gate * torch.sigmoid(gate) * up


def _norm64(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _head64(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    return torch.cat([x @ w[i:i + 16384].double().t() for i in range(0, w.shape[0], 16384)], dim=1)


def _model64(case: dict, seed: int, m: int, head: bool) -> torch.Tensor:
    hidden, inter, heads, kv, _ = MODELS[case["model"]]
    # the embedding comes last in the tensors' order: go over them twice rather than hold them all
    for what, t in _model_raw(case["model"], case["layers"], head, seed):
        if what == "embed":
            h = t[_ids(seed, m)].double()
    residual, lin = torch.zeros_like(h), {}
    for what, t in _model_raw(case["model"], case["layers"], head, seed):
        if what in ("qkv", "o", "gate_up", "down"):
            lin[what] = t
        elif what == "n1":
            n1 = t
        elif what == "n2":
            residual = residual + h
            qkv = _norm64(residual, n1) @ _dense64(lin["qkv"])
            v = qkv[:, 128 * (heads + kv):].view(m, kv, 1, 128).expand(m, kv, heads // kv, 128).reshape(m, 128 * heads)
            residual = residual + v @ _dense64(lin["o"])
            h = _silu_mul64(_norm64(residual, t) @ _dense64(lin["gate_up"])) @ _dense64(lin["down"])
        elif what == "norm":
            h = _norm64(residual + h, t)
        elif what == ("embed" if case["model"] in TIED else "head") and head:
            return _head64(h, t)
    return h


@torch.no_grad()
def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind in ("step", "layers"):
        return _model64(case, seed, case["batch"], kind == "step")
    if kind == "prefill":
        return _model64(case, seed, case["m"], False)
    g = _gen(seed)
    if kind == "mlp":
        hidden, inter = MODELS[case["model"]][:2]
        up, down = _raw(hidden, 2 * inter, g), _raw(inter, hidden, g)
        return _silu_mul64(_randn(g, case["m"], hidden).double() @ _dense64(up)) @ _dense64(down)
    if kind == "head":
        w = _randn(g, case["n"], case["k"]) * 0.02
        return _head64(_randn(g, case["m"], case["k"]).double(), w)
    raw = _raw(case["k"], case["n"], g)
    if kind == "linear":
        y = _randn(g, case["m"], case["k"]).double() @ _dense64(raw)
        return _silu_mul64(y) if case["silu"] else y
    if kind == "dequant":
        return _dense64(raw).t()
    return None
