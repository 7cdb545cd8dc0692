"""The framework's work, as cases to be timed: the two mixers, the key step, chunked and token-by-token decoding, the column.

A case is a dict of plain values with a ``kind``:

- ``scan``: the delta-rule scan (``delta_scan_fused`` / ``delta_scan_fused_fp32``), forward, or forward
  and backward under autograd (``train``);
- ``attn``: window attention over a cache's ``m`` rows and ``n`` new ones (``window_attention``), forward or
  forward and backward;
- ``attend``: a chunk's attention over the carried window and the pushed window (``attend``);
- ``keys``: the causal key filter and normalization (``fused_keys``), forward and backward;
- ``decode``: one token per row through a column's passes (``CapturedDecoder.step``);
- ``column``: the looped column with per-token halting over a whole chunk (``LoopedColumn.forward``).

``exact`` restates each in float64 from the definitions, in plain torch.
"""

from __future__ import annotations

import math
import random
import sys
from pathlib import Path
from typing import Any

import torch
from torch import Tensor

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "vesper-preview_amd"))

from vesper.attention import KVCache, attend  # noqa: E402
from vesper.decode import WARM_STEPS, CapturedDecoder  # noqa: E402
from vesper.kernels.delta_scan import delta_scan_fused, delta_scan_fused_fp32  # noqa: E402
from vesper.kernels.keys import fused_keys  # noqa: E402
from vesper.kernels.window_attn import window_attention  # noqa: E402
from vesper.loop import LoopedColumn  # noqa: E402

Case = dict[str, Any]
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "fp32": torch.float32}
WINDOW = 512  # the window of every configuration
TAPS = 4  # the key filter's width in every configuration
P_HALT = 0.3
BASE = 10000.0


def listed() -> list[Case]:
    return [
        # the smallest call: the first training stage's scan, 88 tokens, two heads of 16, in float32
        {"name": "scan_fp32_train_b32_n88_h2_d16", "kind": "scan", "dtype": "fp32", "train": True, "b": 32, "n": 88,
         "h": 2, "dk": 16},
        # training in float32 on chunks of a ragged length (the default scan of a training run)
        {"name": "scan_fp32_train_b8_n1000_h8_d64", "kind": "scan", "dtype": "fp32", "train": True, "b": 8, "n": 1000,
         "h": 8, "dk": 64},
        # training in bf16: a batch of 1024-token chunks at twelve heads of 64
        {"name": "scan_bf16_train_b16_n1024_h12_d64", "kind": "scan", "dtype": "bf16", "train": True, "b": 16,
         "n": 1024, "h": 12, "dk": 64},
        # prefill of a batch of prompts: the headline shape
        {"name": "scan_bf16_prefill_b8_n4096_h8_d64", "kind": "scan", "dtype": "bf16", "train": False, "b": 8,
         "n": 4096, "h": 8, "dk": 64},
        # prefill of one long document of an odd length: few heads, many chunks
        {"name": "scan_bf16_prefill_b1_n8191_h12_d64", "kind": "scan", "dtype": "bf16", "train": False, "b": 1,
         "n": 8191, "h": 12, "dk": 64},
        # prefill of a batch of prompts: the headline shape
        {"name": "attn_bf16_prefill_b8_n4096_h8_d64", "kind": "attn", "dtype": "bf16", "train": False, "b": 8,
         "n": 4096, "m": 0, "h": 8, "hkv": 8, "dk": 64},
        # training on a chunk after a full cached window, four query heads a key head
        {"name": "attn_bf16_train_b16_n1024_m512_h8_kv2_d64", "kind": "attn", "dtype": "bf16", "train": True, "b": 16,
         "n": 1024, "m": 512, "h": 8, "hkv": 2, "dk": 64},
        # streaming a text in chunks of a ragged length over the carried window, in float16
        {"name": "attend_f16_b4_n777_m512_h12_kv4_d64", "kind": "attend", "dtype": "f16", "b": 4, "n": 777, "m": 512,
         "h": 12, "hkv": 4, "dk": 64},
        # the key step of a training pass
        {"name": "keys_bf16_train_b16_n1024_h12_d64", "kind": "keys", "dtype": "bf16", "b": 16, "n": 1024, "h": 12,
         "dk": 64},
        # serving: one token for each of 64 streams, and for a single one
        {"name": "decode_b64_h8_d64_p8", "kind": "decode", "b": 64, "h": 8, "hkv": 8, "dk": 64, "passes": 8},
        {"name": "decode_b1_h8_d64_p8", "kind": "decode", "b": 1, "h": 8, "hkv": 8, "dk": 64, "passes": 8},
        # the whole column over a batch of prompts, tokens halting one by one
        {"name": "column_b4_n2048_h8_d64_p8", "kind": "column", "b": 4, "n": 2048, "h": 8, "hkv": 8, "dk": 64,
         "passes": 8},
    ]


def _spread(rng: random.Random, lo: int, hi: int) -> int:
    """A whole number of ``lo..hi``, even over its logarithm."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


# the most elements (b * n * h * dk) that a drawn case of a kind holds, from the listed ones
_MOST = {("scan", "bf16", False): 1 << 24, ("scan", "bf16", True): 12 << 20, ("scan", "fp32", False): 4 << 20,
         ("scan", "fp32", True): 4 << 20, ("attn", "bf16", False): 1 << 24, ("attn", "f16", False): 1 << 24,
         ("attn", "bf16", True): 8 << 20, ("attn", "f16", True): 8 << 20}


def draw(rng: random.Random) -> Case:
    kind = rng.choices(["scan", "attn", "attend", "keys", "decode", "column"], [8, 5, 2, 2, 2, 1])[0]
    if kind == "scan":
        dtype, train = rng.choice(["bf16", "fp32"]), rng.random() < 0.5
        while True:
            c = {"kind": kind, "dtype": dtype, "train": train, "b": _spread(rng, 1, 32),
                 "n": _spread(rng, 64, 2048 if dtype == "fp32" else 8192), "h": _spread(rng, 2, 12),
                 "dk": rng.choice([16, 64] if rng.random() < 0.8 else [32])}
            if (1 << 16) <= c["b"] * c["n"] * c["h"] * c["dk"] <= _MOST[kind, dtype, train]:
                return c
    if kind == "attn":
        dtype, train = rng.choice(["bf16", "bf16", "f16"]), rng.random() < 0.5
        while True:
            hkv = rng.choice([2, 4, 8])
            c = {"kind": kind, "dtype": dtype, "train": train, "b": _spread(rng, 1, 16), "n": _spread(rng, 64, 8192),
                 "m": rng.choice([0, WINDOW, rng.randint(1, WINDOW)]), "h": hkv * rng.choice([1, 2, 4] if hkv < 8 else [1]),
                 "hkv": hkv, "dk": 64}
            if (1 << 18) <= c["b"] * c["n"] * c["h"] * c["dk"] <= _MOST[kind, dtype, train]:
                return c
    if kind == "attend":
        hkv = rng.choice([2, 4])
        return {"kind": kind, "dtype": rng.choice(["bf16", "f16"]), "b": _spread(rng, 1, 8), "n": _spread(rng, 64, 2048),
                "m": rng.choice([WINDOW, rng.randint(1, WINDOW)]), "h": hkv * rng.choice([1, 3, 4]), "hkv": hkv, "dk": 64}
    if kind == "keys":
        return {"kind": kind, "dtype": rng.choice(["bf16", "bf16", "fp32"]), "b": _spread(rng, 1, 16),
                "n": _spread(rng, 64, 1024), "h": rng.choice([2, 8, 12]), "dk": rng.choice([16, 64])}
    if kind == "decode":
        return {"kind": kind, "b": _spread(rng, 1, 64), "h": 8, "hkv": rng.choice([2, 8]), "dk": 64,
                "passes": rng.randint(1, 8)}
    return {"kind": kind, "b": _spread(rng, 1, 4), "n": _spread(rng, 128, 2048), "h": 8, "hkv": rng.choice([2, 8]),
            "dk": 64, "passes": rng.randint(2, 8)}


# ---- inputs -----------------------------------------------------------------------------------


def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g: torch.Generator, *shape: int) -> Tensor:
    return torch.randn(*shape, generator=g, device="cuda")


def _unit(x: Tensor) -> Tensor:
    return x / x.norm(dim=-1, keepdim=True).clamp_min(1e-6)


def _scan_inputs(c: Case, seed: int) -> dict[str, Tensor]:
    """Normalized queries and keys, N(0, 1) values, write strengths in (0, 1), a small carried state."""
    g, t, shape = _gen(seed), DTYPES[c["dtype"]], (c["b"], c["n"], c["h"], c["dk"])
    x = {"q": _unit(_randn(g, *shape)).to(t), "k": _unit(_randn(g, *shape)).to(t), "v": _randn(g, *shape).to(t),
         "beta": torch.sigmoid(_randn(g, *shape[:3])).to(t), "state": 0.02 * _randn(g, c["b"], c["h"], c["dk"], c["dk"])}
    if c["train"]:
        x |= {"go": _randn(g, *shape).to(t), "gs": 0.1 * _randn(g, c["b"], c["h"], c["dk"], c["dk"])}
    return x


def _attn_inputs(c: Case, seed: int) -> dict[str, Tensor]:
    g, t = _gen(seed), DTYPES[c["dtype"]]
    x = {"q": _randn(g, c["b"], c["n"], c["h"], c["dk"]).to(t)}
    x |= {name: _randn(g, c["b"], c["m"] + c["n"], c["hkv"], c["dk"]).to(t) for name in ("keys", "values")}
    if c.get("train"):
        x["go"] = _randn(g, c["b"], c["n"], c["h"], c["dk"]).to(t)
    return x


def _keys_inputs(c: Case, seed: int) -> dict[str, Tensor]:
    g, t, d = _gen(seed), DTYPES[c["dtype"]], c["h"] * c["dk"]
    return {"z": _randn(g, c["b"], c["n"], d).to(t), "history": _randn(g, c["b"], TAPS - 1, d),
            "taps": _randn(g, TAPS, d) / math.sqrt(TAPS), "go": _randn(g, c["b"], c["n"], c["h"], c["dk"]).to(t)}


def _column_weights(c: Case, g: torch.Generator) -> tuple[dict[str, list[Tensor]], list[Tensor]]:
    """Projections ~ N(0, 1/d) in bf16 and filter taps ~ U(-1/sqrt(K), 1/sqrt(K)) of every pass."""
    d, kv = c["h"] * c["dk"], c["hkv"] * c["dk"]
    outs = {"wq": d, "wk": d, "wv": d, "wb": c["h"], "waq": d, "wak": kv, "wav": kv}
    weights = {name: [(_randn(g, d, out) / math.sqrt(d)).bfloat16() for _ in range(c["passes"])] for name, out in outs.items()}
    bound = 1 / math.sqrt(TAPS)
    return weights, [(torch.rand(TAPS, d, generator=g, device="cuda") * 2 - 1) * bound for _ in range(c["passes"])]


def _decode_inputs(c: Case, seed: int) -> dict[str, Any]:
    """A column's weights, a hidden state a row and each pass's carried state with its window full."""
    g, b, d = _gen(seed), c["b"], c["h"] * c["dk"]
    weights, taps = _column_weights(c, g)
    flat: list[Tensor] = []
    for _ in range(c["passes"]):
        ring = [_randn(g, b, WINDOW, c["hkv"], c["dk"]).bfloat16() for _ in range(2)]
        flat += [0.02 * _randn(g, b, c["h"], c["dk"], c["dk"]), _randn(g, b, TAPS - 1, d), *ring,
                 torch.arange(WINDOW, device="cuda").expand(b, WINDOW).contiguous(),
                 torch.ones(b, WINDOW, dtype=torch.bool, device="cuda")]
    return {"weights": weights, "taps": taps, "x": _randn(g, b, 1, d),
            "pos": torch.full((b, 1), WINDOW, device="cuda"), "flat": flat}


def _column_inputs(c: Case, seed: int) -> dict[str, Any]:
    g, b, n, d = _gen(seed), c["b"], c["n"], c["h"] * c["dk"]
    weights, taps = _column_weights(c, g)
    return {"weights": weights, "taps": taps, "x": _randn(g, b, n, d),
            "states": [0.02 * _randn(g, b, c["h"], c["dk"], c["dk"]) for _ in range(c["passes"])],
            "histories": [_randn(g, b, TAPS - 1, d) for _ in range(c["passes"])],
            "exits": [torch.rand(b, n, generator=g, device="cuda") < P_HALT for _ in range(c["passes"])]}


def prepare(case: Case, seed: int) -> dict[str, Any]:
    c = case
    if c["kind"] == "scan":
        x = _scan_inputs(c, seed)
        if c["train"]:
            for name in ("q", "k", "v", "beta", "state"):
                x[name].requires_grad_()
        return {"case": c, **x}
    if c["kind"] == "attn":
        x = _attn_inputs(c, seed)
        if c["train"]:
            for name in ("q", "keys", "values"):
                x[name].requires_grad_()
        return {"case": c, **x}
    if c["kind"] == "attend":
        x, b, n, m = _attn_inputs(c, seed), c["b"], c["n"], c["m"]
        pos = torch.arange(m + n, device="cuda").expand(b, m + n)
        cache = KVCache(x["keys"][:, :m].contiguous(), x["values"][:, :m].contiguous(), pos[:, :m].contiguous(), WINDOW)
        return {"case": c, "q": x["q"], "k": x["keys"][:, m:].contiguous(), "v": x["values"][:, m:].contiguous(),
                "pos": pos[:, m:].contiguous(), "cache": cache}
    if c["kind"] == "keys":
        x = _keys_inputs(c, seed)
        for name in ("z", "history", "taps"):
            x[name].requires_grad_()
        return {"case": c, **x}
    if c["kind"] == "decode":
        x = _decode_inputs(c, seed)
        column = LoopedColumn(x["weights"], c["h"], c["hkv"], c["dk"], WINDOW, x["taps"], rotary_base=BASE)
        decoder = CapturedDecoder(column, c["passes"])
        flat = decoder.start(c["b"])
        for t in range(WARM_STEPS + 1):  # the eager steps, then the capture
            _, flat = decoder.step(x["x"], torch.full_like(x["pos"], t), flat)
        for mine, given in zip(flat, x["flat"]):  # a conversation that has filled its windows
            mine.copy_(given)
        return {"case": c, "decoder": decoder, "x": x["x"], "pos": x["pos"], "flat": flat}
    x = _column_inputs(c, seed)
    column = LoopedColumn(x["weights"], c["h"], c["hkv"], c["dk"], WINDOW, x["taps"], rotary_base=BASE)
    return {"case": c, "column": column, **{name: x[name] for name in ("x", "states", "histories", "exits")}}


def run(state: dict[str, Any]) -> Any:
    c, s = state["case"], state
    if c["kind"] == "scan":
        scan = delta_scan_fused if c["dtype"] == "bf16" else delta_scan_fused_fp32
        inputs = (s["q"], s["k"], s["v"], s["beta"], s["state"])
        if not c["train"]:
            return scan(*inputs)
        o, final = scan(*inputs)
        return [o.detach(), final.detach(), *torch.autograd.grad((o, final), inputs, (s["go"], s["gs"]))]
    if c["kind"] == "attn":
        inputs = (s["q"], s["keys"], s["values"])
        o = window_attention(*inputs, WINDOW)
        return [o.detach(), *torch.autograd.grad(o, inputs, s["go"])] if c["train"] else o
    if c["kind"] == "attend":
        o, cache = attend(s["q"], s["k"], s["v"], s["pos"], s["cache"])
        return [o, cache.k, cache.v, cache.pos]
    if c["kind"] == "keys":
        inputs = (s["z"], s["history"], s["taps"])
        k = fused_keys(*inputs, c["h"])
        return [k.detach(), *torch.autograd.grad(k, inputs, s["go"])]
    if c["kind"] == "decode":
        y, s["flat"] = s["decoder"].step(s["x"], s["pos"], s["flat"])
        s["pos"].add_(1)
        return [y, *s["flat"]]
    r = s["column"].forward(s["x"], s["states"], s["exits"], s["histories"])
    return [r.y, r.n_iters, *r.states, *(r.histories or ())]


# ---- what a pass cannot do without ------------------------------------------------------------


def _scan_flops(c: Case) -> float:
    """A token's write (what the key reads, the update) and its query's read: 6 dk^2 a head."""
    return 6.0 * c["b"] * c["n"] * c["h"] * c["dk"] ** 2


def _attn_flops(c: Case) -> float:
    m = c.get("m", 0)
    pairs = sum(min(m + i + 1, WINDOW) for i in range(c["n"]))
    return 4.0 * c["b"] * c["h"] * c["dk"] * pairs


def work(case: Case) -> dict[str, float]:
    c = case
    b, h, dk = c["b"], c["h"], c["dk"]
    d = h * dk
    if c["kind"] == "scan":
        size, rows = (2 if c["dtype"] == "bf16" else 4), b * c["n"] * d
        beta, st = b * c["n"] * h, 4 * b * h * dk * dk
        if c["train"]:  # q, k, v, go read, o, dq, dk, dv written; beta and its gradient; four states
            return {"bytes": size * (8 * rows + 2 * beta) + 4 * st, "flops": 3 * _scan_flops(c)}
        return {"bytes": size * (4 * rows + beta) + 2 * st, "flops": _scan_flops(c)}
    if c["kind"] in ("attn", "attend"):
        q, kv = b * c["n"] * d, b * (c["m"] + c["n"]) * c["hkv"] * dk
        if c["kind"] == "attend":
            kept = b * min(c["m"] + c["n"], WINDOW) * (2 * c["hkv"] * dk * 2 + 8)
            return {"bytes": 2 * (2 * q + 2 * kv) + 8 * b * (c["m"] + c["n"]) + kept, "flops": _attn_flops(c)}
        if c["train"]:  # q, go read and o, dq written; keys, values and their gradients
            return {"bytes": 2 * (4 * q + 4 * kv), "flops": 3.5 * _attn_flops(c)}
        return {"bytes": 2 * (2 * q + 2 * kv), "flops": _attn_flops(c)}
    if c["kind"] == "keys":  # z, the keys' gradient read, the keys and dz written
        size = 2 if c["dtype"] == "bf16" else 4
        return {"bytes": size * 4 * b * c["n"] * d + 8 * TAPS * d + 8 * b * (TAPS - 1) * d,
                "flops": 6.0 * TAPS * b * c["n"] * d}
    kv = c["hkv"] * dk
    columns = 3 * d + h + d + 2 * kv  # projected columns of a pass
    if c["kind"] == "decode":
        one = (2 * d * columns + 8 * b * h * dk * dk + 8 * b * (TAPS - 1) * d + 4 * TAPS * d
               + b * (WINDOW * (2 * kv * 2 + 9) + 2 * kv * 2))
        flops = 2.0 * b * d * columns + 6.0 * b * h * dk * dk + 4.0 * b * d * WINDOW
        return {"bytes": c["passes"] * one + 8 * b * d, "flops": c["passes"] * flops}
    tokens = b * c["n"]
    one = 2 * d * columns + 8 * b * h * dk * dk + 8 * b * (TAPS - 1) * d + 4 * TAPS * d + tokens
    flops = 2.0 * tokens * d * columns + _scan_flops(c) + _attn_flops(c)
    return {"bytes": c["passes"] * one + 8 * tokens * d + 4 * tokens, "flops": c["passes"] * flops}


# four times the largest error of an output against float64 over the listed and several drawn cases
# (float32 scan 5.3e-7 at most, and three times that again for other orders of the sums over longer texts)
_REL = {("scan", "fp32"): 6e-6, ("scan", "bf16"): 2e-2, ("attn", "bf16"): 1e-2, ("attn", "f16"): 1.2e-3,
        ("attend", "bf16"): 1e-2, ("attend", "f16"): 1.2e-3, ("keys", "bf16"): 7e-3, ("keys", "fp32"): 2e-6,
        ("decode", None): 2.7e-2, ("column", None): 3e-2}


def tolerance(case: Case) -> Any:
    return {"rel": _REL[case["kind"], case.get("dtype")]}


# ---- the same, in float64 ---------------------------------------------------------------------


def _scan64(q: Tensor, k: Tensor, v: Tensor, beta: Tensor, state: Tensor) -> tuple[Tensor, Tensor]:
    """The delta rule ``S += beta k (v - S^T k)^T``, ``o = S^T q``, over blocks of 64 tokens: a block's
    writes solve ``(I + tril(diag(beta) K K^T, -1)) D = diag(beta) (V - K S)``."""
    b, n, h, dk = q.shape
    block = 64
    pad = -n % block

    def blocks(x: Tensor) -> Tensor:
        x = torch.nn.functional.pad(x, (0, 0, 0, 0, 0, pad)).transpose(1, 2)
        return x.reshape(b, h, -1, block, x.shape[-1])

    q, k, v, beta = blocks(q), blocks(k), blocks(v), blocks(beta[..., None])
    low = torch.tril(beta * (k @ k.transpose(-1, -2).contiguous()), -1)
    inverse = torch.linalg.solve_triangular(low, torch.diag_embed(beta[..., 0]), upper=False, unitriangular=True)
    w, u = inverse @ k, inverse @ v
    seen = torch.tril(q @ k.transpose(-1, -2).contiguous())
    kt, outs = k.transpose(-1, -2).contiguous(), []
    for i in range(q.shape[2]):
        delta = u[:, :, i] - w[:, :, i] @ state
        outs.append(q[:, :, i] @ state + seen[:, :, i] @ delta)
        state = state + kt[:, :, i] @ delta
    return torch.stack(outs, 2).reshape(b, h, -1, dk)[:, :, :n].transpose(1, 2), state


def _attn64(q: Tensor, keys: Tensor, values: Tensor) -> Tensor:
    """Softmax of each query over the last ``WINDOW`` keys up to its own, in blocks of queries."""
    b, n, h, dk = q.shape
    m, group = keys.shape[1] - n, h // keys.shape[2]
    q = q.transpose(1, 2)
    k, v = (x.transpose(1, 2).repeat_interleave(group, dim=1) for x in (keys, values))
    outs = []
    for s in range(0, n, WINDOW):
        e = min(n, s + WINDOW)
        first = max(0, m + s - WINDOW + 1)
        i = torch.arange(m + s, m + e, device=q.device)[:, None]
        j = torch.arange(first, m + e, device=q.device)[None]
        score = q[:, :, s:e] @ k[:, :, first:m + e].transpose(-1, -2).contiguous() / math.sqrt(dk)
        score = score.masked_fill((j > i) | (j <= i - WINDOW), -math.inf)
        outs.append(torch.softmax(score, -1) @ v[:, :, first:m + e])
    return torch.cat(outs, 2).transpose(1, 2)


def _keys64(z: Tensor, history: Tensor, taps: Tensor, h: int) -> Tensor:
    n, width = z.shape[1], taps.shape[0]
    x = torch.cat([history, z], 1)
    u = sum(taps[r] * x[:, width - 1 - r:width - 1 - r + n] for r in range(width))
    u = u.unflatten(-1, (h, -1))
    return u / u.norm(dim=-1, keepdim=True).clamp_min(1e-6)


def _norm64(x: Tensor) -> Tensor:
    return x / (x.square().mean(-1, keepdim=True) + 1e-6).sqrt()


def _rotary64(x: Tensor, pos: Tensor) -> Tensor:
    dk = x.shape[-1]
    angle = pos.double()[..., None, None] * BASE ** (-torch.arange(0, dk, 2, device=x.device, dtype=torch.float64) / dk)
    a, b, cos, sin = x[..., 0::2], x[..., 1::2], angle.cos(), angle.sin()
    return torch.stack([a * cos - b * sin, a * sin + b * cos], -1).flatten(-2)


def _double(x: Any) -> Any:
    if isinstance(x, Tensor):
        return x.double() if x.is_floating_point() else x
    if isinstance(x, dict):
        return {name: _double(v) for name, v in x.items()}
    return [_double(v) for v in x]


def _grads64(outs: Tensor | tuple[Tensor, ...], inputs: list[Tensor], grads: Tensor | tuple[Tensor, ...]) -> list[Tensor]:
    return list(torch.autograd.grad(outs, inputs, grads))


def _decode64(c: Case, seed: int) -> list[Tensor]:
    s = _double(_decode_inputs(c, seed))
    b, h, hkv, dk = c["b"], c["h"], c["hkv"], c["dk"]
    x, flat, out = s["x"], s["flat"], []
    w = {name: v for name, v in s["weights"].items()}
    for t in range(c["passes"]):
        state, history, rk, rv, rpos, rvalid = flat[6 * t:6 * t + 6]
        xn = _norm64(x)
        z = xn @ w["wk"][t]
        k = _keys64(z, history, s["taps"][t], h)
        o, state = _scan64((xn @ w["wq"][t]).view(b, 1, h, dk), k, (xn @ w["wv"][t]).view(b, 1, h, dk),
                           torch.sigmoid(xn @ w["wb"][t]), state)
        x = x + o.reshape(b, 1, -1)
        xn = _norm64(x)
        aq = _rotary64((xn @ w["waq"][t]).view(b, 1, h, dk), s["pos"])
        ak = _rotary64((xn @ w["wak"][t]).view(b, 1, hkv, dk), s["pos"])
        av = (xn @ w["wav"][t]).view(b, 1, hkv, dk)
        # position WINDOW takes slot 0, whose entry has just left the window
        rk, rv, rpos = torch.cat([ak, rk[:, 1:]], 1), torch.cat([av, rv[:, 1:]], 1), torch.cat([s["pos"], rpos[:, 1:]], 1)
        order = torch.cat([torch.arange(1, WINDOW, device=x.device), torch.zeros(1, dtype=torch.long, device=x.device)])
        x = x + _attn64(aq, rk[:, order], rv[:, order]).reshape(b, 1, -1)
        out += [state, torch.cat([history, z], 1)[:, 1:], rk, rv, rpos, rvalid]
    return [x, *out]


def _column64(c: Case, seed: int) -> list[Tensor]:
    s = _double(_column_inputs(c, seed))
    b, n, h, hkv, dk = c["b"], c["n"], c["h"], c["hkv"], c["dk"]
    x, w = s["x"], s["weights"]
    active = torch.ones(b, n, dtype=torch.bool, device=x.device)
    iters = torch.zeros(b, n, dtype=torch.int32, device=x.device)
    pos = torch.arange(n, device=x.device).expand(b, n)
    held: list[Tensor] | None = None  # what halted tokens go on writing: z, k, v, beta, attention k and v
    states, histories = [], []

    def fresh(a: Tensor, i: int) -> Tensor:
        return a if held is None else torch.where(active.reshape(b, n, *[1] * (a.dim() - 2)), a, held[i])

    for t in range(c["passes"]):
        xn = _norm64(x)
        z = fresh(xn @ w["wk"][t], 0)
        k = fresh(_keys64(z, s["histories"][t], s["taps"][t], h), 1)
        v = fresh((xn @ w["wv"][t]).view(b, n, h, dk), 2)
        beta = fresh(torch.sigmoid(xn @ w["wb"][t]), 3)
        o, state = _scan64((xn @ w["wq"][t]).view(b, n, h, dk), k, v, beta, s["states"][t])
        x1 = x + o.reshape(b, n, -1)
        xn = _norm64(x1)
        aq = _rotary64((xn @ w["waq"][t]).view(b, n, h, dk), pos)
        ak = fresh(_rotary64((xn @ w["wak"][t]).view(b, n, hkv, dk), pos), 4)
        av = fresh((xn @ w["wav"][t]).view(b, n, hkv, dk), 5)
        x1 = x1 + _attn64(aq, ak, av).reshape(b, n, -1)
        states.append(state)
        histories.append(torch.cat([s["histories"][t], z], 1)[:, n:])
        x = torch.where(active[..., None], x1, x)
        iters += active.int()
        # a token that is still active has written what it computed, and would freeze that; a halted one is held already
        held = [z, k, v, beta, ak, av]
        active = active & ~s["exits"][t]
    return [x, iters, *states, *histories]


def exact(case: Case, seed: int) -> Any:
    c = case
    if c["kind"] == "scan":
        x = _double(_scan_inputs(c, seed))
        inputs = [x[name] for name in ("q", "k", "v", "beta", "state")]
        if not c["train"]:
            return _scan64(*inputs)
        inputs = [i.requires_grad_() for i in inputs]
        o, final = _scan64(*inputs)
        return [o.detach(), final.detach(), *_grads64((o, final), inputs, (x["go"], x["gs"]))]
    if c["kind"] in ("attn", "attend"):
        x = _double(_attn_inputs(c, seed))
        inputs = [x[name] for name in ("q", "keys", "values")]
        if c["kind"] == "attend":
            first = max(0, c["m"] + c["n"] - WINDOW)
            pos = torch.arange(first, c["m"] + c["n"], device="cuda").expand(c["b"], -1)
            return [_attn64(*inputs), inputs[1][:, first:], inputs[2][:, first:], pos]
        if not c["train"]:
            return _attn64(*inputs)
        inputs = [i.requires_grad_() for i in inputs]
        o = _attn64(*inputs)
        return [o.detach(), *_grads64(o, inputs, x["go"])]
    if c["kind"] == "keys":
        x = _double(_keys_inputs(c, seed))
        inputs = [x[name].requires_grad_() for name in ("z", "history", "taps")]
        k = _keys64(*inputs, c["h"])
        return [k.detach(), *_grads64(k, inputs, x["go"])]
    return _decode64(c, seed) if c["kind"] == "decode" else _column64(c, seed)
