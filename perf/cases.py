"""Performance cases: what a user of the encoder has it do, and over which ranges.

Every case is one call through a public entry point: a whole forward of
``UserOptimizedTransformer`` (``forward``), or one layer through the native
binding (``attention``, ``ffn``, ``qkv``, ``linear``, ``norm``).  Sizes are the
official matrix's, the encoder configurations' c2 to c5 and sizes between and
around them.  Inputs are made on the GPU from the seed alone; ``exact``
evaluates the same inputs in 64 bits with plain torch operations.
"""

from __future__ import annotations

import math
from typing import Dict, List, Optional

import torch
import torch.nn.functional as F

from tiktoktechjam2026track3_amd import native
from tiktoktechjam2026track3_amd.cases import TransformerConfig
from tiktoktechjam2026track3_amd.models import UserOptimizedTransformer

EPS = 1e-5
BF16 = torch.bfloat16
F64 = torch.float64
# The largest case: one sequence of 100000 tokens through 16 heads of 64.
MAX_FLOPS = 4.2e13
# Elements of fp64 temporaries that exact() keeps at once.
EXACT_BLOCK = 1 << 28


# --------------------------------------------------------------------------
# The cases
# --------------------------------------------------------------------------


def _forward(name: str, batch: int, seq: int, d: int, heads: int, ffn: int, layers: int, causal: bool,
             padding: float = 0.0) -> dict:
    return {"name": name, "kind": "forward", "batch": batch, "seq": seq, "d": d, "heads": heads, "ffn": ffn,
            "layers": layers, "causal": causal, "padding": padding}


def _attention(name: str, batch: int, seq: int, heads: int, hd: int, causal: bool, mask: str = "none",
               online: bool = False) -> dict:
    return {"name": name, "kind": "attention", "batch": batch, "seq": seq, "heads": heads, "hd": hd,
            "causal": causal, "mask": mask, "online": online}


def listed() -> List[dict]:
    return [
        # One short request through a narrow model (official case 2): a whole
        # call whose time is launches, host work and latency.
        _forward("forward_1x128_d128", 1, 128, 128, 4, 128, 4, True),
        # One short request through a six-layer model of ordinary width (c2).
        _forward("forward_1x128_d512", 1, 128, 512, 8, 2048, 6, False),
        # A batch of long prompts through a wide four-layer model (c3).
        _forward("forward_8x1024_d1024", 8, 1024, 1024, 16, 4096, 4, True),
        # Offline scoring of a very large batch with a narrow model: one block
        # at official case 6's sizes.
        _forward("block_10000x128_d128", 10000, 128, 128, 4, 128, 1, True),
        # Longer rows through a narrow block (official case 13).
        _forward("block_64x1024_d128", 64, 1024, 128, 4, 128, 1, True),
        # A wide block with few, wide heads on a padded batch of ragged length
        # (official case 8 is 64 x 128 with 256-wide heads).
        _forward("block_64x125_d1024_padded", 64, 125, 1024, 4, 1024, 1, True, 0.25),
        # Long padded prompts, causal (c4's attention).
        _attention("attention_4x8192_prefix", 4, 8192, 16, 64, True, "prefix"),
        # A whole book at once, every key visible (one of c5's sequences).
        _attention("attention_1x100000", 1, 100000, 16, 64, False),
        # The feed-forward half of c4's block on its padded batch.
        {"name": "ffn_32768_1024_4096_masked", "kind": "ffn", "rows": 32768, "d": 1024, "ffn": 4096, "masked": True},
        # The packed projection of a ragged mid-sized batch.
        {"name": "qkv_3x777_d1024", "kind": "qkv", "batch": 3, "seq": 777, "d": 1024, "heads": 16},
        # The attention output projection of one 1000-token request, residual
        # added, with the weight laid out once as the model lays it out.
        {"name": "linear_1000_1024_1024_residual", "kind": "linear", "rows": 1000, "n": 1024, "k": 1024,
         "epilogue": "residual", "packed": True},
        # LayerNorm of c3's batch.
        {"name": "norm_8192_1024", "kind": "norm", "rows": 8192, "d": 1024, "masked": False},
    ]


def _log_int(rng, low: int, high: int) -> int:
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _draw_once(rng) -> dict:
    kind = rng.choice(["narrow", "narrow", "narrow", "wide", "wide", "attention", "attention", "ffn", "qkv", "linear",
                       "norm"])
    causal = rng.random() < 0.6
    padding = rng.choice([0.0, 0.0, 0.25, 0.5])
    if kind == "narrow":  # the official matrix's models: d_model and ffn up to 128
        d = rng.choice([32, 64, 128, 128, 128])
        hd = rng.choice([h for h in (8, 32, 64, 128) if h <= d])
        seq = _log_int(rng, 16, 1024)
        batch = _log_int(rng, 1, max(1, min(10000, 1280000 // seq)))
        case = _forward("", batch, seq, d, d // hd, rng.choice([f for f in (32, 64, 128) if f >= d // 2]),
                        rng.choice([1, 2, 4]), causal, padding)
    elif kind == "wide":  # d_model 256 and up
        d = rng.choice([256, 512, 1024, 1024, 2048])
        seq = _log_int(rng, 24, 2048)
        batch = _log_int(rng, 1, max(1, min(256, 16384 // seq)))
        case = _forward("", batch, seq, d, d // rng.choice([64, 64, 128]), rng.choice([d, 2 * d, 4 * d]),
                        rng.choice([1, 2]), causal, padding)
    elif kind == "attention":
        hd = rng.choice([8, 32, 64, 64, 64, 128, 256])
        seq = _log_int(rng, 32, 16384)
        seq = seq if seq <= 2048 else seq // 4 * 4
        heads = rng.choice([2, 4, 8, 16])
        batch = _log_int(rng, 1, max(1, min(64, 65536 // seq)))
        mask = rng.choice(["none", "none", "prefix", "bytes"])
        case = _attention("", batch, seq, heads, hd, causal, mask, hd == 64 and rng.random() < 0.25)
    elif kind == "ffn":
        d = rng.choice([256, 512, 1024, 2048])
        case = {"kind": kind, "rows": _log_int(rng, 1, 32768), "d": d, "ffn": rng.choice([d, 2 * d, 4 * d]),
                "masked": padding > 0}
    elif kind == "qkv":
        d = rng.choice([256, 512, 1024, 2048])
        seq = _log_int(rng, 24, 2048)
        case = {"kind": kind, "batch": _log_int(rng, 1, max(1, 32768 // seq)), "seq": seq, "d": d,
                "heads": d // rng.choice([32, 64, 128])}
    elif kind == "linear":
        case = {"kind": kind, "rows": _log_int(rng, 1, 32768), "n": rng.choice([512, 1024, 2048, 4096]),
                "k": rng.choice([512, 1024, 2048]), "epilogue": rng.choice(["bias", "gelu", "residual"]),
                "packed": rng.random() < 0.5}
    else:
        case = {"kind": kind, "rows": _log_int(rng, 1, 262144), "d": rng.choice([32, 128, 256, 512, 1024, 2048]),
                "masked": padding > 0}
    case.pop("name", None)
    return case


def draw(rng) -> dict:
    while True:
        case = _draw_once(rng)
        if work(case)["flops"] <= MAX_FLOPS:
            return case


# --------------------------------------------------------------------------
# Inputs
# --------------------------------------------------------------------------


class _Random:
    """Values on the GPU from one seed, in the order they are asked for."""

    def __init__(self, seed: int) -> None:
        self.device = torch.device("cuda", torch.cuda.current_device())
        self.gen = torch.Generator(device=self.device)
        self.gen.manual_seed(seed)

    def normal(self, *shape: int, scale: float = 1.0) -> torch.Tensor:
        return torch.randn(*shape, generator=self.gen, device=self.device, dtype=BF16).mul_(scale)

    def weight(self, out_features: int, in_features: int) -> torch.Tensor:
        """nn.Linear's default range, +-1/sqrt(in_features)."""
        w = torch.rand(out_features, in_features, generator=self.gen, device=self.device)
        return ((2 * w - 1) / math.sqrt(in_features)).to(BF16)

    def bias(self, out_features: int, in_features: int) -> torch.Tensor:
        b = torch.rand(out_features, generator=self.gen, device=self.device)
        return ((2 * b - 1) / math.sqrt(in_features)).to(BF16)

    def gain(self, width: int) -> torch.Tensor:
        return (1 + 0.1 * torch.randn(width, generator=self.gen, device=self.device)).to(BF16)

    def lengths(self, batch: int, seq: int, padding: float) -> torch.Tensor:
        """Valid lengths, uniform over [seq * (1 - padding), seq]."""
        low = max(1, int(round(seq * (1.0 - padding))))
        return torch.randint(low, seq + 1, (batch,), generator=self.gen, device=self.device)

    def keep(self, *shape: int, share: float) -> torch.Tensor:
        return torch.rand(*shape, generator=self.gen, device=self.device) < share


def _prefix(lengths: torch.Tensor, seq: int) -> torch.Tensor:
    return torch.arange(seq, device=lengths.device)[None, :] < lengths[:, None]


def _forward_inputs(case: dict, seed: int) -> Dict[str, object]:
    r = _Random(seed)
    d, f = case["d"], case["ffn"]
    layers = []
    for _ in range(case["layers"]):
        layers.append({
            "norm1.weight": r.gain(d), "norm1.bias": r.normal(d, scale=0.05),
            "attention.qkv_proj.weight": r.weight(3 * d, d), "attention.qkv_proj.bias": r.bias(3 * d, d),
            "attention.out_proj.weight": r.weight(d, d), "attention.out_proj.bias": r.bias(d, d),
            "norm2.weight": r.gain(d), "norm2.bias": r.normal(d, scale=0.05),
            "ffn_in.weight": r.weight(f, d), "ffn_in.bias": r.bias(f, d),
            "ffn_out.weight": r.weight(d, f), "ffn_out.bias": r.bias(d, f),
        })
    final = {"final_norm.weight": r.gain(d), "final_norm.bias": r.normal(d, scale=0.05)}
    x = r.normal(case["batch"], case["seq"], d)
    if case["padding"] > 0:
        mask = _prefix(r.lengths(case["batch"], case["seq"], case["padding"]), case["seq"])
        x.masked_fill_(~mask[..., None], 0)
    else:
        mask = torch.ones(case["batch"], case["seq"], device=x.device, dtype=torch.bool)
    return {"layers": layers, "final": final, "x": x, "mask": mask}


def _attention_inputs(case: dict, seed: int) -> Dict[str, Optional[torch.Tensor]]:
    """Projections of a normalised activation: entries of about 1/sqrt(3)."""
    r = _Random(seed)
    b, h, s, hd = case["batch"], case["heads"], case["seq"], case["hd"]
    q, k, v = (r.normal(b, h, s, hd, scale=0.58) for _ in range(3))
    v_t = torch.zeros(b, h, hd, native.vt_stride(s), device=q.device, dtype=BF16)
    v_t[..., :s] = v.transpose(2, 3)
    kv_len = key_mask = None
    if case["mask"] == "prefix":
        kv_len = r.lengths(b, s, 0.5).to(torch.int32)
    elif case["mask"] == "bytes":
        key_mask = r.keep(b, s, share=0.9)
        key_mask[:, 0] = True  # no query without a key
    return {"q": q, "k": k, "v": v, "v_t": v_t, "kv_len": kv_len, "key_mask": key_mask}


def _layer_inputs(case: dict, seed: int) -> Dict[str, object]:
    r = _Random(seed)
    kind = case["kind"]
    if kind == "ffn":
        rows, d, f = case["rows"], case["d"], case["ffn"]
        return {"h": r.normal(rows, d), "w_in": r.weight(f, d), "b_in": r.bias(f, d), "w_out": r.weight(d, f),
                "b_out": r.bias(d, f), "residual": r.normal(rows, d),
                "mask": r.keep(rows, share=0.75) if case["masked"] else None}
    if kind == "qkv":
        d = case["d"]
        return {"x": r.normal(case["batch"], case["seq"], d), "w": r.weight(3 * d, d), "b": r.bias(3 * d, d)}
    if kind == "linear":
        rows, n, k = case["rows"], case["n"], case["k"]
        return {"a": r.normal(rows, k), "w": r.weight(n, k), "b": r.bias(n, k),
                "residual": r.normal(rows, n) if case["epilogue"] == "residual" else None}
    rows, d = case["rows"], case["d"]
    return {"x": r.normal(rows, d), "w": r.gain(d), "b": r.normal(d, scale=0.05),
            "mask": r.keep(rows, share=0.75) if case["masked"] else None}


# --------------------------------------------------------------------------
# The measured calls
# --------------------------------------------------------------------------


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    if kind == "forward":
        inputs = _forward_inputs(case, seed)
        config = TransformerConfig(case["batch"], case["seq"], case["d"], case["heads"], case["ffn"], case["layers"],
                                   case["causal"])
        x = inputs["x"]
        with torch.device(x.device):
            model = UserOptimizedTransformer(config).to(BF16).eval()
        values = {f"layers.{i}.{name}": v for i, layer in enumerate(inputs["layers"]) for name, v in layer.items()}
        model.load_state_dict({**values, **inputs["final"]}, strict=True)
        return {"kind": kind, "model": model, "x": x, "mask": inputs["mask"]}
    if kind == "attention":
        state = _attention_inputs(case, seed)
        del state["v"]
        state.update(kind=kind, scale=case["hd"] ** -0.5, causal=case["causal"], online=case["online"])
        return state
    state = _layer_inputs(case, seed)
    state["kind"] = kind
    if kind == "ffn":
        state["hidden"] = torch.empty(case["rows"], case["ffn"], device=state["h"].device, dtype=BF16)
    elif kind == "qkv":
        state["heads"] = case["heads"]
    elif kind == "linear":
        state["packed"] = native.prepack_weight(state["w"]) if case["packed"] else None
        state["epilogue"] = {"bias": native.ENC_EPI_BIAS, "gelu": native.ENC_EPI_BIAS_GELU,
                             "residual": native.ENC_EPI_BIAS_RESIDUAL_KEEP}[case["epilogue"]]
    return state


def run(state: dict):
    kind = state["kind"]
    if kind == "forward":
        with torch.inference_mode():
            return state["model"](state["x"], state["mask"])
    if kind == "attention":
        return native.attention(state["q"], state["k"], state["v_t"], state["scale"], state["causal"],
                                kv_len=state["kv_len"], key_mask=state["key_mask"], online=state["online"])
    if kind == "ffn":
        return native.ffn(state["h"], state["w_in"], state["b_in"], state["w_out"], state["b_out"],
                          state["residual"], row_mask=state["mask"], hidden=state["hidden"])
    if kind == "qkv":
        q, k, v_t = native.qkv_proj(state["x"], state["w"], state["b"], state["heads"])
        # (the columns past seq of V's rows are padding that no caller reads)
        return [q, k, v_t[..., : q.shape[2]]]
    if kind == "linear":
        return native.linear(state["a"], state["w"], state["b"], state["epilogue"], residual=state["residual"],
                             packed_weight=state["packed"])
    return native.layernorm(state["x"], state["w"], state["b"], EPS, row_mask=state["mask"])


# --------------------------------------------------------------------------
# What a call cannot do without
# --------------------------------------------------------------------------


def _live_scores(seq: int, causal: bool, mask: str, padding: float) -> float:
    """Mean query-key pairs of one head and sequence that take part."""
    low = 1.0 - padding if mask == "prefix" else 1.0
    mean_square = (1.0 + low + low * low) / 3.0  # of a length uniform over [low, 1]
    pairs = seq * seq * mean_square
    return (pairs + seq) / 2 if causal else pairs


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "forward":
        d, f, s, t = case["d"], case["ffn"], case["seq"], case["batch"] * case["seq"]
        scores = case["batch"] * _live_scores(s, case["causal"], "prefix", case["padding"])
        layer = 2.0 * t * (4 * d * d + 2 * d * f) + 4.0 * d * scores
        weights = case["layers"] * (4 * d * d + 2 * d * f + 9 * d + f) + 2 * d
        return {"bytes": 2.0 * (2 * t * d + weights) + t, "flops": case["layers"] * layer}
    if kind == "attention":
        b, h, s, hd = case["batch"], case["heads"], case["seq"], case["hd"]
        return {"bytes": 2.0 * 4 * b * h * s * hd + (b * s if case["mask"] == "bytes" else 0),
                "flops": 4.0 * hd * b * h * _live_scores(s, case["causal"], case["mask"], 0.5)}
    if kind == "ffn":
        rows, d, f = case["rows"], case["d"], case["ffn"]
        return {"bytes": 2.0 * (3 * rows * d + 2 * d * f + d + f), "flops": 4.0 * rows * d * f}
    if kind == "qkv":
        t, d = case["batch"] * case["seq"], case["d"]
        return {"bytes": 2.0 * (4 * t * d + 3 * d * d + 3 * d), "flops": 6.0 * t * d * d}
    if kind == "linear":
        m, n, k = case["rows"], case["n"], case["k"]
        residual = m * n if case["epilogue"] == "residual" else 0
        return {"bytes": 2.0 * (m * k + n * k + m * n + n + residual), "flops": 2.0 * m * n * k}
    return {"bytes": 4.0 * case["rows"] * case["d"] + 4.0 * case["d"], "flops": 0.0}


def tolerance(case: dict) -> dict:
    """About four times what the path measured against exact(): bf16 outputs of
    one layer are 1.6e-3 to 2.4e-3 off (the rounding of scores, weights and
    results to bf16), a block and its final norm 3e-3, four to six layers
    5e-3 to 6e-3."""
    if case["kind"] != "forward":
        return {"rel": 8e-3}
    return {"rel": 1.2e-2 if case["layers"] == 1 else 2e-2}


# --------------------------------------------------------------------------
# The same in 64 bits
# --------------------------------------------------------------------------


def _linear64(x: torch.Tensor, w: torch.Tensor, b: torch.Tensor) -> torch.Tensor:
    return torch.matmul(x, w.to(F64).t().contiguous()) + b.to(F64)


def _norm64(x: torch.Tensor, w: torch.Tensor, b: torch.Tensor) -> torch.Tensor:
    return F.layer_norm(x, (x.shape[-1],), w.to(F64), b.to(F64), EPS)


def _attention64(q, k, v, scale: float, causal: bool, keys_ok: Optional[torch.Tensor]) -> torch.Tensor:
    """[B, H, S, hd] in and out, fp64; keys_ok [B, S] or None."""
    s = q.shape[2]
    out = torch.empty_like(q)
    for b in range(q.shape[0]):
        heads = max(1, min(q.shape[1], EXACT_BLOCK // (s * s)))
        for h in range(0, q.shape[1], heads):
            k_t = k[b, h:h + heads].transpose(1, 2).contiguous()
            rows = max(1, min(s, EXACT_BLOCK // (s * heads)))
            for r in range(0, s, rows):
                scores = torch.matmul(q[b, h:h + heads, r:r + rows], k_t).mul_(scale)
                if causal:
                    at = torch.arange(r, r + scores.shape[1], device=q.device)
                    scores.masked_fill_(torch.arange(s, device=q.device)[None, :] > at[:, None], -math.inf)
                if keys_ok is not None:
                    scores.masked_fill_(~keys_ok[b], -math.inf)
                out[b, h:h + heads, r:r + rows] = torch.matmul(torch.softmax(scores, dim=-1), v[b, h:h + heads])
    return out


def _small_attention64(q, k, v, scale: float, causal: bool, keys_ok: Optional[torch.Tensor]) -> torch.Tensor:
    """The same with many sequences at once."""
    scores = torch.matmul(q, k.transpose(2, 3).contiguous()).mul_(scale)
    s = q.shape[2]
    if causal:
        scores.masked_fill_(torch.ones(s, s, device=q.device, dtype=torch.bool).triu_(1), -math.inf)
    if keys_ok is not None:
        scores.masked_fill_(~keys_ok[:, None, None, :], -math.inf)
    return torch.matmul(torch.softmax(scores, dim=-1), v)


def _forward64(case: dict, inputs: dict) -> torch.Tensor:
    b, s, d, h = case["batch"], case["seq"], case["d"], case["heads"]
    hd = d // h
    out = []
    step = max(1, min(b, EXACT_BLOCK // (h * s * s), EXACT_BLOCK // (s * max(3 * d, case["ffn"]))))
    for at in range(0, b, step):
        mask = inputs["mask"][at:at + step]
        x = inputs["x"][at:at + step].to(F64)
        pad = ~mask[..., None]
        for p in inputs["layers"]:
            y = _linear64(_norm64(x, p["norm1.weight"], p["norm1.bias"]), p["attention.qkv_proj.weight"],
                          p["attention.qkv_proj.bias"])
            q, k, v = (t.view(-1, s, h, hd).transpose(1, 2).contiguous() for t in y.split(d, dim=-1))
            core = _attention64 if s > 4096 else _small_attention64
            context = core(q, k, v, hd ** -0.5, case["causal"], mask).transpose(1, 2).reshape(-1, s, d)
            y = _linear64(context, p["attention.out_proj.weight"], p["attention.out_proj.bias"])
            x = x + y.masked_fill_(pad, 0)
            y = F.gelu(_linear64(_norm64(x, p["norm2.weight"], p["norm2.bias"]), p["ffn_in.weight"], p["ffn_in.bias"]))
            x = (x + _linear64(y, p["ffn_out.weight"], p["ffn_out.bias"])).masked_fill_(pad, 0)
        final = inputs["final"]
        out.append(_norm64(x, final["final_norm.weight"], final["final_norm.bias"]).masked_fill_(pad, 0))
    return torch.cat(out)


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "forward":
        return _forward64(case, _forward_inputs(case, seed))
    if kind == "attention":
        i = _attention_inputs(case, seed)
        b, s, h, hd = case["batch"], case["seq"], case["heads"], case["hd"]
        keys_ok = i["key_mask"] if i["kv_len"] is None else _prefix(i["kv_len"], s)
        out = _attention64(i["q"].to(F64), i["k"].to(F64), i["v"].to(F64), hd ** -0.5, case["causal"], keys_ok)
        out = out.transpose(1, 2).reshape(b, s, h * hd)
        if i["kv_len"] is not None:  # rows past a sequence's length are padding, written as zeros
            out.masked_fill_(~keys_ok[..., None], 0)
        return out
    i = _layer_inputs(case, seed)
    if kind == "ffn":
        hidden = F.gelu(_linear64(i["h"].to(F64), i["w_in"], i["b_in"]))
        out = i["residual"].to(F64) + _linear64(hidden, i["w_out"], i["b_out"])
        return out if i["mask"] is None else out.masked_fill_(~i["mask"][:, None], 0)
    if kind == "qkv":
        b, s, d, h = case["batch"], case["seq"], case["d"], case["heads"]
        q, k, v = (t.view(b, s, h, d // h).transpose(1, 2).contiguous()
                   for t in _linear64(i["x"].to(F64), i["w"], i["b"]).split(d, dim=-1))
        return [q, k, v.transpose(2, 3).contiguous()]
    if kind == "linear":
        y = _linear64(i["a"].to(F64), i["w"], i["b"])
        if case["epilogue"] == "gelu":
            return F.gelu(y)
        return y if i["residual"] is None else i["residual"].to(F64) + y
    out = _norm64(i["x"].to(F64), i["w"], i["b"])
    return out if i["mask"] is None else out.masked_fill_(~i["mask"][:, None], 0)
