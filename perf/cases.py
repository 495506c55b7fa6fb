"""The calls whose time matters to a program that serves the 26B-A4B text stack
with this package, as cases that can be prepared, run and checked one by one.

A case is a dict of plain values; its "kind" picks the entry point:

  decode        one sampled step of Engine.decode_fn (a step of generate())
  prefill       Engine.prefill_fn on one prompt
  attn_prefill  ops.prefill_attention of one layer's prompt rows
  attn_decode   ops.decode_attention of one layer for B sequences
  moe_decode    ops.moe_block of two layers for a few tokens
  moe_prefill   ops.moe_router_topk + ops.moe_prefill of one layer
  products      every dense product of a sliding and a full layer, as the
                batched prefill and the batched decode call them
  sample        ops.sample on one logits row

The layer widths are those of gemma4_26b_a4b_config; the two whole-model kinds
keep its first six layers (five sliding, one full), which hold every kernel
that the thirty layers run.  Sizes that a program varies (prompt lengths,
positions, rows, sequences) are the case's own.  Inputs come from the seed
alone.  `exact` restates each case in float64 torch.
"""

from __future__ import annotations

import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "kaggle-tpu-inference_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from gemma4_mi import _lib, model, ops  # noqa: E402
from gemma4_mi.config import FULL, SLIDING, gemma4_26b_a4b_config  # noqa: E402
from gemma4_mi.engine import Engine  # noqa: E402

DEV = "cuda:0"
BF16 = torch.bfloat16
LAYERS = 6           # of the whole-model kinds: layers 0-4 sliding, layer 5 full
MAX_LEN = 32768      # the cache length the decode workload is served with
PAGE = model.PAGE_SIZE


def _cfg(layers: int = LAYERS):
    full = gemma4_26b_a4b_config()
    return full.replace(num_hidden_layers=layers, layer_types=full.layer_types[:layers])


CFG = _cfg()
H, NH, E, TOPK = CFG.hidden_size, CFG.num_attention_heads, CFG.num_experts, CFG.top_k_experts
F, I = CFG.moe_intermediate_size, CFG.intermediate_size
EPS = CFG.rms_norm_eps


# ------------------------------------------------------------------------ cases
def listed() -> list[dict]:
    return [
        # the step that a chat session repeats for every token: a short
        # context, generate()'s default temperature and top_p
        {"name": "decode_700", "kind": "decode", "pos": 700, "temperature": 1.0, "top_p": 0.95},
        # time to first token of a long prompt (not a multiple of any tile)
        {"name": "prefill_2000", "kind": "prefill", "n": 2000},
        # a full-attention layer of a long document's prompt
        {"name": "attn_prefill_full_4096", "kind": "attn_prefill", "layer": FULL, "t": 4096, "p0": 0,
         "softcap": 0.0},
        # a sliding layer of an ordinary long prompt
        {"name": "attn_prefill_sliding_2000", "kind": "attn_prefill", "layer": SLIDING, "t": 2000, "p0": 0,
         "softcap": 0.0},
        # one sequence at the end of the 32K cache (softcap as in the
        # attention workload of the benchmark)
        {"name": "attn_decode_full_32k", "kind": "attn_decode", "layer": FULL, "b": 1, "max_len": MAX_LEN,
         "shortest": 32767, "softcap": 50.0},
        # eight served sequences of different lengths up to 8K
        {"name": "attn_decode_full_b8", "kind": "attn_decode", "layer": FULL, "b": 8, "max_len": 8704,
         "shortest": 2000, "softcap": 0.0},
        # the MoE blocks of a decode step of sixteen sequences
        {"name": "moe_decode_16", "kind": "moe_decode", "n": 16},
        # the experts of an ordinary chat prompt: about 19 rows per expert
        {"name": "moe_prefill_300", "kind": "moe_prefill", "n": 300},
        # the experts of a long document
        {"name": "moe_prefill_4096", "kind": "moe_prefill", "n": 4096},
        # projections and dense MLPs of a decode step of eight sequences
        {"name": "products_8", "kind": "products", "n": 8},
        # the same of a long prompt
        {"name": "products_2000", "kind": "products", "n": 2000},
        # the sampler on its own: every stochastic step ends with it
        {"name": "sample_262144", "kind": "sample", "vocab": 262144, "top_k": 64, "temperature": 1.0, "top_p": 0.95},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng) -> dict:
    kind = rng.choice(["decode", "prefill", "attn_prefill", "attn_decode", "moe_decode", "moe_prefill", "products",
                       "sample"])
    if kind == "decode":
        return {"kind": kind, "pos": _log_int(rng, 16, MAX_LEN - 2), "temperature": rng.choice([0.0, 0.7, 1.0]),
                "top_p": rng.choice([0.9, 0.95, 1.0])}
    if kind == "prefill":
        return {"kind": kind, "n": _log_int(rng, 2, 2000)}
    if kind == "attn_prefill":
        layer = rng.choice([FULL, SLIDING])
        t = _log_int(rng, 17, 4096)
        # a prompt from its start, or the rows after a cached prefix
        p0 = rng.choice([0, 0, rng.randint(1, 4096)])
        p0 = min(p0, 4096 - t) if layer == FULL else p0
        return {"kind": kind, "layer": layer, "t": t, "p0": p0, "softcap": rng.choice([0.0, 0.0, 50.0])}
    if kind == "attn_decode":
        b = rng.choice([1, 1, 2, 3, 4, 6, 8, 12, 16])
        longest = _log_int(rng, 64, MAX_LEN if b == 1 else 65536 // max(b, 8))
        return {"kind": kind, "layer": rng.choice([FULL, SLIDING]), "b": b, "max_len": longest,
                "shortest": rng.randint(1, longest), "softcap": rng.choice([0.0, 0.0, 50.0])}
    if kind == "moe_decode":
        return {"kind": kind, "n": _log_int(rng, 1, 32)}
    if kind == "moe_prefill":
        return {"kind": kind, "n": _log_int(rng, 17, 4096)}
    if kind == "products":
        return {"kind": kind, "n": _log_int(rng, 1, 2000)}
    return {"kind": "sample", "vocab": _log_int(rng, 4096, 262144), "top_k": rng.randint(1, 64),
            "temperature": rng.choice([0.0, 0.5, 1.0, 1.3]), "top_p": rng.choice([0.5, 0.9, 0.95, 1.0])}


# ----------------------------------------------------------------------- inputs
class _Rand:
    """Device tensors from one seed, in the order they are asked for."""

    def __init__(self, seed: int):
        self.g = torch.Generator(device=DEV).manual_seed(int(seed) * 7919 + 17)

    def normal(self, *shape, std=1.0, mean=0.0, dtype=BF16):
        t = torch.empty(shape, dtype=dtype, device=DEV)
        return t.normal_(mean, std, generator=self.g)

    def ints(self, hi, *shape):
        return torch.randint(0, hi, shape, device=DEV, dtype=torch.int32, generator=self.g)

    def perm(self, n):
        return torch.randperm(n, device=DEV, generator=self.g).to(torch.int32)


def _std(name: str) -> tuple[float, float]:
    """(mean, std) of a parameter: unit norms with some spread, query/key norms
    that keep the scores of a 256- or 512-wide head within a few units, a
    router whose logits spread over a few units, block outputs that add to the
    residual without drowning it, N(0, 0.02) matrices."""
    if name.endswith("layer_scalar"):
        return 1.0, 0.0
    if name.endswith(("q_norm", "k_norm")):
        return 0.3, 0.02
    if name.endswith(("post_attention_layernorm", "post_feedforward_layernorm")):
        return 0.3, 0.03
    if name.endswith(("layernorm", "layernorm_1", "layernorm_2", "router.scale", "router.per_expert_scale")) \
            or name == "norm":
        return 1.0, 0.1
    if name.endswith("router.proj"):
        return 0.0, 2.0
    return 0.0, 0.02


def _params(r: _Rand) -> dict:
    out = {}
    for name, shape in model.param_shapes(CFG).items():
        mean, std = _std(name)
        out[name] = r.normal(*shape, std=std, mean=mean)
    return out


def _geometry(layer: str) -> tuple[int, int, int]:
    """(KV heads, head_dim, window) of a layer type."""
    return CFG.kv_heads_for(layer), CFG.head_dim_for(layer), CFG.sliding_window if layer == SLIDING else 0


def _lengths(case) -> list[int]:
    """Positions of the B sequences: evenly from the shortest to the longest."""
    b, lo, hi = case["b"], case["shortest"] - 1, case["max_len"] - 1
    return [hi - (hi - lo) * i // max(b - 1, 1) for i in range(b)]


def _model_inputs(case, seed):
    r = _Rand(seed)
    p = _params(r)
    n = case["n"] if case["kind"] == "prefill" else 1
    return r, p, r.ints(CFG.vocab_size, n)


def _attn_prefill_inputs(case, seed):
    r = _Rand(seed)
    kv, d, _ = _geometry(case["layer"])
    pages = (case["p0"] + case["t"] + PAGE - 1) // PAGE
    # normed and rotated rows: q as after q_norm_rope, the cache as after kv_append
    return (r.normal(case["t"], NH, d, std=0.3), r.normal(pages, kv, PAGE, d, std=0.3),
            r.normal(pages, kv, PAGE, d), r.perm(pages))


def _attn_decode_inputs(case, seed):
    r = _Rand(seed)
    kv, d, _ = _geometry(case["layer"])
    b, mp = case["b"], (case["max_len"] + PAGE - 1) // PAGE
    q, k = r.normal(b, NH, d), r.normal(b, kv, d)
    v = r.normal(b, kv, d) if case["layer"] == SLIDING else None
    qn, kn = r.normal(d, mean=0.3, std=0.02), r.normal(d, mean=0.3, std=0.02)
    kp, vp = r.normal(b * mp, kv, PAGE, d, std=0.3), r.normal(b * mp, kv, PAGE, d)
    pt = r.perm(b * mp).reshape(b, mp).contiguous()
    pos = torch.tensor(_lengths(case), dtype=torch.int32, device=DEV)
    return q, k, v, qn, kn, kp, vp, pt, pos


def _moe_inputs(case, seed):
    r = _Rand(seed)
    layers = []
    for _ in range(2 if case["kind"] == "moe_decode" else 1):
        layers.append({"x": r.normal(case["n"], H), "scale": r.normal(H, mean=1.0, std=0.1),
                       "proj": r.normal(E, H, std=2.0), "pes": r.normal(E, mean=1.0, std=0.1),
                       "gate_up": r.normal(E, 2, F, H, std=0.02), "down": r.normal(E, H, F, std=0.02)})
    return layers


def _products_inputs(case, seed):
    r = _Rand(seed)
    n, layers = case["n"], []
    for layer in (SLIDING, FULL):
        kv, d, _ = _geometry(layer)
        w = [r.normal(NH * d, H, std=0.02), r.normal(kv * d, H, std=0.02)]
        if layer == SLIDING:
            w.append(r.normal(kv * d, H, std=0.02))
        layers.append({"xn": r.normal(n, H), "qkv": w, "ctx": r.normal(n, NH * d, std=0.5),
                       "o": r.normal(H, NH * d, std=0.02), "xm": r.normal(n, H),
                       "gate_up": r.normal(2 * I, H, std=0.02), "down": r.normal(H, I, std=0.02)})
    return layers


def _sample_inputs(case, seed):
    r = _Rand(seed)
    v = case["vocab"]
    logits = 30.0 * torch.tanh(r.normal(v, std=3.0, dtype=torch.float32) / 30.0)
    # the few tokens a language model holds likely
    logits[r.ints(v, 24).long()] += r.normal(24, mean=9.0, std=2.0, dtype=torch.float32)
    return logits


# ---------------------------------------------------------------------- prepare
def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, seed)


def _engine(p, max_len):
    eng = Engine(None, max_len, 1, 64, cfg=CFG, params=p, device=DEV)
    eng.compile_all(256)  # what a server does once, before its first request
    return eng


def _prepare_decode(case, seed):
    r, p, tok = _model_inputs(case, seed)
    eng = _engine(p, MAX_LEN)
    pos = case["pos"]
    pages = (pos + PAGE - 1) // PAGE
    for kp, vp in zip(eng.cache["k"], eng.cache["v"]):  # the earlier positions of the session
        kp[:pages].normal_(0.0, 0.3, generator=r.g)
        vp[:pages].normal_(0.0, 1.0, generator=r.g)
    row = lambda t: t[pos // PAGE, :, pos % PAGE]  # noqa: E731
    return {"eng": eng, "step": eng.decode_fn(), "tok": tok.reshape(1, 1), "pos": pos, "seed": int(seed),
            "t": case["temperature"], "p": case["top_p"],
            "out": {"logits": eng._runner.logits, "k": [row(t) for t in eng.cache["k"]],
                    "v": [row(t) for t in eng.cache["v"]]}}


def _prepare_prefill(case, seed):
    _, p, tok = _model_inputs(case, seed)
    n = case["n"]
    eng = _engine(p, 2048)
    bucket = max(256, (n + 255) // 256 * 256)
    pages = (n + PAGE - 1) // PAGE
    return {"eng": eng, "fn": eng.prefill_fn(bucket), "tok": tok.cpu().reshape(1, n), "n": n,
            "out": {"logits": eng._runner.logits, "k": eng.cache["k"][-1][:pages], "v": eng.cache["v"][-1][:pages]}}


def _prepare_attn_prefill(case, seed):
    q, kp, vp, pt = _attn_prefill_inputs(case, seed)
    return {"q": q, "k": kp, "v": vp, "pt": pt, "ctx": torch.empty_like(q), "p0": case["p0"],
            "window": _geometry(case["layer"])[2], "cap": case["softcap"] or None}


def _rope(layer, n):
    partial = CFG.rope_partial_rotary_factor_full if layer == FULL else 1.0
    theta = CFG.rope_theta_full if layer == FULL else CFG.rope_theta_sliding
    return model.rope_table(CFG.head_dim_for(layer), theta, partial, n, DEV)


def _prepare_attn_decode(case, seed):
    q, k, v, qn, kn, kp, vp, pt, pos = _attn_decode_inputs(case, seed)
    b, n = case["b"], case["max_len"]
    cos, sin = _rope(case["layer"], n)
    splits = max(ops.attention_min_splits(n), 1)
    ws = int(_lib.lib().g4mi_decode_attention_workspace_bytes(b, NH, q.shape[2], n, splits))
    return {"args": (q, k, v, qn, kn, cos, sin, kp, vp, pt, pos, _geometry(case["layer"])[2], case["softcap"], EPS, n),
            "ctx": torch.zeros_like(q), "ws": torch.zeros(ws, dtype=torch.uint8, device=DEV), "k": kp, "v": vp}


def _prepare_moe_decode(case, seed):
    n = case["n"]
    layers = _moe_inputs(case, seed)
    for lp in layers:
        lp["out"] = torch.empty(n, H, dtype=BF16, device=DEV)
        lp["route"] = (torch.empty(n, TOPK, dtype=torch.float32, device=DEV),
                       torch.empty(n, TOPK, dtype=torch.int32, device=DEV))
    return layers


_prepare_moe_prefill = _prepare_moe_decode


def _prepare_products(case, seed):
    n = case["n"]
    layers = _products_inputs(case, seed)
    for lp in layers:
        new = lambda cols: torch.empty(n, cols, dtype=BF16, device=DEV)  # noqa: E731
        lp["y"] = {"qkv": [new(w.shape[0]) for w in lp["qkv"]], "o": new(H), "act": new(I), "mlp": new(H)}
    return layers


def _prepare_sample(case, seed):
    logits = _sample_inputs(case, seed)
    return {"logits": logits, "k": case["top_k"], "tok": torch.zeros(1, dtype=torch.int32, device=DEV),
            "params": ops.sample_params(case["temperature"], case["top_p"], int(seed), DEV),
            "ws": torch.zeros(ops.sample_workspace_bytes(case["vocab"]), dtype=torch.uint8, device=DEV)}


# -------------------------------------------------------------------------- run
def run(state):
    if isinstance(state, list):
        return [_run_products(lp) if "qkv" in lp else _run_moe(lp, len(state) == 2) for lp in state]
    if "step" in state:
        eng = state["eng"]
        state["step"](eng.params, state["tok"], eng.cache, state["pos"], state["seed"], state["t"], state["p"])
        return state["out"]
    if "fn" in state:
        eng = state["eng"]
        state["fn"](eng.params, state["tok"], eng.cache, state["n"], 0, 0.0, 1.0)
        return state["out"]
    if "q" in state:
        return ops.prefill_attention(state["q"], state["k"], state["v"], state["pt"], state["p0"], state["window"],
                                     state["cap"], ctx=state["ctx"])
    if "args" in state:
        ops.decode_attention(*state["args"], ctx=state["ctx"], ws=state["ws"])
        return {"ctx": state["ctx"], "k": state["k"], "v": state["v"]}
    return ops.sample(state["logits"], state["k"], state["params"], state["tok"], counter_mode=0, ws=state["ws"])


def _run_moe(lp, decode: bool):
    if decode:
        ops.moe_block(lp["x"], lp["scale"], lp["proj"], lp["pes"], lp["gate_up"], lp["down"], TOPK, EPS,
                      out=lp["out"], route=lp["route"])
    else:
        ops.moe_router_topk(lp["x"], lp["scale"], lp["proj"], lp["pes"], TOPK, EPS, out=lp["route"])
        ops.moe_prefill(lp["x"], *lp["route"], lp["gate_up"], lp["down"], out=lp["out"])
    return {"out": lp["out"], "w": lp["route"][0], "i": lp["route"][1]}


def _run_products(lp):
    y = lp["y"]
    if lp["xn"].shape[0] <= 16:  # decode rows: one launch for q, k and v
        ops.gemm_segments(lp["xn"], lp["qkv"], y["qkv"])
    else:
        for w, out in zip(lp["qkv"], y["qkv"]):
            ops.prefill_gemm(lp["xn"], w, out)
    ops.prefill_gemm(lp["ctx"], lp["o"], y["o"])
    ops.prefill_gemm(lp["xm"], lp["gate_up"], y["act"], epilogue=ops.EP_GATED, pair_offset=I * H, n=I)
    ops.prefill_gemm(y["act"], lp["down"], y["mlp"])
    return y


# ------------------------------------------------------------------------- work
def _attended(layer: str, positions) -> int:
    w = _geometry(layer)[2]
    return sum(min(p + 1, w) if w else p + 1 for p in positions)


def _layer_weights(layer: str) -> int:
    """Values of a layer's dense projections and MLP."""
    kv, d, _ = _geometry(layer)
    return H * (2 * NH * d + kv * d * (2 if layer == SLIDING else 1) + 3 * I)


def _experts_read(n: int) -> float:
    """Experts of E that n tokens of TOPK each select, routing evenly."""
    return E * (1.0 - (1.0 - TOPK / E) ** n)


EXPERT = 3 * F * H  # values of one expert


def _model_work(positions, n: int, head_rows: int):
    wb = CFG.vocab_size * H * 2.0
    fl = 2.0 * head_rows * CFG.vocab_size * H
    for layer in CFG.layer_types:
        kv, d, _ = _geometry(layer)
        wb += 2.0 * (_layer_weights(layer) + E * H + _experts_read(n) * EXPERT)
        fl += 2.0 * n * (_layer_weights(layer) + E * H + TOPK * EXPERT)
        att = _attended(layer, positions)
        fl += 4.0 * NH * d * att
        lo = max(0, positions[0] + 1 - _geometry(layer)[2]) if layer == SLIDING else 0
        wb += 2 * 2.0 * kv * d * (positions[-1] + 1 - lo)
    return {"bytes": wb, "flops": fl}


def work(case):
    kind = case["kind"]
    if kind == "decode":
        return _model_work([case["pos"]], 1, 1)
    if kind == "prefill":
        return _model_work(range(case["n"]), case["n"], 1)
    if kind == "attn_prefill":
        kv, d, w = _geometry(case["layer"])
        t, p0 = case["t"], case["p0"]
        keys = p0 + t - (max(0, p0 + 1 - w) if w else 0)
        return {"bytes": 2.0 * (2 * t * NH * d + 2 * keys * kv * d),
                "flops": 4.0 * NH * d * _attended(case["layer"], range(p0, p0 + t))}
    if kind == "attn_decode":
        kv, d, _ = _geometry(case["layer"])
        att = _attended(case["layer"], _lengths(case))
        return {"bytes": 2.0 * (2 * att * kv * d + 2 * case["b"] * NH * d), "flops": 4.0 * NH * d * att}
    if kind in ("moe_decode", "moe_prefill"):
        n, layers = case["n"], 2 if kind == "moe_decode" else 1
        return {"bytes": layers * 2.0 * (_experts_read(n) * EXPERT + E * H + 2 * n * H),
                "flops": layers * 2.0 * n * (TOPK * EXPERT + E * H)}
    if kind == "products":
        n, b, fl = case["n"], 0.0, 0.0
        for layer in (SLIDING, FULL):
            kv, d, _ = _geometry(layer)
            cols = 2 * NH * d + kv * d * (2 if layer == SLIDING else 1) + 4 * H + 2 * I
            b += 2.0 * (_layer_weights(layer) + n * cols)
            fl += 2.0 * n * _layer_weights(layer)
        return {"bytes": b, "flops": fl}
    return {"bytes": 4.0 * case["vocab"] + 4, "flops": 0.0}


def tolerance(case):
    # measured against `exact`: attention 0.004-0.012 (probabilities and ctx in
    # bf16), experts 0.0045-0.0064, products 0.0017-0.0039; the whole models
    # 0.01-0.05: every layer's bf16 rounding, and now and then an expert that is
    # chosen by a hair, go through the layers that follow
    return {"decode": {"rel": 0.15}, "prefill": {"rel": 0.15}, "attn_prefill": {"rel": 0.03},
            "attn_decode": {"rel": 0.04}, "moe_decode": {"rel": 0.02}, "moe_prefill": {"rel": 0.02},
            "products": {"rel": 0.015}, "sample": "exact"}[case["kind"]]


# ------------------------------------------------------------------------ exact
def exact(case, seed):
    fn = globals().get("_exact_" + case["kind"])
    return None if fn is None else fn(case, seed)  # sample: a drawn index, no value in 64 bits


def _mm(a, b):
    """a [n, k] . b [m, k]^T in float64, b in pieces of at most 64 MB."""
    step = max(1, (8 << 20) // b.shape[1])
    return torch.cat([a @ b[i:i + step].double().T for i in range(0, b.shape[0], step)], dim=1)


def _norm(x, w=None):
    y = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)
    return y if w is None else y * w.double()


def _gelu(x):
    return 0.5 * x * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (x + 0.044715 * x**3)))


def _rotate(x, layer, positions):
    """RoPE of x [n, heads, d] at positions [n]."""
    d = x.shape[-1]
    part = CFG.rope_partial_rotary_factor_full if layer == FULL else 1.0
    theta = CFG.rope_theta_full if layer == FULL else CFG.rope_theta_sliding
    rot = int(part * d // 2)
    inv = torch.zeros(d // 2, dtype=torch.float64, device=x.device)
    inv[:rot] = 1.0 / theta ** (torch.arange(rot, dtype=torch.float64, device=x.device) * 2.0 / d)
    ang = positions.double()[:, None] * inv[None]
    c, s = torch.cos(ang)[:, None], torch.sin(ang)[:, None]
    a, b = x[..., : d // 2], x[..., d // 2:]
    return torch.cat([a * c - b * s, b * c + a * s], dim=-1)


def _attend(q, k, v, q_pos, k_pos, window, cap):
    """q [t, NH, d], k and v [s, KV, d] -> [t, NH, d]; rows in pieces."""
    g = NH // k.shape[1]
    out = torch.empty_like(q)
    for t0 in range(0, q.shape[0], 512):
        qp = q_pos[t0:t0 + 512, None]
        mask = (k_pos[None] <= qp) & ((k_pos[None] > qp - window) if window else True)
        for h in range(NH):
            s = q[t0:t0 + 512, h] @ k[:, h // g].T
            s = torch.tanh(s / cap) * cap if cap else s
            out[t0:t0 + 512, h] = torch.softmax(s.masked_fill(~mask, -math.inf), -1) @ v[:, h // g]
    return out


def _unpage(pages, row):
    """[n, KV, PAGE, d] through a page-table row -> [positions, KV, d]."""
    t = pages[row.long()]
    return t.permute(0, 2, 1, 3).reshape(-1, t.shape[1], t.shape[3]).double()


def _exact_attn_prefill(case, seed):
    q, kp, vp, pt = _attn_prefill_inputs(case, seed)
    n = case["p0"] + case["t"]
    k_pos = torch.arange(n, device=DEV)
    return _attend(q.double(), _unpage(kp, pt)[:n], _unpage(vp, pt)[:n], k_pos[case["p0"]:], k_pos,
                   _geometry(case["layer"])[2], case["softcap"])


def _exact_attn_decode(case, seed):
    q, k, v, qn, kn, kp, vp, pt, pos = _attn_decode_inputs(case, seed)
    layer = case["layer"]
    q = _rotate(_norm(q.double(), qn), layer, pos)
    v = _norm((k if v is None else v).double())
    k = _rotate(_norm(k.double(), kn), layer, pos)
    kp, vp, ctx = kp.double(), vp.double(), torch.empty_like(q)
    for b, p in enumerate(_lengths(case)):
        page = int(pt[b, p // PAGE])
        kp[page, :, p % PAGE], vp[page, :, p % PAGE] = k[b], v[b]
        k_pos = torch.arange(p + 1, device=DEV)
        ctx[b] = _attend(q[b:b + 1], _unpage(kp, pt[b])[:p + 1], _unpage(vp, pt[b])[:p + 1], pos[b:b + 1], k_pos,
                         _geometry(layer)[2], case["softcap"])[0]
    return {"ctx": ctx, "k": kp, "v": vp}


def _route(x, scale, proj, pes):
    """The router's selection on bf16 rows: its input and its logits are bf16
    by definition (they decide which experts run), ties go to the lower
    index; the weights in float64."""
    r = lambda t: t.to(BF16).double()  # noqa: E731
    x2 = r(r(r(_norm(x.double())) * scale.double()) * r(torch.tensor(H**-0.5, dtype=torch.float64)).to(x.device))
    p = torch.softmax(r(_mm(x2, proj).float()), -1)
    top = torch.sort(p, dim=-1, descending=True, stable=True).indices[:, :TOPK]
    w = torch.gather(p, 1, top)
    return w / w.sum(-1, keepdim=True) * pes.double()[top], top


def _experts(x, w, top, gate_up, down):
    out = torch.zeros(x.shape[0], H, dtype=torch.float64, device=x.device)
    for e in torch.unique(top).tolist():
        rows, slots = (top == e).nonzero(as_tuple=True)
        xe = x[rows]
        act = _gelu(_mm(xe, gate_up[e, 0])) * _mm(xe, gate_up[e, 1]) * w[rows, slots][:, None]
        out.index_add_(0, rows, _mm(act, down[e]))
    return out


def _exact_moe_decode(case, seed):
    got = []
    for lp in _moe_inputs(case, seed):
        w, top = _route(lp["x"], lp["scale"], lp["proj"], lp["pes"])
        got.append({"out": _experts(lp["x"].double(), w, top, lp["gate_up"], lp["down"]), "w": w,
                    "i": top.to(torch.int32)})
    return got


_exact_moe_prefill = _exact_moe_decode


def _exact_products(case, seed):
    got = []
    for lp in _products_inputs(case, seed):
        xm = lp["xm"].double()
        act = _gelu(_mm(xm, lp["gate_up"][:I])) * _mm(xm, lp["gate_up"][I:])
        got.append({"qkv": [_mm(lp["xn"].double(), w) for w in lp["qkv"]], "o": _mm(lp["ctx"].double(), lp["o"]),
                    "act": act, "mlp": _mm(act, lp["down"])})
    return got


def _exact_model(p, tok, p0, past):
    """The six layers and the head on tok [n] at positions p0 .. after the
    cached (k, v) [p0, KV, d] of each layer: (logits of the last row, k, v
    per layer)."""
    n = tok.numel()
    positions = torch.arange(p0, p0 + n, device=DEV)
    k_pos = torch.arange(p0 + n, device=DEV)
    x = p["embed"][tok.long()].double() * float(torch.tensor(math.sqrt(H)).to(BF16))
    ks, vs = [], []
    for i, layer in enumerate(CFG.layer_types):
        lp = {k[len(f"layers.{i}."):]: v for k, v in p.items() if k.startswith(f"layers.{i}.")}
        kv, d, window = _geometry(layer)
        h = _norm(x, lp["input_layernorm"])
        k = _mm(h, lp["k_proj"].reshape(kv * d, H)).reshape(n, kv, d)
        v = _mm(h, lp["v_proj"].reshape(kv * d, H)).reshape(n, kv, d) if "v_proj" in lp else k
        q = _rotate(_norm(_mm(h, lp["q_proj"].reshape(NH * d, H)).reshape(n, NH, d), lp["q_norm"]), layer, positions)
        k, v = _rotate(_norm(k, lp["k_norm"]), layer, positions), _norm(v)
        ks.append(k)
        vs.append(v)
        ctx = _attend(q, torch.cat([past[i][0], k]), torch.cat([past[i][1], v]), positions, k_pos, window, None)
        x = x + _norm(_mm(ctx.reshape(n, NH * d), lp["o_proj"].reshape(H, NH * d)), lp["post_attention_layernorm"])
        xm = _norm(x, lp["pre_feedforward_layernorm"])
        mlp = _mm(_gelu(_mm(xm, lp["mlp.gate_proj"])) * _mm(xm, lp["mlp.up_proj"]), lp["mlp.down_proj"])
        xe = _norm(x, lp["pre_feedforward_layernorm_2"])
        w, top = _route(xe.to(BF16), lp["router.scale"], lp["router.proj"], lp["router.per_expert_scale"])
        moe = _experts(xe, w, top, lp["experts.gate_up_proj"], lp["experts.down_proj"])
        ff = _norm(mlp, lp["post_feedforward_layernorm_1"]) + _norm(moe, lp["post_feedforward_layernorm_2"])
        x = (x + _norm(ff, lp["post_feedforward_layernorm"])) * lp["layer_scalar"].double()
    logits = _mm(_norm(x[-1:], p["norm"]), p["embed"])[0]
    cap = CFG.final_logit_softcapping
    return torch.tanh(logits / cap) * cap, ks, vs


def _exact_decode(case, seed):
    r, p, tok = _model_inputs(case, seed)
    pos, past = case["pos"], []
    pages = (pos + PAGE - 1) // PAGE
    order = torch.arange(pages, device=DEV)
    for layer in CFG.layer_types:
        kv, d, _ = _geometry(layer)
        k = r.normal(pages, kv, PAGE, d, std=0.3)
        v = r.normal(pages, kv, PAGE, d)
        past.append((_unpage(k, order)[:pos], _unpage(v, order)[:pos]))
    logits, ks, vs = _exact_model(p, tok, pos, past)
    return {"logits": logits, "k": [k[0] for k in ks], "v": [v[0] for v in vs]}


def _exact_prefill(case, seed):
    _, p, tok = _model_inputs(case, seed)
    none = [(torch.empty(0, *_geometry(t)[:2], dtype=torch.float64, device=DEV),) * 2 for t in CFG.layer_types]
    logits, ks, vs = _exact_model(p, tok, 0, none)
    pages = (case["n"] + PAGE - 1) // PAGE

    def page(t):  # [n, KV, d] -> the pages, zero past the prompt
        full = torch.zeros(pages * PAGE, *t.shape[1:], dtype=t.dtype, device=t.device)
        full[: t.shape[0]] = t
        return full.reshape(pages, PAGE, *t.shape[1:]).permute(0, 2, 1, 3).contiguous()

    return {"logits": logits, "k": page(ks[-1]), "v": page(vs[-1])}
