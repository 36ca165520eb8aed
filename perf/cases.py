"""The work whose speed this framework is judged by, as cases that a timing
program can list, draw, prepare, run and check.

The framework is a W4A16 AWQ GEMM for a Qwen2-7B-shaped model, the kernels
around it, and the greedy decode engine that calls them.  The cases are what
its users have it do:

* ``linear``: one call on one projection (the smallest unit of work);
* ``layers``: the projections of some decoder layers on one batch of tokens,
  as an engine issues them -- fused QKV with its bias, o_proj and down_proj
  with their residual, fused gate||up; or the seven unfused projections of the
  reference's model.  Each layer has its own weights, so a decode step reads
  them from memory and not from a cache, as in a model;
* ``lm_head``: the logits of the last position;
* ``silu_mul``: SiLU * up over a prompt's fused gate||up output;
* ``prefill``, ``decode`` and ``generate``: the engine's three entry points.

Sizes are those of the Qwen2-7B configuration (hidden 3584, intermediate
18944, 28 / 4 heads of 128, vocabulary 152064, 28 layers), with prompt and
batch sizes from one token to a few thousand.
"""
import math
import os
import sys

import torch

# The package's folder name is no Python identifier: its parts are imported from inside it.
_PKG = os.path.abspath("qwen2-7b-triton_engine_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from engine.qwen2_decode import Qwen2AwqDecoder, Qwen2Shape  # noqa: E402
from kernels.awq_gemm import awq_gemm_forward, awq_gemm_forward_ex  # noqa: E402
from kernels.lm_head import lm_head_forward  # noqa: E402
from kernels.silu_mul import silu_mul_gate_up  # noqa: E402

HIDDEN, INTER, QKV, KV, VOCAB, LAYERS = 3584, 18944, 4608, 512, 152064, 28
HEADS, KV_HEADS, HEAD_DIM, EPS, THETA = 28, 4, 128, 1e-6, 1e6

# (name, K, N, epilogue) of one decoder layer's projections, as the engine
# fuses them and as the reference's model holds them.
FUSED = (("qkv", HIDDEN, QKV, "bias"), ("o", HIDDEN, HIDDEN, "residual"), ("gate_up", HIDDEN, 2 * INTER, ""),
         ("down", INTER, HIDDEN, "residual"))
UNFUSED = (("q", HIDDEN, HIDDEN, ""), ("k", HIDDEN, KV, ""), ("v", HIDDEN, KV, ""), ("o", HIDDEN, HIDDEN, ""),
           ("gate", HIDDEN, INTER, ""), ("up", HIDDEN, INTER, ""), ("down", INTER, HIDDEN, ""))


def listed():
    return [
        # The smallest call: k_proj of one token.
        {"name": "k_proj_m1", "kind": "linear", "m": 1, "k": HIDDEN, "n": KV, "epilogue": ""},
        # One token through the projections of 16 layers (1.9 GB of weights): batch-1 decoding.
        {"name": "layers_m1", "kind": "layers", "m": 1, "layers": 16, "fused": True},
        # Three sequences at once on the unfused projections, the reference's own modules.
        {"name": "layers_m3_unfused", "kind": "layers", "m": 3, "layers": 9, "fused": False},
        # A small serving batch.
        {"name": "layers_m16", "kind": "layers", "m": 16, "layers": 12, "fused": True},
        # A short prompt of ragged length.
        {"name": "layers_m77", "kind": "layers", "m": 77, "layers": 8, "fused": True},
        # An ordinary prompt of ragged length.
        {"name": "layers_m700", "kind": "layers", "m": 700, "layers": 3, "fused": True},
        # A long prompt.
        {"name": "layers_m2048", "kind": "layers", "m": 2048, "layers": 2, "fused": True},
        # The logits of one sequence's last position.
        {"name": "lm_head_m1", "kind": "lm_head", "m": 1, "n": VOCAB},
        # The MLP's activation over an ordinary prompt.
        {"name": "silu_mul_m1021", "kind": "silu_mul", "m": 1021, "i": INTER},
        # A long ragged prompt into a stack of a few layers: the attention's share grows with the prompt.
        {"name": "prefill_s1777", "kind": "prefill", "layers": 4, "prompt": 1777, "max_seq": 2048},
        # A given continuation scored token by token after a prompt (eager decode steps).
        {"name": "decode_s900", "kind": "decode", "layers": 4, "prompt": 900, "steps": 8, "max_seq": 2048},
        # The whole model: a 1024-token prompt and greedy tokens after it.
        {"name": "generate_28", "kind": "generate", "layers": LAYERS, "prompt": 1024, "steps": 48, "max_seq": 1152},
    ]


def _log_int(rng, lo, hi):
    """A whole number of [lo, hi], spread evenly over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "layers", "layers", "lm_head", "silu_mul", "prefill", "decode",
                       "generate"])
    if kind == "linear":
        if rng.random() < 0.5:
            _, k, n, _ = rng.choice(FUSED + UNFUSED)
        else:       # generic weights: K in groups of 128, N in packed words of 8
            k, n = 128 * _log_int(rng, 2, 148), 8 * _log_int(rng, 8, 4736)
        return {"kind": kind, "m": _log_int(rng, 1, 2048), "k": k, "n": n,
                "epilogue": rng.choice(["", "", "bias", "residual"])}
    if kind == "layers":
        return {"kind": kind, "m": _log_int(rng, 1, 2048), "layers": rng.randint(1, 2), "fused": rng.random() < 0.7}
    if kind == "lm_head":
        return {"kind": kind, "m": rng.randint(1, 8), "n": _log_int(rng, 1000, VOCAB)}
    if kind == "silu_mul":
        return {"kind": kind, "m": _log_int(rng, 1, 2048), "i": 8 * _log_int(rng, 64, INTER // 8)}
    prompt = _log_int(rng, 1, 1900)
    case = {"kind": kind, "layers": rng.randint(1, 5), "prompt": prompt}
    if kind != "prefill":
        case["steps"] = rng.randint(2, 24)
    case["max_seq"] = prompt + case.get("steps", 0) + rng.randint(1, 700)
    return case


# ---- inputs ----------------------------------------------------------------------


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _awq(k, n, g, lo=0.002, hi=0.02):
    """AWQ operands: uniform codes and zero codes, scales U[lo, hi]."""
    word = dict(generator=g, device="cuda", dtype=torch.int32)
    return (torch.randint(-2**31, 2**31 - 1, (k, n // 8), **word),
            torch.randint(-2**31, 2**31 - 1, (k // 128, n // 8), **word),
            (torch.rand((k // 128, n), generator=g, device="cuda") * (hi - lo) + lo).half())


def _normal(shape, g, std=1.0):
    return (torch.randn(shape, generator=g, device="cuda") * std).half()


def _linear_inputs(m, k, n, epilogue, g):
    return {"x": _normal((m, k), g), "w": _awq(k, n, g),
            "bias": _normal((n,), g, 0.02) if epilogue == "bias" else None,
            "residual": _normal((m, n), g) if epilogue == "residual" else None}


def _layers_inputs(case, g):
    m = case["m"]
    x = {HIDDEN: _normal((m, HIDDEN), g), INTER: _normal((m, INTER), g)}
    residual = _normal((m, HIDDEN), g)
    calls = []
    for _ in range(case["layers"]):
        for _, k, n, epilogue in FUSED if case["fused"] else UNFUSED:
            calls.append({"x": x[k], "w": _awq(k, n, g), "bias": _normal((n,), g, 0.02) if epilogue == "bias" else None,
                          "residual": residual if epilogue == "residual" else None})
    return calls


def _model_inputs(case, g):
    """Weights of a model with the structure a trained one shows: weights of
    standard deviation 0.01 that let the embedding show through to the last
    layer, and an output projection that answers each token with one clear
    successor -- so that greedy tokens do not hang on roundings."""
    embed = torch.randn((VOCAB, HIDDEN), generator=g, device="cuda").half()
    successor = torch.randperm(VOCAB, generator=g, device="cuda")
    lm_head = torch.empty_like(embed)
    lm_head[successor] = embed * 0.02
    layers = []
    for _ in range(case["layers"]):
        lw = {"ln1": (1.0 + 0.1 * torch.randn(HIDDEN, generator=g, device="cuda")).half(),
              "ln2": (1.0 + 0.1 * torch.randn(HIDDEN, generator=g, device="cuda")).half(),
              "qkv_bias": _normal((QKV,), g, 0.5)}
        for name, k, n, _ in FUSED:
            lw[name] = _awq(k, n, g, 0.0005, 0.003)
        layers.append(lw)
    weights = {"embed": embed, "lm_head": lm_head, "final_norm": torch.ones(HIDDEN, dtype=torch.float16, device="cuda"),
               "layers": layers}
    prompt = torch.randint(0, VOCAB, (case["prompt"],), generator=g, device="cuda")
    forced = torch.randint(0, VOCAB, (case.get("steps", 0),), generator=g, device="cuda")
    return weights, successor, prompt, forced


def _shape(case):
    return Qwen2Shape(vocab_size=VOCAB, hidden_size=HIDDEN, intermediate_size=INTER, num_layers=case["layers"],
                      num_heads=HEADS, num_kv_heads=KV_HEADS, rms_norm_eps=EPS, rope_theta=THETA)


def prepare(case, seed):
    g = _generator(seed)
    kind = case["kind"]
    if kind == "linear":
        return {"kind": kind, **_linear_inputs(case["m"], case["k"], case["n"], case["epilogue"], g)}
    if kind == "layers":
        return {"kind": kind, "calls": _layers_inputs(case, g)}
    if kind == "lm_head":
        return {"kind": kind, "x": _normal((case["m"], HIDDEN), g), "weight": _normal((case["n"], HIDDEN), g, 0.02)}
    if kind == "silu_mul":
        return {"kind": kind, "gate_up": _normal((case["m"], 2 * case["i"]), g, 4.0)}
    weights, _, prompt, forced = _model_inputs(case, g)
    model = Qwen2AwqDecoder(_shape(case), max_seq_len=case["max_seq"], device="cuda:0", weights=weights)
    if kind == "decode":
        model.prefill(prompt)
    return {"kind": kind, "model": model, "prompt": prompt, "forced": forced, "steps": case.get("steps", 0)}


def _call(c):
    if c["bias"] is None and c["residual"] is None:
        return awq_gemm_forward(c["x"], *c["w"])
    return awq_gemm_forward_ex(c["x"], *c["w"], bias=c["bias"], residual=c["residual"])


def run(state):
    kind = state["kind"]
    if kind == "linear":
        return _call(state)
    if kind == "layers":
        return [_call(c) for c in state["calls"]]
    if kind == "lm_head":
        return lm_head_forward(state["x"], state["weight"])
    if kind == "silu_mul":
        return silu_mul_gate_up(state["gate_up"])
    model, prompt = state["model"], state["prompt"]
    if kind == "prefill":
        return {"logits": model.prefill(prompt), "k": model.k_cache, "v": model.v_cache}
    if kind == "decode":
        start = prompt.shape[0]
        logits = [model.decode_logits(state["forced"][i], start + i) for i in range(state["steps"])]
        return {"logits": torch.stack(logits), "k": model.k_cache, "v": model.v_cache}
    # The tokens, then the logits that follow the last of them.
    tokens = model.generate(prompt, state["steps"])["tokens"]
    logits = model.decode_logits(tokens[-1], prompt.shape[0] + state["steps"] - 1)
    return {"tokens": tokens, "logits": logits, "k": model.k_cache, "v": model.v_cache}


# ---- what a pass cannot do without --------------------------------------------------


def _linear_work(m, k, n, extra=0):
    return k * n // 2 + (k // 128) * n * 5 // 2 + 2 * m * (k + n) + 2 * extra, 2 * m * k * n


def _model_step_work(layers, new, context):
    """(bytes, flops) of `new` positions that end at `context` positions,
    through `layers` layers and the last position's logits."""
    b, f = 2 * VOCAB * HIDDEN + 2 * VOCAB, 2 * VOCAB * HIDDEN
    pairs = sum(range(context - new + 1, context + 1))
    for _, k, n, _ in FUSED:
        lb, lf = _linear_work(0, k, n)
        b, f = b + layers * lb, f + layers * 2 * new * k * n
    b += layers * 2 * 2 * KV * context                       # the keys and values read and written
    f += layers * 4 * HIDDEN * pairs
    return b, f


def work(case):
    kind = case["kind"]
    if kind == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        b, f = _linear_work(m, k, n, {"": 0, "bias": n, "residual": m * n}[case["epilogue"]])
    elif kind == "layers":
        m, b, f = case["m"], 0, 0
        for _, k, n, epilogue in FUSED if case["fused"] else UNFUSED:
            lb, lf = _linear_work(m, k, n, {"": 0, "bias": n, "residual": m * n}[epilogue])
            b, f = b + case["layers"] * lb, f + case["layers"] * lf
    elif kind == "lm_head":
        m, n = case["m"], case["n"]
        b, f = 2 * (n * HIDDEN + m * HIDDEN + m * n), 2 * m * n * HIDDEN
    elif kind == "silu_mul":
        b, f = 6 * case["m"] * case["i"], 4 * case["m"] * case["i"]
    else:
        b = f = 0
        if kind != "decode":
            b, f = _model_step_work(case["layers"], case["prompt"], case["prompt"])
        # generate: steps - 1 graph replays and the closing step; decode: one for each given token.
        for i in range(case.get("steps", 0)):
            sb, sf = _model_step_work(case["layers"], 1, case["prompt"] + i + 1)
            b, f = b + sb, f + sf
    return {"bytes": b, "flops": f}


def tolerance(case):
    """About four times the largest distance from ``exact`` measured over the
    listed and some drawn cases: one fp16 rounding of each output (and, for the
    bias and the residual, of the sum), and for the engine's calls the fp16
    activations of the layers before."""
    kind = case["kind"]
    if kind in ("linear", "layers"):
        return {"rel": 1.5e-3, "max": 6e-3}
    if kind in ("lm_head", "silu_mul"):
        return {"rel": 8e-4, "max": 2e-3}
    return {"rel": 8e-3, "max": 0.1}


# ---- the same in 64 bits, in plain torch ------------------------------------------------


def _unpack(words):
    """Codes of logical columns: column c of a packed word is nibble (0,4,1,5,2,6,3,7)[c]."""
    shifts = torch.tensor([0, 16, 4, 20, 8, 24, 12, 28], dtype=torch.int32, device=words.device)
    return ((words.unsqueeze(-1) >> shifts) & 15).reshape(words.shape[0], -1)


def _dense(w):
    """fp16((q - z) * s), the weight that the operands stand for, in 64 bits."""
    qweight, qzeros, scales = w
    q = _unpack(qweight).view(scales.shape[0], 128, -1)
    return ((q - _unpack(qzeros).unsqueeze(1)).half() * scales.unsqueeze(1)).double().view(qweight.shape[0], -1)


def _exact_linear(x, w, bias=None, residual=None):
    y = x.double() @ _dense(w)
    if bias is not None:
        y = y + bias.double()
    return y if residual is None else y + residual.double()


def _exact_norm(h, w):
    return h * torch.rsqrt(h.pow(2).mean(-1, keepdim=True) + EPS) * w.double()


def _exact_model(weights, ids, max_seq):
    """Last hidden states [S, hidden] and the caches after the positions of `ids`."""
    S = ids.shape[0]
    h = weights["embed"][ids].double()
    inv = THETA ** (-torch.arange(0, HEAD_DIM, 2, device="cuda", dtype=torch.float64) / HEAD_DIM)
    angle = torch.outer(torch.arange(S, device="cuda", dtype=torch.float64), inv)
    cos, sin = torch.cat((angle, angle), -1).cos().unsqueeze(1), torch.cat((angle, angle), -1).sin().unsqueeze(1)

    def rope(t):
        return t * cos + torch.cat((-t[..., HEAD_DIM // 2:], t[..., :HEAD_DIM // 2]), -1) * sin

    mask = torch.ones((S, S), dtype=torch.bool, device="cuda").triu(1)
    cache = torch.zeros((2, len(weights["layers"]), KV_HEADS, max_seq, HEAD_DIM), dtype=torch.float64, device="cuda")
    for li, p in enumerate(weights["layers"]):
        qkv = _exact_linear(_exact_norm(h, p["ln1"]), p["qkv"], bias=p["qkv_bias"])
        q = rope(qkv[:, :HIDDEN].view(S, HEADS, HEAD_DIM)).transpose(0, 1)
        k = rope(qkv[:, HIDDEN:HIDDEN + KV].view(S, KV_HEADS, HEAD_DIM)).transpose(0, 1)
        v = qkv[:, HIDDEN + KV:].view(S, KV_HEADS, HEAD_DIM).transpose(0, 1)
        cache[0, li, :, :S], cache[1, li, :, :S] = k, v
        att = torch.empty((S, HEADS, HEAD_DIM), dtype=torch.float64, device="cuda")
        for head in range(HEADS):
            g = head // (HEADS // KV_HEADS)
            scores = (q[head] @ k[g].t().contiguous() / math.sqrt(HEAD_DIM)).masked_fill(mask, float("-inf"))
            att[:, head] = torch.softmax(scores, -1) @ v[g].contiguous()
        h = _exact_linear(att.view(S, HIDDEN), p["o"], residual=h)
        gate_up = _exact_linear(_exact_norm(h, p["ln2"]), p["gate_up"])
        h = _exact_linear(torch.nn.functional.silu(gate_up[:, :INTER]) * gate_up[:, INTER:], p["down"], residual=h)
    return h, cache[0], cache[1]


def exact(case, seed):
    g = _generator(seed)
    kind = case["kind"]
    if kind == "linear":
        c = _linear_inputs(case["m"], case["k"], case["n"], case["epilogue"], g)
        return _exact_linear(c["x"], c["w"], c["bias"], c["residual"])
    if kind == "layers":
        return [_exact_linear(c["x"], c["w"], c["bias"], c["residual"]) for c in _layers_inputs(case, g)]
    if kind == "lm_head":
        x, weight = _normal((case["m"], HIDDEN), g), _normal((case["n"], HIDDEN), g, 0.02)
        return x.double() @ weight.double().t()
    if kind == "silu_mul":
        gate, up = _normal((case["m"], 2 * case["i"]), g, 4.0).double().chunk(2, -1)
        return torch.nn.functional.silu(gate) * up
    weights, successor, prompt, forced = _model_inputs(case, g)
    if kind == "generate":      # the greedy tokens are the chain of successors; checked below
        forced = [successor[prompt[-1]]]
        while len(forced) < case["steps"]:
            forced.append(successor[forced[-1]])
        forced = torch.stack(forced)
    h, k, v = _exact_model(weights, torch.cat([prompt, forced]), case["max_seq"])
    last = _exact_norm(h[case["prompt"] - 1:], weights["final_norm"])     # the prompt's last position onwards
    head = weights["lm_head"].double().t()
    if kind == "prefill":
        return {"logits": (last[:1] @ head)[0], "k": k, "v": v}
    logits = last @ head
    if kind == "decode":
        return {"logits": logits[1:], "k": k, "v": v}
    tokens = logits[:-1].argmax(-1)
    if not torch.equal(tokens, forced):
        return None
    return {"tokens": tokens.cpu(), "logits": logits[-1], "k": k, "v": v}
