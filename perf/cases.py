"""Performance cases of the backend: the calls a program that serves Qwen3.5
makes, each through a public entry point, over the sizes it meets.

Kinds (`kind` of a case):
  attend  KvAppend + CausalGqa of one layer (ops.kv_append_causal_gqa), or,
          with `gated`, the whole attention block around it
          (ops.gated_attention): one token is a decode step, more a prompt
          chunk against `past` cached rows;
  mixer   the row work of one Gated DeltaNet layer between its projections:
          convolution + SiLU, the q / k / v views, the gates, L2Norm +
          DeltaUpdate, the gated norm (bound calls, as a serving loop keeps);
  mlp     the SwiGLU MLP of one layer, W8A8 (`w8`) or fp16 (bound calls);
  model   a step of the whole Qwen3.5-4B W8A8 session: `prompt` starts a new
          sequence and returns the last row's logits, else one decode step
          after `past` tokens.

Widths are Qwen3.5-4B's (hidden 2560, MLP 9216, 16 query / 4 KV heads of 256,
DeltaNet 16 key / 32 value heads of 128, convolution over 8192 channels), and
the 128-wide attention heads of the tests.
"""
import math

import torch

from llminfer_amd import _lib, ops

HIDDEN, INTER = 2560, 9216
HK, HV, DK, DV, TAPS = 16, 32, 128, 128, 4
CHANNELS = 2 * HK * DK + HV * DV
ROTARY_SHARE, THETA, EPS = 0.25, 1e7, 1e-6


def listed():
    return [
        # a token of a chat at a medium context: the smallest attention call
        attend("attend_decode_4k", 1, 4096),
        # a token of a long conversation or document, at no round length
        attend("attend_decode_32k", 1, 32749),
        # the next message of a conversation: a short chunk, a long history
        attend("attend_turn_16k", 61, 16411),
        # a large chunk of a long prompt
        attend("attend_chunk_2k", 2048, 2048),
        # a first message through the whole attention block
        attend("block_prompt_333", 333, 0, gated=True),
        # one token, and one prompt chunk, through a DeltaNet layer
        {"name": "mixer_decode", "kind": "mixer", "tokens": 1},
        {"name": "mixer_chunk_1k", "kind": "mixer", "tokens": 1024},
        # the MLP for one token, a short message and a prompt chunk
        {"name": "mlp_w8_turn", "kind": "mlp", "w8": True, "tokens": 13},
        {"name": "mlp_w8_chunk", "kind": "mlp", "w8": True, "tokens": 512},
        # an unquantized checkpoint's MLP for a message
        {"name": "mlp_f16_turn", "kind": "mlp", "w8": False, "tokens": 93},
        # the whole model: a decode step, a prompt
        {"name": "model_decode", "kind": "model", "prompt": False, "tokens": 1, "past": 512},
        {"name": "model_prompt_512", "kind": "model", "prompt": True, "tokens": 512, "past": 0},
    ]


def attend(name, tokens, past, gated=False, dim=256):
    case = {"kind": "attend", "tokens": tokens, "past": past, "gated": gated, "q_heads": 16,
            "kv_heads": 4, "dim": dim}
    return case if name is None else {"name": name, **case}


def _log(rng, low, high):
    """A whole number from low to high, spread evenly over its logarithm."""
    return min(high, max(low, int(math.exp(rng.uniform(math.log(low), math.log(high + 1))))))


def draw(rng):
    kind = rng.choices(["attend", "mixer", "mlp", "model"], [40, 20, 30, 10])[0]
    if kind == "attend":
        # half decode steps, half chunks of any length; contexts to 32K rows
        # (a chunk's work at most that of the largest listed one)
        tokens = 1 if rng.random() < 0.4 else _log(rng, 2, 2048)
        past = rng.choice([0, _log(rng, 1, 32768), _log(rng, 256, 32768)])
        past = min(past, 2048 * 3072 // tokens)
        return attend(None, tokens, past, rng.random() < 0.3, rng.choice([256, 256, 128]))
    if kind == "mixer":
        return {"kind": "mixer", "tokens": 1 if rng.random() < 0.3 else _log(rng, 2, 2048)}
    if kind == "mlp":
        w8 = rng.random() < 0.7
        tokens = 1 if rng.random() < 0.25 else _log(rng, 2, 1024 if w8 else 128)
        return {"kind": "mlp", "w8": w8, "tokens": tokens}
    if rng.random() < 0.5:
        return {"kind": "model", "prompt": False, "tokens": 1, "past": _log(rng, 16, 1024)}
    return {"kind": "model", "prompt": True, "tokens": _log(rng, 2, 512), "past": 0}


# ----------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn16(g, *shape):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).half()


def _attend_inputs(case, seed):
    g = _gen(seed)
    T, P, hq, hkv, d = (case[k] for k in ("tokens", "past", "q_heads", "kv_heads", "dim"))
    x = {"k": _randn16(g, T, hkv, d), "v": _randn16(g, T, hkv, d),
         "k_cache": _randn16(g, P + T, hkv, d), "v_cache": _randn16(g, P + T, hkv, d)}
    if case["gated"]:
        x["q"] = _randn16(g, T, hq, 2 * d)
        x["q_weight"] = 0.1 * torch.randn(d, generator=g, device="cuda")
        x["k_weight"] = 0.1 * torch.randn(d, generator=g, device="cuda")
    else:
        x["q"] = _randn16(g, T, hq, d)
    return x


def _mixer_inputs(case, seed):
    g = _gen(seed)
    T = case["tokens"]
    return {"x": _randn16(g, T, CHANNELS), "history": _randn16(g, CHANNELS, TAPS - 1),
            "w": (0.5 * torch.randn(CHANNELS, TAPS, generator=g, device="cuda")).half(),
            "a": _randn16(g, T, HV), "b": _randn16(g, T, HV),
            "a_log": 0.5 * torch.randn(HV, generator=g, device="cuda"),
            "dt_bias": 0.5 * torch.randn(HV, generator=g, device="cuda"),
            "state": 0.1 * torch.randn(HV, DK, DV, generator=g, device="cuda"),
            "z": _randn16(g, T * HV, DV),
            "norm": 1 + 0.2 * torch.randn(DV, generator=g, device="cuda")}


def _mlp_inputs(case, seed):
    g = _gen(seed)
    x = {"x": _randn16(g, case["tokens"], HIDDEN)}
    for name, columns, width in (("up", INTER, HIDDEN), ("gate", INTER, HIDDEN),
                                 ("down", HIDDEN, INTER)):
        if case["w8"]:
            w = torch.randint(-127, 128, (columns, width), generator=g, device="cuda",
                              dtype=torch.int8)
            scale = torch.rand(columns, width // 32, generator=g, device="cuda")
            x[name] = (w, (scale * 6e-4 + 1e-4).half())
        else:
            x[name] = ((0.02 * torch.randn(columns, width, generator=g, device="cuda")).half(),)
    return x


def prepare(case, seed):
    return {"attend": _prepare_attend, "mixer": _prepare_mixer, "mlp": _prepare_mlp,
            "model": _prepare_model}[case["kind"]](case, seed)


def _prepare_attend(case, seed):
    return {"case": case, **_attend_inputs(case, seed)}


def _prepare_mixer(case, seed):
    x = _mixer_inputs(case, seed)
    T = case["tokens"]
    half = lambda *shape: torch.empty(shape, dtype=torch.float16, device="cuda")
    full = lambda *shape: torch.empty(shape, dtype=torch.float32, device="cuda")
    y, q, k, v, mixed = half(T, CHANNELS), half(T, HK * DK), half(T, HK * DK), \
        half(T, HV * DV), half(T, HV * DV)
    beta, decay, out = full(T, HV), full(T, HV), half(T * HV, DV)
    x.update(case=case, out=out, keep=(y, q, k, v, mixed, beta, decay))
    x["calls"] = [
        ops.bind_causal_conv(x["x"], x["w"], x["history"], y, True),
        ops.bind_copy_half_view(y, q, (T, HK * DK), (CHANNELS, 1), 0),
        ops.bind_copy_half_view(y, k, (T, HK * DK), (CHANNELS, 1), HK * DK),
        ops.bind_copy_half_view(y, v, (T, HV * DV), (CHANNELS, 1), 2 * HK * DK),
        ops.bind_delta_gates(x["a"], x["b"], x["a_log"], x["dt_bias"], beta, decay),
        ops.bind_l2_norm_delta_update(q, k, v, beta, decay, x["state"], mixed),
        ops.bind_gated_rms_norm(mixed.view(T * HV, DV), x["z"], x["norm"], out)]
    return x


def _prepare_mlp(case, seed):
    x = _mlp_inputs(case, seed)
    T = case["tokens"]
    half = lambda width: torch.empty(T, width, dtype=torch.float16, device="cuda")
    up, act, out = half(INTER), half(INTER), half(HIDDEN)
    x.update(case=case, act=act, out=out, keep=[up])
    if case["w8"]:
        rows = [(torch.empty(T, w, dtype=torch.int8, device="cuda"),
                 torch.empty(T, w // 32, dtype=torch.float32, device="cuda"))
                for w in (HIDDEN, INTER)]
        x["keep"] += rows
        x["calls"] = [
            ops.bind_quantize_activation(x["x"], *rows[0]),
            ops.bind_linear_w8a8(*rows[0], *x["up"], up),
            ops.bind_linear_w8a8(*rows[0], *x["gate"], act, _lib.LINEAR_SILU_MUL, 0, up),
            ops.bind_quantize_activation(act, *rows[1]),
            ops.bind_linear_w8a8(*rows[1], *x["down"], out)]
    else:
        x["calls"] = [
            ops.bind_linear_f16(x["x"], *x["up"], up),
            ops.bind_linear_f16(x["x"], *x["gate"], act, _lib.LINEAR_SILU_MUL, 0, up),
            ops.bind_linear_f16(act, *x["down"], out)]
    return x


# The session's cache rows: a decode case starts over when it is full.
CAPACITY = 4096


def _prepare_model(case, seed):
    from llminfer_amd.graph import qwen35_4b
    from llminfer_amd.plan import ModelSession, random_weights
    c = qwen35_4b()
    device = torch.device("cuda", 0)
    session = ModelSession(c, random_weights(c, True, device, int(seed)), CAPACITY, True, device)
    g = torch.Generator().manual_seed(int(seed))
    ids = torch.randint(0, c.vocabulary, (case["past"] + case["tokens"],), generator=g).numpy()
    if case["past"]:
        session.step(ids[:case["past"]], "none")
    return {"case": case, "session": session, "ids": ids}


# -------------------------------------------------------------------- run

def run(state):
    case = state["case"]
    if case["kind"] == "attend":
        return _run_attend(case, state)
    if case["kind"] == "model":
        return _run_model(case, state)
    for call in state["calls"]:
        call()
    if case["kind"] == "mixer":
        return [state["out"], state["state"], state["history"]]
    return [state["act"], state["out"]]


def _run_attend(case, x):
    if case["gated"]:
        out = ops.gated_attention(x["q"], x["k"], x["v"], x["q_weight"], x["k_weight"],
                                  x["k_cache"], x["v_cache"], case["past"],
                                  int(case["dim"] * ROTARY_SHARE), EPS, THETA)
    else:
        out = ops.kv_append_causal_gqa(x["q"], x["k"], x["v"], x["k_cache"], x["v_cache"],
                                       case["past"])
    return [out, x["k_cache"], x["v_cache"]]


def _run_model(case, x):
    s = x["session"]
    if case["prompt"]:
        s.reset()
        return [s.step(x["ids"], "last").logits]
    if s.past >= CAPACITY:  # the cache is full: the sequence starts over
        s.reset()
    return [s.step(x["ids"][case["past"]:], "last").logits]


# ------------------------------------------------- what a pass cannot avoid

def work(case):
    T = case["tokens"]
    if case["kind"] == "attend":
        P, hq, hkv, d = (case[k] for k in ("past", "q_heads", "kv_heads", "dim"))
        rows = T * hq * d * (3 if case["gated"] else 2) + 2 * P * hkv * d + 4 * T * hkv * d
        return {"bytes": 2 * rows, "flops": 4 * hq * d * (T * P + T * (T + 1) // 2)}
    if case["kind"] == "mixer":
        rows = T * CHANNELS + 2 * T * HV * DV + 2 * T * HV + CHANNELS * (TAPS + 2 * (TAPS - 1))
        return {"bytes": 2 * rows + 8 * HV * DK * DV, "flops": 6 * T * HV * DK * DV}
    if case["kind"] == "mlp":
        weights = 3 * HIDDEN * INTER
        return {"bytes": (weights * 34 // 32 if case["w8"] else 2 * weights) + 4 * T * HIDDEN,
                "flops": 2 * T * weights}
    from llminfer_amd.graph import EMBEDDING_ID, Element, qwen35_4b, qwen35_tensors
    c = qwen35_4b()
    projections = sum(math.prod(shape) for name, (element, shape) in
                      qwen35_tensors(c, True).items()
                      if element == Element.I8 and name != EMBEDDING_ID)
    head = c.vocabulary * c.hidden
    gqa = sum(k == "gqa" for k in c.layers)
    delta = len(c.layers) - gqa
    rows = case["past"] + T
    moved = (projections + head) * 34 // 32 + gqa * 2 * rows * c.kv_heads * c.head_dim * 2 + \
        delta * 2 * c.value_heads * c.key_dim * c.value_dim * 4 + 4 * c.vocabulary
    flops = 2 * T * projections + 2 * head + \
        gqa * 4 * c.q_heads * c.head_dim * (T * case["past"] + T * (T + 1) // 2) + \
        delta * 6 * T * c.value_heads * c.key_dim * c.value_dim
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    """About four times what was measured: against 64 bits for the layers; for
    the model between splits of one prompt into chunks (256 + 256, 500 + 12,
    511 + 1 tokens), which sum in other orders."""
    if case["kind"] == "attend":
        # fp16 inputs, probabilities and outputs: 4e-4 (largest 3e-3)
        return {"rel": 1.5e-3, "max": 0.015}
    if case["kind"] == "mixer":
        # rows divided by their own root mean square, so an ulp of a small
        # row becomes one of a row of ones: 2.5e-4 (largest 4e-3)
        return {"rel": 1e-3, "max": 0.02}
    if case["kind"] == "mlp":
        # int8 levels of the product flip with its last bit: 1.7e-3 (largest
        # 2e-2); fp16 2e-4 (6e-4)
        return {"rel": 7e-3, "max": 0.08} if case["w8"] else {"rel": 1e-3, "max": 3e-3}
    # every flipped level travels through the layers that follow: 3e-2 - 7e-2
    return {"rel": 0.25}


# ------------------------------------------------------------ in 64 bits

def _h(x):
    """A stored fp16 value, in 64 bits."""
    return x.half().double()


def exact(case, seed):
    return {"attend": _exact_attend, "mixer": _exact_mixer, "mlp": _exact_mlp,
            "model": lambda case, seed: None}[case["kind"]](case, seed)


def _norm_rope(x, weight, past, d):
    """The norm of each row by 1 + weight, its first channels rotated by the
    row's position; rounded to fp16 where the layer's rows are stored."""
    x = x.double()
    x = _h(x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * (1 + weight.double()))
    rot = int(d * ROTARY_SHARE)
    at = torch.arange(past, past + x.shape[0], device=x.device, dtype=torch.float64)
    freq = THETA ** (-2 * torch.arange(rot // 2, device=x.device, dtype=torch.float64) / rot)
    angle = (at[:, None] * freq).unsqueeze(1)
    a, b = x[..., :rot // 2], x[..., rot // 2:rot]
    c, s = angle.cos(), angle.sin()
    return _h(torch.cat([a * c - b * s, b * c + a * s, x[..., rot:]], -1))


def _exact_attend(case, seed):
    x = _attend_inputs(case, seed)
    T, P, hq, hkv, d = (case[k] for k in ("tokens", "past", "q_heads", "kv_heads", "dim"))
    q, k = x["q"].double(), x["k"].double()
    if case["gated"]:
        q = _norm_rope(x["q"][..., :d], x["q_weight"], P, d)
        k = _norm_rope(x["k"], x["k_weight"], P, d)
    x["k_cache"][P:] = k.half()
    x["v_cache"][P:] = x["v"]
    out = torch.empty(T, hq, d, dtype=torch.float64, device="cuda")
    hidden = torch.arange(P + T, device="cuda")[None, :] > \
        torch.arange(P, P + T, device="cuda")[:, None]
    for h in range(hq):
        keys = x["k_cache"][:, h // (hq // hkv)].double().t().contiguous()
        values = x["v_cache"][:, h // (hq // hkv)].double().contiguous()
        score = (q[:, h].contiguous() @ keys) / math.sqrt(d)
        out[:, h] = torch.softmax(score.masked_fill(hidden, -math.inf), -1) @ values
    if case["gated"]:
        out = _h(out) * _h(torch.sigmoid(x["q"][..., d:].double()))
    return [out, x["k_cache"].double(), x["v_cache"].double()]


def _exact_mixer(case, seed):
    x = _mixer_inputs(case, seed)
    T = case["tokens"]
    w = x["w"].double()
    rows = torch.cat([x["history"].double().t(), x["x"].double()])
    y = _h(sum(rows[j:j + T] * w[:, j] for j in range(TAPS)))
    y = _h(y * torch.sigmoid(y))
    unit = lambda r: r * torch.rsqrt((r * r).sum(-1, keepdim=True) + EPS)
    share = HV // HK
    q = unit(y[:, :HK * DK].reshape(T, HK, DK)).repeat_interleave(share, 1) / math.sqrt(DK)
    k = unit(y[:, HK * DK:2 * HK * DK].reshape(T, HK, DK)).repeat_interleave(share, 1)
    v = y[:, 2 * HK * DK:].reshape(T, HV, DV)
    beta = _h(torch.sigmoid(x["b"].double()))
    decay = torch.exp(-x["a_log"].double().exp() * torch.nn.functional.softplus(
        x["a"].double() + x["dt_bias"].double(), threshold=200.0))
    s = x["state"].double()
    mixed = torch.empty(T, HV, DV, dtype=torch.float64, device="cuda")
    for t in range(T):
        s = s * decay[t, :, None, None]
        delta = (v[t] - (s * k[t, :, :, None]).sum(1)) * beta[t, :, None]
        s = s + k[t, :, :, None] * delta[:, None, :]
        mixed[t] = (s * q[t, :, :, None]).sum(1)
    m = _h(mixed).reshape(T * HV, DV)
    m = _h(m * torch.rsqrt((m * m).mean(-1, keepdim=True) + EPS))
    z = x["z"].double()
    return [m * x["norm"].double() * z * torch.sigmoid(z), s,
            rows[-(TAPS - 1):].t().contiguous()]


def _quantized(x):
    """Rows as 32-wide groups of 127 levels, and back."""
    groups = x.reshape(x.shape[0], -1, 32)
    scale = groups.abs().amax(-1, keepdim=True) / 127
    scale = torch.where(scale > 0, scale, torch.ones_like(scale)).float().double()
    return ((groups / scale).clamp(-127, 127).round() * scale).reshape(x.shape)


def _exact_mlp(case, seed):
    x = _mlp_inputs(case, seed)

    def project(rows, name):
        w = x[name][0].double()
        if case["w8"]:
            rows = _quantized(rows)
            w = (w.reshape(w.shape[0], -1, 32) * x[name][1].double()[:, :, None]).reshape(w.shape)
        return rows @ w.t().contiguous()

    rows = x["x"].double()
    up, gate = _h(project(rows, "up")), _h(project(rows, "gate"))
    act = _h(_h(gate * torch.sigmoid(gate)) * up)
    return [act, project(act, "down")]
