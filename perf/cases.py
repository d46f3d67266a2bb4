"""The work a program has the quantized-matmul hot path do, as timed cases.

The sizes are those of the model the library serves (hidden 2048, vocabulary
128000, 64 experts top-4 of intermediate 1536, dense intermediate 11776, f32
sigmoid router with a selection bias) and of the benchmark's configurations
(65536-row heads, bf16 softmax router); the drawn cases spread over the
smaller and odd sizes in between.  Kinds:

  conv_mixer   decode, one token: the short-conv mixer's input projection with
               the conv fused, then its output projection (30 of 40 layers).
  dense_ffn    decode, one token: gate/up + SwiGLU, then the down projection.
  moe_decode   decode, one token: router, top-k, experts, combine.
  head         decode: the LM head's logits and the greedy token ids.
  sample       decode: the temperature / top-k / top-p draw over the stored
               logits, the token, and its mark in the seen set.
  moe_prefill  prefill: the MoE block of one layer over m prompt tokens.
  project      prefill: one dense projection of m prompt rows.
"""
import math

import torch

from molten_amd import hip

HIDDEN = 2048
GROUP = 64


def listed():
    return [
        # decode, one token: latency and launches count
        {"name": "conv_mixer", "kind": "conv_mixer", "h": 2048},
        {"name": "dense_ffn", "kind": "dense_ffn", "h": 2048, "inter": 11776},
        {"name": "moe_decode", "kind": "moe_decode", "h": 2048, "inter": 1536, "experts": 64, "topk": 4,
         "router": "f32", "mode": 0},
        # the model's own head, and the benchmark's batched one (8 sequences)
        {"name": "head_q6", "kind": "head", "n": 128000, "h": 2048, "bits": 6, "batch": 1},
        {"name": "head_q6_batch8", "kind": "head", "n": 65536, "h": 2048, "bits": 6, "batch": 8},
        # a sampled token instead of the greedy one
        {"name": "sample", "kind": "sample", "n": 128000, "top_k": 40, "top_p": 0.9, "temperature": 0.8,
         "penalty": 1.05},
        # a prompt's last token is decoded alone: 256-, 1K- and 4K-token prompts
        # prefill 255, 1023 and 4095 rows; 21 is a short follow-up message in a
        # chat.  The 4096-row case is the benchmark's (bf16 softmax router).
        {"name": "moe_prefill_21", "kind": "moe_prefill", "m": 21, "h": 2048, "inter": 1536, "experts": 64,
         "topk": 4, "router": "f32", "mode": 0},
        {"name": "moe_prefill_255", "kind": "moe_prefill", "m": 255, "h": 2048, "inter": 1536, "experts": 64,
         "topk": 4, "router": "f32", "mode": 0},
        {"name": "moe_prefill_1023", "kind": "moe_prefill", "m": 1023, "h": 2048, "inter": 1536, "experts": 64,
         "topk": 4, "router": "f32", "mode": 0},
        {"name": "moe_prefill_4096", "kind": "moe_prefill", "m": 4096, "h": 2048, "inter": 1536, "experts": 64,
         "topk": 4, "router": "bf16", "mode": 1},
        # the attention / conv output projection of a short prompt, and the
        # conv input projection of a long one
        {"name": "project_255", "kind": "project", "m": 255, "n": 2048, "k": 2048},
        {"name": "project_4095", "kind": "project", "m": 4095, "n": 6144, "k": 2048},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["conv_mixer", "dense_ffn", "moe_decode", "head", "sample", "moe_prefill", "moe_prefill",
                       "moe_prefill", "project", "project"])
    if kind == "conv_mixer":
        return {"kind": kind, "h": 128 * rng.randint(4, 16)}
    if kind == "dense_ffn":
        return {"kind": kind, "h": rng.choice([1024, 2048]), "inter": 64 * rng.randint(40, 184)}
    if kind in ("moe_decode", "moe_prefill"):
        c = {"kind": kind, "h": rng.choice([1024, 2048, 2048]), "inter": rng.choice([512, 1024, 1536, 1536]),
             "experts": rng.choice([16, 32, 64, 64]), "topk": rng.choice([2, 4, 4])}
        c["router"], c["mode"] = rng.choice([("f32", 0), ("f32", 0), ("bf16", 1)])
        if kind == "moe_prefill":
            c["m"] = _log_int(rng, 2, 4096)
        return c
    if kind == "head":
        return {"kind": kind, "n": _log_int(rng, 8000, 128000) // 2 * 2, "h": rng.choice([1024, 2048, 2048]),
                "bits": rng.choice([4, 6]), "batch": rng.choice([1, 1, 2, 4, 5, 8])}
    if kind == "sample":
        return {"kind": kind, "n": _log_int(rng, 8000, 128000) // 4 * 4, "top_k": rng.choice([0, 20, 40, 50]),
                "top_p": rng.choice([0.8, 0.9, 0.95, 1.0]), "temperature": rng.choice([0.3, 0.7, 1.0]),
                "penalty": rng.choice([1.0, 1.05])}
    # project: the dense projections' widths (k, v; q, o, conv out; conv in; dense FFN)
    n, k = rng.choice([(512, 2048), (2048, 2048), (2048, 2048), (6144, 2048), (6144, 2048), (11776, 2048),
                       (2048, 11776)])
    return {"kind": "project", "m": _log_int(rng, 2, 4096), "n": n, "k": k}


# ------------------------------------------------------------------ inputs --

def _weights(gen, n, k, bits):
    """An affine-quantized matrix with entries around zero, as a trained one:
    uniform codes, positive scales that vary by group, biases near minus half
    the code range (so the weights' standard deviation is about 0.7/sqrt(k))."""
    dev = gen.device
    levels = 2 ** bits
    codes = torch.randint(-2 ** 31, 2 ** 31, (n, k * bits // 32), dtype=torch.int64, device=dev, generator=gen)
    codes = codes.to(torch.int32)
    unit = 0.7 * math.sqrt(12.0 / k) / levels
    s = unit * (0.5 + torch.rand((n, k // GROUP), device=dev, generator=gen))
    b = s * (-levels / 2) * (1.0 + 0.1 * torch.randn((n, k // GROUP), device=dev, generator=gen))
    return hip.QuantWeights(codes, s.to(torch.bfloat16), b.to(torch.bfloat16), n, k, GROUP, bits)


def _randn(gen, *shape):
    return torch.randn(shape, device=gen.device, generator=gen).to(torch.bfloat16)


def _empty(gen, *shape, dtype=torch.bfloat16):
    return torch.empty(shape, dtype=dtype, device=gen.device)


def _moe(case, gen):
    e, h, i = case["experts"], case["h"], case["inter"]
    s = {"gate": _weights(gen, e * i, h, 4), "up": _weights(gen, e * i, h, 4), "down": _weights(gen, e * h, i, 4)}
    # router rows of length about 1 over unit-variance inputs; some experts
    # are chosen more often than others (the selection bias)
    router = torch.randn((e, h), device=gen.device, generator=gen) / math.sqrt(h)
    if case["router"] == "f32":
        s["router"] = router
        s["bias"] = 0.05 * torch.randn(e, device=gen.device, generator=gen)
    else:
        s["router"], s["bias"] = router.to(torch.bfloat16), None
    return s


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    kind = case["kind"]
    s = {"case": case}
    if kind == "conv_mixer":
        h = case["h"]
        s["w_in"], s["w_out"] = _weights(gen, 3 * h, h, 4), _weights(gen, h, h, 4)
        s["x"], s["taps"], s["conv_state"] = _randn(gen, h), _randn(gen, h, 3), _randn(gen, 2, h)
        s["mixed"], s["new_state"], s["y"] = _empty(gen, h), _empty(gen, 2, h), _empty(gen, h)
    elif kind == "dense_ffn":
        h, i = case["h"], case["inter"]
        s["gate"], s["up"], s["down"] = _weights(gen, i, h, 4), _weights(gen, i, h, 4), _weights(gen, h, i, 4)
        s["x"], s["act"], s["y"] = _randn(gen, h), _empty(gen, i), _empty(gen, h)
    elif kind == "moe_decode":
        s.update(_moe(case, gen))
        e, k = case["experts"], case["topk"]
        s["x"], s["out"] = _randn(gen, case["h"]), _empty(gen, case["h"])
        s["logits"], s["ids"] = _empty(gen, e, dtype=torch.float32), _empty(gen, k, dtype=torch.int32)
        s["gw"], s["act"] = _empty(gen, k), _empty(gen, k, case["inter"])
        s["scratch"] = torch.zeros(hip.MOE_DECODE_SCRATCH_WORDS, dtype=torch.int32, device=gen.device)
    elif kind == "head":
        b, n, h = case["batch"], case["n"], case["h"]
        s["w"], s["x"] = _weights(gen, n, h, case["bits"]), _randn(gen, b, h)
        s["logits"], s["ids"] = _empty(gen, b, n), _empty(gen, b, dtype=torch.int32)
        s["scratch"] = torch.zeros(hip.argmax_scratch_words(b), dtype=torch.int64, device=gen.device)
    elif kind == "sample":
        n = case["n"]
        # logits as a head gives them: a bulk and a tail of likely tokens
        bulk = 1.5 * torch.randn(n, device=gen.device, generator=gen)
        rare = torch.rand(n, device=gen.device, generator=gen) < 0.002
        tail = 6.0 * torch.rand(n, device=gen.device, generator=gen)
        s["logits"] = (bulk + rare * tail).to(torch.bfloat16)
        # a few hundred tokens already seen
        words = (n + 31) // 32
        bit = 1 << torch.randint(0, 31, (words,), device=gen.device, generator=gen)
        s["seen"] = (bit * (torch.rand(words, device=gen.device, generator=gen) < 0.1)).to(torch.int32)
        s["params"] = hip.sample_params(case["temperature"], seed, 17, case["penalty"], case["top_k"],
                                        case["top_p"])
        s["best"] = torch.zeros(1, dtype=torch.int64, device=gen.device)
        s["tok"] = _empty(gen, 1, dtype=torch.int32)
        s["ws_bytes"] = hip.sample_workspace_bytes(n)
        s["ws"] = torch.zeros(s["ws_bytes"], dtype=torch.uint8, device=gen.device)
    elif kind == "moe_prefill":
        s.update(_moe(case, gen))
        m = case["m"]
        s["x"], s["out"] = _randn(gen, m, case["h"]), _empty(gen, m, case["h"])
        s["ws_bytes"], _ = hip.moe_prefill_workspace(m, case["experts"], case["topk"], case["h"], case["inter"])
        s["ws"] = torch.empty(s["ws_bytes"], dtype=torch.uint8, device=gen.device)
    else:
        s["w"], s["x"] = _weights(gen, case["n"], case["k"], 4), _randn(gen, case["m"], case["k"])
        s["y"] = _empty(gen, case["m"], case["n"])
    return s


# -------------------------------------------------------------------- pass --

def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "conv_mixer":
        hip.conv3_gemv(s["w_in"], s["x"], s["taps"], s["conv_state"], s["mixed"], s["new_state"])
        hip.gemv_quant(s["w_out"], s["mixed"], s["y"])
        return {"mixed": s["mixed"], "new_state": s["new_state"], "y": s["y"]}
    if kind == "dense_ffn":
        hip.gemv_gu_act(s["gate"], s["up"], s["x"], s["act"])
        hip.gemv_quant(s["down"], s["act"], s["y"])
        return {"act": s["act"], "y": s["y"]}
    if kind == "moe_decode":
        hip.moe_decode(s["router"], s["bias"], s["gate"], s["up"], s["down"], c["experts"], c["topk"], s["x"],
                       s["out"], s["logits"], s["ids"], s["gw"], s["act"], s["scratch"], mode=c["mode"])
        return {"out": s["out"], "logits": s["logits"], "ids": s["ids"], "gw": s["gw"], "act": s["act"]}
    if kind == "head":
        hip.gemv_quant_argmax(s["w"], s["x"], s["logits"], s["scratch"], s["ids"], c["batch"])
        return {"logits": s["logits"], "ids": s["ids"]}
    if kind == "sample":
        hip.sample_draw(s["logits"], c["n"], s["seen"], s["params"], s["best"], s["ws"], s["ws_bytes"])
        hip.token_tail(s["best"], s["tok"])
        hip.sample_mark(s["tok"], s["seen"], c["n"])
        return {"tok": s["tok"], "seen": s["seen"]}
    if kind == "moe_prefill":
        hip.moe_prefill(s["router"], s["bias"], s["gate"], s["up"], s["down"], c["experts"], c["topk"], s["x"],
                        c["m"], s["out"], s["ws"], s["ws_bytes"], mode=c["mode"])
        return {"out": s["out"]}
    hip.gemm_q4_dense(s["x"], c["m"], s["w"], s["y"])
    return {"y": s["y"]}


# -------------------------------------------------------------------- work --

def _q_bytes(n, k, bits):
    return n * (k * bits // 8 + 4 * (k // GROUP))


def work(case):
    kind = case["kind"]
    if kind == "conv_mixer":
        h = case["h"]
        return {"bytes": _q_bytes(4 * h, h, 4) + 2 * h * (1 + 3 + 2 + 1 + 2 + 1), "flops": 8 * h * h}
    if kind == "dense_ffn":
        h, i = case["h"], case["inter"]
        return {"bytes": 2 * _q_bytes(i, h, 4) + _q_bytes(h, i, 4) + 2 * (2 * h + i), "flops": 6 * h * i}
    if kind in ("moe_decode", "moe_prefill"):
        e, k, h, i = case["experts"], case["topk"], case["h"], case["inter"]
        m = case.get("m", 1)
        hit = e * (1.0 - (1.0 - k / e) ** m)  # experts that some token chooses
        one = 2 * _q_bytes(i, h, 4) + _q_bytes(h, i, 4)
        router = e * h * (4 if case["router"] == "f32" else 2)
        return {"bytes": hit * one + router + 4 * m * h, "flops": m * (6 * k * h * i + 2 * e * h)}
    if kind == "head":
        n, h, b = case["n"], case["h"], case["batch"]
        return {"bytes": _q_bytes(n, h, case["bits"]) + 2 * b * (h + n) + 4 * b, "flops": 2 * b * n * h}
    if kind == "sample":
        return {"bytes": 2 * case["n"] + case["n"] // 8, "flops": 2 * case["n"]}
    m, n, k = case["m"], case["n"], case["k"]
    return {"bytes": _q_bytes(n, k, 4) + 2 * m * (n + k), "flops": 2 * m * n * k}


def tolerance(case):
    """About four times what the outputs differ from exact()'s: the bf16 store
    itself is 1.7e-3 (2-norm) and 3.9e-3 (half a unit of the last place); in
    the prefill's MoE block a stored intermediate that rounds the other way
    moves single outputs by up to 1.8e-2 of their root mean square."""
    kind = case["kind"]
    if kind == "sample":
        return "exact"
    if kind == "moe_prefill":
        return {"rel": 6e-3, "max": 7e-2}
    # the greedy ids (head) and the routed ids (moe_decode) are whole numbers
    return {"rel": 6e-3, "max": 1.6e-2, "differ": 0.0}


# ------------------------------------------------------- 64-bit references --

def _bf16(v):
    return v.to(torch.float32).to(torch.bfloat16).to(torch.float64)


def _codes(w):
    if w.bits == 4:
        sh = torch.arange(0, 32, 4, device=w.codes.device, dtype=torch.int32)
        return ((w.codes[:, :, None] >> sh) & 15).reshape(w.codes.shape[0], -1)
    by = w.codes.view(torch.uint8).to(torch.int32).reshape(w.codes.shape[0], -1, 3)
    v = by[:, :, 0] | (by[:, :, 1] << 8) | (by[:, :, 2] << 16)
    sh = torch.arange(0, 24, 6, device=w.codes.device, dtype=torch.int32)
    return ((v[:, :, None] >> sh) & 63).reshape(w.codes.shape[0], -1)


def _rows(w, lo=0, hi=None):
    """Rows lo..hi of s * q + b in 64 bits."""
    hi = w.codes.shape[0] if hi is None else hi
    part = hip.QuantWeights(w.codes[lo:hi], w.scales[lo:hi], w.biases[lo:hi], hi - lo, w.in_features, GROUP, w.bits)
    q = _codes(part).to(torch.float64).reshape(hi - lo, -1, GROUP)
    return (q * part.scales.double()[:, :, None] + part.biases.double()[:, :, None]).reshape(hi - lo, -1)


def _swiglu(g, u):
    return _bf16(_bf16(g / (1.0 + torch.exp(-g))) * u)


def _route(s, c, x):
    z = x @ s["router"].double().T
    if c["mode"] == 0:
        p = torch.sigmoid(z)
        ids = torch.topk(p + s["bias"].double(), c["topk"], dim=1).indices
        top = torch.gather(p, 1, ids)
        return z, ids, top / (1e-6 + top.sum(1, keepdim=True))
    top, ids = torch.topk(z, c["topk"], dim=1)
    return z, ids, torch.softmax(top, dim=1)


def exact(case, seed):
    """run()'s results in 64 bits, with the roundings to bf16 that the
    operators define between their steps (stored intermediates, and the
    weights that the matrix products of the prefill take as bf16)."""
    kind = case["kind"]
    if kind == "sample":
        return None
    s = prepare(case, seed)
    x = s["x"].double()
    if kind == "conv_mixer":
        h = case["h"]
        b, c, xx = _bf16(_rows(s["w_in"]) @ x).reshape(3, h)
        v = _bf16(b * xx)
        t, st = s["taps"].double(), s["conv_state"].double()
        mixed = c * _bf16(t[:, 0] * st[0] + t[:, 1] * st[1] + t[:, 2] * v)
        return {"mixed": mixed, "new_state": torch.stack([st[1], v]), "y": _rows(s["w_out"]) @ _bf16(mixed)}
    if kind == "dense_ffn":
        act = _swiglu(_bf16(_rows(s["gate"]) @ x), _bf16(_rows(s["up"]) @ x))
        return {"act": act, "y": _rows(s["down"]) @ act}
    if kind == "head":
        n = case["n"]
        z = torch.cat([x @ _rows(s["w"], lo, min(lo + 16384, n)).T for lo in range(0, n, 16384)], dim=1)
        return {"logits": z, "ids": _bf16(z).argmax(1).to(torch.int32)}
    if kind == "project":
        return {"y": x @ _bf16(_rows(s["w"])).T}
    e, h, i = case["experts"], case["h"], case["inter"]
    if kind == "moe_decode":
        z, ids, gw = _route(s, case, x[None])
        acts, out = [], 0.0
        for r, j in enumerate(ids[0].tolist()):
            act = _swiglu(_bf16(_rows(s["gate"], j * i, (j + 1) * i) @ x), _bf16(_rows(s["up"], j * i, (j + 1) * i) @ x))
            out = out + _bf16(_bf16(gw[0, r]) * _bf16(_rows(s["down"], j * h, (j + 1) * h) @ act))
            acts.append(act)
        return {"out": out, "logits": z[0], "ids": ids[0].to(torch.int32), "gw": gw[0], "act": torch.stack(acts)}
    _, ids, gw = _route(s, case, x)
    out, gw = torch.zeros_like(x), _bf16(gw)
    for j in range(e):
        tok, slot = (ids == j).nonzero(as_tuple=True)
        if tok.numel() == 0:
            continue
        xs = x[tok]
        g = _bf16(xs @ _bf16(_rows(s["gate"], j * i, (j + 1) * i)).T)
        u = _bf16(xs @ _bf16(_rows(s["up"], j * i, (j + 1) * i)).T)
        d = _bf16(_swiglu(g, u) @ _bf16(_rows(s["down"], j * h, (j + 1) * h)).T)
        out.index_add_(0, tok, _bf16(gw[tok, slot][:, None] * d))
    return {"out": out}
