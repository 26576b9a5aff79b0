"""Performance cases of the Qwen3-0.6B Q4 library: what its users run, over the sizes they run it at.

A case is one call of a public entry point (the drop-in functions of ``common`` and
``quantize``, the decoders of ``decode``, or the C ABI of ``include/q4dec.h``), with inputs
made on the GPU from a seed.  Weights are N(0, 0.03) matrices quantised by the Q4 rule
(one Q2.14 scale per 64 columns), K/V rows N(0, 1) in fp16, norm weights 1 + N(0, 0.1).
"""

import ctypes
import math

import numpy as np
import torch

from llm_accelerator_amd import _lib, common
from llm_accelerator_amd.decode import BatchedDecoder, Prefill
from llm_accelerator_amd.fixed import FixedKVCache, FixedQ4Model
from llm_accelerator_amd.model import (KVCache, Q4Tensor, Qwen3Config, Workspace, batched_step_bytes, build_model,
                                       current_stream, prefill_flops)
from llm_accelerator_amd.quantize import quantize_weight_q4

CFG = Qwen3Config()
H, I, D = CFG.hidden_size, CFG.intermediate_size, CFG.head_dim
QH, KVH, LAYERS, VOCAB = CFG.num_attention_heads, CFG.num_key_value_heads, CFG.num_hidden_layers, CFG.vocab_size
MATS = {"q_proj": (QH * D, H), "k_proj": (KVH * D, H), "v_proj": (KVH * D, H), "o_proj": (H, QH * D),
        "gate_proj": (I, H), "up_proj": (I, H), "down_proj": (H, I)}
PROJECTIONS = ("q_proj", "k_proj", "o_proj", "gate_proj", "down_proj")  # one of each shape


def listed():
    return [
        # one token's activations through one projection: the smallest call, all latency
        {"name": "linear_token", "op": "linear", "proj": "gate_proj", "rows": 1},
        # a prompt's activations through one projection in fp32 (the step-by-step validators)
        {"name": "linear_prompt", "op": "linear", "proj": "down_proj", "rows": 211},
        # the same contraction with fp16 activations, a long prompt
        {"name": "gemm_prompt", "op": "gemm", "proj": "gate_proj", "rows": 2000, "y": "f16"},
        # causal attention of two prompts
        {"name": "attention_prompt", "op": "attention_prompt", "batch": 2, "seq": 1500},
        # decode attention of a serving batch, every sequence at a position of its own
        {"name": "attention_cached", "op": "attention_cached", "batch": 24, "pos": 1500, "step": 37, "cap": 2048},
        # final norm, LM head and argmax of a serving batch
        {"name": "head_batch", "op": "head", "batch": 24},
        # one generated token of a chat: the whole model, batch 1
        {"name": "step_token", "op": "step", "pos": 1500, "cap": 4096},
        # one generated token for each of 16 users
        {"name": "step_batch", "op": "step_batch", "batch": 16, "pos": 1500, "step": 61, "cap": 2048},
        # a short chat prompt through the whole model
        {"name": "prefill_short", "op": "prefill", "n": 75, "start": 0},
        # a long document through the whole model
        {"name": "prefill_long", "op": "prefill", "n": 2048, "start": 0},
        # one token in the integer arithmetic of the hardware datapath
        {"name": "fixed_token", "op": "fixed", "pos": 700, "cap": 1024},
        # a checkpoint's largest matrix to Q4
        {"name": "quantize_table", "op": "quantize", "rows": VOCAB, "cols": H, "dtype": "bf16"},
    ]


def _log(rng, lo, hi):
    """An integer of [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _ragged(rng, cap_lo, cap_hi, tokens):
    """A batch of 1 .. 64 sequences at positions pos, pos - step, ... within ``tokens`` in all."""
    batch = _log(rng, 1, 64)
    cap = 64 * _log(rng, cap_lo // 64, max(cap_lo, min(cap_hi, tokens // batch)) // 64)
    pos = rng.randrange(cap // 4, cap)
    return {"batch": batch, "pos": pos, "step": rng.randrange(0, pos // batch + 1), "cap": cap}


def draw(rng):
    op = rng.choice(("linear", "gemm", "attention_prompt", "attention_cached", "head", "step", "step_batch",
                     "prefill", "fixed", "quantize"))
    if op == "linear":
        return {"op": op, "proj": rng.choice(PROJECTIONS), "rows": _log(rng, 1, 1024)}
    if op == "gemm":
        return {"op": op, "proj": rng.choice(PROJECTIONS), "rows": _log(rng, 1, 2048),
                "y": rng.choice(("f16", "f32", "resid"))}
    if op == "attention_prompt":
        batch = _log(rng, 1, 8)
        return {"op": op, "batch": batch, "seq": _log(rng, 1, int(3000 / math.sqrt(batch)))}
    if op == "attention_cached":
        return {"op": op, **_ragged(rng, 64, 8192, 131072)}
    if op == "head":
        return {"op": op, "batch": _log(rng, 1, 64)}
    if op == "step":
        cap = 64 * _log(rng, 4, 128)
        return {"op": op, "pos": rng.randrange(0, cap), "cap": cap}
    if op == "step_batch":
        return {"op": op, **_ragged(rng, 256, 4096, 65536)}
    if op == "prefill":
        start = rng.choice((0, 0, rng.randrange(1, 1500)))
        return {"op": op, "n": _log(rng, 1, 1024 if start else 2048), "start": start}
    if op == "fixed":
        cap = 64 * _log(rng, 4, 32)
        return {"op": op, "pos": rng.randrange(0, cap), "cap": cap}
    return {"op": op, "rows": _log(rng, 64, 50000), "cols": rng.choice((1024, 2048, 3072)),
            "dtype": rng.choice(("bf16", "f32"))}


# ---------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device="cuda")


def _q4(g, rows, cols):
    """(packed, scale code) of a quantised N(0, 0.03) matrix, on the GPU."""
    packed, codes = [], []
    for r0 in range(0, rows, 16384):
        w = _randn(g, min(16384, rows - r0), cols // 64, 64) * 0.03
        code = torch.clamp(torch.round(w.abs().amax(-1) * (16384.0 / 7)), min=1)
        q = torch.clamp(torch.round(w * (16384.0 / code)[..., None]), -8, 7).to(torch.int16).reshape(len(w), cols) & 15
        packed.append((q[:, 0::2] | (q[:, 1::2] << 4)).to(torch.uint8))
        codes.append(code.to(torch.int16))
    return torch.cat(packed), torch.cat(codes)


def _weight(g, rows, cols):
    packed, code = _q4(g, rows, cols)
    return Q4Tensor(packed, code.view(torch.uint16))


def _host_q4(g, rows, cols):
    packed, code = _q4(g, rows, cols)
    return packed.cpu().numpy(), code.cpu().numpy().view(np.uint16)


def _gamma(g, n):
    return (1 + 0.1 * _randn(g, n)).cpu().numpy()


def _host_weights(g, layers):
    out = []
    for _ in range(layers):
        L = {n: _host_q4(g, *s) for n, s in MATS.items()}
        for n, k in (("input_layernorm", H), ("post_attention_layernorm", H), ("q_norm", D), ("k_norm", D)):
            L[n] = _gamma(g, k)
        out.append(L)
    return {"layers": out, "embed_tokens": _host_q4(g, VOCAB, H), "norm": _gamma(g, H)}


def _model(g, layers, max_ctx):
    """(device model, host weights)"""
    host = _host_weights(g, layers)
    cfg = Qwen3Config(num_hidden_layers=layers)
    return build_model(cfg, host, max_ctx), host


def _tokens(g, n):
    return torch.randint(0, VOCAB, (n,), generator=g, device="cuda", dtype=torch.int32)


def _positions(case):
    return [case["pos"] - b * case["step"] for b in range(case["batch"])]


def _cache(g, layers, batch, cap):
    kv = KVCache(CFG, layers, batch, cap)
    for plane in kv.data:
        plane.normal_(generator=g)
    return kv


def _new_rows(data, case):
    """The K/V rows a step writes: [layers, 2, batch, kv heads, head dim], sequence b at position pos - step b."""
    s = data.stride()
    return data.as_strided(data.shape[:4] + data.shape[5:], (s[0], s[1], s[2] - case.get("step", 0) * s[4], s[3], s[5]),
                           data.storage_offset() + case["pos"] * s[4])


def prepare(case, seed):
    g = _gen(seed)
    op = case["op"]
    if op == "linear":
        rows, cols = MATS[case["proj"]]
        return {"op": op, "w": _weight(g, rows, cols), "x": _randn(g, 1, case["rows"], cols)}
    if op == "gemm":
        rows, cols = MATS[case["proj"]]
        m, w = case["rows"], _weight(g, rows, cols)
        f16 = case["y"] == "f16"
        return {"op": op, "w": w, "desc": w.descriptor(), "x": _randn(g, m, cols).half(), "m": m,
                "y": torch.empty(m, rows, dtype=torch.float16 if f16 else torch.float32, device="cuda"),
                "dtype": _lib.Q4D_F16 if f16 else _lib.Q4D_F32,
                "resid": _randn(g, m, rows) if case["y"] == "resid" else None}
    if op == "attention_prompt":
        b, s = case["batch"], case["seq"]
        return {"op": op, "q": _randn(g, b, QH, s, D), "k": _randn(g, b, KVH, s, D), "v": _randn(g, b, KVH, s, D)}
    if op == "quantize":
        w = _randn(g, case["rows"], case["cols"]) * 0.03
        return {"op": op, "w": w.bfloat16() if case["dtype"] == "bf16" else w}

    if op == "attention_cached":
        b = case["batch"]
        model, _ = _model(g, 1, case["cap"])
        kv = _cache(g, 1, b, case["cap"])
        return {"op": op, "model": model, "desc": model.descriptor(), "kv": kv, "kvd": kv.descriptor(),
                "ws": Workspace(model, b), "q": _randn(g, b, QH, D),
                "pos": torch.tensor(_positions(case), dtype=torch.int32, device="cuda"),
                "out": torch.empty(b, QH * D, device="cuda")}
    if op == "head":
        b = case["batch"]
        model, _ = _model(g, 1, 64)
        return {"op": op, "model": model, "desc": model.descriptor(), "ws": Workspace(model, b), "batch": b,
                "hidden": 3 * _randn(g, b, H), "token": torch.zeros(b, dtype=torch.int32, device="cuda"),
                "score": torch.zeros(b, device="cuda"), "logits": torch.empty(b, VOCAB, device="cuda")}
    if op == "step":
        model, _ = _model(g, LAYERS, case["cap"])
        kv = _cache(g, LAYERS, 1, case["cap"])
        return {"op": op, "model": model, "desc": model.descriptor(), "kv": kv, "kvd": kv.descriptor(),
                "ws": Workspace(model, 1), "tok": _tokens(g, 1),
                "pos": torch.tensor([case["pos"]], dtype=torch.int32, device="cuda"),
                "next": torch.zeros(1, dtype=torch.int32, device="cuda"), "score": torch.zeros(1, device="cuda"),
                "logits": torch.empty(VOCAB, device="cuda"), "new": _new_rows(kv.data, case)}
    if op == "step_batch":
        b = case["batch"]
        model, _ = _model(g, LAYERS, case["cap"])
        kv = _cache(g, LAYERS, b, case["cap"])
        return {"op": op, "dec": BatchedDecoder(model, b, kv), "tok": _tokens(g, b),
                "pos": torch.tensor(_positions(case), dtype=torch.int32, device="cuda"),
                "logits": torch.empty(b, VOCAB, device="cuda"), "new": _new_rows(kv.data, case)}
    if op == "prefill":
        n, start = case["n"], case["start"]
        cap = 64 * -(-(n + start + 64) // 64)
        model, _ = _model(g, LAYERS, cap)
        kv = _cache(g, LAYERS, 1, cap)
        return {"op": op, "run": Prefill(model, kv, n), "tok": _tokens(g, n), "start": start,
                "next": torch.zeros(1, dtype=torch.int32, device="cuda"), "score": torch.zeros(1, device="cuda"),
                "logits": torch.empty(VOCAB, device="cuda"), "new": kv.data[:, :, 0, :, start:start + n]}
    model, host = _model(g, LAYERS, case["cap"])
    fixed = FixedQ4Model(model, host)
    kv = FixedKVCache(LAYERS, KVH, case["cap"])
    for plane in kv.data:
        plane.copy_(_randn(g, *plane.shape) * 4096)
    return {"op": op, "fixed": fixed, "kv": kv, "tok": _tokens(g, 1),
            "pos": torch.tensor([case["pos"]], dtype=torch.int32, device="cuda"),
            "new": kv.data[:, :, :, case["pos"]]}


# ---------------------------------------------------------------- one pass
def run(state):
    s, op = state, state["op"]
    if op == "linear":
        return common.manual_linear_from_weight(s["x"], s["w"])
    if op == "attention_prompt":
        return common.manual_causal_attention(s["q"], common.manual_repeat_kv(s["k"], QH // KVH),
                                              common.manual_repeat_kv(s["v"], QH // KVH), CFG.scaling)[0]
    if op == "quantize":
        return quantize_weight_q4(s["w"], return_codes=False)
    if op == "step_batch":
        _, score = s["dec"].step(s["tok"], s["pos"], s["logits"])
        return {"logits": s["logits"], "score": score, "kv": s["new"]}
    if op == "prefill":
        _, score = s["run"].run(s["tok"], start_pos=s["start"], next_token=s["next"], score=s["score"],
                                logits=s["logits"])
        return {"logits": s["logits"], "score": score, "kv": s["new"]}
    if op == "fixed":
        token, score, logits, hidden = s["fixed"].run_one_token(s["tok"], s["pos"], s["kv"], want_logits=True)
        return {"token": token, "score": score, "logits": logits, "hidden": hidden, "kv": s["new"]}
    lib = _lib.load()
    if op == "gemm":
        _lib.check(lib.q4d_gemm(ctypes.byref(s["desc"]), s["x"].data_ptr(), s["m"], s["y"].data_ptr(), s["dtype"],
                                s["resid"].data_ptr() if s["resid"] is not None else None, current_stream()),
                   "q4d_gemm")
        return s["y"]
    ws = s["ws"]
    if op == "attention_cached":
        _lib.check(lib.q4d_cached_attention(ctypes.byref(s["desc"]), ctypes.byref(s["kvd"]), 0, s["q"].data_ptr(),
                                            s["pos"].data_ptr(), s["out"].data_ptr(), _lib.Q4D_F32, ws.ptr,
                                            ws.nbytes, current_stream()), "q4d_cached_attention")
        return s["out"]
    if op == "head":
        _lib.check(lib.q4d_lm_head_argmax_batch(ctypes.byref(s["desc"]), s["hidden"].data_ptr(), s["batch"],
                                                s["token"].data_ptr(), s["score"].data_ptr(),
                                                s["logits"].data_ptr(), ws.ptr, ws.nbytes, current_stream()),
                   "q4d_lm_head_argmax_batch")
        return {"logits": s["logits"], "score": s["score"]}
    _lib.check(lib.q4d_run_one_token(ctypes.byref(s["desc"]), s["tok"].data_ptr(), s["pos"].data_ptr(),
                                     ctypes.byref(s["kvd"]), s["next"].data_ptr(), s["score"].data_ptr(),
                                     s["logits"].data_ptr(), ws.ptr, ws.nbytes, current_stream()),
               "q4d_run_one_token")
    return {"logits": s["logits"], "score": s["score"], "kv": s["new"]}


# ---------------------------------------------------------------- what a pass cannot do without
def _matrix_bytes(rows, cols):
    return rows * cols // 2 + 2 * rows * (cols // 64)


LAYER_WEIGHTS = sum(r * c for r, c in MATS.values())
LAYER_BYTES = sum(_matrix_bytes(r, c) for r, c in MATS.values())


def work(case):
    op = case["op"]
    if op in ("linear", "gemm"):
        rows, cols = MATS[case["proj"]]
        m = case["rows"]
        xb, yb = (4, 4) if op == "linear" else (2, {"f16": 2, "f32": 4, "resid": 8}[case["y"]])
        return {"bytes": _matrix_bytes(rows, cols) + m * (cols * xb + rows * yb), "flops": 2 * m * rows * cols}
    if op == "attention_prompt":
        b, s = case["batch"], case["seq"]
        return {"bytes": 4 * b * s * D * (2 * QH + 2 * KVH), "flops": 4 * D * QH * b * (s * (s + 1) // 2)}
    if op == "attention_cached":
        t = sum(p + 1 for p in _positions(case))
        return {"bytes": t * 2 * KVH * D * 2 + case["batch"] * QH * D * 8, "flops": 4 * D * QH * t}
    if op == "head":
        b = case["batch"]
        return {"bytes": _matrix_bytes(VOCAB, H) + 4 * b * (H + VOCAB), "flops": 2 * b * VOCAB * H}
    if op in ("step", "step_batch"):
        pos = _positions(case) if op == "step_batch" else [case["pos"]]
        t, b = sum(p + 1 for p in pos), len(pos)
        return {"bytes": batched_step_bytes(CFG, 1, t) + 4 * b * VOCAB,
                "flops": 2 * b * (LAYERS * LAYER_WEIGHTS + VOCAB * H) + 4 * D * QH * LAYERS * t}
    if op == "prefill":
        n, s0 = case["n"], case["start"]
        return {"bytes": LAYERS * LAYER_BYTES + _matrix_bytes(VOCAB, H) + LAYERS * 2 * KVH * D * 2 * (n + s0) +
                4 * VOCAB, "flops": prefill_flops(CFG, n) + 4 * D * QH * LAYERS * n * s0}
    if op == "fixed":
        return {"bytes": LAYERS * (LAYER_BYTES + 2 * KVH * D * 4 * (case["pos"] + 1)) + _matrix_bytes(VOCAB, H) +
                8 * VOCAB, "flops": 2 * (LAYERS * LAYER_WEIGHTS + VOCAB * H) + 4 * D * QH * LAYERS * (case["pos"] + 1)}
    n = case["rows"] * case["cols"]
    return {"bytes": n * (2 if case["dtype"] == "bf16" else 4) + _matrix_bytes(case["rows"], case["cols"]), "flops": 4 * n}


def tolerance(case):
    """About four times the distance from the 64-bit values that the data types give: fp32 sums (linear,
    attention_cached), weights and activations rounded to fp16 once (gemm, head, attention_prompt), fp16 K/V
    (step), and fp16 activations through all layers (step_batch, prefill)."""
    return {
        "linear": {"rel": 3e-5, "max": 3e-4},
        "gemm": {"rel": 1e-3, "max": 1e-2},
        "attention_prompt": {"rel": 2e-3, "max": 3e-2},
        "attention_cached": {"rel": 1e-6, "max": 1e-5},
        "head": {"rel": 1e-3, "max": 1e-2},
        "step": {"rel": 1.2e-3, "max": 1.2e-2},
        "step_batch": {"rel": 1.2e-2, "max": 1.2e-1},
        "prefill": {"rel": 8e-3, "max": 1.2e-1},
    }.get(case["op"], "exact")


# ---------------------------------------------------------------- the same values in 64 bits
def _dense(packed, code):
    """A Q4 matrix as float64 on the GPU."""
    packed = torch.as_tensor(packed, device="cuda")
    code = torch.as_tensor(np.asarray(code).astype(np.int64) if isinstance(code, np.ndarray) else code.to(torch.int64),
                           device="cuda")
    q = torch.stack([packed & 15, packed >> 4], dim=-1).reshape(packed.shape[0], -1).to(torch.int8)
    q = torch.where(q >= 8, q - 16, q).double().reshape(len(q), -1, 64)
    return (q * (code.double() / 16384)[..., None]).reshape(len(q), -1)


def _matmul(x, packed, code):
    out = torch.empty(len(x), len(packed), dtype=torch.float64, device="cuda")
    for r0 in range(0, len(packed), 16384):
        out[:, r0:r0 + 16384] = x @ _dense(packed[r0:r0 + 16384], code[r0:r0 + 16384]).t().contiguous()
    return out


def _rms(x, gamma):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + CFG.rms_norm_eps) * torch.as_tensor(gamma, device="cuda").double()


def _rope(x, pos):
    """x [tokens, heads, D] at positions pos [tokens]; the angles in fp32, as the model's tables hold them."""
    inv = 1.0 / (CFG.rope_theta ** (torch.arange(0, D, 2, dtype=torch.int64).float() / D))
    f = (pos.cpu().float()[:, None] * inv[None, :].float()).to("cuda")
    c, s = f.cos().double()[:, None], f.sin().double()[:, None]
    a, b = x[..., :D // 2], x[..., D // 2:]
    return torch.cat([a * c - b * s, b * c + a * s], dim=-1)


def _attend(q, k, v, visible):
    """q [n, QH, D], k, v [KVH, t, D]; visible [n, t] or None."""
    out = torch.empty_like(q)
    for h in range(QH):
        s = (q[:, h] @ k[h // 2].t().contiguous()) * CFG.scaling
        if visible is not None:
            s = s.masked_fill(~visible, -math.inf)
        out[:, h] = torch.softmax(s, dim=-1) @ v[h // 2]
    return out


def _exact_layers(host, tokens, seqs):
    """All layers over the tokens of ``seqs``: per sequence (rows of its tokens, positions, K/V cache of layer l).
    Returns (hidden, new K/V rows [layers, 2, tokens, KVH, D])."""
    packed, code = host["embed_tokens"]
    idx = tokens.cpu().long().numpy()
    x = _dense(packed[idx], code[idx])
    new = []
    for l, L in enumerate(host["layers"]):
        h = _rms(x, L["input_layernorm"])
        q, k, v = (_matmul(h, *L[n]).reshape(len(x), -1, D) for n in ("q_proj", "k_proj", "v_proj"))
        pos = torch.cat([p for _, p, _ in seqs])
        q, k = _rope(_rms(q, L["q_norm"]), pos), _rope(_rms(k, L["k_norm"]), pos)
        new.append(torch.stack([k, v]))
        att = torch.empty_like(q)
        for rows, p, cache in seqs:
            first = int(p[0])
            kk, vv = (torch.cat([cache[l, i, :, :first].double(), t[rows].transpose(0, 1)], dim=1)
                      for i, t in enumerate((k, v)))
            visible = None if len(p) == 1 else torch.arange(kk.shape[1], device="cuda")[None, :] <= p[:, None]
            att[rows] = _attend(q[rows], kk, vv, visible)
        x = x + _matmul(att.reshape(len(x), -1), *L["o_proj"])
        h = _rms(x, L["post_attention_layernorm"])
        a = torch.nn.functional.silu(_matmul(h, *L["gate_proj"])) * _matmul(h, *L["up_proj"])
        x = x + _matmul(a, *L["down_proj"])
    return x, torch.stack(new)


def exact(case, seed):
    g = _gen(seed)
    op = case["op"]
    if op in ("linear", "gemm"):
        rows, cols = MATS[case["proj"]]
        w = _q4(g, rows, cols)
        if op == "linear":
            return _matmul(_randn(g, 1, case["rows"], cols)[0].double(), *w)[None]
        y = _matmul(_randn(g, case["rows"], cols).half().double(), *w)
        return y + _randn(g, case["rows"], rows).double() if case["y"] == "resid" else y
    if op == "attention_prompt":
        b, s = case["batch"], case["seq"]
        q, k, v = (_randn(g, b, n, s, D).double() for n in (QH, KVH, KVH))
        t = torch.arange(s, device="cuda")
        return torch.stack([_attend(q[i].transpose(0, 1).contiguous(), k[i], v[i], t[None, :] <= t[:, None]).transpose(0, 1)
                            for i in range(b)])
    if op in ("quantize", "fixed"):
        return None  # whole numbers
    layers = 1 if op in ("attention_cached", "head") else LAYERS
    host = _host_weights(g, layers)
    if op == "attention_cached":
        kv = _cache(g, 1, case["batch"], case["cap"]).data[0]
        q = _randn(g, case["batch"], QH, D).double()
        return torch.cat([_attend(q[b:b + 1], kv[0, b, :, :p + 1].double(), kv[1, b, :, :p + 1].double(), None)
                          for b, p in enumerate(_positions(case))]).reshape(case["batch"], -1)
    if op == "head":
        logits = _matmul(_rms(3 * _randn(g, case["batch"], H).double(), host["norm"]), *host["embed_tokens"])
        return {"logits": logits, "score": logits.amax(-1)}
    if op == "prefill":
        n, start = case["n"], case["start"]
        kv = _cache(g, LAYERS, 1, 64 * -(-(n + start + 64) // 64)).data
        tokens = _tokens(g, n)
        x, new = _exact_layers(host, tokens, [(slice(0, n), torch.arange(start, start + n, device="cuda"), kv[:, :, 0])])
        logits = _matmul(_rms(x[-1:], host["norm"]), *host["embed_tokens"])[0]
        return {"logits": logits, "score": logits.amax().reshape(1), "kv": new.transpose(2, 3)}
    pos = _positions(case) if op == "step_batch" else [case["pos"]]
    kv = _cache(g, LAYERS, len(pos), case["cap"]).data
    tokens = _tokens(g, len(pos))
    x, new = _exact_layers(host, tokens, [(slice(b, b + 1), torch.tensor([p], device="cuda"), kv[:, :, b])
                                          for b, p in enumerate(pos)])
    logits = _matmul(_rms(x, host["norm"]), *host["embed_tokens"])
    if op == "step":
        return {"logits": logits[0], "score": logits[0].amax().reshape(1), "kv": new}
    return {"logits": logits, "score": logits.amax(-1), "kv": new}
