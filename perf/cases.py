"""Performance cases of the RWKV-7 inference path.

Each case is one call that a serving program makes, from a one-row decode
product to a batch prefill, with the sizes of this repository's models: the
0.1B architecture (hidden 768), the 1.5B and 2.9B widths (2048, 2560) and the
7.2B width (4096, FFN 16384, 64 heads, vocabulary 65536).

``listed()`` gives the fixed cases, ``draw(rng)`` one more of the same ranges,
``prepare`` the inputs and handles, ``run`` one pass, ``exact`` the pass in
64-bit torch without this package, ``work`` the bytes and operations that a
pass cannot do without, ``tolerance`` the error bound of its results.
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

if str(Path.cwd() / "hf-adapter_amd") not in sys.path:
    sys.path.insert(0, str(Path.cwd() / "hf-adapter_amd"))

DEV = "cuda"
VOCAB = 65536
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}
RANKS = (64, 64, 128, 32)  # W, A, G, V LoRA ranks of every width here


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # One token of a single chat through a 7.2B MM8 feed-forward block:
        # latency, launches and the weight stream.
        {"name": "mm8_ffn_decode_1", "kind": "mm8_ffn", "rows": 1, "hidden": 4096, "ffn": 16384, "dtype": "fp16"},
        # The same block with 16 chats decoding together.
        {"name": "mm8_ffn_decode_16", "kind": "mm8_ffn", "rows": 16, "hidden": 4096, "ffn": 16384, "dtype": "fp16"},
        # A short prompt (a ragged 200 tokens) through a 1.5B block, bf16.
        {"name": "mm8_ffn_prompt_200", "kind": "mm8_ffn", "rows": 200, "hidden": 2048, "ffn": 8192, "dtype": "bf16"},
        # An ordinary prompt of 1000 tokens through a 7.2B block.
        {"name": "mm8_ffn_prompt_1000", "kind": "mm8_ffn", "rows": 1000, "hidden": 4096, "ffn": 16384, "dtype": "fp16"},
        # A prefill batch of 4 x 4096 tokens: the largest product.
        {"name": "mm8_ffn_batch_16384", "kind": "mm8_ffn", "rows": 16384, "hidden": 4096, "ffn": 16384,
         "dtype": "fp16"},
        # The vocabulary head in min/max affine 4-bit (group 128), 4 chats decoding.
        {"name": "w4_head_decode_4", "kind": "w4", "rows": 4, "inputs": 4096, "outputs": VOCAB, "affine": True,
         "dtype": "fp16"},
        # A 384-token prompt through the FFN key in symmetric 4-bit (group 128).
        {"name": "w4_key_prompt_384", "kind": "w4", "rows": 384, "inputs": 4096, "outputs": 16384, "affine": False,
         "dtype": "fp16"},
        # The recurrence of one 1000-token prompt (ragged: not a multiple of the chunk).
        {"name": "scan_prompt_1x1000", "kind": "scan", "batch": 1, "tokens": 1000, "heads": 32, "dtype": "fp16"},
        # The recurrence of a prefill batch at the 7.2B head count.
        {"name": "scan_batch_8x4096", "kind": "scan", "batch": 8, "tokens": 4096, "heads": 64, "dtype": "fp16"},
        # The W/A/G/V LoRA projections of a 700-token prompt at the 7.2B width.
        {"name": "lora_prompt_700", "kind": "lora", "rows": 700, "hidden": 4096, "dtype": "fp16"},
        # A chat turn on the whole 0.1B model (fp16, unquantised): prompt, then
        # decode steps on the captured graph.  Small kernels: launches count.
        {"name": "chat_0p1b", "kind": "chat", "layers": 12, "hidden": 768, "mm8": False, "batch": 1, "prompt": 512,
         "steps": 8},
        # A chat turn on two layers of the 7.2B MM8 model with its head.
        {"name": "chat_7p2b_2l", "kind": "chat", "layers": 2, "hidden": 4096, "mm8": True, "batch": 2, "prompt": 300,
         "steps": 8},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["mm8_ffn", "mm8_ffn", "w4", "scan", "lora", "chat"])
    if kind == "mm8_ffn":
        hidden = rng.choice([2048, 2560, 4096])
        return {"kind": kind, "rows": _log_int(rng, 1, 16000), "hidden": hidden, "ffn": 4 * hidden,
                "dtype": rng.choice(["fp16", "fp16", "bf16"])}
    if kind == "w4":
        n, m = rng.choice([(4096, 4096), (4096, 16384), (16384, 4096), (4096, VOCAB)])
        # only last tokens reach the vocabulary head: decode rows
        return {"kind": kind, "rows": _log_int(rng, 1, 16 if m == VOCAB else 1000), "inputs": n, "outputs": m,
                "affine": rng.random() < 0.5, "dtype": rng.choice(["fp16", "fp16", "bf16"])}
    if kind == "scan":
        return {"kind": kind, "batch": rng.randint(1, 8), "tokens": _log_int(rng, 16, 4000),
                "heads": rng.choice([12, 32, 40, 64]), "dtype": rng.choice(["fp16", "fp16", "bf16"])}
    if kind == "lora":
        return {"kind": kind, "rows": _log_int(rng, 1, 16000), "hidden": rng.choice([768, 2048, 2560, 4096]),
                "dtype": rng.choice(["fp16", "fp16", "bf16"])}
    small = rng.random() < 0.5
    return {"kind": kind, "layers": 12 if small else 2, "hidden": 768 if small else 4096, "mm8": not small,
            "batch": rng.randint(1, 8), "prompt": _log_int(rng, 16, 512), "steps": rng.randint(2, 12)}


# ------------------------------------------------------------------ inputs
def _gen(seed, salt):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 1000003 + salt) & 0x7FFFFFFF)
    return g


def _randn(gen, *shape, scale=1.0, dtype=torch.float32):
    return (torch.randn(*shape, generator=gen, device=DEV) * scale).to(dtype)


def _mm8_weight(gen, n, m, dtype):
    """A packed MM8 weight [n inputs, m outputs] whose dequantised values
    (w + 0.5) ry rx + my + mx are about N(0, 0.02): the bytes and the four
    scale vectors as a prepacked checkpoint holds them."""
    u8 = torch.empty(n, m, device=DEV, dtype=torch.uint8)
    for r in range(0, n, 4096):
        blk = torch.randn(min(4096, n - r), m, generator=gen, device=DEV, dtype=torch.float16)
        u8[r:r + 4096] = blk.mul_(32).add_(128).round_().clamp_(0, 255).to(torch.uint8)
    s = math.sqrt(0.02 / 32)
    a = 0.05 * torch.randn(n, generator=gen, device=DEV)
    b = 0.05 * torch.randn(m, generator=gen, device=DEV)
    ry, rx = s * (1 + a), s * (1 + b)
    my, mx = -128.5 * s * s * (0.5 + a), -128.5 * s * s * (0.5 + b)
    return u8, mx.to(dtype), rx.to(dtype), my.reshape(n, 1).to(dtype), ry.reshape(n, 1).to(dtype)


def _mm8_dense(packed):
    """The weight [n, m] that the packed form stands for, in 64 bits."""
    u8, mx, rx, my, ry = packed
    w = u8.double().add_(0.5).mul_(ry.double()).mul_(rx.double())
    return w.add_(my.double()).add_(mx.double())


def _mm8_module(packed):
    from rwkv7mi.native_quant_mm8 import MM8Linear, mm8_block

    u8, mx, rx, my, ry = packed
    n, m = (int(s) for s in u8.shape)
    return MM8Linear.from_packed(mm8_block(u8), mx, rx, my, ry, n, m)


def _ffn_inputs(case, seed):
    dt, d, f = DTYPES[case["dtype"]], case["hidden"], case["ffn"]
    g = _gen(seed, 1)
    return {"x": _randn(g, case["rows"], d, dtype=dt), "residual": _randn(g, case["rows"], d, dtype=dt),
            "key": _mm8_weight(g, d, f, dt), "value": _mm8_weight(g, f, d, dt)}


def _w4_inputs(case, seed):
    dt, n, m = DTYPES[case["dtype"]], case["inputs"], case["outputs"]
    g = _gen(seed, 2)
    q = torch.empty(m, n // 2, device=DEV, dtype=torch.uint8)
    for r in range(0, m, 8192):  # nibbles of a normal weight: about +-3 sigma over the 16 codes
        c = torch.randn(min(8192, m - r), n, generator=g, device=DEV, dtype=torch.float16)
        c = c.mul_(2.6).add_(8 if not case["affine"] else 7.5).round_().clamp_(0, 15).to(torch.uint8)
        q[r:r + 8192] = c[:, 0::2] | (c[:, 1::2] << 4)
    scales = (0.0077 * (1 + 0.1 * torch.randn(m, n // 128, generator=g, device=DEV))).to(dt)
    out = {"x": _randn(g, case["rows"], n, dtype=dt), "q": q, "scales": scales}
    if case["affine"]:
        out["biases"] = (-7.5 * scales.float() + 0.002 * torch.randn(m, n // 128, generator=g, device=DEV)).to(dt)
    return out


def _scan_inputs(case, seed):
    dt = DTYPES[case["dtype"]]
    shape = (case["batch"], case["tokens"], case["heads"], 64)
    g = _gen(seed, 3)
    k = torch.nn.functional.normalize(torch.randn(*shape, generator=g, device=DEV), dim=-1)
    return {"r": _randn(g, *shape, dtype=dt),
            "w": torch.exp(-torch.exp(-0.5 + 0.5 * torch.randn(*shape, generator=g, device=DEV))),
            "k": k.to(dt), "v": _randn(g, *shape, dtype=dt), "kk": k.to(dt),
            "a": torch.sigmoid(torch.randn(*shape, generator=g, device=DEV)).to(dt),
            "state": _randn(g, case["batch"], case["heads"], 64, 64, scale=0.1)}


def _lora_inputs(case, seed):
    dt, d, rows = DTYPES[case["dtype"]], case["hidden"], case["rows"]
    g = _gen(seed, 4)
    return {"xs": [_randn(g, rows, d, dtype=dt) for _ in RANKS],
            "downs": [_randn(g, r, d, scale=0.02, dtype=dt) for r in RANKS],
            "ups": [_randn(g, d, r, scale=0.02, dtype=dt) for r in RANKS],
            "biases": [None if p == 2 else _randn(g, d, scale=0.01, dtype=dt) for p in range(4)]}


def _chat_inputs(case, seed):
    """The named weights of the model (a converted checkpoint's names) in fp16,
    its packed MM8 projections, and the token ids of the turn."""
    d, f, layers, dt = case["hidden"], 4 * case["hidden"], case["layers"], torch.float16
    g = _gen(seed, 5)
    w, packed = {}, {}

    def linear(name, out, inp):
        if case["mm8"]:
            packed[name] = _mm8_weight(g, inp, out, dt)
        else:
            w[name + ".weight"] = _randn(g, out, inp, scale=0.02, dtype=dt)

    def norm(name):
        w[name + ".weight"] = (1 + 0.1 * torch.randn(d, generator=g, device=DEV)).to(dt)
        w[name + ".bias"] = _randn(g, d, scale=0.02, dtype=dt)

    w["model.embeddings.weight"] = _randn(g, VOCAB, d, dtype=dt)
    for i in range(layers):
        p = f"model.layers.{i}."
        for n in (["pre_norm"] if i == 0 else []) + ["attn_norm", "ffn_norm", "attn.g_norm"]:
            norm(p + n)
        for n in ("x_r", "x_w", "x_k", "x_v", "x_a", "x_g"):
            w[p + "attn." + n] = torch.rand(1, 1, d, generator=g, device=DEV).to(dt)
        w[p + "ffn.x_k"] = torch.rand(d, generator=g, device=DEV).to(dt)
        w[p + "attn.k_k"] = (0.85 + 0.1 * torch.randn(d, generator=g, device=DEV)).to(dt)
        w[p + "attn.k_a"] = (1 + 0.1 * torch.randn(d, generator=g, device=DEV)).to(dt)
        w[p + "attn.r_k"] = _randn(g, d // 64, 64, scale=0.1, dtype=dt)
        for n, r in zip("wagv", RANKS):
            if n == "v" and i == 0:
                continue
            w[p + f"attn.{n}_lora.lora.0.weight"] = _randn(g, r, d, scale=0.02, dtype=dt)
            w[p + f"attn.{n}_lora.lora.2.weight"] = _randn(g, d, r, scale=0.02, dtype=dt)
            if n != "g":
                w[p + f"attn.{n}_lora.lora.2.bias"] = _randn(g, d, scale=0.01, dtype=dt)
        for n in ("r", "k", "v", "o"):
            linear(p + f"attn.{n}_proj", d, d)
        linear(p + "ffn.key", f, d)
        linear(p + "ffn.value", d, f)
    norm("model.norm")
    linear("lm_head", VOCAB, d)
    ids = torch.randint(0, VOCAB, (case["batch"], case["prompt"] + case["steps"]), generator=g, device=DEV)
    return {"weights": w, "packed": packed, "ids": ids}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "mm8_ffn":
        s = _ffn_inputs(case, seed)
        s["key"], s["value"] = _mm8_module(s["key"]), _mm8_module(s["value"])
    elif kind == "w4":
        s = _w4_inputs(case, seed)
    elif kind == "scan":
        s = _scan_inputs(case, seed)
    elif kind == "lora":
        s = _lora_inputs(case, seed)
    else:
        from rwkv7mi.model import NativeRWKV7Config, NativeRWKV7ForCausalLM

        inp = _chat_inputs(case, seed)
        cfg = NativeRWKV7Config(vocab_size=VOCAB, hidden_size=case["hidden"], num_hidden_layers=case["layers"],
                                intermediate_size=4 * case["hidden"], decay_low_rank_dim=RANKS[0],
                                a_low_rank_dim=RANKS[1], gate_low_rank_dim=RANKS[2], v_low_rank_dim=RANKS[3],
                                use_native_mm8=case["mm8"])
        model = NativeRWKV7ForCausalLM(cfg, inp["weights"], device=DEV, dtype=torch.float16,
                                       prepacked={n: _mm8_module(p) for n, p in inp["packed"].items()})
        model.graph_runner(case["batch"])  # a server captures its decode step once
        s = {"model": model, "ids": inp["ids"]}
    s["case"] = case
    return s


# ------------------------------------------------------------------ the pass
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "mm8_ffn":
        return s["key"].rwkv7_forward_ffn(s["x"], s["value"], s["residual"])
    if kind == "w4":
        from rwkv7mi.sm70_quant import w4_affine_groupwise_linear, w4_groupwise_linear

        if case["affine"]:
            return w4_affine_groupwise_linear(s["x"], s["q"], s["scales"], s["biases"], case["outputs"],
                                              case["inputs"])
        return w4_groupwise_linear(s["x"], s["q"], s["scales"], case["outputs"], case["inputs"])
    if kind == "scan":
        from rwkv7mi import dplr_chunk_scan

        return dplr_chunk_scan(s["r"], s["w"], s["k"], s["v"], s["kk"], s["a"], s["state"])
    if kind == "lora":
        from rwkv7mi.fused_lora import fused_wavg_lora

        return fused_wavg_lora(*s["xs"], *s["downs"], *s["ups"], *s["biases"])
    model, ids, t = s["model"], s["ids"], case["prompt"]
    out = model.forward(ids[:, :t], logits_to_keep=1)
    cache, logits = out.past_key_values, [out.logits]
    for i in range(case["steps"]):  # a scored continuation: the next token is given
        logits.append(model.forward(ids[:, t + i:t + i + 1], past_key_values=cache).logits)
    state, xpa, xpf, _ = cache
    return {"logits": torch.cat(logits, 1), "state": torch.stack(list(state)), "shift": torch.stack([*xpa, *xpf])}


# ------------------------------------------------------------------ 64-bit results
def _recurrence(r, w, k, v, kk, a, state):
    """S <- S diag(w) - (S kk) (kk a)^T + v k^T, y = S r, token by token."""
    y = torch.empty_like(r)
    b = kk * a
    for t in range(r.shape[1]):
        sa = torch.matmul(state, kk[:, t].unsqueeze(-1))
        state = state * w[:, t].unsqueeze(-2)
        state -= sa * b[:, t].unsqueeze(-2)
        state += v[:, t].unsqueeze(-1) * k[:, t].unsqueeze(-2)
        y[:, t] = torch.matmul(state, r[:, t].unsqueeze(-1)).squeeze(-1)
    return y, state


def _exact_chat(case, seed):
    inp = _chat_inputs(case, seed)
    d, n, b = case["hidden"], 64, case["batch"]
    h, t, steps = d // n, case["prompt"], case["steps"]
    w = {k: v.double() for k, v in inp["weights"].items() if k != "model.embeddings.weight"}
    lin = {k: _mm8_dense(p) for k, p in inp["packed"].items()}
    ln = lambda x, name: torch.nn.functional.layer_norm(x, (d,), w[name + ".weight"], w[name + ".bias"], 1e-5)
    proj = lambda name, x: x @ (lin[name] if name in lin else w[name + ".weight"].t())
    lead = lambda x: torch.cat([torch.zeros_like(x[:, :1]), x[:, :-1]], 1)
    x = inp["weights"]["model.embeddings.weight"][inp["ids"]].double()
    states, xpa, xpf, first = [], [], [], None
    for i in range(case["layers"]):
        p = f"model.layers.{i}."
        if i == 0:
            x = ln(x, p + "pre_norm")
        z = ln(x, p + "attn_norm")
        xpa.append(z[:, -1])
        dz = lead(z) - z
        mix = {c: z + dz * w[p + "attn.x_" + c] for c in "rwkvag"}
        r, k, v = (proj(p + f"attn.{c}_proj", mix[c]) for c in "rkv")

        def lora(c, mid):
            return mid(mix[c] @ w[p + f"attn.{c}_lora.lora.0.weight"].t()) @ w[p + f"attn.{c}_lora.lora.2.weight"].t()

        wd = lora("w", torch.tanh) + w[p + "attn.w_lora.lora.2.bias"]
        a = torch.sigmoid(lora("a", lambda m: m) + w[p + "attn.a_lora.lora.2.bias"])
        g = lora("g", torch.sigmoid)
        kk = (k * w[p + "attn.k_k"]).view(b, -1, h, n)
        kk = kk / kk.norm(dim=-1, keepdim=True).clamp_min(1e-12)
        k = k * (1 + (a - 1) * w[p + "attn.k_a"])
        if i == 0:
            first = v
        else:
            v = v + (first - v) * torch.sigmoid(lora("v", lambda m: m) + w[p + "attn.v_lora.lora.2.bias"])
        heads = lambda q: q.reshape(b, -1, h, n)
        s0 = torch.zeros(b, h, n, n, device=DEV, dtype=torch.float64)
        y, s1 = _recurrence(heads(r), heads(torch.exp(-0.606531 * torch.sigmoid(wd))), heads(k), heads(v), kk,
                            heads(a), s0)
        states.append(s1)
        y = (y - y.mean(-1, keepdim=True)) / torch.sqrt(y.var(-1, unbiased=False, keepdim=True) + n * 1e-5)
        y = y.reshape(b, -1, d) * w[p + "attn.g_norm.weight"] + w[p + "attn.g_norm.bias"]
        bonus = (heads(r) * heads(k) * w[p + "attn.r_k"]).sum(-1, keepdim=True) * heads(v)
        x = x + proj(p + "attn.o_proj", (y + bonus.reshape(b, -1, d)) * g)
        z = ln(x, p + "ffn_norm")
        xpf.append(z[:, -1])
        z = z + (lead(z) - z) * w[p + "ffn.x_k"]
        x = x + proj(p + "ffn.value", torch.relu(proj(p + "ffn.key", z)) ** 2)
    logits = proj("lm_head", ln(x[:, t - 1:], "model.norm"))
    return {"logits": logits, "state": torch.stack(states), "shift": torch.stack([*xpa, *xpf])}


def exact(case, seed):
    kind = case["kind"]
    if kind == "mm8_ffn":
        s = _ffn_inputs(case, seed)
        hidden = torch.relu(s["x"].double() @ _mm8_dense(s["key"])).square_()
        return s["residual"].double() + hidden @ _mm8_dense(s["value"])
    if kind == "w4":
        s = _w4_inputs(case, seed)
        n, m = case["inputs"], case["outputs"]
        out = torch.empty(case["rows"], m, device=DEV, dtype=torch.float64)
        x = s["x"].double()
        for r in range(0, m, 8192):
            q = s["q"][r:r + 8192]
            u = torch.stack((q & 15, q >> 4), -1).reshape(q.shape[0], n // 128, 128).double()
            sc = s["scales"][r:r + 8192].double().unsqueeze(-1)
            u = u * sc + s["biases"][r:r + 8192].double().unsqueeze(-1) if case["affine"] else (u - 8) * sc
            out[:, r:r + 8192] = x @ u.reshape(-1, n).t()
        return out
    if kind == "scan":
        s = _scan_inputs(case, seed)
        return _recurrence(*(s[n].double() for n in ("r", "w", "k", "v", "kk", "a", "state")))
    if kind == "lora":
        s = _lora_inputs(case, seed)
        mids = (torch.tanh, lambda m: m, torch.sigmoid, lambda m: m)
        outs = []
        for x, dn, up, bias, mid in zip(s["xs"], s["downs"], s["ups"], s["biases"], mids):
            y = mid(x.double() @ dn.double().t()) @ up.double().t()
            outs.append(y if bias is None else y + bias.double())
        outs[3] = torch.sigmoid(outs[3])
        return tuple(outs)
    return _exact_chat(case, seed)


# ------------------------------------------------------------------ what a pass needs
def work(case):
    kind = case["kind"]
    if kind == "mm8_ffn":
        r, d, f = case["rows"], case["hidden"], case["ffn"]
        return {"bytes": 2 * d * f + 8 * (d + f) + 6 * r * d, "flops": 4 * r * d * f}
    if kind == "w4":
        r, n, m = case["rows"], case["inputs"], case["outputs"]
        meta = (4 if case["affine"] else 2) * m * (n // 128)
        return {"bytes": n * m // 2 + meta + 2 * r * (n + m), "flops": 2 * r * n * m}
    if kind == "scan":
        th = case["batch"] * case["tokens"] * case["heads"]
        return {"bytes": th * 64 * 16 + case["batch"] * case["heads"] * 32768, "flops": th * 64 * 64 * 7}
    if kind == "lora":
        r, d, ranks = case["rows"], case["hidden"], sum(RANKS)
        return {"bytes": 16 * r * d + 4 * ranks * d, "flops": 4 * r * d * ranks}
    d, layers, b, t, steps = case["hidden"], case["layers"], case["batch"], case["prompt"], case["steps"]
    esz = 1 if case["mm8"] else 2
    per_layer = 12 * d * d * esz + 4 * sum(RANKS) * d
    state = layers * b * d * 64 * 4
    weights = layers * per_layer + VOCAB * d * esz
    # prompt: weights once, state out; each step: weights, state in and out
    nbytes = (1 + steps) * weights + (1 + 2 * steps) * state
    flops = 2 * layers * (12 * d * d + 2 * sum(RANKS) * d + 7 * 32 * d) * b * (t + steps)
    return {"bytes": nbytes, "flops": flops + 2 * VOCAB * d * b * (1 + steps)}


def tolerance(case):
    """About four times the error against ``exact`` (2-norm) that an fp16 and a
    bf16 pass show: an output's rounding alone is 2.1e-4 and 1.7e-3, the MM8
    pair adds its rounded hidden row and, for prompts, its rounded weight."""
    bf16 = case.get("dtype") == "bf16"
    rel = {"mm8_ffn": (1.8e-3, 1.4e-2), "w4": (8.5e-4, 7e-3), "scan": (8.5e-4, 7e-3), "lora": (1.2e-3, 9e-3),
           "chat": (5e-3, 5e-3)}[case["kind"]][int(bf16)]
    return {"rel": rel}
