"""What the speed of this engine is judged by: passes of whole requests through a loaded model.

A pass is what a server does with a batch of requests that arrive together: their prompts go in, in portions under
the step's token budget, prompts that are through decode beside those that are not, and the requests are given back.
The continuations are given ahead, as in a trace replay: a pass asks for the same numbers whatever a close argmax does.
Entry points: `LLM(model, random_weights=True)` and `Replayer.run(record)`.

A model is loaded once per process and serves all cases of its name, as in a server; a state is the requests' tokens.
"""

from __future__ import annotations

import math
import random

import torch

from llmserve import LLM, EngineConfig
from llmserve.config import preset
from llmserve.engine.replay import Replayer

# Widths, heads, vocabularies and so on are those of the named sizes of `llmserve.config`.  The Llama shapes run with fewer
# layers, all alike: over the full depth of a model of random weights rounding to bfloat16 grows until two right answers
# differ by 3 to 7 percent, which would hide a wrong one.
DEPTH = {"tinyllama-1.1b": 12, "llama2-7b": 4}
# (the pages hold the largest case)
PAGES = {"tinyllama-1.1b": 4096, "llama2-7b": 1024, "dibepel-1b": 1024, "ramolix-1b": 1024}
BLOCK = 16


def _config(model: str) -> dict:
    cfg = dict(preset(model))
    if model in DEPTH:
        cfg["num_hidden_layers"] = DEPTH[model]
    return cfg


def listed() -> list[dict]:
    def case(name, model, requests, shortest, longest, new, budget=2048, dtype="bfloat16", spread=1):
        return dict(name=name, model=model, dtype=dtype, requests=requests, shortest=shortest, longest=longest, new=new,
                    budget=budget, spread=spread)

    small, large = "tinyllama-1.1b", "llama2-7b"
    return [
        # one user, a short question, a short answer: the latency of a step
        case("one short chat", small, 1, 11, 11, 16),
        # the batch the engine's benchmark quotes, prompts of a line to a paragraph
        case("8 streams", small, 8, 24, 160, 32),
        # as many live requests as the default engine has slots
        case("64 streams", small, 64, 12, 48, 24),
        # questions about a document: long ragged prompts in portions of 512, then answers behind long contexts
        case("long contexts", small, 4, 1200, 1900, 24, budget=512),
        # the benchmark's prompt in one step
        case("prompt of 2048", small, 1, 2048, 2048, 1),
        # an ordinary prompt of no particular size
        case("prompt of 333", small, 1, 333, 333, 1),
        # a server under load: portions of prompts and decoding requests in the same steps
        case("mixed steps", small, 24, 64, 700, 20, budget=512),
        # the larger shape: three prompts, and eight streams
        case("7b prompts", large, 3, 400, 1500, 1),
        case("7b 8 streams", large, 8, 30, 120, 12),
        # the 32-bit engine
        case("32-bit", small, 2, 40, 90, 8, dtype="float32"),
        # the other decoders: one of attention with two score maps and mixed heads, one of state-space layers, windowed
        # attention and latent attention.  (Those with experts are left out here: where two router scores are close,
        # rounding alone sends a token elsewhere, and two right answers differ by as much as two wrong ones.)
        case("dibepel", "dibepel-1b", 4, 150, 1100, 12),
        case("ramolix", "ramolix-1b", 4, 150, 1100, 12),
    ]


def draw(rng: random.Random) -> dict:
    most = max(_estimate(c) for c in listed())

    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    while True:
        model = rng.choice(["tinyllama-1.1b"] * 6 + ["llama2-7b"] * 2 + ["dibepel-1b", "ramolix-1b"])
        dtype = "float32" if model == "tinyllama-1.1b" and rng.random() < 0.15 else "bfloat16"
        requests = log_int(1, 64)
        shortest = log_int(8, 1900)
        longest = min(1900, log_int(shortest, max(shortest, 8 * shortest)))
        c = dict(model=model, dtype=dtype, requests=requests, shortest=shortest, longest=longest, new=log_int(1, 32),
                 budget=rng.choice([512, 1024, 2048]), spread=rng.randrange(1 << 16))
        if dtype == "float32" and (requests > 4 or longest > 160 or c["new"] > 12):
            continue
        if model in ("dibepel-1b", "ramolix-1b") and (requests > 8 or longest > 1100):
            continue
        pages = sum(-(-(n + c["new"]) // BLOCK) for n in _lengths(c))
        if pages <= PAGES[model] - 8 and _estimate(c) <= most:
            return c


# ---------------------------------------------------------------------------------------------- the requests of a case
def _lengths(case: dict) -> list[int]:
    """Prompt lengths: the shortest, the longest, and between them, spread over their logarithm."""
    rng = random.Random(case["spread"])
    lo, hi, n = case["shortest"], case["longest"], case["requests"]
    between = [int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))))) for _ in range(max(0, n - 2))]
    return ([lo] + between + [hi])[:n] if n > 1 else [hi]


def _schedule(case: dict) -> list[list[tuple[int, int, int, bool]]]:
    """The steps of a pass: (request, first position, number of tokens, whether the last one's logits are wanted) each.
    Decoding requests take a token of the budget, the rest goes to prompts in the order of arrival."""
    lengths, new, budget = _lengths(case), case["new"], case["budget"]
    at = [0] * len(lengths)  # tokens that are in
    steps = []
    while any(a < n + new - 1 for a, n in zip(at, lengths)):
        step, left = [], budget
        for r, n in enumerate(lengths):
            if n <= at[r] < n + new - 1:
                step.append((r, at[r], 1, True))
                left -= 1
        for r, n in enumerate(lengths):
            if at[r] < n and left > 0:
                take = min(left, n - at[r])
                step.append((r, at[r], take, at[r] + take == n))
                left -= take
        for r, start, count, _ in step:
            at[r] = start + count
        steps.append(step)
    return steps


def _tokens(case: dict, seed: int) -> list[list[int]]:
    cfg = _config(case["model"])
    vocab = cfg.get("vocab_size") or cfg["vocab"]
    g = torch.Generator().manual_seed(seed)
    return [torch.randint(0, vocab, (n + case["new"],), generator=g).tolist() for n in _lengths(case)]


_SERVERS: dict[tuple[str, str], LLM] = {}


def _server(model: str, dtype: str) -> LLM:
    if (model, dtype) not in _SERVERS:
        with torch.inference_mode():
            _SERVERS[(model, dtype)] = LLM(_config(model), random_weights=True, seed=0, engine=EngineConfig(
                dtype=dtype, block_size=BLOCK, num_blocks=PAGES[model], max_num_seqs=64, max_num_batched_tokens=2048))
    return _SERVERS[(model, dtype)]


def prepare(case: dict, seed: int) -> dict:
    llm = _server(case["model"], case["dtype"])
    tokens = _tokens(case, seed)
    records, last = [], {}
    steps = _schedule(case)
    for s, step in enumerate(steps):
        for r, *_ in step:
            last[r] = s
    for s, step in enumerate(steps):
        records.append({"step": s, "end": [r for r in last if last[r] == s], "entries": [
            {"id": r, "tokens": tokens[r][start:start + count], "want": [count - 1] if want else []}
            for r, start, count, want in step]})
    return {"replayer": Replayer(llm.runner), "records": records}


def run(state: dict) -> torch.Tensor:
    """Every wanted row of logits, in the order of the steps."""
    return torch.cat([state["replayer"].run(record) for record in state["records"]])


# -------------------------------------------------------------------------------------------------- what a pass costs
def _layers(model: str) -> list[dict]:
    """Per layer: matrix elements that every token meets, and per (query, visible key) the multiply-adds of attention and
    the numbers a key keeps in the cache; `keys(n)` of n earlier ones that are visible."""
    cfg = _config(model)
    if "hidden_size" in cfg:
        h, ff, heads, kv = (cfg[k] for k in ("hidden_size", "intermediate_size", "num_attention_heads", "num_key_value_heads"))
        d = h // heads
        return [dict(matrix=h * (heads + 2 * kv) * d + heads * d * h + 3 * h * ff, pair=2 * heads * d, row=2 * kv * d,
                     window=None)] * cfg["num_hidden_layers"]
    out, w = [], cfg["width"]
    for e in cfg["layers"]:
        m, ff = e["mixer"], 3 * w * e["mlp"]["ff"]
        window = (m.get("mask") or {}).get("size")
        if e["type"] == "mamba2":
            inner, bc = m["heads"] * m["vdim"], 2 * m["groups"] * m["state"]
            # (the recurrence: a state of heads x state x vdim numbers, multiplied and read once a token)
            out.append(dict(matrix=w * (2 * inner + bc + m["heads"]) + inner * w + ff + 2 * inner * m["state"], pair=0, row=0,
                            window=1))
            continue
        H, dk, dv = m["heads"], m["dim"], m["vdim"]
        if e["type"] == "latent_attention":
            r = m["kv_rank"]
            out.append(dict(matrix=w * H * dk + (0 if "kv_from" in m else w * r) + H * r * (dk + dv) + H * dv * w + ff,
                            pair=2 * H * r, row=r, window=window))
        elif cfg["architecture"] == "Ramolix":
            out.append(dict(matrix=w * (H + m["kv_heads"]) * dk + H * dv * w + ff, pair=2 * H * dk, row=2 * m["kv_heads"] * dk,
                            window=window))
        else:
            maps = 2 if e["type"] == "attention" else 1
            mix = H if e["type"] == "attention_2" else 0
            out.append(dict(matrix=w * (maps * (H + m["kv_heads"]) * dk + m["kv_heads"] * dv) + H * dv * w + 2 * w * w + ff,
                            pair=H * maps * (dk + dv) + H * mix, row=m["kv_heads"] * (maps * dk + dv), window=window))
    return out


def work(case: dict) -> dict:
    """Every step reads the weights it uses and the visible keys and values of its requests once and writes its logits."""
    cfg = _config(case["model"])
    vocab = cfg.get("vocab_size") or cfg["vocab"]
    width = cfg.get("hidden_size") or cfg["width"]
    layers, elem = _layers(case["model"]), 4 if case["dtype"] == "float32" else 2
    weights = sum(layer["matrix"] for layer in layers)
    kinds: dict[tuple, int] = {}
    for layer in layers:
        key = (layer["pair"], layer["row"], layer["window"])
        kinds[key] = kinds.get(key, 0) + 1
    total_bytes = total_flops = 0.0
    for step in _schedule(case):
        rows, wanted = sum(c for _, _, c, _ in step), sum(1 for e in step if e[3])
        total_bytes += weights * elem + rows * width * elem + (wanted > 0) * vocab * width * elem + wanted * vocab * 4
        total_flops += 2.0 * rows * weights + 2.0 * wanted * vocab * width
        for _, start, count, _ in step:
            for (pair, row, window), times in kinds.items():
                end = start + count
                seen = end if window is None else min(end, window + count - 1)
                pairs = sum(min(p + 1, window or p + 1) for p in (start, end - 1)) / 2.0 * count
                total_bytes += times * (seen + count) * row * elem
                total_flops += times * 2.0 * pairs * pair
    return {"bytes": total_bytes, "flops": total_flops}


def _estimate(case: dict) -> float:
    w = work(case)
    rate = 60e12 if case["dtype"] == "float32" else 800e12
    return w["bytes"] / 4e12 + w["flops"] / rate


def tolerance(case: dict) -> dict:
    # bfloat16: the step with other kernels for the same products (sums in another order) is 0.012 to 0.016 off, either is 0.02
    # to 0.03 off the 64-bit result; 32-bit: 5e-6 off the 64-bit result
    if case["dtype"] == "float32":
        return {"rel": 2e-5}
    return {"rel": 0.03}


# ---------------------------------------------------------------------------------------------- the same in 64 bits
F64 = torch.float64


def _rms(x, eps, weight=None):
    y = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)
    return y if weight is None else y * weight


def _softmax_values(scores, seen, v):
    """scores [G, R, T, T], v [G, T, dv] -> [T, G * R * dv]."""
    a = torch.softmax(scores.masked_fill(~seen, -math.inf), -1)
    return (a @ v[:, None]).permute(2, 0, 1, 3).reshape(scores.shape[2], -1)


def _grouped(x, heads):
    return x.view(x.shape[0], heads, -1).transpose(0, 1)


def _turned(x, freq, halves):
    """x [heads, T, d]: dimension i turns together with dimension i + halves."""
    angle = torch.arange(x.shape[1], device=x.device, dtype=F64)[:, None] * freq
    c, s = torch.cos(angle), torch.sin(angle)
    a, b = x[..., :halves], x[..., halves:2 * halves]
    return torch.cat([a * c - b * s, b * c + a * s, x[..., 2 * halves:]], -1)


def _causal(n, device):
    i = torch.arange(n, device=device)
    return i[:, None], i[None, :], i[None, :] <= i[:, None]


def _causal_conv(x, w, bias=None):
    taps = w.shape[1]
    padded = torch.cat([x.new_zeros(taps - 1, x.shape[1]), x])
    y = sum(padded[j:j + x.shape[0]] * w[:, j] for j in range(taps))
    return y if bias is None else y + bias


def _llama_layer(cfg, w, i, x):
    p, h = f"model.layers.{i}.", cfg["hidden_size"]
    H, G, eps = cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["rms_norm_eps"]
    d, n = h // H, x.shape[0]
    freq = cfg["rope_theta"] ** (-torch.arange(0, d, 2, device=x.device, dtype=F64) / d)
    y = _rms(x, eps, w(p + "input_layernorm.weight"))
    q = _turned(_grouped(y @ w(p + "self_attn.q_proj.weight").T, H), freq, d // 2).view(G, H // G, n, d)
    k = _turned(_grouped(y @ w(p + "self_attn.k_proj.weight").T, G), freq, d // 2)
    v = _grouped(y @ w(p + "self_attn.v_proj.weight").T, G)
    a = _softmax_values(q @ k[:, None].transpose(-1, -2) * d ** -0.5, _causal(n, x.device)[2], v)
    x = x + a @ w(p + "self_attn.o_proj.weight").T
    y = _rms(x, eps, w(p + "post_attention_layernorm.weight"))
    return x + (torch.nn.functional.silu(y @ w(p + "mlp.gate_proj.weight").T) * (y @ w(p + "mlp.up_proj.weight").T)) @ w(
        p + "mlp.down_proj.weight").T


def _dibepel_layer(cfg, w, i, x):
    entry, owner, eps = cfg["layers"][i], i, cfg["norm"]["eps"]
    while cfg["layers"][owner].get("weights_of") is not None:
        owner = cfg["layers"][owner]["weights_of"]
    p, m = f"l{owner}.", entry["mixer"]
    H, G, dk = m["heads"], m["kv_heads"], m["dim"]
    n, mask = x.shape[0], m.get("mask") or {}
    row, col, seen = _causal(n, x.device)
    y = _rms(x, eps, 1.0 + w(p + "norm1"))
    mix = p + "mix."
    if entry["type"] == "attention":  # two score maps per head over the same values
        if mask.get("size") is not None:
            seen = seen & ((row - col < mask["size"]) | (col < int(mask.get("keep_first") or 0)))
        q = (y @ w(mix + "q").T).view(n, G, H // G, 2, dk)
        k = (y @ w(mix + "k").T).view(n, G, 2, dk)
        v = _grouped(y @ w(mix + "v").T, G)
        one, two = (_softmax_values(q[..., c, :].permute(1, 2, 0, 3) @ k[:, :, c].permute(1, 2, 0)[:, None] * m["scale"],
                                    seen, v).view(n, H, -1) for c in range(2))
        lam = torch.exp((w(mix + "lq1") * w(mix + "lk1")).sum()) - torch.exp((w(mix + "lq2") * w(mix + "lk2")).sum()) + m["diff"]
        a = _rms(one - lam * two, eps) * (1.0 - m["diff"])
    else:  # short convolutions, a distance bias, the query's own chunk, the heads' weights mixed
        if mask.get("size") is not None:
            seen = seen & (row // mask["size"] == col // mask["size"])
        q, k, v = (_causal_conv(y @ w(mix + c).T, w(mix + c + ".conv")) if m.get("conv") else y @ w(mix + c).T for c in "qkv")
        q, k, v = _grouped(q, H).view(G, H // G, n, dk), _grouped(k, G), _grouped(v, G)
        slopes = 2.0 ** (-8.0 * torch.arange(1, H + 1, device=x.device, dtype=F64) / H)
        s = q @ k[:, None].transpose(-1, -2) * m["scale"] - slopes.view(G, H // G, 1, 1) * (row - col)
        a = torch.softmax(s.masked_fill(~seen, -math.inf), -1).view(H, n * n)
        a = (w(mix + "talk") @ a).view(G, H // G, n, n)
        a = (a @ v[:, None]).permute(2, 0, 1, 3)
    total = torch.sigmoid(y @ w(p + "rg1").T + w(p + "rg1.b")) * (a.reshape(n, -1) @ w(mix + "o").T)
    f = (torch.nn.functional.silu(y @ w(p + "mlp.gate").T) * (y @ w(p + "mlp.up").T)) @ w(p + "mlp.down").T
    return x + total + torch.sigmoid(y @ w(p + "rg2").T + w(p + "rg2.b")) * f


def _stretched(rot, device):
    out = []
    for i in range(rot["dims"] // 2):
        f = rot["base"] ** (-2.0 * i / rot["dims"])
        s = rot.get("scaling")
        if s:
            wave = 2.0 * math.pi / f
            if wave > s["original"] / s["low"]:
                f = f / s["factor"]
            elif wave >= s["original"] / s["high"]:
                t = (s["original"] / wave - s["low"]) / (s["high"] - s["low"])
                f = (1.0 - t) * f / s["factor"] + t * f
        out.append(f)
    return torch.tensor(out, dtype=F64, device=device)


def _ramolix_layer(cfg, w, i, x, kept):
    entry, eps, mult = cfg["layers"][i], cfg["norm"]["eps"], cfg["residual_mult"]
    p, m, n = f"l{i}.", entry["mixer"], x.shape[0]
    mix, (row, col, seen) = p + "mix.", _causal(n, x.device)
    if entry["type"] == "attention":  # the values are the keys as projected
        H, G, d, size = m["heads"], m["kv_heads"], m["dim"], (m.get("mask") or {}).get("size")
        q, k = x @ w(mix + "q").T + w(mix + "q.b"), x @ w(mix + "k").T + w(mix + "k.b")
        freq = _stretched(m["rot"], x.device)
        v = _grouped(k, G)
        q = _turned(_grouped(_rms(q, eps, w(mix + "q.norm")), H), freq, freq.numel()).view(G, H // G, n, d)
        k = _turned(_grouped(_rms(k, eps, w(mix + "k.norm")), G), freq, freq.numel())
        if size is not None:
            seen = seen & (row - col < size)
        y = _softmax_values(q @ k[:, None].transpose(-1, -2) * m["scale"], seen, v) @ w(mix + "o").T
    elif entry["type"] == "latent_attention":
        H = m["heads"]
        if m.get("kv_from") is None:
            kept[i] = _rms(x @ w(mix + "dkv").T, eps, w(mix + "dkv.norm"))
        c = kept[m["kv_from"] if m.get("kv_from") is not None else i]
        q, k, v = _grouped(x @ w(mix + "q").T, H), _grouped(c @ w(mix + "uk").T, H), _grouped(c @ w(mix + "uv").T, H)
        y = _softmax_values(q[:, None] @ k[:, None].transpose(-1, -2) * m["scale"], seen, v) @ w(mix + "o").T
    else:  # the recurrence, as the sum over earlier tokens that it is
        H, P, N, G = m["heads"], m["vdim"], m["state"], m["groups"]
        inner = H * P
        z, u, dt = (x @ w(mix + "in").T).split([inner, inner + 2 * G * N, H], -1)
        u = torch.nn.functional.silu(_causal_conv(u, w(mix + "conv"), w(mix + "conv.b")))
        dt = torch.nn.functional.softplus(dt + w(mix + "dt_bias"))
        v, B, C = _grouped(u[:, :inner], H), _grouped(u[:, inner:inner + G * N], G), _grouped(u[:, inner + G * N:], G)
        passed = torch.cumsum(-torch.exp(w(mix + "A_log")) * dt, 0).T  # [H, n]
        y = v * w(mix + "D")[:, None, None]
        for g in range(G):
            heads = slice(g * (H // G), (g + 1) * (H // G))
            left = torch.exp((passed[heads, :, None] - passed[heads, None, :]).masked_fill(~seen, -math.inf))
            y[heads] += (left * (C[g] @ B[g].T) * dt.T[heads, None, :]) @ v[heads]
        y = y.transpose(0, 1).reshape(n, inner) * torch.nn.functional.silu(z)
        y = _rms(y.view(n, m["norm_groups"], -1), eps).reshape(n, inner) * w(mix + "norm")
        y = y @ w(mix + "o").T
    x = x + mult * _rms(y, eps, w(p + "norm1"))
    f = torch.nn.functional.gelu(x @ w(p + "mlp.gate").T, approximate="tanh") * (x @ w(p + "mlp.up").T)
    return x + mult * _rms(f @ w(p + "mlp.down").T, eps, w(p + "norm2"))


def exact(case: dict, seed: int) -> torch.Tensor:
    """The logits of a pass from whole sequences in 64 bits: no cache, no steps.  The weights are the random ones that the
    named size gives (drawn again, tensor by tensor); the arithmetic is torch's."""
    from llmserve.weights.random import random_tensor

    cfg, dtype = _config(case["model"]), torch.float32 if case["dtype"] == "float32" else torch.bfloat16
    infos = _server(case["model"], case["dtype"]).runner.model.param_infos()
    device = torch.device("cuda:0")

    drawn: dict[str, torch.Tensor] = {}

    def w(name):
        if name not in drawn:  # (one layer's tensors at a time are kept)
            drawn[name] = random_tensor(name, infos[name], 0, dtype, device).to(F64)
        return drawn[name]

    lengths = _lengths(case)
    ids = [torch.tensor(t[:n + case["new"] - 1], device=device) for t, n in zip(_tokens(case, seed), lengths)]
    llama = "hidden_size" in cfg
    embed = w("model.embed_tokens.weight" if llama else "embed")
    xs = [embed[t] * (1.0 if llama else cfg["embedding"]["scale"]) for t in ids]
    kept: list[dict] = [{} for _ in xs]
    for i in range(cfg["num_hidden_layers"] if llama else len(cfg["layers"])):
        drawn.clear()
        for r, x in enumerate(xs):
            xs[r] = (_llama_layer(cfg, w, i, x) if llama else _dibepel_layer(cfg, w, i, x) if cfg["architecture"] == "Dibepel"
                     else _ramolix_layer(cfg, w, i, x, kept[r]))
    drawn.clear()
    if llama:
        xs = [_rms(x, cfg["rms_norm_eps"], w("model.norm.weight")) for x in xs]
        head = w("lm_head.weight")
    elif cfg["architecture"] == "Dibepel":
        xs, head = [_rms(x, cfg["norm"]["eps"], 1.0 + w("final.norm")) for x in xs], w("head")
    else:
        xs, head = [_rms(x, cfg["norm"]["eps"], w("final.norm")) for x in xs], embed
    rows = [xs[r][start + count - 1] for step in _schedule(case) for r, start, count, want in step if want]
    return torch.stack(rows) @ head.T
