"""The calls whose speed this framework is judged by: what its users run, over the sizes they run it at.

Three kinds, after the framework's three programs:
  * "generate" -- prompts in, new tokens out (generate.py, its batched form, the hybrid models' sessions): a prompt call,
    then one captured step per token;
  * "window" -- the logits of every position of one text window without a cache (evaluate/full.py);
  * "quantize" -- one Linear through the GPTQ producer (quantize/gptq.py).

Weights and inputs are random, made on the GPU from the seed alone, with the properties of trained models that the paths
depend on: round-to-nearest integer codes of bell-shaped rows with integer zeros, a few large norm gains (the outlier
columns of LLM.int8), sublayer outputs that are small beside the residual, and an output head that is sure of the next
token (so that greedy tokens are the same for every correct implementation). Every token has one successor: `_chain`.

`exact` restates the models in float64 with torch alone, layer by layer, on the whole sequence at once.
"""
from __future__ import annotations

import gc
import math
import sys
from pathlib import Path

import torch
import torch.nn.functional as F

sys.path.insert(0, str(Path.cwd() / "lit-llama-ja_amd"))  # the package of the tree this is run from

# Finished programs (reference cycles that own a captured graph) are collected between programs, in prepare(): freeing a
# graph synchronizes the device, which must not happen while another one is being captured.
gc.disable()

DEV = "cuda"

# name -> (layers, heads, width, vocabulary): lit_llama.model.llama_configs
LLAMA = {"19M": (6, 8, 512, 35000), "49M": (10, 10, 640, 35000), "125M": (12, 10, 780, 35000), "7B": (32, 32, 4096, 32000),
         "13B": (40, 40, 5120, 32000)}
# the hybrid benchmark's sizes: width, layers, heads, feed-forward, window, key / value heads, gated feed-forward
HYBRID = {"1B": (2048, 24, 16, 8448, 1024, 4, 6656), "7B": (4096, 32, 32, 16512, 2048, 8, 13056)}
QUANTIZE = {"int4": "gptq.int4", "int8": "llm.int8", "code8": "gptq.int8"}  # mode -> --quantize
BLOCK = 2048


def listed() -> list:
    return [
        # the fork's small model answering a short prompt: launch latencies are all there is
        _generate("49M-chat", "llama", "49M", "bf16", 1, 24, 32),
        # the fork's largest own model (780 wide, heads of 78: the any-shape kernels)
        _generate("125M-chat", "llama", "125M", "bf16", 1, 100, 32),
        # the headline: one user on the 4-bit model
        _generate("7B-int4-chat", "llama", "7B", "int4", 1, 16, 64),
        # several users together on the 4-bit model, prompts of a sentence or two
        _generate("7B-int4-batch", "llama", "7B", "int4", 8, 37, 48),
        # unquantized weights, a long prompt, the command line's sampling
        _generate("7B-bf16-long", "llama", "7B", "bf16", 1, 1001, 32, top_k=200, temperature=0.8),
        # LLM.int8 for eight users
        _generate("7B-int8-batch", "llama", "7B", "int8", 8, 16, 32),
        # 8-bit GPTQ codes, two users
        _generate("7B-code8-pair", "llama", "7B", "code8", 2, 77, 32),
        # perplexity: one full window of the 4-bit model, and the last, ragged one in the program's default precision
        _window("7B-int4-window", "7B", "int4", 2048),
        _window("7B-f32-window", "7B", "f32", 301),
        # the hybrid families: prompts of different lengths together, and one user after a long prompt
        _generate("1B-mugivik-ragged", "mugivik", "1B", "bf16", 8, 1000, 32),
        _generate("7B-bobasun-chat", "bobasun", "7B", "bf16", 1, 1000, 32),
        # GPTQ of an attention projection from four calibration windows
        {"name": "7B-quantize-linear", "kind": "quantize", "rows": 4096, "columns": 4096, "windows": 4, "tokens": 2048, "bits": 4},
    ]


def _generate(name, family, size, mode, batch, prompt, new, top_k=1, temperature=1.0) -> dict:
    """batch prompts of `prompt` tokens (hybrid models: of prompt / 2 .. prompt), `new` tokens each."""
    return {"name": name, "kind": "generate", "family": family, "size": size, "mode": mode, "batch": batch, "prompt": prompt,
            "new": new, "top_k": top_k, "temperature": temperature}


def _window(name, size, mode, tokens) -> dict:
    return {"name": name, "kind": "window", "family": "llama", "size": size, "mode": mode, "batch": 1, "prompt": tokens}


def draw(rng) -> dict:
    """One more case of the listed ranges."""

    def spread(lo, hi):  # over the logarithm
        return min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))

    kind = rng.choice(["chat", "chat", "batch", "batch", "window", "hybrid", "hybrid", "quantize"])
    if kind == "chat":
        size = rng.choice(["19M", "49M", "125M", "7B", "7B", "13B"])
        mode = rng.choice(["int4", "bf16", "int8", "code8"]) if size == "7B" else "int4" if size == "13B" else "bf16"
        sampled = rng.random() < 0.5
        case = _generate("", "llama", size, mode, 1, spread(1, 500 if size == "125M" else 1500), spread(8, 48),
                         200 if sampled else 1, 0.8 if sampled else 1.0)
    elif kind == "batch":
        mode = rng.choice(["int4", "int4", "int8", "code8", "bf16"])
        batch = rng.randint(2, 12)
        case = _generate("", "llama", rng.choice(["49M", "7B"]) if mode == "bf16" else "7B", mode, batch,
                         spread(4, 1200 // batch), spread(8, 32))
    elif kind == "window":
        size, mode = rng.choice([("7B", "int4"), ("7B", "bf16"), ("7B", "int8"), ("7B", "f32"), ("125M", "f32")])
        case = _window("", size, mode, spread(20, 2048 if mode != "f32" else 301 if size == "7B" else 1000))
    elif kind == "hybrid":
        case = _generate("", rng.choice(["mugivik", "bobasun"]), rng.choice(["1B", "1B", "7B"]), "bf16",
                         rng.choice([1, 1, 2, 3, 5, 8]), spread(2, 1000), spread(8, 32))
    else:
        case = {"kind": "quantize", "rows": 16 * rng.randint(16, 256), "columns": 128 * rng.randint(4, 32), "windows": rng.randint(1, 4),
                "tokens": spread(256, 2048), "bits": rng.choice([4, 4, 8])}
    case.pop("name", None)
    return case


# ------------------------------------------------------------------------------------------- weights and inputs
def _generator(seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _chain(vocab: int, seed: int):
    """(successor of every token, its inverse)."""
    g = torch.Generator().manual_seed(int(seed) + 77)
    perm = torch.randperm(vocab, generator=g)
    inv = torch.empty_like(perm)
    inv[perm] = torch.arange(vocab)
    return perm, inv


def _hidden(width: int) -> int:
    n = int(2 * (4 * width) / 3)
    return n + (-n) % 256


def _llama_tensors(case: dict, seed: int) -> dict:
    """State dict of a LLaMA checkpoint: dense weights, or 4- / 8-bit codes packed as the GPTQ producer packs them."""
    layers, _, C, vocab = LLAMA[case["size"]]
    mode, H, V = case["mode"], _hidden(C), vocab + (-vocab) % 64
    dt = torch.float32 if mode == "f32" else torch.bfloat16
    g, sd = _generator(seed), {}

    def put(name, w):
        if mode not in ("int4", "code8"):
            sd[name + ".weight"] = w.to(dt)
            return
        bits = 4 if mode == "int4" else 8
        low, high = w.amin(1, keepdim=True).clamp(max=0), w.amax(1, keepdim=True).clamp(min=0)
        scale = ((high - low) / (2 ** bits - 1)).to(dt)
        zero = torch.round(-low / scale.float())
        q = torch.round(w / scale.float() + zero).clamp_(0, 2 ** bits - 1).to(torch.uint8)
        sd[name + ".quant_weight"] = q[:, 0::2] | (q[:, 1::2] << 4) if bits == 4 else q
        sd[name + ".scales"], sd[name + ".zeros"] = scale, zero.to(dt)

    def linear(name, rows, cols, gain=1.0):
        put(name, torch.randn(rows, cols, generator=g, device=DEV) * (gain * cols ** -0.5))

    def norm(name):
        w = 1.0 + 0.1 * torch.randn(C, generator=g, device=DEV)
        if mode == "int8":
            w[torch.arange(6, device=DEV) * (C // 6) + 7] = 20.0
        sd[name + ".scale"] = w.to(dt)

    wte = torch.randn(V, C, generator=g, device=DEV)
    sd["transformer.wte.weight"] = wte.to(dt)
    for i in range(layers):
        p = f"transformer.h.{i}."
        norm(p + "rms_1")
        linear(p + "attn.c_attn", 3 * C, C)
        linear(p + "attn.c_proj", C, C, (2 * layers) ** -0.5)
        norm(p + "rms_2")
        linear(p + "mlp.c_fc1", H, C)
        linear(p + "mlp.c_fc2", H, C)
        linear(p + "mlp.c_proj", C, H, (2 * layers) ** -0.5)
    norm("transformer.ln_f")
    _, inv = _chain(vocab, seed)
    head = torch.randn(V, C, generator=g, device=DEV) * 0.1
    head[:vocab] = wte[inv.to(DEV)]
    put("lm_head", head * C ** -0.5)
    return sd


def _hybrid_config(case: dict) -> dict:
    """config.json of the hybrid models as the benchmark sizes them."""
    C, layers, heads, ff, window, kv, glu = HYBRID[case["size"]]
    out, owner = [], None
    for i in range(layers):
        if case["family"] == "bobasun":
            mixer = {"heads": heads, "kv_heads": kv, "dim": 128, "vdim": 128, "scale": 0.1, "v_mix": True,
                     "rot": {"base": 10000.0, "dims": 128, "scaling": {"factor": 2.0}}}
            out.append({"type": "attention", "mixer": mixer, "mlp": {"ff": glu, "kind": "dense", "limit": 7.0}})
            continue
        if i % 6 == 2:
            mixer = {"heads": heads, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 512, "mask": {"size": window},
                     "scale": 192 ** -0.5, "rot": {"base": 10000.0, "dims": 64}}
            if (i // 6) % 2:
                mixer["kv_from"] = owner
            else:
                owner = i
            out.append({"type": "latent_attention", "mixer": mixer, "mlp": {"ff": ff, "kind": "dense"}})
        else:
            out.append({"type": "gla", "mixer": {"heads": heads, "dim": 64, "vdim": 128, "tau": 8.0}, "mlp": {"ff": ff, "kind": "dense"}})
    cfg = {"architecture": "Bobasun" if case["family"] == "bobasun" else "Mugivik", "layers": out, "norm": {"eps": 1e-5},
           "vocab": 32000, "width": C}
    if case["family"] == "bobasun":
        return {**cfg, "embedding": {"scale": 8.0}, "streams": 4}
    return {**cfg, "embedding": {"bigram": {"buckets": 65537, "mul_cur": 11, "mul_prev": 127}}}


def _hybrid_shapes(cfg: dict) -> dict:
    """Checkpoint names and shapes of a hybrid model."""
    C, bobasun = cfg["width"], cfg["architecture"] == "Bobasun"
    out = {"embed": (cfg["vocab"], C)}
    if not bobasun:
        out.update({"bigram": (cfg["embedding"]["bigram"]["buckets"] + 1, C), "embed.norm": (C,)})
    for i, layer in enumerate(cfg["layers"]):
        m, ff = layer["mixer"], layer["mlp"]["ff"]
        H, D, V = m["heads"], m["dim"], m["vdim"]
        if bobasun:
            G, S = m["kv_heads"], cfg["streams"]
            part = {"q": (H * D, C), "k": (G * D, C), "v": (G * V, C), "g": (H, C), "o": (C, H * V), "q.b": (H * D,),
                    "k.b": (G * D,), "v.b": (G * V,), "o.b": (C,), "vmix": ()}
            mlp = {"gate": (ff, C), "gate.b": (ff,), "up": (ff, C), "up.b": (ff,), "down": (C, ff), "down.b": (C,)}
            for q in (1, 2):
                out.update({f"l{i}.hc{q}.in": (S,), f"l{i}.hc{q}.out": (S,), f"l{i}.hc{q}.mix": (S, S)})
        elif layer["type"] == "gla":
            part = {"q": (H * D, C), "k": (H * D, C), "v": (H * V, C), "g": (H * V, C), "o": (C, H * V), "norm": (V,),
                    "a1": (16, C), "a2": (H * D, 16), "a2.b": (H * D,)}
            mlp = {"up": (ff, C), "down": (C, ff)}
        else:
            R, rd = m["kv_rank"], m["rot_dim"]
            part = {"q": (H * (D + rd), C), "uk": (H * D, R), "uv": (H * V, R), "g": (H * V, C), "o": (C, H * V)}
            if "kv_from" not in m:
                part.update({"dkv": (R + rd, C), "dkv.norm": (R,)})
            mlp = {"up": (ff, C), "down": (C, ff)}
        out.update({f"l{i}.norm1": (C,), f"l{i}.norm2": (C,)})
        out.update({f"l{i}.mix.{k}": s for k, s in part.items()})
        out.update({f"l{i}.mlp.{k}": s for k, s in mlp.items()})
    out["final.norm"] = (C,)
    if bobasun:
        out["head"] = (cfg["vocab"], C)
    return out


def _hybrid_tensors(cfg: dict, seed: int) -> dict:
    g, t, bobasun, C = _generator(seed), {}, cfg["architecture"] == "Bobasun", cfg["width"]
    for name, shape in _hybrid_shapes(cfg).items():
        r = torch.randn(shape, generator=g, device=DEV)
        if ".hc" in name:  # streams: a mixing near the identity
            S = cfg["streams"]
            r = (torch.eye(S, device=DEV) * 0.9 + 0.1 / S + 0.01 * r if name.endswith(".mix") else
                 (1.0 / S if name.endswith(".in") else 1.0) + 0.1 * r)
        elif name.endswith(".vmix"):
            r = 0.4 + 0.1 * r
        elif len(shape) == 1:
            if bobasun:
                base = 0.0 if name.endswith(".b") else 1.0
            else:  # norm weights are stored around zero; a sublayer adds a quarter of the residual's size
                base = (1.0 if name.endswith((".mix.norm", ".dkv.norm")) else 2.0 if name.endswith(".b") else
                        -0.75 if name.endswith((".norm1", ".norm2")) else 0.0)
            r = base + 0.1 * r
        elif bobasun and name == "embed":
            pass
        elif name == "head":
            r = t["embed"].float()[_chain(cfg["vocab"], seed)[1].to(DEV)] * C ** -0.5
        else:
            r = r * ((0.3 if name == "bigram" else 1.0) * shape[1] ** -0.5)
        t[name] = (r if r.dim() == 0 or ".hc" in name else r.to(torch.bfloat16))
    return t


def _prompts(case: dict, seed: int) -> list:
    """Token ids of every prompt, on the host as a tokenizer gives them."""
    g, B, n = torch.Generator().manual_seed(int(seed) + 13), case["batch"], case["prompt"]
    vocab = LLAMA[case["size"]][3] if case["family"] == "llama" else 32000
    lens = [n - (0 if case["family"] == "llama" else b * n // (2 * B)) for b in range(B)]
    return [torch.randint(3, vocab, (k,), generator=g) for k in lens]


def _calibration(case: dict, seed: int):
    """(weight, calibration windows): activations with correlated columns of different sizes."""
    g, N, K, T = _generator(seed), case["rows"], case["columns"], case["tokens"]
    w = torch.randn(N, K, generator=g, device=DEV) * K ** -0.5
    basis = torch.randn(32, K, generator=g, device=DEV) * 0.3
    size = torch.exp(0.5 * torch.randn(K, generator=g, device=DEV))
    x = [(torch.randn(1, T, K, generator=g, device=DEV) + torch.randn(1, T, 32, generator=g, device=DEV) @ basis) * size
         for _ in range(case["windows"])]
    return w, x


# ------------------------------------------------------------------------------------------- the calls
def prepare(case: dict, seed: int) -> dict:
    gc.collect()
    if case["kind"] == "quantize":
        w, x = _calibration(case, seed)
        lin = torch.nn.Linear(case["columns"], case["rows"], bias=False, device=DEV)
        with torch.no_grad():
            lin.weight.copy_(w)
        return {"case": case, "linear": lin, "windows": x}
    prompts = _prompts(case, seed)
    if case["family"] == "llama":
        from lit_llama import LLaMA
        from lit_llama.utils import EmptyInitOnDevice

        dt = torch.float32 if case["mode"] == "f32" else torch.bfloat16
        with EmptyInitOnDevice(device=torch.device(DEV), dtype=dt, quantization_mode=QUANTIZE.get(case["mode"])):
            model = LLaMA.from_name(case["size"])
        model.load_state_dict(_llama_tensors(case, seed))
        prompts = torch.stack(prompts).to(DEV)
    else:
        from lit_llama import Bobasun, Mugivik

        cls, cfg = Bobasun if case["family"] == "bobasun" else Mugivik, _hybrid_config(case)
        model = cls.from_tensors(cls.config_from_dict(cfg), _hybrid_tensors(cfg, seed), torch.bfloat16, DEV)
        prompts = [p.tolist() for p in prompts]
    return {"case": case, "model": model.eval(), "prompts": prompts, "seed": int(seed)}


def run(state: dict):
    case = state["case"]
    if case["kind"] == "quantize":
        from lit_llama.quantization import GPTQQuantizer

        q = GPTQQuantizer(state["linear"], bits=case["bits"], actorder=True)
        for x in state["windows"]:
            q.collect_input_stats(None, (x,), None)
        packed, error = q.quantize()
        return [packed.quant_weight, packed.scales, packed.zeros, error]
    model, prompts = state["model"], state["prompts"]
    if case["kind"] == "window":
        return model(prompts)
    from lit_llama.engine import DecodeSession

    total = case["prompt"] + case["new"]
    sess = DecodeSession(model, case["batch"], total, total, temperature=case["temperature"], top_k=case["top_k"], seed=state["seed"])
    sess.prefill(prompts)
    sess.decode(case["new"] - 1)
    return [sess.output(), sess.logits]


def work(case: dict) -> dict:
    """Weights once per call and step, keys and values read per step and written, the head's logits; products counted once."""
    if case["kind"] == "quantize":
        N, K, T = case["rows"], case["columns"], case["windows"] * case["tokens"]
        return {"bytes": 4 * T * K + 4 * N * K + N * K * case["bits"] // 8, "flops": 2 * T * K * K + 2 * K ** 3 + N * K * K}
    B, P = case["batch"], case["prompt"]
    if case["family"] == "llama":
        L, _, C, vocab = LLAMA[case["size"]]
        V = vocab + (-vocab) % 64
        mats, head = L * (4 * C * C + 3 * C * _hidden(C)), V * C
        width = {"f32": 4, "bf16": 2, "int8": 1, "code8": 1, "int4": 0.5}[case["mode"]]
        kv, att, act = 2 * L * C, 4 * L * C, 4 if case["mode"] == "f32" else 2
    else:
        C, L, heads, ff, window, kvh, glu = HYBRID[case["size"]]
        V, width, act = 32000, 2, 2
        shapes = _hybrid_shapes(_hybrid_config(case))
        head = V * C
        mats = sum(math.prod(s) for n, s in shapes.items() if len(s) == 2 and n not in ("embed", "bigram", "head"))
        if case["family"] == "bobasun":
            kv, att = L * kvh * 256, 4 * L * heads * 128
        else:  # latents of every second latent layer; the recurrence's state instead of keys elsewhere
            kv, att = (L // 12) * 576, 4 * (L // 6) * heads * 160
    if case["kind"] == "window":
        return {"bytes": int((mats + head) * width + B * P * V * act), "flops": int(2 * B * P * (mats + head) + att * B * P * P / 2)}
    mean = 0.75 * P if case["family"] != "llama" and B > 1 else P  # ragged prompts
    steps = case["new"] - 1
    bytes_ = (mats + head) * width * (1 + steps) + B * kv * act * (mean + steps * (mean + steps / 2)) + B * V * act * (1 + steps)
    flops = 2 * B * mats * (mean + steps) + 2 * B * head * (1 + steps) + att * B * (mean * mean / 2 + steps * (mean + steps / 2))
    return {"bytes": int(bytes_), "flops": int(flops)}


def tolerance(case: dict):
    if case["kind"] == "quantize":
        return {"rel": 1e-4, "max": 1e-3, "differ": 0.01}
    if case["mode"] == "f32":
        return {"rel": 5e-6, "max": 1e-3}
    # bf16 against float64: 0.003 (Bobasun) .. 0.014 (LLaMA, Mugivik), LLM.int8 0.03
    return {"rel": 0.012 if case["family"] == "bobasun" else 0.03, "max": 0.5, "differ": 0.0}


# ------------------------------------------------------------------------------------------- float64
def exact(case: dict, seed: int):
    with torch.no_grad():
        if case["kind"] == "quantize":
            return _exact_quantize(case, seed)
        logits_of = _exact_llama(case, seed) if case["family"] == "llama" else _exact_hybrid(case, seed)
        prompts = _prompts(case, seed)
        if case["kind"] == "window":
            return logits_of(torch.stack(prompts).to(DEV), None)
        lens, new, T = [len(p) for p in prompts], case["new"], max(len(p) for p in prompts) + case["new"] - 1
        vocab = 32000 if case["family"] != "llama" else LLAMA[case["size"]][3]
        succ = torch.arange(vocab) if case["family"] == "mugivik" else _chain(vocab, seed)[0]
        rows = []
        for p in prompts:  # every token followed by its successor, then checked against the logits
            row = p.tolist()
            for _ in range(new):
                row.append(int(succ[row[-1]]))
            rows.append(row)
        ids = torch.stack([F.pad(torch.tensor(r[:-1]), (0, T + 1 - len(r))) for r in rows]).to(DEV)
        at = torch.tensor([[n - 1 + j for j in range(new)] for n in lens], device=DEV)
        logits = logits_of(ids, at)  # (B, new, V)
        if not torch.equal(logits.argmax(-1).cpu(), torch.tensor([r[-new:] for r in rows])):
            return None  # a draw of weights whose head is not sure of the successor
        tokens = [torch.tensor(r, dtype=torch.int32) for r in rows]
        return [torch.stack(tokens) if len(set(lens)) == 1 else tokens, logits[:, -1].contiguous()]


def _rotate(x, base, pairs, factor=1.0):
    """Rotary positions 0.. over the last axis of x (B, H, T, D); pairs: dimensions (2 i, 2 i + 1), else (i, i + D / 2)."""
    D, T = x.shape[-1], x.shape[-2]
    f = base ** (-2.0 * torch.arange(D // 2, device=DEV, dtype=torch.float64) / D) / factor
    a = torch.arange(T, device=DEV, dtype=torch.float64)[:, None] * f
    c, s = a.cos(), a.sin()
    u, v = (x[..., 0::2], x[..., 1::2]) if pairs else (x[..., :D // 2], x[..., D // 2:])
    u, v = u * c - v * s, v * c + u * s
    return torch.stack([u, v], -1).flatten(-2) if pairs else torch.cat([u, v], -1)


def _rms(x, eps=1e-5):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _heads(x, n):
    return x.unflatten(-1, (n, -1)).transpose(1, 2)


def _attend(q, k, v, scale, window=None, sink=False):
    """Causal attention over (B, H, T, D), one head at a time."""
    T, out = q.shape[2], torch.empty(*q.shape[:3], v.shape[-1], dtype=torch.float64, device=DEV)
    i = torch.arange(T, device=DEV)
    hidden = i[None, :] > i[:, None]
    if window is not None:
        hidden |= i[None, :] <= i[:, None] - window
    for b in range(q.shape[0]):
        for h in range(q.shape[1]):
            s = (q[b, h] @ k[b, h % k.shape[1] if k.shape[1] == 1 else h * k.shape[1] // q.shape[1]].T) * scale
            s.masked_fill_(hidden, -math.inf)
            m = s.amax(-1, keepdim=True)
            m = m.clamp(min=0.0) if sink else m
            e = torch.exp(s - m)
            z = e.sum(-1, keepdim=True) + (torch.exp(-m) if sink else 0.0)
            out[b, h] = (e / z) @ v[b, h * v.shape[1] // q.shape[1]]
    return out.transpose(1, 2).flatten(2)


def _exact_llama(case: dict, seed: int):
    layers, nh, C, _ = LLAMA[case["size"]]
    sd, mode, first = _llama_tensors(case, seed), case["mode"], case["prompt"]

    def weight(name):
        if name + ".weight" in sd:
            return sd[name + ".weight"].double()
        q = sd[name + ".quant_weight"]
        w = torch.stack([q & 15, q >> 4], -1).flatten(1) if mode == "int4" else q
        return (w.double() - sd[name + ".zeros"].double()) * sd[name + ".scales"].double()

    def linear(x, name):
        w = weight(name)
        if mode != "int8":
            return x @ w.T
        # LLM.int8: columns with an entry of 6 or more among the rows of one call (the prompts, then every step) stay
        # unquantized, the others become row-wise 8-bit codes
        big = x.abs() >= 6.0
        n = first if x.shape[1] >= first else 0
        cols = torch.cat([big[:, :n].flatten(0, 1).any(0, keepdim=True).expand(n, -1), big[:, n:].any(0)])
        sa = x.abs().masked_fill(big, 0.0).amax(-1, keepdim=True)
        sa = torch.where(sa == 0, 1.0, sa)
        sw = w.abs().amax(1)
        cw = torch.round(w * (127.0 / sw[:, None]))
        ca = torch.round(x * (127.0 / sa)).masked_fill(cols, 0.0)
        return (ca @ cw.T) * (sa * sw / 127.0 ** 2) + x.masked_fill(~cols, 0.0) @ (cw * (sw[:, None] / 127.0)).T

    def logits(ids, at):
        x = sd["transformer.wte.weight"][ids].double()
        for i in range(layers):
            p = f"transformer.h.{i}."
            q, k, v = linear(_rms(x) * sd[p + "rms_1.scale"].double(), p + "attn.c_attn").split(C, -1)
            q, k = (_rotate(_heads(t, nh), 10000.0, True) for t in (q, k))
            x = x + linear(_attend(q, k, _heads(v, nh), (C // nh) ** -0.5), p + "attn.c_proj")
            h = _rms(x) * sd[p + "rms_2.scale"].double()
            x = x + linear(F.silu(linear(h, p + "mlp.c_fc1")) * linear(h, p + "mlp.c_fc2"), p + "mlp.c_proj")
        x = _rms(x) * sd["transformer.ln_f.scale"].double()
        return linear(x if at is None else x.gather(1, at[..., None].expand(-1, -1, C)), "lm_head")

    return logits


def _exact_hybrid(case: dict, seed: int):
    cfg = _hybrid_config(case)
    t, C = _hybrid_tensors(cfg, seed), cfg["width"]

    def par(name):
        return t[name].double()

    def linear(x, name):
        y = x @ par(name).T
        return y + par(name + ".b") if name + ".b" in t else y

    def recurrence(h, m, p):
        H, D, V = m["heads"], m["dim"], m["vdim"]
        B, T, _ = h.shape
        q, k, v = (linear(h, p + n).view(B, T, H, -1) for n in "qkv")
        z = h @ par(p + "a1").T @ par(p + "a2").T + par(p + "a2.b")
        a = torch.exp(F.logsigmoid(z) / m["tau"]).view(B, T, H, D)
        S, o = torch.zeros(B, H, D, V, dtype=torch.float64, device=DEV), torch.empty_like(v)
        for j in range(T):
            S = a[:, j, :, :, None] * S + k[:, j, :, :, None] * v[:, j, :, None]
            o[:, j] = (q[:, j, :, None] @ S)[:, :, 0]
        o = (_rms(o * D ** -0.5) * par(p + "norm")).flatten(2)
        return linear(o * F.silu(linear(h, p + "g")), p + "o")

    def latent(h, m, p, i, kept):
        H, D, R = m["heads"], m["dim"], m["kv_rank"]
        if "kv_from" not in m:
            r = linear(h, p + "dkv")
            kept[i] = (_rms(r[..., :R]) * par(p + "dkv.norm"), _rotate(r[:, None, :, R:], m["rot"]["base"], True))
        c, kr = kept[m.get("kv_from", i)]
        q = _heads(linear(h, p + "q"), H)
        q = torch.cat([q[..., :D], _rotate(q[..., D:], m["rot"]["base"], True)], -1)
        k = torch.cat([_heads(linear(c, p + "uk"), H), kr.expand(-1, H, -1, -1)], -1)
        y = _attend(q, k, _heads(linear(c, p + "uv"), H), m["scale"], m["mask"]["size"])
        return linear(y * torch.sigmoid(linear(h, p + "g")), p + "o")

    def mugivik(ids):
        big = cfg["embedding"]["bigram"]
        prev = F.pad(ids, (1, 0))[:, :-1]
        row = (prev * big["mul_prev"] + ids * big["mul_cur"]) % big["buckets"]
        row[:, 0] = big["buckets"]
        x = _rms(t["embed"][ids].double() + t["bigram"][row].double()) * (1.0 + par("embed.norm"))
        kept = {}
        for i, layer in enumerate(cfg["layers"]):
            p, m = f"l{i}.mix.", layer["mixer"]
            y = recurrence(x, m, p) if layer["type"] == "gla" else latent(x, m, p, i, kept)
            x = x + _rms(y) * (1.0 + par(f"l{i}.norm1"))
            y = linear(torch.relu(linear(x, f"l{i}.mlp.up")) ** 2, f"l{i}.mlp.down")
            x = x + _rms(y) * (1.0 + par(f"l{i}.norm2"))
        return _rms(x) * (1.0 + par("final.norm"))

    def layer_norm(x, name):
        d = x - x.mean(-1, keepdim=True)
        return _rms(d) * par(name)

    def bobasun(ids):
        X = (t["embed"][ids].double() * cfg["embedding"]["scale"]).expand(cfg["streams"], *ids.shape, C)
        first = None

        def sublayer(X, hc, norm, f):
            y = f(layer_norm(torch.tensordot(par(hc + "in"), X, 1), norm))
            return torch.tensordot(par(hc + "mix").T.contiguous(), X, 1) + par(hc + "out")[:, None, None, None] * y

        def attention(h, i, m):
            nonlocal first
            p, H, G = f"l{i}.mix.", m["heads"], m["kv_heads"]
            q, k, v = (_heads(linear(h, p + n), g) for n, g in (("q", H), ("k", G), ("v", G)))
            q, k = (_rms(_rotate(z, m["rot"]["base"], False, m["rot"]["scaling"]["factor"])) for z in (q, k))
            first = v if first is None else first
            v = v + par(p + "vmix") * (first - v)
            y = _attend(q, k, v, m["scale"], sink=True).unflatten(-1, (H, -1)) * torch.sigmoid(linear(h, p + "g"))[..., None]
            return linear(y.flatten(2), p + "o")

        def gated(h, i, limit):
            g = linear(h, f"l{i}.mlp.gate").clamp(max=limit)
            u = linear(h, f"l{i}.mlp.up").clamp(-limit, limit)
            return linear(g * torch.sigmoid(1.702 * g) * (u + 1.0), f"l{i}.mlp.down")

        for i, layer in enumerate(cfg["layers"]):
            X = sublayer(X, f"l{i}.hc1.", f"l{i}.norm1", lambda h: attention(h, i, layer["mixer"]))
            X = sublayer(X, f"l{i}.hc2.", f"l{i}.norm2", lambda h: gated(h, i, layer["mlp"]["limit"]))
        return layer_norm(X.sum(0), "final.norm")

    def logits(ids, at):
        x = bobasun(ids) if cfg["architecture"] == "Bobasun" else mugivik(ids)
        x = x.gather(1, at[..., None].expand(-1, -1, C))
        return x @ par("head" if "head" in t else "embed").T

    return logits


def _exact_quantize(case: dict, seed: int):
    """GPTQ in float64: scales, zeros and the total error. The codes have no such value: one rounding that falls the
    other way changes every later column of its row."""
    w, windows = _calibration(case, seed)
    W, most = w.double(), 2 ** case["bits"] - 1
    low, high = W.amin(1).clamp(max=0), W.amax(1).clamp(min=0)
    scale = (high - low) / most
    zero = torch.round(-low / scale)
    H = sum(2.0 / len(windows) * (x[0].double().T @ x[0].double()) for x in windows)
    order = torch.argsort(torch.diag(H), descending=True, stable=True)
    W, H = W[:, order], H[order][:, order]
    H.diagonal().add_(0.01 * H.diagonal().mean())
    U = torch.linalg.cholesky(torch.cholesky_inverse(torch.linalg.cholesky(H)), upper=True)
    W, loss, B = W.T.contiguous(), 0.0, 128
    for i in range(0, W.shape[0], B):
        part, u = W[i:i + B].clone(), U[i:i + B, i:i + B]
        err = torch.empty_like(part)
        for j in range(B):
            q = scale * (torch.round(part[j] / scale + zero).clamp(0, most) - zero)
            err[j] = (part[j] - q) / u[j, j]
            part[j + 1:] -= u[j, j + 1:, None] * err[j]
        loss = loss + (err ** 2).sum()
        W[i + B:] -= U[i:i + B, i + B:].T @ err
    return [None, scale[:, None], zero[:, None], float(loss) / 2]
