"""What is measured: the work a program built on this library has it do, through its public entry points.

Three kinds of work:

* requests: a prompt goes in, tokens come out one at a time, on models in the storage formats that GGUF files use (Q8_0, Q4_0,
  llama.cpp's Q4_K_M recipe) in the fast and the order-faithful mode, and on dense model folders of both designs;
* single operations, as a program calls them that owns its own loop: quantised matrix times vector or rows, attention of a
  prompt and of one query over an fp16 cache;
* the host's share of sampling with a temperature.

The models have the shapes of the benchmark configurations and random weights.  The rows of the output matrix are the embedding
rows moved by one, and what a sublayer adds to the residual stream is small beside it, as in a trained network: the next token is
then decided clearly, so tokens do not hang on the last bits of a sum, and logits can be compared closely.
"""
import math
import os
import shutil
import tempfile

import numpy as np
import torch

from __graft_entry__ import load_package

Q4_0, Q8_0, Q4_K, Q6_K = 2, 8, 12, 14
FORMATS = {"q8_0": Q8_0, "q4_0": Q4_0, "q4_k": Q4_K, "q6_k": Q6_K}
ROW_BYTES = {Q8_0: (32, 34), Q4_0: (32, 18), Q4_K: (256, 144), Q6_K: (256, 210)}      # weights and bytes of a block
FOLDERS = ("kakirax_135m", "kakirax_1b", "vabirax_135m")

# rows to columns of the projections of the configured models: (K, N)
PROJECTIONS = ((576, 576), (576, 1536), (1536, 576), (2048, 512), (2048, 2048), (2048, 8192), (8192, 2048), (3072, 1024), (3072, 8192), (8192, 3072))
HEADS = ((9, 3, 64), (32, 8, 64), (24, 8, 128), (32, 32, 96), (32, 8, 128), (12, 2, 128))


def listed():
    return [
        # one projection of a decode step called on its own: the smallest call, all latency
        {"name": "vec-q8-2048x2048", "kind": "vec", "fmt": "q8_0", "K": 2048, "N": 2048},
        # the output matrix of a 128 k vocabulary as a K-quant: the largest matrix-vector product of a step
        {"name": "vec-q6k-head", "kind": "vec", "fmt": "q6_k", "K": 2048, "N": 128256},
        # a projection for a ragged handful of rows (a short message, a few sequences side by side)
        {"name": "mat-q4-37", "kind": "mat", "fmt": "q4_0", "M": 37, "K": 2048, "N": 8192, "exact": False},
        # the same for the rows of a long message, the depth-8192 projection
        {"name": "mat-q8-902", "kind": "mat", "fmt": "q8_0", "M": 902, "K": 8192, "N": 2048, "exact": False},
        # attention of a long prompt; heads of 96 without sharing, a length that is no multiple of any tile
        {"name": "attn-prompt-3001", "kind": "attn", "heads": 32, "kv_heads": 32, "head_dim": 96, "rows": 3001, "base": 0, "window": 0, "exact": False},
        # attention of one query over a long cache, grouped heads
        {"name": "attn-step-8192", "kind": "attn", "heads": 32, "kv_heads": 8, "head_dim": 64, "rows": 1, "base": 8191, "window": 0, "exact": False},
        # what the server does on the host for every token of a request with a temperature
        {"name": "sample-128k", "kind": "sample", "vocab": 128256, "temperature": 0.8, "top_k": 0, "top_p": 0.9, "recent": 300},
        # a short exchange on the smallest model in the mode that reproduces the CPU path's bits
        {"name": "request-135m-exact", "kind": "request", "model": "smollm2_135m", "fmt": "q8_0", "exact": True, "prompt": 32, "new": 64},
        # a short exchange in the default mode: launches and small batches count
        {"name": "request-1b-short", "kind": "request", "model": "llama32_1b", "fmt": "q8_0", "exact": False, "prompt": 33, "new": 16},
        # a long document and an answer: the prompt dominates, the steps run at a long context
        {"name": "request-1b-long", "kind": "request", "model": "llama32_1b", "fmt": "q4_k_m", "exact": False, "prompt": 2502, "new": 16},
        # dense folders: gated linear attention with a middle-sized prompt, latent attention with a long one
        {"name": "folder-kakirax-1b", "kind": "folder", "model": "kakirax_1b", "dtype": "bfloat16", "prompt": 902, "new": 8},
        {"name": "folder-vabirax-135m", "kind": "folder", "model": "vabirax_135m", "dtype": "bfloat16", "prompt": 2502, "new": 8},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("vec", "mat", "mat", "attn", "attn", "sample", "request", "request", "folder"))
    if kind == "vec":
        K, N = rng.choice(PROJECTIONS)
        fmt = rng.choice(sorted(f for f in FORMATS if K % ROW_BYTES[FORMATS[f]][0] == 0))
        return {"kind": kind, "fmt": fmt, "K": K, "N": rng.choice((N, _log_int(rng, 64, 128256)))}
    if kind == "mat":
        K, N = rng.choice(PROJECTIONS)
        return {"kind": kind, "fmt": rng.choice(("q8_0", "q4_0")), "M": _log_int(rng, 2, 2502), "K": K, "N": N, "exact": rng.random() < 0.25}
    if kind == "attn":
        heads, kv_heads, head_dim = rng.choice(HEADS)
        one = rng.random() < 0.5
        rows = 1 if one else _log_int(rng, 3, 3001)
        base = _log_int(rng, 1, 8191) if one else rng.choice((0, 0, _log_int(rng, 1, 2000)))
        window = rng.choice((0, 0, 0, _log_int(rng, 64, 4096)))
        return {"kind": kind, "heads": heads, "kv_heads": kv_heads, "head_dim": head_dim, "rows": rows, "base": base, "window": window,
                "exact": window == 0 and rng.random() < 0.25}
    if kind == "sample":
        return {"kind": kind, "vocab": rng.choice((32000, 49152, 128256, _log_int(rng, 1000, 128256))), "temperature": round(rng.uniform(0.3, 1.5), 2),
                "top_k": rng.choice((0, 0, 40, _log_int(rng, 2, 1000))), "top_p": rng.choice((0.9, 0.95, 1.0, round(rng.uniform(0.1, 0.99), 2))),
                "recent": _log_int(rng, 1, 3000)}
    if kind == "request":
        model = rng.choice(("smollm2_135m", "smollm2_135m", "llama32_1b"))
        fmt = rng.choice(("q8_0", "q4_0") if model == "smollm2_135m" else ("q8_0", "q4_0", "q4_k_m"))
        exact = rng.random() < 0.3
        return {"kind": kind, "model": model, "fmt": fmt, "exact": exact, "prompt": _log_int(rng, 3, 1200 if exact else 2400), "new": _log_int(rng, 2, 16)}
    dtype = rng.choice(("bfloat16", "bfloat16", "float32"))
    model = rng.choice(FOLDERS if dtype == "bfloat16" else ("kakirax_135m", "vabirax_135m"))
    return {"kind": "folder", "model": model, "dtype": dtype, "prompt": _log_int(rng, 3, 2000 if dtype == "bfloat16" else 700), "new": _log_int(rng, 2, 8)}


# ---- weights --------------------------------------------------------------------------------------------------------------

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 11)


def _ids(seed, n, vocab):
    return np.random.default_rng(int(seed) + 5).integers(0, vocab, n).astype(np.uint32)


def _f16_bytes(x):
    return x.to(torch.float16).contiguous().view(torch.uint8).view(*x.shape, 2)


def _blocks(gen, fmt, n, k, std):
    """An [n][k] matrix as GGUF blocks, uint8 [n][row bytes] on the GPU: normal weights quantised (Q8_0, Q4_0), or random super-blocks
    whose weights have that spread (Q4_K, Q6_K)."""
    per, size = ROW_BYTES[fmt]
    if fmt in (Q8_0, Q4_0):
        x = torch.randn(n, k // per, per, generator=gen, device="cuda") * std
        scale = x.abs().amax(-1) / (127.0 if fmt == Q8_0 else 8.0)
        code = torch.round(x / scale[..., None])
        if fmt == Q8_0:
            body = code.clamp(-127, 127).to(torch.int8).view(torch.uint8)
        else:
            code = (code + 8).clamp(0, 15).to(torch.uint8)
            body = code[..., :16] | (code[..., 16:] << 4)
        return torch.cat([_f16_bytes(scale), body], -1).reshape(n, -1)
    raw = torch.randint(0, 256, (n, k // per, size), generator=gen, device="cuda", dtype=torch.uint8)
    d = torch.empty(n, k // per, device="cuda").uniform_(0.7, 1.3, generator=gen) * (std / (258.0 if fmt == Q4_K else 165.0))
    if fmt == Q4_K:
        raw[..., 0:2] = _f16_bytes(d)
        raw[..., 2:4] = _f16_bytes(7.5 * d)
    else:
        raw[..., 192:208] = torch.randint(-15, 16, (n, k // per, 16), generator=gen, device="cuda", dtype=torch.int8).view(torch.uint8)
        raw[..., 208:210] = _f16_bytes(d)
    return raw.reshape(n, -1)


def _f16_at(raw, at):
    return raw[..., at:at + 2].contiguous().view(torch.float16).to(torch.float64)


def _dequant(raw, fmt):
    """The weights that GGUF blocks stand for, in 64 bits: uint8 [n][row bytes] -> [n][k]."""
    per, size = ROW_BYTES[fmt]
    raw = raw.view(raw.shape[0], -1, size)
    if fmt == Q8_0:
        w = raw[..., 2:].contiguous().view(torch.int8).to(torch.float64) * _f16_at(raw, 0)
    elif fmt == Q4_0:
        w = (torch.cat([raw[..., 2:] & 15, raw[..., 2:] >> 4], -1).to(torch.float64) - 8.0) * _f16_at(raw, 0)
    elif fmt == Q4_K:
        s = raw[..., 4:16].to(torch.int32)
        sc = torch.cat([s[..., 0:4] & 63, (s[..., 8:12] & 15) | ((s[..., 0:4] >> 6) << 4)], -1).to(torch.float64)
        mn = torch.cat([s[..., 4:8] & 63, (s[..., 8:12] >> 4) | ((s[..., 4:8] >> 6) << 4)], -1).to(torch.float64)
        qs = raw[..., 16:].view(*raw.shape[:2], 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 3).reshape(*raw.shape[:2], 8, 32).to(torch.float64)
        w = q * (_f16_at(raw, 0) * sc)[..., None] - (_f16_at(raw, 2) * mn)[..., None]
    else:
        ql, qh = raw[..., :128].view(*raw.shape[:2], 2, 64).to(torch.int32), raw[..., 128:192].view(*raw.shape[:2], 2, 32).to(torch.int32)
        low = torch.stack([ql[..., :32] & 15, ql[..., 32:] & 15, ql[..., :32] >> 4, ql[..., 32:] >> 4], 3)
        high = torch.stack([(qh >> t) & 3 for t in (0, 2, 4, 6)], 3)
        q = (low | (high << 4)).reshape(*raw.shape[:2], 16, 16).to(torch.float64) - 32.0
        sc = raw[..., 192:208].contiguous().view(torch.int8).to(torch.float64)
        w = q * (_f16_at(raw, 208) * sc)[..., None]
    return w.reshape(raw.shape[0], -1)


def _llama_config(case):
    """(forge_hip_config fields, formats of q, k, v, o, gate, up, down)."""
    fh = load_package()
    recipe = case["fmt"] == "q4_k_m"
    fmt = Q8_0 if recipe else FORMATS[case["fmt"]]
    room = case["prompt"] + case["new"]
    cfg = getattr(fh.synth, case["model"])(wdtype=fmt, max_seq=max(1024, (room + 63) // 64 * 64))
    cfg["flags"] = fh.FLAG_EXACT if case["exact"] else 0
    if recipe:
        cfg["lm_head_dtype"] = Q6_K
        return cfg, [Q4_K, Q4_K, Q6_K, Q4_K, Q4_K, Q4_K, Q6_K]
    return cfg, [fmt] * 7


def _llama_parts(cfg, formats, seed):
    """The model's tensors in the order of weights.bin: [(name, f32 vector or table | (blocks, format))]."""
    gen = _generator(seed)
    H, I, V = cfg["hidden"], cfg["inter"], cfg["vocab"]
    Q, KV = cfg["heads"] * cfg["head_dim"], cfg["kv_heads"] * cfg["head_dim"]
    small = 0.02 / math.sqrt(2.0 * cfg["layers"])                    # what a layer adds stays small beside the stream

    def norm():
        return 1.0 + 0.1 * torch.randn(H, generator=gen, device="cuda")

    head = _blocks(gen, cfg["lm_head_dtype"], V, H, 0.02)
    table = torch.empty(V, H, device="cuda")
    for a in range(0, V, 16384):                                     # row t of the table: row t + 1 of the output matrix
        rows = (torch.arange(a, min(a + 16384, V), device="cuda") + 1) % V
        table[a:a + 16384] = _dequant(head[rows], cfg["lm_head_dtype"]) * 50.0
    parts = [("embed", table)]
    shapes = ((Q, H, 0.02), (KV, H, 0.02), (KV, H, 0.02), (H, Q, small), (I, H, 0.02), (I, H, 0.02), (H, I, small))
    for layer in range(cfg["layers"]):
        parts.append(("attn_norm", norm()))
        for i, (name, (n, k, std)) in enumerate(zip(("q", "k", "v", "o", "gate", "up", "down"), shapes)):
            if i == 4:
                parts.append(("ffn_norm", norm()))
            parts.append((name, (_blocks(gen, formats[i], n, k, std), formats[i])))
    return parts + [("final_norm", norm()), ("head", (head, cfg["lm_head_dtype"]))]


_staging = None


def _to_host(tensors):
    """The bytes of the tensors one behind the other, in a host buffer that is kept for the next model's weights."""
    global _staging
    size = sum(t.numel() * t.element_size() for t in tensors)
    if _staging is None or _staging.numel() < size:
        _staging = None
        _staging = torch.empty(size, dtype=torch.uint8, pin_memory=True)
    at = 0
    for t in tensors:
        b = t.contiguous().view(-1).view(torch.uint8)
        _staging[at:at + b.numel()].copy_(b, non_blocking=True)
        at += b.numel()
    torch.cuda.synchronize()
    return _staging[:size].numpy()


def _folder_tensors(config, seed):
    """Random weights of a model folder, bfloat16 on the GPU by name."""
    fh = load_package()
    gen = _generator(seed)
    shapes = fh.synth.folder_shapes(config)
    width, small = config["width"], (2.0 * len(config["layers"])) ** -0.5
    out = {}
    for name, shape in shapes.items():
        if name == "embed":
            v = torch.randn(shape, generator=gen, device="cuda") / config["embedding"]["scale"]
        elif name == "head":                                         # row t + 1 answers row t of the embedding
            v = torch.roll(out["embed"].float(), 1, 0) * config["embedding"]["scale"] * width ** -0.5
        elif name == "loop.in":                                      # a pass starts near the mean of both inputs
            v = torch.randn(shape, generator=gen, device="cuda") * (0.1 * shape[1] ** -0.5)
            v += 0.6 * torch.eye(width, device="cuda").repeat(1, 2)
        elif len(shape) == 2:
            v = torch.randn(shape, generator=gen, device="cuda") * shape[1] ** -0.5
            if config["architecture"] == "Kakirax" and name.endswith((".o", ".down")):
                v *= small
        elif name.endswith(".alpha"):
            v = torch.empty(shape, device="cuda").uniform_(0.5, 1.2, generator=gen)
        elif name.endswith(".b"):
            v = torch.randn(shape, generator=gen, device="cuda") * (2.0 if name.endswith(".a2.b") else 0.02)
        else:
            v = torch.empty(shape, device="cuda").uniform_(0.5, 1.5, generator=gen)
            if name.endswith(("norm1b", "norm2b")):                  # the norm behind a sublayer of the Vabirax design
                v *= small
        out[name] = v.to(torch.bfloat16)
    return out


# ---- inputs ---------------------------------------------------------------------------------------------------------------

def prepare(case, seed):
    fh = load_package()
    kind = case["kind"]
    if kind in ("vec", "mat"):
        gen, fmt = _generator(seed), FORMATS[case["fmt"]]
        raw = _blocks(gen, fmt, case["N"], case["K"], 0.02)
        shape = (case["K"],) if kind == "vec" else (case["M"], case["K"])
        x = torch.randn(shape, generator=gen, device="cuda")
        return {"case": case, "w": fh.ops.QWeight(fmt, raw.cpu().numpy(), case["K"], case["N"]), "x": x}
    if kind == "attn":
        gen = _generator(seed)
        q = torch.randn(case["rows"], case["heads"] * case["head_dim"], generator=gen, device="cuda")
        caches = [torch.randn(case["base"] + case["rows"], case["kv_heads"] * case["head_dim"], generator=gen, device="cuda").half().view(torch.int16)
                  for _ in range(2)]
        return {"case": case, "q": q[0].contiguous() if case["rows"] == 1 else q, "k": caches[0], "v": caches[1]}
    if kind == "sample":
        rng = np.random.default_rng(int(seed))
        logits = (rng.standard_normal(case["vocab"]) * 2.0).astype(np.float32)
        logits[rng.integers(0, case["vocab"], 12)] += 8.0            # a few candidates stand out
        recent = rng.integers(0, case["vocab"], case["recent"]).astype(np.uint32)
        return {"case": case, "logits": logits, "recent": recent, "rng": int(rng.integers(1, 1 << 62))}
    if kind == "request":
        cfg, formats = _llama_config(case)
        blob = _to_host([p[0] if isinstance(p, tuple) else p for _, p in _llama_parts(cfg, formats, seed)])
        model = fh.HipModel(cfg, blob, formats if case["fmt"] == "q4_k_m" else None)
        return {"case": case, "model": model, "prompt": _ids(seed, case["prompt"], cfg["vocab"])}
    config = getattr(fh.synth, case["model"])()
    tensors = {n: t.view(torch.int16).cpu().numpy().view(np.uint16) for n, t in _folder_tensors(config, seed).items()}
    folder = tempfile.mkdtemp(dir="/dev/shm" if os.path.isdir("/dev/shm") else None)
    try:
        fh.synth.write_model_folder(folder, config, tensors)
        model = fh.HipModel.from_folder(folder, max_seq=case["prompt"] + case["new"], dtype=case["dtype"])
    finally:
        shutil.rmtree(folder)
    return {"case": case, "model": model, "prompt": _ids(seed, case["prompt"], config["vocab"])}


def run(state):
    fh = load_package()
    case = state["case"]
    kind = case["kind"]
    if kind == "vec":
        return fh.ops.matmul_vec_q(state["w"], state["x"])
    if kind == "mat":
        return fh.ops.matmul_mat_q(state["w"], state["x"], fh.FLAG_EXACT if case["exact"] else 0)
    if kind == "attn":
        flags = fh.FLAG_EXACT if case["exact"] else 0
        heads = (case["heads"], case["kv_heads"], case["head_dim"])
        q, k, v, seq = state["q"], state["k"], state["v"], case["base"] + case["rows"]
        if case["rows"] == 1:
            if case["window"]:
                return fh.ops.attention_sliding(q, k, v, seq, case["window"], *heads, flags)
            return fh.ops.attention_flash(q, k, v, seq, *heads, flags)
        if case["window"]:
            return fh.ops.attention_sliding_batch(q, k, v, case["base"], case["window"], *heads, flags)
        return fh.ops.attention_flash_batch(q, k, v, case["base"], *heads, flags)
    if kind == "sample":
        probs = state["logits"].copy()                               # a step's logits arrive in a buffer of their own
        fh.ops.apply_repeat_penalty(probs, state["recent"], 1.1)
        token, rng = fh.ops.sample(probs, case["temperature"], case["top_k"], case["top_p"], state["rng"])
        return {"probs": probs, "token": token, "rng": np.array(rng, np.uint64).view(np.int64)}
    model = state["model"]
    model.reset()
    first = model.forward_prefill(state["prompt"])
    tokens = [fh.ops.argmax_host(first)]
    for _ in range(case["new"] - 1):
        tokens.append(model.forward_greedy(tokens[-1]))
    return {"first": first, "tokens": np.array(tokens, np.int64), "last": model.forward(tokens[-1])}


# ---- what a pass cannot do without ----------------------------------------------------------------------------------------

def _matrix_bytes(fmt, n, k):
    per, size = ROW_BYTES[fmt]
    return n * (k // per) * size


def _pairs(rows, base, window):
    """Sum over the query rows of the cache rows that each sees."""
    if not window:
        return rows * base + rows * (rows + 1) // 2
    return sum(min(base + r + 1, window) for r in range(rows))


def work(case):
    kind = case["kind"]
    if kind in ("vec", "mat"):
        M, K, N = case.get("M", 1), case["K"], case["N"]
        return {"bytes": _matrix_bytes(FORMATS[case["fmt"]], N, K) + 4 * M * (K + N), "flops": 2 * M * K * N}
    if kind == "attn":
        width, kv = case["heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"]
        seen = case["base"] + case["rows"]
        if case["window"]:
            seen = min(seen, case["window"] + case["rows"] - 1)
        return {"bytes": 4 * seen * kv + 8 * case["rows"] * width, "flops": 4 * width * _pairs(case["rows"], case["base"], case["window"])}
    if kind == "sample":
        return {"bytes": 8 * case["vocab"] + 4 * case["recent"], "flops": 4 * case["vocab"]}
    P, new = case["prompt"], case["new"]
    if kind == "request":
        cfg, formats = _llama_config(case)
        H, I, V = cfg["hidden"], cfg["inter"], cfg["vocab"]
        Q, KV = cfg["heads"] * cfg["head_dim"], cfg["kv_heads"] * cfg["head_dim"]
        shapes = ((Q, H), (KV, H), (KV, H), (H, Q), (I, H), (I, H), (H, I))
        layer = sum(_matrix_bytes(f, n, k) for f, (n, k) in zip(formats, shapes))
        macs = cfg["layers"] * sum(n * k for n, k in shapes)
        head = _matrix_bytes(cfg["lm_head_dtype"], V, H)
        cache = cfg["layers"] * 4 * KV
        attention = cfg["layers"] * 4 * Q * _pairs(P + new, 0, 0)
        steps = sum(range(P + 1, P + new + 1))
        return {"bytes": (1 + new) * (cfg["layers"] * layer + head + 4 * V) + cache * (P + new + steps), "flops": 2 * macs * (P + new) + 2 * V * H * (1 + new) + attention}
    fh = load_package()
    config = getattr(fh.synth, case["model"])()
    shapes = fh.synth.folder_shapes(config)
    size = 2 if case["dtype"] == "bfloat16" else 4
    loop = config.get("loop") or {"start": 0, "stop": 0, "times": 1}
    matrices = attention = states = cache = 0
    for i, layer in enumerate(config["layers"]):
        times = loop["times"] if loop["start"] <= i < loop["stop"] else 1
        matrices += times * sum(math.prod(s) for n, s in shapes.items() if n.startswith("l%d." % i) and len(s) == 2)
        m = layer["mixer"]
        window = (m.get("mask") or {}).get("size", 0)
        if layer["type"] == "gla":
            states += times * m["heads"] * m["dim"] * m["vdim"]
        else:
            attention += times * 2 * m["heads"] * (m["dim"] + m.get("rot_dim", 0) + m["vdim"]) * _pairs(P + new, 0, window)
            row = m["kv_heads"] * (m["dim"] + m["vdim"]) if layer["type"] == "attention" else m["kv_rank"] + m["rot_dim"]
            cache += times * size * row * (P + new + _pairs(new, P, window))
    head = config["vocab"] * config["width"]
    return {"bytes": (1 + new) * (size * (matrices + head) + 4 * config["vocab"] + 8 * states) + cache,
            "flops": 2 * matrices * (P + new) + 2 * head * (1 + new) + attention + 8 * states * (P + new)}


def tolerance(case):
    kind = case["kind"]
    if kind == "sample" or case.get("exact"):
        return "exact"                                               # defined down to the order of every sum
    if kind == "vec":
        return {"rel": 1e-6}                                         # exact block sums, a 32-bit sum over the blocks
    if kind == "mat":
        return {"rel": 1e-4}                                         # the fast mode's biased 32-bit accumulation
    if kind == "attn":
        return {"rel": 1e-3}                                         # softmax weights in 16 bits
    if kind == "request":
        return {"rel": 3e-2, "differ": 0.01}                         # a last bit moves 8-bit activation codes
    return {"rel": 1e-2 if case["dtype"] == "bfloat16" else 5e-6, "differ": 0.01}


# ---- the same in 64 bits ---------------------------------------------------------------------------------------------------

def _quantised(x):
    """Activations as the 8-bit blocks of 32 with a 16-bit scale that the quantised products are defined on, in 64 bits."""
    b = x.reshape(*x.shape[:-1], -1, 32)
    scale = b.abs().amax(-1, keepdim=True) / 127.0
    inv = torch.where(scale > 0, 1.0 / scale, 0.0)
    code = b * inv
    code = torch.trunc(code + torch.copysign(torch.full_like(code, 0.5), code)).clamp(-127, 127)
    return (code * scale.to(torch.float16).to(x.dtype)).reshape(x.shape)


def _rms(x, w, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _attend(q, k, v, scale, base, window):
    """Causal attention, one head after the other: q [T, heads, d], k and v [S, kv heads, d], query t at position base + t."""
    at = torch.arange(q.shape[0], device=q.device)[:, None] + base
    to = torch.arange(k.shape[0], device=q.device)[None, :]
    hidden = to > at
    if window:
        hidden |= at - to >= window
    out = torch.empty(q.shape[0], q.shape[1], v.shape[2], device=q.device, dtype=q.dtype)
    for h in range(q.shape[1]):
        g = h // (q.shape[1] // k.shape[1])
        s = (q[:, h] @ k[:, g].T * scale).masked_fill(hidden, -math.inf)
        out[:, h] = torch.softmax(s, -1) @ v[:, g]
    return out


def _answer(forward, prompt, new, vocab, step):
    """A request's outputs from one pass over the prompt and the tokens that follow it, each `step` after the one before."""
    chain = (int(prompt[-1]) + step * (1 + np.arange(new))) % vocab
    ids = torch.from_numpy(np.concatenate([prompt.astype(np.int64), chain])).cuda()
    logits = forward(ids)[-(new + 1):]
    tokens = logits[:-1].argmax(-1)
    if tokens.tolist() != chain.tolist():
        return None
    return {"first": logits[0], "tokens": None, "last": logits[-1]}


def _llama(case, seed):
    cfg, formats = _llama_config(case)
    parts = iter(_llama_parts(cfg, formats, seed))
    hd = cfg["head_dim"]

    def take():
        p = next(parts)[1]
        return _dequant(*p) if isinstance(p, tuple) else p.double()

    def forward(ids):
        x = take()[ids]
        T = ids.numel()
        angle = torch.arange(T, device="cuda", dtype=torch.float64)[:, None] * cfg["rope_theta"] ** (
            -torch.arange(0, hd, 2, device="cuda", dtype=torch.float64) / hd)
        cos, sin = angle.cos()[:, None], angle.sin()[:, None]

        def turned(z):
            a, b = z[..., 0::2], z[..., 1::2]
            return torch.stack([a * cos - b * sin, a * sin + b * cos], -1).reshape(z.shape)

        for _ in range(cfg["layers"]):
            h = _quantised(_rms(x, take(), cfg["rms_eps"]))
            q, k, v = ((h @ take().T).reshape(T, -1, hd) for _ in range(3))
            k, v = (z.half().double() for z in (turned(k), v))       # the cache holds 16-bit rows
            a = _attend(turned(q), k, v, hd ** -0.5, 0, 0).reshape(T, -1)
            x = x + _quantised(a) @ take().T
            h = _quantised(_rms(x, take(), cfg["rms_eps"]))
            g, u = h @ take().T, h @ take().T
            x = x + _quantised(torch.nn.functional.silu(g) * u) @ take().T
        x = x[-(case["new"] + 1):]
        return _quantised(_rms(x, take(), cfg["rms_eps"])) @ take().T

    return _answer(forward, _ids(seed, case["prompt"], cfg["vocab"]), case["new"], cfg["vocab"], 1)


def _frequencies(rot):
    f = rot["base"] ** (-torch.arange(0, rot["dims"], 2, device="cuda", dtype=torch.float64) / rot["dims"])
    s = rot.get("scaling")
    if s is None:
        return f
    turns = s["original"] * f / (2.0 * math.pi)
    blend = ((turns - s["low"]) / (s["high"] - s["low"])).clamp(0.0, 1.0)
    return (1.0 - blend) * f / s["factor"] + blend * f


def _turned_halves(z, rot):
    half = rot["dims"] // 2
    angle = torch.arange(z.shape[0], device="cuda", dtype=torch.float64)[:, None] * _frequencies(rot)
    cos, sin = angle.cos()[:, None], angle.sin()[:, None]
    a, b = z[..., :half], z[..., half:2 * half]
    return torch.cat([a * cos - b * sin, b * cos + a * sin, z[..., 2 * half:]], -1)


def _latent_mixer(h, p, m, eps):
    T, H, rank = h.shape[0], m["heads"], m["kv_rank"]
    q = (_rms(h @ p["dq"].T, p["dq.norm"], eps) @ p["uq"].T).reshape(T, H, -1)
    q = torch.cat([q[..., :m["dim"]], _turned_halves(q[..., m["dim"]:], m["rot"])], -1)
    kv = h @ p["dkv"].T
    c = _rms(kv[:, :rank], p["dkv.norm"], eps)
    shared = _turned_halves(kv[:, None, rank:], m["rot"]).expand(T, H, -1)
    k = torch.cat([(c @ p["uk"].T).reshape(T, H, -1), shared], -1)
    v = (c @ p["uv"].T).reshape(T, H, -1)
    o = _attend(q, k, v, m["scale"], 0, (m.get("mask") or {}).get("size", 0))
    return (o.reshape(T, -1) * torch.sigmoid(h @ p["g"].T)) @ p["o"].T


def _grouped_mixer(h, p, m, eps):
    T = h.shape[0]
    q = _turned_halves(_rms((h @ p["q"].T).reshape(T, m["heads"], -1), p["q.norm"], eps), m["rot"])
    k = _turned_halves(_rms((h @ p["k"].T).reshape(T, m["kv_heads"], -1), p["k.norm"], eps), m["rot"])
    o = _attend(q, k, (h @ p["v"].T).reshape(T, m["kv_heads"], -1), m["scale"], 0, 0)
    return (o.reshape(T, -1) * torch.sigmoid(h @ p["g"].T)) @ p["o"].T


def _linear_mixer(h, p, m, eps):
    T, H = h.shape[0], m["heads"]
    q = (h @ p["q"].T).reshape(T, H, -1) * m["dim"] ** -0.5
    k, v = (h @ p["k"].T).reshape(T, H, -1), (h @ p["v"].T).reshape(T, H, -1)
    a = torch.exp(torch.nn.functional.logsigmoid(h @ p["a1"].T @ p["a2"].T + p["a2.b"]) / m["tau"]).reshape(T, H, -1)
    state, o = torch.zeros(H, m["dim"], m["vdim"], device="cuda", dtype=torch.float64), torch.empty_like(v)
    for t in range(T):
        state = torch.addcmul(a[t][..., None] * state, k[t][..., None], v[t][:, None])
        o[t] = (q[t][:, None] @ state)[:, 0]
    return (_rms(o, p["norm"], eps).reshape(T, -1) * torch.nn.functional.silu(h @ p["g"].T)) @ p["o"].T


def _folder(case, seed):
    config = getattr(load_package().synth, case["model"])()
    t = {n: v.double() for n, v in _folder_tensors(config, seed).items()}
    eps, latent = config["norm"]["eps"], config["architecture"] == "Vabirax"
    mixers = {"latent_attention": _latent_mixer, "attention": _grouped_mixer, "gla": _linear_mixer}

    def norm(x, name):
        if latent:
            return torch.tanh(t[name + ".alpha"] * x) * t[name] + t[name + ".b"]
        return torch.nn.functional.layer_norm(x, x.shape[-1:], t[name], t[name + ".b"], eps)

    loop = config.get("loop") or {"start": 0, "stop": 0, "times": 1}
    body = list(range(loop["start"], loop["stop"]))
    order = list(range(loop["start"])) + body * loop["times"] + list(range(loop["stop"], len(config["layers"])))

    def forward(ids):
        x0 = x = t["embed"][ids] * config["embedding"]["scale"]
        for i in order:
            layer, n = config["layers"][i], "l%d." % i
            if body and i == body[0]:
                x = torch.cat([x, x0], -1) @ t["loop.in"].T
            p = {k[len(n) + 4:]: v for k, v in t.items() if k.startswith(n + "mix.")}
            y = mixers[layer["type"]](norm(x, n + "norm1"), p, layer["mixer"], eps)
            x = x + (norm(y, n + "norm1b") if latent else y)
            h = norm(x, n + "norm2")
            g, u = h @ t[n + "mlp.gate"].T, h @ t[n + "mlp.up"].T
            g = torch.nn.functional.silu(g) if latent else torch.nn.functional.gelu(g, approximate="tanh")
            y = (g * u) @ t[n + "mlp.down"].T
            x = x + (norm(y, n + "norm2b") if latent else y)
        x = norm(x[-(case["new"] + 1):], "final.norm")
        if latent:
            return x @ t["head"].T
        return config["logit_softcap"] * torch.tanh(x @ t["embed"].T / config["logit_softcap"])

    return _answer(forward, _ids(seed, case["prompt"], config["vocab"]), case["new"], config["vocab"], 1 if latent else 0)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("vec", "mat"):
        gen, fmt = _generator(seed), FORMATS[case["fmt"]]
        w = _dequant(_blocks(gen, fmt, case["N"], case["K"], 0.02), fmt)
        x = torch.randn((case["K"],) if kind == "vec" else (case["M"], case["K"]), generator=gen, device="cuda").double()
        return _quantised(x) @ w.T
    if kind == "attn":
        s = prepare(case, seed)
        T, hd = case["rows"], case["head_dim"]
        k, v = (c.view(torch.float16).double().reshape(-1, case["kv_heads"], hd) for c in (s["k"], s["v"]))
        o = _attend(s["q"].double().reshape(T, case["heads"], hd), k, v, hd ** -0.5, case["base"], case["window"])
        return o.reshape(s["q"].shape)
    if kind == "sample":
        s = prepare(case, seed)
        l = s["logits"].astype(np.float64)
        for i in s["recent"]:
            l[i] = l[i] / 1.1 if l[i] > 0 else l[i] * 1.1
        p = np.exp((l - l.max()) / case["temperature"])
        p /= p.sum()
        order = np.argsort(-p, kind="stable")
        if 0 < case["top_k"] < p.size:
            p[order[case["top_k"]:]] = 0.0
        if 0.0 < case["top_p"] < 1.0:
            p[order[np.cumsum(p[order]) > case["top_p"]]] = 0.0
        return {"probs": p / p.sum() if p.sum() > 0 else p, "token": None, "rng": None}
    if kind == "request":
        return _llama(case, seed)
    return _folder(case, seed)
