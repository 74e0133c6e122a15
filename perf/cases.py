"""The forward calls that programs built on this package make, as measurable cases.

Every case is one ``HipBackend.forward`` call (Engine::eval_tokens, eval_next and
the perplexity loop are made of it) on a model of one of the package's presets: a
single token after a context (chat decoding), a prompt or a later chunk of one, or
a handful of tokens whose logits are all wanted (checking drafted tokens).  Two
cases are whole models.  The others are a few layers of one under a small
vocabulary, so that a case is the layers' own work, and their prompts ask for every
row's logits, so that all of the last layer's rows are wanted too.

Weights are drawn on the GPU as quantized blocks (codes about normal, block scales
of varying size, values of standard deviation about 0.02) and written to a GGUF
image.  ``exact`` computes the same call from the same weights in float64.  It
rounds keys and values to the cache's format, which the caller chooses, but leaves
out the 8-bit rounding of activations that quantized weights imply: the distance
of either side to it then holds that rounding, and not the lottery of which few
codes next to a rounding boundary the last bits of an f32 sum move.
"""
import math
import struct
import zlib

import numpy as np
import torch

import rust_interference_engine_amd as R

GPU = "cuda:0"

# arch, embedding, layers, heads, KV heads, head dim, FFN, vocabulary, tied head
PRESETS = {
    "smollm2-360m": ("llama", 960, 32, 15, 5, 64, 2560, 49152, True),
    "qwen2.5-0.5b": ("qwen2", 896, 24, 14, 2, 64, 4864, 151936, True),
    "qwen2.5-1.5b": ("qwen2", 1536, 28, 12, 2, 128, 8960, 151936, True),
    "qwen3-0.6b": ("qwen3", 1024, 28, 16, 8, 128, 3072, 151936, True),
    "qwen3-1.7b": ("qwen3", 2048, 28, 16, 8, 128, 6144, 151936, True),
    "qwen3-4b": ("qwen3", 2560, 36, 32, 8, 128, 9728, 151936, True),
    "llama-3.2-1b": ("llama", 2048, 16, 32, 8, 64, 8192, 128256, True),
    "llama-3.2-3b": ("llama", 3072, 28, 24, 8, 128, 8192, 128256, True),
    "llama-3.1-8b": ("llama", 4096, 32, 32, 8, 128, 14336, 128256, False),
    "gemma-3-1b": ("gemma3", 1152, 26, 4, 1, 256, 6912, 262144, True),
    "qwen3-30b-a3b": ("qwen3moe", 2048, 48, 32, 4, 128, 768, 151936, False),
}
EXPERTS, USED = 128, 8  # qwen3-30b-a3b (its FFN width above is an expert's)
WINDOW = 512            # gemma-3-1b's sliding window; every sixth layer is global
CACHE = {"f16": R.KvType.F16, "q8_0": R.KvType.Q8_0, "turbo4": R.KvType.TURBO4}
EPS = 1e-6


def listed():
    def case(name, model, weights, n, pos, layers=2, vocab=1024, cache="f16", every=True):
        return {"name": name, "model": model, "weights": weights, "cache": cache, "layers": layers, "vocab": vocab,
                "pos": pos, "n": n, "all": every}

    return [
        # the smallest call: the next token of a short chat with a small whole model
        case("token-smollm2-360m-q8_0", "smollm2-360m", "q8_0", 1, 60, layers=32, vocab=49152, every=False),
        # the first prompt of a chat through a whole model
        case("prompt-llama-3.2-1b-q4_0", "llama-3.2-1b", "q4_0", 333, 0, layers=16, vocab=128256, every=False),
        # chat decoding, the benchmark's model
        case("token-llama-3.1-8b-q4_0", "llama-3.1-8b", "q4_0", 1, 700),
        # a long document's next token, 4-bit cache
        case("token-llama-3.2-3b-q4_k_m-turbo4", "llama-3.2-3b", "q4_k_m", 1, 16011, cache="turbo4"),
        # decoding with a mixture of experts
        case("token-qwen3-30b-a3b-q4_k", "qwen3-30b-a3b", "q4_k", 1, 300),
        # a few drafted tokens checked in one call
        case("check-qwen3-4b-q4_k_m", "qwen3-4b", "q4_k_m", 5, 900),
        # the benchmark's prompt
        case("prompt-llama-3.1-8b-q4_0", "llama-3.1-8b", "q4_0", 512, 0),
        # a prompt of any length, the common 5-bit mix
        case("prompt-llama-3.2-3b-q5_k_m", "llama-3.2-3b", "q5_k_m", 421, 0),
        # a question after a system prompt, unquantized weights
        case("prompt-qwen3-4b-bf16", "qwen3-4b", "bf16", 203, 300),
        # a chunk in the middle of a long document, 8-bit weights and cache
        case("prompt-llama-3.1-8b-q8_0-cache-q8_0", "llama-3.1-8b", "q8_0", 512, 7680, cache="q8_0"),
        # a prompt through a mixture of experts
        case("prompt-qwen3-30b-a3b-q4_k", "qwen3-30b-a3b", "q4_k", 384, 0, layers=1),
        # 256-wide heads, five window layers and a global one
        case("prompt-gemma-3-1b-q8_0", "gemma-3-1b", "q8_0", 650, 0, layers=6),
    ]


def draw(rng):
    most = max(_size(c) for c in listed())
    while True:
        model = rng.choice([m for m in PRESETS if m != "qwen3-30b-a3b"] + ["qwen3-30b-a3b"] * 2)
        weights = rng.choice(["q4_k", "q4_0", "q8_0", "q4_k"] if model == "qwen3-30b-a3b" else
                             ["q4_0", "q4_0", "q4_k_m", "q4_k_m", "q5_k_m", "q6_k", "q8_0", "q5_0", "f16", "bf16"])
        kind = rng.choice(["token", "token", "few", "prompt", "prompt"])
        n = {"token": 1, "few": rng.randint(2, 8), "prompt": round(math.exp(rng.uniform(math.log(9), math.log(1024))))}[kind]
        floats = weights in ("f16", "bf16")
        pos = round(math.exp(rng.uniform(math.log(8), math.log(2000 if floats else 16000))))
        if kind == "prompt" and rng.random() < 0.5:
            pos = 0
        c = {"model": model, "weights": weights, "cache": rng.choice(["f16", "f16", "f16", "q8_0", "turbo4"]),
             "layers": {"gemma-3-1b": 6, "qwen3-30b-a3b": 1}.get(model, 2), "vocab": rng.choice([512, 1024, 2048]),
             "pos": pos, "n": n, "all": True}
        if _size(c) <= most:
            return c


def _size(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 50)


# ---- weights -------------------------------------------------------------------
# Each maker returns the blocks' bytes [blocks, bytes] and a function giving their
# values in float64.

def _scale(g, nb, at):
    """f16 scales around `at`"""
    return (at * (0.75 + 0.5 * torch.rand(nb, 1, device=GPU, generator=g))).half()


def _codes(g, shape, std, mean, lo, hi):
    return (torch.randn(shape, device=GPU, generator=g) * std + mean).round_().clamp_(lo, hi).to(torch.int16)


def _u8(t):
    return t.contiguous().view(torch.uint8)


def _q4_0(g, n):
    d, q = _scale(g, n // 32, 0.008), _codes(g, (n // 32, 32), 2.5, 8, 0, 15)
    return torch.cat([_u8(d), (q[:, :16] | q[:, 16:] << 4).to(torch.uint8)], 1), lambda: d.double() * (q - 8)


def _q5_0(g, n):
    d, q = _scale(g, n // 32, 0.004), _codes(g, (n // 32, 32), 5, 16, 0, 31)
    high = ((q >> 4).long() << torch.arange(32, device=GPU)).sum(1, keepdim=True)
    high = torch.cat([(high >> s) & 255 for s in (0, 8, 16, 24)], 1).to(torch.uint8)
    return torch.cat([_u8(d), high, (q[:, :16] & 15 | (q[:, 16:] & 15) << 4).to(torch.uint8)], 1), lambda: d.double() * (q - 16)


def _q8_0(g, n):
    d, q = _scale(g, n // 32, 0.0005), _codes(g, (n // 32, 32), 40, 0, -127, 127).to(torch.int8)
    return torch.cat([_u8(d), q.view(torch.uint8)], 1), lambda: d.double() * q


def _q45_k(g, n, bits):
    nb, half = n // 256, 2 ** (bits - 1) - 0.5
    d = _scale(g, nb, 0.02 / (half / 3) / 48)
    dmin = (d.float() * half).half()
    sc = torch.randint(32, 64, (nb, 8), device=GPU, generator=g, dtype=torch.int16)
    mn = (sc + torch.randint(-2, 3, (nb, 8), device=GPU, generator=g, dtype=torch.int16)).clamp_(0, 63)
    q = _codes(g, (nb, 4, 2, 32), half / 3, half, 0, 2 ** bits - 1)
    packed = torch.cat([sc[:, :4] | sc[:, 4:] >> 4 << 6, mn[:, :4] | mn[:, 4:] >> 4 << 6, sc[:, 4:] & 15 | (mn[:, 4:] & 15) << 4], 1)
    parts = [_u8(d), _u8(dmin), packed.to(torch.uint8)]
    if bits == 5:
        plane = 2 * torch.arange(4, device=GPU).view(1, 4, 1, 1) + torch.arange(2, device=GPU).view(1, 1, 2, 1)
        parts.append(((q >> 4).int() << plane).sum((1, 2)).to(torch.uint8))
    parts.append((q[:, :, 0] & 15 | (q[:, :, 1] & 15) << 4).to(torch.uint8).view(nb, 128))
    return torch.cat(parts, 1), lambda: (d.double() * sc).view(nb, 8, 1) * q.view(nb, 8, 32) - (dmin.double() * mn).view(nb, 8, 1)


def _q6_k(g, n):
    nb = n // 256
    d = _scale(g, nb, 0.02 / 10 / 64)
    sc = torch.randint(40, 96, (nb, 16), device=GPU, generator=g, dtype=torch.int16) * (torch.randint(0, 2, (nb, 16), device=GPU, generator=g, dtype=torch.int16) * 2 - 1)
    q = _codes(g, (nb, 2, 4, 32), 10, 32, 0, 63)
    low = q & 15
    ql = torch.cat([low[:, :, 0] | low[:, :, 2] << 4, low[:, :, 1] | low[:, :, 3] << 4], 2).to(torch.uint8).view(nb, 128)
    qh = (q[:, :, 0] >> 4 | q[:, :, 1] >> 4 << 2 | q[:, :, 2] >> 4 << 4 | q[:, :, 3] >> 4 << 6).to(torch.uint8).view(nb, 64)
    return torch.cat([ql, qh, sc.to(torch.int8).view(torch.uint8), _u8(d)], 1), lambda: (d.double() * sc).view(nb, 16, 1) * (q.view(nb, 16, 16) - 32)


def _float(g, n, dtype, std):
    x = (torch.randn(n, device=GPU, generator=g) * std).to(dtype)
    return _u8(x), x.double


# name: (ggml type id, values and bytes of a block, maker)
TYPES = {
    "f32": (0, 1, 4, None), "f16": (1, 1, 2, lambda g, n: _float(g, n, torch.float16, 0.02)),
    "bf16": (30, 1, 2, lambda g, n: _float(g, n, torch.bfloat16, 0.02)),
    "q4_0": (2, 32, 18, _q4_0), "q5_0": (6, 32, 22, _q5_0), "q8_0": (8, 32, 34, _q8_0),
    "q4_k": (12, 256, 144, lambda g, n: _q45_k(g, n, 4)), "q5_k": (13, 256, 176, lambda g, n: _q45_k(g, n, 5)), "q6_k": (14, 256, 210, _q6_k),
}


def _tensors(case):
    """name -> (type, dims with the row length first) of the model's GGUF file"""
    arch, E, whole, H, KV, hd, ff, _, tied = PRESETS[case["model"]]
    L, V, w = case["layers"], case["vocab"], case["weights"]
    blocked = w not in ("f16", "bf16")
    if w in ("q4_k", "q4_k_m", "q5_k_m", "q6_k") and (E % 256 or ff % 256):
        w = "q8_0"  # as the presets do: no 256-value blocks in these rows
    more = w.endswith("_m")  # the mixes hold attn_v and half of ffn_down in q6_k
    base = w[:-2] if more else w
    embd = ("q6_k" if E % 256 == 0 else "q8_0") if blocked else base
    t = {"token_embd.weight": (embd, (E, V)), "output_norm.weight": ("f32", (E,))}
    if not tied:
        t["output.weight"] = (embd, (E, V))
    for i in range(L):
        p = "blk.%d." % i
        t[p + "attn_norm.weight"] = t[p + "ffn_norm.weight"] = ("f32", (E,))
        t[p + "attn_q.weight"], t[p + "attn_k.weight"] = (base, (E, H * hd)), (base, (E, KV * hd))
        t[p + "attn_v.weight"] = ("q6_k" if more else base, (E, KV * hd))
        t[p + "attn_output.weight"] = (base, (H * hd, E))
        if arch == "qwen2":
            t[p + "attn_q.bias"], t[p + "attn_k.bias"], t[p + "attn_v.bias"] = ("f32", (H * hd,)), ("f32", (KV * hd,)), ("f32", (KV * hd,))
        if arch in ("qwen3", "qwen3moe", "gemma3"):
            t[p + "attn_q_norm.weight"] = t[p + "attn_k_norm.weight"] = ("f32", (hd,))
        if arch == "gemma3":
            t[p + "post_attention_norm.weight"] = t[p + "post_ffw_norm.weight"] = ("f32", (E,))
        if arch == "qwen3moe":
            t[p + "ffn_gate_inp.weight"] = ("f32", (E, EXPERTS))
            t[p + "ffn_gate_exps.weight"] = t[p + "ffn_up_exps.weight"] = (base, (E, ff, EXPERTS))
            t[p + "ffn_down_exps.weight"] = (base, (ff, E, EXPERTS))
        else:
            t[p + "ffn_gate.weight"] = t[p + "ffn_up.weight"] = (base, (E, ff))
            t[p + "ffn_down.weight"] = ("q6_k" if more and 2 * i >= L else base, (ff, E))
    return t


def _bytes(ty, dims):
    return math.prod(dims) // TYPES[ty][1] * TYPES[ty][2]


def _make(seed, name, ty, dims):
    g = torch.Generator(GPU).manual_seed((seed * 1000003 + zlib.crc32(name.encode())) % (1 << 62))
    n = math.prod(dims)
    if ty == "f32" and len(dims) == 2:  # router: logits of standard deviation 2
        return _float(g, n, torch.float32, 2 / math.sqrt(dims[0]))
    if ty == "f32":
        x = torch.rand(n, device=GPU, generator=g) * 0.2 - 0.1 + (0 if name.endswith("bias") else 1)
        return _u8(x), x.double
    return TYPES[ty][3](g, n)


def _image(case, seed):
    arch, E, _, H, KV, hd, ff, _, _ = PRESETS[case["model"]]

    def text(s):
        return struct.pack("<Q", len(s)) + s.encode()

    u32 = {".embedding_length": E, ".block_count": case["layers"], ".attention.head_count": H, ".attention.head_count_kv": KV,
           ".attention.key_length": hd, ".attention.value_length": hd, ".feed_forward_length": ff, ".vocab_size": case["vocab"],
           ".context_length": 1 << 17, ".rope.dimension_count": hd}
    if arch == "qwen3moe":
        u32.update({".expert_count": EXPERTS, ".expert_used_count": USED, ".expert_feed_forward_length": ff})
    if arch == "gemma3":
        u32[".attention.sliding_window"] = WINDOW
    kv = [text("general.architecture") + struct.pack("<I", 8) + text(arch)]
    kv += [text(arch + k) + struct.pack("<II", 4, v) for k, v in u32.items()]
    kv += [text(arch + k) + struct.pack("<If", 6, v) for k, v in ((".rope.freq_base", 1e6), (".attention.layer_norm_rms_epsilon", EPS))]
    tensors, infos, at = _tensors(case), [], 0
    offsets = {}
    for name, (ty, dims) in tensors.items():
        infos.append(text(name) + struct.pack("<I%dQIQ" % len(dims), len(dims), *dims, TYPES[ty][0], at))
        offsets[name] = at
        at += (_bytes(ty, dims) + 31) // 32 * 32
    head = struct.pack("<IIQQ", 0x46554747, 3, len(tensors), len(kv)) + b"".join(kv + infos)
    start = (len(head) + 31) // 32 * 32
    img = np.empty(start + at, np.uint8)
    img[:start] = np.frombuffer(head.ljust(start, b"\0"), np.uint8)
    host = torch.from_numpy(img)
    for name, (ty, dims) in tensors.items():
        o = start + offsets[name]
        host[o:o + _bytes(ty, dims)] = _make(seed, name, ty, dims)[0].view(-1).cpu()
    return img


def _tokens(case, seed):
    return np.random.default_rng(seed).integers(0, case["vocab"], case["pos"] + case["n"]).astype(np.uint32)


# ---- the call ------------------------------------------------------------------

def prepare(case, seed):
    pos, n = case["pos"], case["n"]
    chunk = max(n, 512)
    be = R.HipBackend(_image(case, seed), n_ctx=pos + n + 128, max_batch=chunk, kv_type=CACHE[case["cache"]])
    tokens = _tokens(case, seed)
    logits = np.zeros((n if case["all"] else 1) * case["vocab"], np.float32)
    for p in range(0, pos, chunk):
        be.forward(tokens[p:min(p + chunk, pos)], p, False, logits[:case["vocab"]])
    return {"backend": be, "tokens": tokens[pos:], "pos": pos, "all": case["all"], "logits": logits}


def run(state):
    return state["backend"].forward(state["tokens"], state["pos"], state["all"], state["logits"])


def work(case):
    arch, E, _, H, KV, hd, ff, _, _ = PRESETS[case["model"]]
    n, pos, V, L = case["n"], case["pos"], case["vocab"], case["layers"]
    rows = n if case["all"] else 1
    nbytes = flops = 0.0
    for name, (ty, dims) in _tensors(case).items():
        b, f = _bytes(ty, dims), 2.0 * n * math.prod(dims)
        if name == "token_embd.weight":
            nbytes += n * b / V
            if PRESETS[case["model"]][8]:
                nbytes, flops = nbytes + b, flops + 2.0 * rows * E * V
        elif name == "output.weight":
            nbytes, flops = nbytes + b, flops + 2.0 * rows * E * V
        elif len(dims) == 3:  # the experts that n tokens of 8 each choose
            nbytes += b * (1 - (1 - USED / EXPERTS) ** n)
            flops += f * USED / EXPERTS
        else:
            nbytes += b
            flops += f if len(dims) == 2 else 0
    row = {"f16": 2 * hd, "q8_0": hd // 32 * 34, "turbo4": hd // 2 + 2}[case["cache"]]
    for i in range(L):
        window = WINDOW if arch == "gemma3" and i % 6 < 5 else pos + n
        seen = sum(min(pos + t + 1, window) for t in range(n))
        nbytes += 2 * KV * row * (min(pos, window) + n)
        flops += 4.0 * H * hd * seen
    return {"bytes": nbytes + 4.0 * rows * V, "flops": flops}


def tolerance(case):
    """Four times what a call's tokens as one batch and as two differ by (other kernels,
    other orders of the f32 sums): 5e-7 to 2e-5 with unquantized weights, 7e-3 to 1.5e-2
    where an 8-bit activation code or a 4- or 8-bit cache code moves."""
    if case["weights"] in ("f16", "bf16"):
        return {"rel": 1e-4, "max": 1e-2} if case["cache"] == "f16" else {"rel": 0.03, "max": 0.3}
    return {"rel": 0.03, "max": 0.3}


# ---- the same call in float64 ----------------------------------------------------

def _norm(x, w):
    return x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * w


def _rope(x, base, neox):
    """x [T, heads, hd]; the angles are f32 products, as every engine's tables hold them"""
    T, hd = x.shape[0], x.shape[2]
    inv = (base ** (-torch.arange(0, hd, 2, device=GPU, dtype=torch.float64) / hd)).float()
    th = (torch.arange(T, device=GPU).float()[:, None] * inv).double()[:, None]
    a, b = (x[..., :hd // 2], x[..., hd // 2:]) if neox else (x[..., 0::2], x[..., 1::2])
    c, s = a * th.cos() - b * th.sin(), a * th.sin() + b * th.cos()
    return torch.cat([c, s], -1) if neox else torch.stack([c, s], -1).flatten(-2)


def _fwht(x):
    n, h = x.shape[-1], 1
    while h < n:
        y = x.view(*x.shape[:-1], n // (2 * h), 2, h)
        x = torch.stack([y[..., 0, :] + y[..., 1, :], y[..., 0, :] - y[..., 1, :]], -2).reshape(x.shape)
        h *= 2
    return x / math.sqrt(n)


def _turbo_signs(hd):
    m, out = (1 << 64) - 1, []
    for i in range(hd):
        z = (0x75426F5175616E74 + i * 0x9E3779B97F4A7C15) & m
        z = ((z ^ z >> 30) * 0xBF58476D1CE4E5B9) & m
        z = ((z ^ z >> 27) * 0x94D049BB133111EB) & m
        out.append(1.0 if (z ^ z >> 31) & 1 == 0 else -1.0)
    return torch.tensor(out, device=GPU, dtype=torch.float64)


def _stored(x, cache):
    """keys or values [T, heads, hd] as the cache holds them"""
    if cache == "f16":
        return x.half().double()
    if cache == "q8_0":
        b = x.view(*x.shape[:2], -1, 32)
        d = b.abs().amax(-1, keepdim=True) / 127
        q = torch.where(d > 0, b / d, torch.zeros_like(b))
        return (d.half().double() * (q.abs() + 0.5).floor().clamp(max=127) * q.sign()).view(x.shape)
    levels = torch.tensor([-126, -95, -74, -58, -43, -30, -18, -6, 6, 18, 30, 43, 58, 74, 95, 126], device=GPU, dtype=torch.float64) / 46
    signs = _turbo_signs(x.shape[-1])
    block = x.shape[-1] & -x.shape[-1]  # rotated in blocks of the largest power of two
    y = _fwht((x * signs).view(*x.shape[:2], -1, block))
    c = levels[torch.bucketize(y / y.square().mean(-1, keepdim=True).sqrt(), (levels[:-1] + levels[1:]) / 2)]
    s = ((y * c).sum(-1, keepdim=True) / c.square().sum(-1, keepdim=True)).half().double()
    return _fwht(s * c).reshape(x.shape) * signs


def _attend(q, k, v, window):
    """q [T, H, hd] scaled, k and v [T, KV, hd]: causal, over the last `window` positions"""
    T, H, hd = q.shape
    KV = k.shape[1]
    out = torch.empty_like(q)
    kt, vt = k.permute(1, 2, 0).contiguous(), v.permute(1, 0, 2).contiguous()
    step = max(1, min(T, (1 << 28) // (T * H)))
    for t in range(0, T, step):
        e = min(T, t + step)
        qs = q[t:e].view(e - t, KV, H // KV, hd).permute(1, 0, 2, 3).reshape(KV, -1, hd)
        s = torch.bmm(qs, kt).view(KV, e - t, H // KV, T)
        i, j = torch.arange(t, e, device=GPU)[:, None], torch.arange(T, device=GPU)[None]
        s.masked_fill_(((j > i) | (j <= i - window))[None, :, None], -math.inf)
        p = torch.softmax(s, -1).view(KV, -1, T)
        out[t:e] = torch.bmm(p, vt).view(KV, e - t, H // KV, hd).permute(1, 0, 2, 3).reshape(e - t, H, hd)
    return out


def exact(case, seed):
    arch, E, _, H, KV, hd, ff, _, tied = PRESETS[case["model"]]
    pos, n, tensors = case["pos"], case["n"], _tensors(case)

    def weight(name):
        ty, dims = tensors[name]
        return _make(seed, name, ty, dims)[1]().view(*reversed(dims))

    gemma, neox = arch == "gemma3", arch != "llama"
    embd = weight("token_embd.weight")
    tokens = torch.from_numpy(_tokens(case, seed).astype(np.int64)).to(GPU)
    x = embd[tokens] * (math.sqrt(E) if gemma else 1.0)
    T = x.shape[0]
    for i in range(case["layers"]):
        p = "blk.%d." % i
        windowed = gemma and i % 6 < 5
        a = _norm(x, weight(p + "attn_norm.weight"))
        q, k, v = (a @ weight(p + "attn_%s.weight" % c).T for c in "qkv")
        if arch == "qwen2":
            q, k, v = q + weight(p + "attn_q.bias"), k + weight(p + "attn_k.bias"), v + weight(p + "attn_v.bias")
        q, k, v = q.view(T, H, hd), k.view(T, KV, hd), v.view(T, KV, hd)
        if arch in ("qwen3", "qwen3moe", "gemma3"):
            q, k = _norm(q, weight(p + "attn_q_norm.weight")), _norm(k, weight(p + "attn_k_norm.weight"))
        base = 1e4 if windowed else 1e6
        q, k = _rope(q, base, neox) / math.sqrt(hd), _rope(k, base, neox)
        o = _attend(q, _stored(k, case["cache"]), _stored(v, case["cache"]), WINDOW if windowed else T)
        o = o.view(T, H * hd) @ weight(p + "attn_output.weight").T
        x = x + (_norm(o, weight(p + "post_attention_norm.weight")) if gemma else o)
        a = _norm(x, weight(p + "ffn_norm.weight"))
        if arch == "qwen3moe":
            prob = torch.softmax(a @ weight(p + "ffn_gate_inp.weight").T, -1)
            top, which = prob.topk(USED, -1)
            top = top / top.sum(-1, keepdim=True)
            gate, up, down = (weight(p + "ffn_%s_exps.weight" % c) for c in ("gate", "up", "down"))
            o = torch.zeros_like(x)
            for e in range(EXPERTS):
                t, j = (which == e).nonzero(as_tuple=True)
                if len(t):
                    h = torch.nn.functional.silu(a[t] @ gate[e].T) * (a[t] @ up[e].T)
                    o.index_add_(0, t, (h @ down[e].T) * top[t, j, None])
            del gate, up, down
        else:
            g = a @ weight(p + "ffn_gate.weight").T
            g = torch.nn.functional.gelu(g, approximate="tanh") if gemma else torch.nn.functional.silu(g)
            o = (g * (a @ weight(p + "ffn_up.weight").T)) @ weight(p + "ffn_down.weight").T
        x = x + (_norm(o, weight(p + "post_ffw_norm.weight")) if gemma else o)
    x = _norm(x[pos if case["all"] else -1:], weight("output_norm.weight"))
    return (x @ (embd if tied else weight("output.weight")).T).view(-1).cpu().numpy()
