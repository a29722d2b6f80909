"""The calls whose speed matters to a user of this package, as cases that can be timed and checked.

Every case is one pass through a public entry point: the C ABI of include/tnhip.h on buffers that the
caller owns (what a host binding calls), or the resident decoder of torchnative_amd.decoder. The ranges
below are the sizes that the package's own benchmark, tests and configurations use, widened to what a
program that serves or runs such models asks for: one activation row to a long prompt, ragged row counts,
output widths that are no multiple of a tile, every weight format, every attention dtype, head dim and mask
kind, short and long caches.
"""

from __future__ import annotations

import ctypes
import functools
import math

import numpy as np
import torch

from torchnative_amd import _lib
from torchnative_amd._lib import check, lib
from torchnative_amd.decoder import LlamaConfig, Q4Llama, inv_freq
from torchnative_amd.tensor import Stream

_TORCH = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
_CODE = {"f32": _lib.TN_F32, "bf16": _lib.TN_BF16, "f16": _lib.TN_F16}
_SIZE = {"f32": 4, "bf16": 2, "f16": 2}
# weight bytes per element as stored: 18 bytes per 32, 34 per 32, 144 per 256
_WEIGHT = {"q4_0": 18 / 32, "q8_0": 34 / 32, "q4_k": 144 / 256, "f32": 4, "f16": 2, "bf16": 2}
_BLOCK = {"q4_0": 32, "q8_0": 32, "q4_k": 256, "f32": 1, "f16": 1, "bf16": 1}
_GGML = ("q4_0", "q8_0", "q4_k")


def listed():
    return [
        # one activation row through a small model's projection: the smallest call, all latency
        _linear("q4_0 one row small", "q4_0", 1, 576, 1536, "f32", "f32"),
        # sixteen sequences decoded together through a large model's MLP projection
        _linear("q4_0 batched decode", "q4_0", 16, 4096, 14336, "bf16", "bf16"),
        # a prompt of 512 tokens through the same projection
        _linear("q4_0 prompt", "q4_0", 512, 4096, 14336, "bf16", "bf16"),
        # a ragged prompt through an 8-bit projection with a bias
        _linear("q8_0 ragged prompt", "q8_0", 200, 1536, 5000, "f32", "f32", bias=True),
        # one row through a large q4_k projection: decoding one sequence from a q4_k file
        _linear("q4_k one row", "q4_k", 1, 4096, 14336, "f32", "f32"),
        # a dense layer (kept dense, or the dense formats of quantize_) over a ragged batch
        _linear("dense f16 batch", "f16", 200, 2048, 2048, "f32", "f32", bias=True),
        # causal grouped-query prefill of a 2048-token prompt, the benchmark's headline
        _sdpa("sdpa causal d64", "bf16", 1, 9, 3, 2048, 2048, 64, True, "none"),
        # two padded prompts at head dim 128: a boolean key padding mask
        _sdpa("sdpa padded d128", "f16", 2, 16, 4, 1000, 1000, 128, False, "key"),
        # a head dim other than 64 and 128, a ragged prompt
        _sdpa("sdpa causal d96", "bf16", 1, 12, 12, 777, 777, 96, True, "none"),
        # sixteen sequences of 512 to 4096 cached tokens, one query token each
        {"name": "decode attention", "op": "decode", "dtype": "bf16", "B": 16, "Hq": 32, "Hkv": 8, "D": 128,
         "cap": 4096, "lo": 512, "hi": 4096},
        # a request to the resident 30-layer decoder: a batched prompt, then steps from a captured graph
        {"name": "prompt and steps", "op": "llama", "layers": 30, "prompt": 400, "steps": 24, "cap": 448},
        # quantising a layer's weight at load time with the search of the q4_k writer
        {"name": "quantize q4_k", "op": "codec", "way": "quantize", "fmt": "q4_k", "n": 4096, "k": 4096},
    ]


def _linear(name, fmt, m, k, n, x, y, bias=False):
    return {"name": name, "op": "linear", "fmt": fmt, "m": m, "k": k, "n": n, "x": x, "y": y, "bias": bias}


def _sdpa(name, dtype, B, Hq, Hkv, L, S, D, causal, mask):
    return {"name": name, "op": "sdpa", "dtype": dtype, "B": B, "Hq": Hq, "Hkv": Hkv, "L": L, "S": S, "D": D,
            "causal": causal, "mask": mask}


def draw(rng):
    """One more case of the ranges above, sizes spread over their logarithm."""
    def log(lo, hi):
        return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))

    op = rng.choice(["linear"] * 4 + ["sdpa"] * 3 + ["decode"] * 2 + ["llama", "codec"])
    while op == "linear":
        fmt = rng.choice(["q4_0", "q4_0", "q8_0", "q4_k", "f32", "f16", "bf16"])
        blk = 256 if fmt == "q4_k" else 32
        k = max(1, log(256, 8192) // blk) * blk
        if fmt not in _GGML and rng.random() < 0.3:
            k += rng.randrange(1, 32)  # a dense layer takes any width
        m, n = (1 if rng.random() < 0.25 else log(1, 1024)), log(64, 16384)
        if rng.random() < 0.6:
            n = max(64, n // 64 * 64)
        most = 512 * 4096 * 14336 if fmt in _GGML else 200 * 2048 * 2048
        if m * k * n > most or n * k > 4096 * 14336:
            continue
        kind = rng.choice(["f32", "bf16"]) if fmt in _GGML else "f32"
        c = _linear("", fmt, m, k, n, kind, kind, rng.random() < 0.3)
        break
    while op == "sdpa":
        D = rng.choice([64, 64, 64, 128, 128, 128, 32, 72, 80, 96, 256])
        dtype = rng.choice(["bf16", "bf16", "f16", "f32"])
        Hkv, rep, B = rng.choice([1, 2, 3, 4, 8]), rng.choice([1, 1, 2, 3, 4]), rng.choice([1, 1, 2, 4])
        S = log(16, 4096)
        L = S if rng.random() < 0.7 else log(1, S)
        causal = L == S and rng.random() < 0.6  # a prompt; fewer queries than keys: a chunk's cross part
        mask = rng.choice(["none", "none", "key", "full"])
        flops = 4 * B * Hkv * rep * D * L * S
        if flops > (16e9 if D in (64, 128) and dtype != "f32" else 3e9):
            continue
        c = _sdpa("", dtype, B, Hkv * rep, Hkv, L, S, D, causal, mask)
        break
    while op == "decode":
        D = rng.choice([64, 64, 128, 128, 96])
        dtype = rng.choice(["bf16", "bf16", "f16", "f32"])
        B, Hkv, rep, cap = log(1, 64), rng.choice([1, 2, 3, 4, 8]), rng.choice([1, 3, 4, 8]), log(64, 16384)
        hi = rng.randrange(max(1, cap // 2), cap + 1)
        lo = rng.randrange(1, hi + 1)
        if B * Hkv * cap * D * _SIZE[dtype] * 2 > (300e6 if D != 96 else 60e6):
            continue
        c = {"op": "decode", "dtype": dtype, "B": B, "Hq": Hkv * rep, "Hkv": Hkv, "D": D, "cap": cap, "lo": lo,
             "hi": hi}
        break
    if op == "llama":
        long_cache = rng.random() < 0.3  # past 512 positions the step's attention takes another path
        prompt, steps = log(1, 400), rng.randrange(0, 9 if long_cache else 25)
        cap = rng.randrange(520, 1500) if long_cache else rng.randrange(prompt + steps, 512)
        c = {"op": "llama", "layers": rng.randrange(16, 31), "prompt": prompt, "steps": steps, "cap": cap}
    if op == "codec":
        fmt = rng.choice(["q4_0", "q8_0", "q4_k"])
        k = max(1, log(256, 8192) // _BLOCK[fmt]) * _BLOCK[fmt]
        c = {"op": "codec", "way": rng.choice(["quantize", "quantize", "dequantize", "upload"]), "fmt": fmt,
             "n": min(log(64, 16384), 4096 * 4096 // k), "k": k}
    c.pop("name", None)
    return c


# --- inputs ------------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) % (1 << 62))


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)


def _f16_bytes(d):
    return d.to(torch.float16).view(torch.uint8).reshape(*d.shape, 2)


def _blocks(fmt, n, k, g):
    """A weight [n, k] as GGML blocks (uint8 [n * k / block, bytes]) and its values in float64 [n, k]: normal
    weights for the 32-element formats, random super-blocks for q4_k. Plain torch throughout."""
    if fmt == "q4_k":
        nb = n * k // 256
        raw = torch.randint(0, 256, (nb, 144), generator=g, device="cuda", dtype=torch.int32).to(torch.uint8)
        raw[:, 0:2] = _f16_bytes(_randn(g, nb).abs() * (0.02 / 63))
        raw[:, 2:4] = _f16_bytes(_randn(g, nb).abs() * (0.002 / 63))
        return raw
    w = (_randn(g, n, k) * 0.02).view(-1, 32)
    if fmt == "q8_0":
        d = w.abs().amax(1) / 127
        q = torch.round(w * torch.where(d > 0, 1 / d, d)[:, None]).clamp(-127, 127).to(torch.int8)
        return torch.cat([_f16_bytes(d), q.view(torch.uint8)], 1)
    d = w.gather(1, w.abs().argmax(1, keepdim=True)).squeeze(1) / -8
    q = (w * torch.where(d != 0, 1 / d, d)[:, None] + 8.5).clamp(0, 15).to(torch.uint8)
    return torch.cat([_f16_bytes(d), q[:, :16] | (q[:, 16:] << 4)], 1)


def _values(fmt, raw, n, k):
    """The float64 values of GGML blocks."""
    f16 = lambda b: b.contiguous().view(torch.float16).to(torch.float64)  # noqa: E731
    if fmt == "q8_0":
        return (raw[:, 2:].contiguous().view(torch.int8).to(torch.float64) * f16(raw[:, 0:2])).view(n, k)
    if fmt == "q4_0":
        q = torch.cat([raw[:, 2:] & 15, raw[:, 2:] >> 4], 1)
        return ((q.to(torch.float64) - 8) * f16(raw[:, 0:2])).view(n, k)
    d, dmin, s = f16(raw[:, 0:2]), f16(raw[:, 2:4]), raw[:, 4:16]
    scale = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).to(torch.float64)
    low = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).to(torch.float64)
    q = raw[:, 16:].view(-1, 4, 32)
    q = torch.stack([q & 15, q >> 4], 2).view(-1, 8, 32).to(torch.float64)
    return (q * (scale * d)[:, :, None] - (low * dmin)[:, :, None]).view(n, k)


def _planes(fmt, raw, n, k):
    """The device planes of GGML blocks, through the upload entry point."""
    blk = _BLOCK[fmt]
    nb = n * k // blk
    if fmt == "q4_k":
        planes = (torch.empty(nb * 144, dtype=torch.uint8, device="cuda"),)
    else:
        planes = (torch.empty(nb * (16 if fmt == "q4_0" else 32), dtype=torch.uint8, device="cuda"),
                  torch.empty(nb, dtype=torch.int16, device="cuda"))
    check(getattr(lib(), f"tn_{fmt}_from_blob")(_stream(), raw.data_ptr(), n, k, *(p.data_ptr() for p in planes)))
    return planes


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _call(fn, *args):
    """One C ABI call with its arguments bound, as a host binding holds them."""
    return functools.partial(fn, *args)


def _linear_inputs(c, seed):
    g = _gen(seed)
    m, k, n, fmt = c["m"], c["k"], c["n"], c["fmt"]
    x = _randn(g, m, k).to(_TORCH[c["x"]])
    bias = _randn(g, n) if c["bias"] else None
    w = _blocks(fmt, n, k, g) if fmt in _GGML else (_randn(g, n, k) * 0.02).to(_TORCH[fmt])
    return x, bias, w


def _prepare_linear(c, seed):
    x, bias, w = _linear_inputs(c, seed)
    m, k, n, fmt = c["m"], c["k"], c["n"], c["fmt"]
    y = torch.empty(m, n, dtype=_TORCH[c["y"]], device="cuda")
    bp = bias.data_ptr() if bias is not None else None
    if fmt in _GGML:
        planes = _planes(fmt, w, n, k)
        call = _call(getattr(lib(), f"tn_{fmt}_linear"), _stream(), x.data_ptr(), _CODE[c["x"]], m, k,
                     *(p.data_ptr() for p in planes), n, bp, y.data_ptr(), _CODE[c["y"]])
    else:
        planes = (w,)
        call = _call(lib().tn_dense_linear, _stream(), x.data_ptr(), m, k, w.data_ptr(), _CODE[fmt], n, bp,
                     y.data_ptr())
    return {"call": call, "out": y, "keep": (x, bias, planes)}


def _exact_linear(c, seed):
    x, bias, w = _linear_inputs(c, seed)
    fmt = c["fmt"]
    x = x.to(torch.float32)
    if fmt in _GGML:
        x, w = _activation(x, fmt), _values(fmt, w, c["n"], c["k"])
    y = x.to(torch.float64) @ w.to(torch.float64).t()
    return y + bias.to(torch.float64) if bias is not None else y


def _round_away(v):
    t = torch.trunc(v)
    return t + torch.where((v - t).abs() >= 0.5, torch.sign(v), torch.zeros_like(v))


def _activation(x, fmt="q4_0"):
    """The float64 values of the block-quantised activation that the linear contracts with: 32-element blocks
    with an f16 scale, for q4_k 256-element ones with an f32 scale of the signed extreme over -127."""
    if fmt == "q4_k":
        b = x.reshape(-1, 256)
        ext = b.gather(1, b.abs().argmax(1, keepdim=True))
        inv = torch.where(ext != 0, -127 / ext, torch.zeros_like(ext))
        q = _round_away(b * inv).clamp(-128, 127)
        scale = torch.where(inv != 0, 1 / inv, inv)
        return (q.to(torch.float64) * scale.to(torch.float64)).reshape(x.shape)
    b = x.reshape(-1, 32)
    d = b.abs().amax(1, keepdim=True) / 127
    q = _round_away(b * torch.where(d != 0, 1 / d, d)).clamp(-128, 127)
    return (q.to(torch.float64) * d.to(torch.float16).to(torch.float64)).reshape(x.shape)


# --- attention ------------------------------------------------------------------------


def _sdpa_inputs(c, seed):
    g = _gen(seed)
    B, Hq, Hkv, L, S, D = (c[i] for i in ("B", "Hq", "Hkv", "L", "S", "D"))
    q, k, v = (_randn(g, B, h, t, D).to(_TORCH[c["dtype"]]) for h, t in ((Hq, L), (Hkv, S), (Hkv, S)))
    mask = None
    if c["mask"] == "key":  # each sequence hides its padding at the end
        keep = torch.randint(max(1, S // 2), S + 1, (B, 1, 1, 1), generator=g, device="cuda")
        mask = torch.arange(S, device="cuda").view(1, 1, 1, S) < keep
    elif c["mask"] == "full":  # an additive bias per (query, key), the same for every head
        mask = _randn(g, B, 1, L, S).to(_TORCH[c["dtype"]])
    return q, k, v, mask


def _prepare_sdpa(c, seed):
    q, k, v, mask = _sdpa_inputs(c, seed)
    B, Hq, Hkv, L, S, D = (c[i] for i in ("B", "Hq", "Hkv", "L", "S", "D"))
    out = torch.empty_like(q)
    lse = torch.empty(B, Hq, L, dtype=torch.float32, device="cuda")
    strides, code = None, 0
    if mask is not None:
        shape = tuple(mask.shape)
        strides = (ctypes.c_int64 * 4)(*(0 if s == 1 else mask.stride(i) for i, s in enumerate(shape)))
        code = _lib.TN_BOOL if mask.dtype == torch.bool else _CODE[c["dtype"]]
    call = _call(lib().tn_sdpa_fwd, _stream(), _CODE[c["dtype"]], q.data_ptr(), k.data_ptr(), v.data_ptr(), B, Hq,
                 Hkv, L, S, D, mask.data_ptr() if mask is not None else None, code, strides, int(c["causal"]),
                 float("nan"), out.data_ptr(), lse.data_ptr())
    return {"call": call, "out": (out, lse), "keep": (q, k, v, mask)}


def _attend(q, k, v, add):
    s = (q @ k.transpose(-1, -2)) / math.sqrt(q.shape[-1])
    if add is not None:
        s = s + add
    return torch.softmax(s, -1) @ v, torch.logsumexp(s, -1)


def _exact_sdpa(c, seed):
    q, k, v, mask = _sdpa_inputs(c, seed)
    B, Hq, Hkv, L, S = (c[i] for i in ("B", "Hq", "Hkv", "L", "S"))
    add = torch.zeros(B, 1, L, S, dtype=torch.float64, device="cuda")
    if mask is not None and mask.dtype == torch.bool:
        add = add.masked_fill(~mask, -math.inf)
    elif mask is not None:
        add = add + mask.to(torch.float64)
    if c["causal"]:
        t = torch.arange(L, device="cuda")[:, None] < torch.arange(S, device="cuda")[None]
        add = add.masked_fill(t, -math.inf)
    q, k, v = (t.to(torch.float64) for t in (q, k, v))
    outs, lses = [], []
    for b in range(B):
        for h in range(Hq):
            kv = h // (Hq // Hkv)
            o, e = _attend(q[b, h], k[b, kv].contiguous(), v[b, kv].contiguous(), add[b, 0])
            outs.append(o)
            lses.append(e)
    return torch.stack(outs).view(q.shape), torch.stack(lses).view(B, Hq, L)


def _lengths(c):
    """Cached lengths spread evenly from lo to hi: the same total for every seed."""
    return [c["lo"] + (c["hi"] - c["lo"]) * (2 * b + 1) // (2 * c["B"]) for b in range(c["B"])]


def _decode_inputs(c, seed):
    g = _gen(seed)
    B, Hq, Hkv, D, cap = (c[i] for i in ("B", "Hq", "Hkv", "D", "cap"))
    q, k, v = (_randn(g, *s).to(_TORCH[c["dtype"]]) for s in ((B, Hq, D), (B, Hkv, cap, D), (B, Hkv, cap, D)))
    order = torch.randperm(B, generator=g, device="cuda")
    lens = torch.tensor(_lengths(c), dtype=torch.int32, device="cuda")[order]
    return q, k, v, lens


def _prepare_decode(c, seed):
    q, k, v, lens = _decode_inputs(c, seed)
    out = torch.empty_like(q)
    lse = torch.empty(c["B"], c["Hq"], dtype=torch.float32, device="cuda")
    call = _call(lib().tn_sdpa_decode, _stream(), _CODE[c["dtype"]], q.data_ptr(), k.data_ptr(), v.data_ptr(),
                 c["B"], c["Hq"], c["Hkv"], c["cap"], c["D"], lens.data_ptr(), max(_lengths(c)), float("nan"),
                 out.data_ptr(), lse.data_ptr())
    return {"call": call, "out": (out, lse), "keep": (q, k, v, lens)}


def _exact_decode(c, seed):
    q, k, v, lens = _decode_inputs(c, seed)
    rep = c["Hq"] // c["Hkv"]
    out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
    lse = torch.empty(q.shape[:2], dtype=torch.float64, device="cuda")
    for b, n in enumerate(lens.tolist()):
        for h in range(c["Hkv"]):
            rows = slice(h * rep, (h + 1) * rep)
            out[b, rows], lse[b, rows] = _attend(q[b, rows].double(), k[b, h, :n].double(), v[b, h, :n].double(),
                                                 None)
    return out, lse


# --- the resident decoder ----------------------------------------------------------------


def _config(c):
    return LlamaConfig(n_layers=c["layers"])


def _llama_weights(cfg, seed):
    """N(0, 0.02) weights by layer, as (layer function, top) of host arrays; the norm weights near one."""
    H, D, I = cfg.hidden, cfg.head_dim, cfg.inter
    g = _gen(seed)

    def w(*shape):
        return (_randn(g, *shape) * 0.02).cpu().numpy()

    def norm():
        return (1 + 0.1 * _randn(g, H)).cpu().numpy()

    layers = [{"qkv": w((cfg.n_heads + 2 * cfg.n_kv_heads) * D, H), "o": w(H, cfg.n_heads * D),
               "gate_up": w(2 * I, H), "down": w(H, I), "ln1": norm(), "ln2": norm()} for _ in range(cfg.n_layers)]
    return layers, {"embed": w(cfg.vocab, H), "norm": norm(), "lm_head": w(cfg.vocab, H)}


def _prompt(c, seed):
    cfg = _config(c)
    return np.random.default_rng(seed).integers(0, cfg.vocab, c["prompt"] + c["steps"]).astype(np.int32)


class _Memory:
    """Device memory of the model's, as torch can look at it."""

    def __init__(self, ptr, shape, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f4", "data": (ptr, False), "version": 2}


def _prepare_llama(c, seed):
    cfg = _config(c)
    layers, top = _llama_weights(cfg, seed)
    model = Q4Llama(cfg, cap=c["cap"], weights=(lambda i: layers[i], top))
    prompt = _prompt(c, seed)
    graph = None
    if c["steps"]:
        model.start(prompt)
        stream = Stream()  # the default stream cannot be captured
        graph = model.capture(c["steps"], stream.handle)
    look = lambda p, *s: torch.as_tensor(_Memory(p, s, model), device="cuda")  # noqa: E731
    n, out = c["prompt"] + c["steps"], {"logits": look(model.logits.data_ptr(), cfg.vocab)}
    for i in (0, cfg.n_layers // 2, cfg.n_layers - 1):  # the cache rows that the request wrote
        L = model._layers[i]
        out[f"k{i}"], out[f"v{i}"] = (look(p, cfg.n_kv_heads, c["cap"], cfg.head_dim)[:, :n]
                                      for p in (L.k_cache, L.v_cache))
    return {"model": model, "prompt": prompt, "graph": graph, "n": c["prompt"], "out": out}


def _run_llama(s):
    # the prompt's rows in one batched pass, then the steps; the later tokens are given, so that every pass does
    # the same work whatever the arg-max of a random model is
    s["model"].start(s["prompt"])
    s["model"].prefill(s["n"])
    if s["graph"] is not None:
        s["graph"].launch(None)
    return s["out"]


def _exact_llama(c, seed):
    cfg = _config(c)
    layers, top = _llama_weights(cfg, seed)
    n, D, Hq, Hkv = c["prompt"] + c["steps"], cfg.head_dim, cfg.n_heads, cfg.n_kv_heads

    def q4(w):
        w = torch.from_numpy(w).cuda().view(-1, 32)
        d = w.gather(1, w.abs().argmax(1, keepdim=True)) / -8
        q = (w * torch.where(d != 0, 1 / d, d) + 8.5).clamp(0, 15).trunc()
        return (q.double() - 8) * d.to(torch.float16).double()

    def lin(x, w):
        return _activation(x) @ q4(w).view(w.shape).t()

    def norm(x, w):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + cfg.eps) * torch.from_numpy(w).cuda().double()

    ang = torch.arange(n, device="cuda").double()[:, None] * torch.from_numpy(inv_freq(cfg)).cuda().double()[None]
    cos, sin = torch.cat([ang.cos()] * 2, 1), torch.cat([ang.sin()] * 2, 1)
    rope = lambda t: t * cos + torch.cat([-t[..., D // 2:], t[..., :D // 2]], -1) * sin  # noqa: E731
    causal = torch.zeros(n, n, device="cuda", dtype=torch.float64).masked_fill(
        torch.ones(n, n, device="cuda", dtype=torch.bool).triu(1), -math.inf)
    h = torch.from_numpy(top["embed"][_prompt(c, seed)]).cuda().double()
    out = {}
    for i, w in enumerate(layers):
        qkv = lin(norm(h, w["ln1"]), w["qkv"]).view(n, Hq + 2 * Hkv, D).transpose(0, 1)
        q, k, v = rope(qkv[:Hq]), rope(qkv[Hq:Hq + Hkv]), qkv[Hq + Hkv:]
        if i in (0, cfg.n_layers // 2, cfg.n_layers - 1):
            out[f"k{i}"], out[f"v{i}"] = k, v
        a = [_attend(q[j], k[j // (Hq // Hkv)], v[j // (Hq // Hkv)], causal)[0] for j in range(Hq)]
        h = h + lin(torch.stack(a, 1).reshape(n, Hq * D), w["o"])
        gate, up = lin(norm(h, w["ln2"]), w["gate_up"]).split(cfg.inter, 1)
        h = h + lin(torch.nn.functional.silu(gate) * up, w["down"])
    out["logits"] = lin(norm(h[-1:], top["norm"]), top["lm_head"])[0]
    return out


# --- weights at load time ----------------------------------------------------------------


def _prepare_codec(c, seed):
    g, fmt, n, k = _gen(seed), c["fmt"], c["n"], c["k"]
    if c["way"] == "quantize":
        w = _randn(g, n, k) * 0.02
        nb = n * k // _BLOCK[fmt]
        out = ((torch.empty(nb * 144, dtype=torch.uint8, device="cuda"),) if fmt == "q4_k" else
               (torch.empty(nb * (16 if fmt == "q4_0" else 32), dtype=torch.uint8, device="cuda"),
                torch.empty(nb, dtype=torch.int16, device="cuda")))
        call = _call(getattr(lib(), f"tn_{fmt}_quantize"), _stream(), w.data_ptr(), n, k,
                     *(o.data_ptr() for o in out))
        return {"call": call, "out": out, "keep": w}
    raw = _blocks(fmt, n, k, g)
    planes = _planes(fmt, raw, n, k)
    if c["way"] == "upload":
        call = _call(getattr(lib(), f"tn_{fmt}_from_blob"), _stream(), raw.data_ptr(), n, k,
                     *(p.data_ptr() for p in planes))
        return {"call": call, "out": planes, "keep": raw}
    out = torch.empty(n, k, dtype=torch.float32, device="cuda")
    call = _call(getattr(lib(), f"tn_{fmt}_dequantize"), _stream(), *(p.data_ptr() for p in planes), n, k,
                 out.data_ptr())
    return {"call": call, "out": out, "keep": planes}


def _exact_codec(c, seed):
    if c["way"] != "dequantize":
        return None  # bytes
    return _values(c["fmt"], _blocks(c["fmt"], c["n"], c["k"], _gen(seed)), c["n"], c["k"])


# --- what a measuring program calls ---------------------------------------------------------

_PREPARE = {"linear": _prepare_linear, "sdpa": _prepare_sdpa, "decode": _prepare_decode, "llama": _prepare_llama,
            "codec": _prepare_codec}
_EXACT = {"linear": _exact_linear, "sdpa": _exact_sdpa, "decode": _exact_decode, "llama": _exact_llama,
          "codec": _exact_codec}


def prepare(case, seed):
    return _PREPARE[case["op"]](case, seed)


def run(state):
    call = state.get("call")
    if call is None:
        return _run_llama(state)
    status = call()
    if status:
        check(status)
    return state["out"]


def exact(case, seed):
    return _EXACT[case["op"]](case, seed)


def work(case):
    c = case
    if c["op"] == "linear":
        m, k, n = c["m"], c["k"], c["n"]
        return {"bytes": n * k * _WEIGHT[c["fmt"]] + m * k * _SIZE[c["x"]] + m * n * _SIZE[c["y"]]
                + (4 * n if c["bias"] else 0), "flops": 2 * m * k * n}
    if c["op"] == "sdpa":
        B, Hq, Hkv, L, S, D = (c[i] for i in ("B", "Hq", "Hkv", "L", "S", "D"))
        full = min(L, S)
        pairs = full * (full + 1) / 2 + max(0, L - S) * S if c["causal"] else L * S
        if c["mask"] == "key":
            pairs *= 0.75  # the padding hides a quarter of the keys on average
        size = _SIZE[c["dtype"]]
        mask = {"none": 0, "key": B * S, "full": B * L * S * size}[c["mask"]]
        return {"bytes": size * D * B * (2 * Hq * L + 2 * Hkv * S) + 4 * B * Hq * L + mask,
                "flops": 4 * B * Hq * D * pairs}
    if c["op"] == "decode":
        tokens, size = sum(_lengths(c)), _SIZE[c["dtype"]]
        return {"bytes": 2 * tokens * c["Hkv"] * c["D"] * size + c["B"] * c["Hq"] * (2 * c["D"] * size + 4),
                "flops": 4 * tokens * c["Hq"] * c["D"]}
    if c["op"] == "llama":
        cfg = _config(c)
        per_layer = cfg.hidden * ((2 * cfg.n_heads + 2 * cfg.n_kv_heads) * cfg.head_dim + 3 * cfg.inter)
        body, head = cfg.n_layers * per_layer, cfg.vocab * cfg.hidden
        p, s = c["prompt"], c["steps"]
        row = 2 * cfg.n_layers * cfg.n_kv_heads * cfg.head_dim * 4  # one position's cache rows
        read = sum(range(p + 1, p + s + 1)) * row  # the cached rows that the steps read
        pairs = (p + s) * (p + s + 1) / 2
        return {"bytes": (1 + s) * (body + head) * 18 / 32 + read + (p + s) * (row + cfg.hidden * 4)
                + (1 + s) * cfg.vocab * 4,
                "flops": 2 * (p + s) * body + 2 * (1 + s) * head + 4 * cfg.n_layers * cfg.n_heads * cfg.head_dim * pairs}
    size = {"quantize": 4 + _WEIGHT[c["fmt"]], "dequantize": 4 + _WEIGHT[c["fmt"]], "upload": 2 * _WEIGHT[c["fmt"]]}
    return {"bytes": c["n"] * c["k"] * size[c["way"]], "flops": 0}


def tolerance(case):
    """Block-quantised linears, the dense linear and the weight codecs have one defined sequence of roundings
    (include/tnhip.h), so their results are the same bits. The attention's order of sums is free: f32 sums, and
    for 16-bit inputs the probabilities and the output rounded to that type. The decoder requantises every
    activation to 8 bits, so a difference in the last bit moves codes in all later layers, until after some
    ten layers the whole rounding noise of the codes (1.3e-2 of a result) is another."""
    if case["op"] in ("linear", "codec"):
        return "exact"
    if case["op"] == "llama":
        return {"rel": 0.03, "max": 0.25}
    return {"bf16": {"rel": 7e-3, "max": 0.05}, "f16": {"rel": 1e-3, "max": 0.01},
            "f32": {"rel": 5e-6, "max": 5e-5}}[case["dtype"]]
