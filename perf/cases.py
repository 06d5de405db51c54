"""What is measured: the calls that a serving program makes on this library.

Kinds of cases, each through the public entry points:

* ``decode``  one decode-attention step of a batch over its filled cache
  (``TQKVPool.decode``);
* ``prefill`` a batch's prompt appended in chunks, coded on flush
  (``TQKVPool.append``);
* ``chat``    one conversation through the drop-in cache: the prompt, then one
  append and one decode per new token (``TurboQuantKVCache``);
* ``save``    one layer block quantized into its containers for the block
  store (the ``per_channel`` and ``polar`` plugins' ``compress``);
* ``load``    the same containers back to dense K/V (``decompress``);
* ``dense``   a prompt through the HF cache layer, which returns dense K/V for
  the prefill's attention (``TurboQuantLayer.update``).

Inputs: keys N(0,1) times a lognormal scale per channel, 2 % of the channels
ten times larger, with RoPE; values and queries N(0,1).  ``exact`` restates
the codecs and the attention in plain 64-bit torch.
"""

from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(1, os.path.join(os.getcwd(), "turboquant-pro_amd"))

CHUNK = 4096
# Lloyd-Max N(0,1) levels and NormalFloat-4 levels: the formats' tables
LLOYD_MAX = {
    2: (-1.510, -0.453, 0.453, 1.510),
    3: (-1.748, -1.050, -0.500, -0.069, 0.069, 0.500, 1.050, 1.748),
    4: (-2.401, -1.844, -1.437, -1.099, -0.800, -0.524, -0.262, -0.066,
        0.066, 0.262, 0.524, 0.800, 1.099, 1.437, 1.844, 2.401),
}
NF4 = (-1.0, -0.6961928009986877, -0.5250730514526367, -0.39491748809814453, -0.28444138169288635,
       -0.18477343022823334, -0.09105003625154495, 0.0, 0.07958029955625534, 0.16093020141124725,
       0.24611230194568634, 0.33791524171829224, 0.44070982933044434, 0.5626170039176941,
       0.7229568362236023, 1.0)


def _decode(name, **kw):
    case = dict(name=name, kind="decode", batch=16, kv_heads=8, q_heads=32, head_dim=128, length=32768,
                ragged=False, page=0, hot_window=512, grid="nf4_asym", key_bits=4, value_bits=3,
                outliers=0.02, dtype="float16")
    case.update(kw)
    return case


def _prefill(name, **kw):
    case = _decode(name, kind="prefill", length=8192, chunk=CHUNK)
    case.update(kw)
    return case


def listed():
    return [
        # a short chat on one multi-head sequence with the robust preset: a
        # few thousand tokens, where launches and set-up count
        _decode("decode_b1_4k", batch=1, kv_heads=32, length=4096, value_bits=4),
        # the headline serving step: 16 sequences at full context, 32 / 8 heads
        _decode("decode_b16_32k"),
        # one very long context: the chip filled by splitting one sequence
        _decode("decode_b1_128k", batch=1, length=131072),
        # continuous batching: ragged lengths in 16-token pages of a shuffled table
        _decode("decode_ragged", batch=32, ragged=True, page=16),
        # head_dim 256 (gemma-2-9b's 16 / 8 heads)
        _decode("decode_d256_8k", q_heads=16, head_dim=256, length=8192),
        # a bf16 or fp32 model's cache kept exactly: fp32 hot window and queries
        _decode("decode_f32_8k", length=8192, dtype="float32"),
        # a batch of long prompts, appended in chunks
        _prefill("prefill_b16_8k"),
        # prompts of a bf16 or fp32 model kept exactly, an odd length
        _prefill("prefill_f32", batch=4, length=5000, dtype="float32"),
        # one conversation: a prompt, then token by token (host path and launches)
        dict(name="chat", kind="chat", kv_heads=8, q_heads=32, head_dim=128, prompt=1000, steps=32),
        # a whole request's layer block into the store (which hands the
        # quantizers fp32 tokens), and a block back out of it
        dict(name="block_save", kind="save", batch=1, kv_heads=8, head_dim=128, length=16000,
             value_bits=3, dtype="float32"),
        dict(name="block_load", kind="load", batch=1, kv_heads=8, head_dim=128, length=4000,
             value_bits=3, dtype="float16"),
        # an HF model's prompt: coded, and dense K/V back for the prefill's attention
        dict(name="dense_prefill", kind="dense", batch=2, kv_heads=8, head_dim=128, length=4000,
             value_bits=4, dtype="bfloat16"),
    ]


def _log(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "chat", "save", "load", "dense"])
    D = rng.choice([64, 128, 128, 128, 256])
    H = rng.choice([1, 2, 4, 8, 8, 16])
    if kind == "chat":
        return dict(kind=kind, kv_heads=H, q_heads=H * rng.choice([1, 2, 4, 7, 8]), head_dim=D,
                    prompt=_log(rng, 20, 3000), steps=rng.randint(3, 40))
    if kind in ("save", "load", "dense"):
        B = rng.choice([1, 1, 2])
        top = {"save": 16000, "load": 4000, "dense": 8000}[kind] * 8 * 128 // (B * H * D)
        return dict(kind=kind, batch=B, kv_heads=H, head_dim=D, length=_log(rng, 40, min(top, 32000)),
                    value_bits=rng.choice([2, 3, 4]),
                    dtype={"save": "float32", "load": rng.choice(["float16", "float32"]),
                           "dense": rng.choice(["float16", "bfloat16"])}[kind])
    grid, kb, out = rng.choice([("nf4_asym", 4, 0.02), ("nf4_asym", 4, 0.02), ("nf4_asym", 4, 0.0),
                                ("uniform", 4, 0.0), ("uniform", 3, 0.0), ("uniform", 2, 0.02),
                                ("polar", 3, 0.0), ("polar", 4, 0.0)])
    dtype = rng.choice(["float16", "float16", "float16", "float32"])
    W, page = rng.choice([(512, 0), (512, 0), (512, 16), (256, 0), (64, 0), (48, 0)])
    case = _decode("", kind=kind, batch=_log(rng, 1, 32), kv_heads=H, q_heads=H * rng.choice([1, 2, 4, 7, 8]),
                   head_dim=D, ragged=rng.random() < 0.3, hot_window=W, page=page, grid=grid, key_bits=kb,
                   value_bits=kb if grid == "polar" else rng.choice([2, 3, 4]), outliers=out, dtype=dtype)
    # at most the largest listed case's tokens; a quarter of them off the
    # head_dim-128 fp16 path
    cells = (16 * 32768 if kind == "decode" else 16 * 8192) * 8 * 128
    if dtype == "float32" or D != 128 or W < 256:
        cells //= 4
    top = max(700, min(65536, cells // (case["batch"] * H * D)))
    case["length"] = _log(rng, 600, top)
    if kind == "prefill":
        case["chunk"] = rng.choice([500, 2048, 4096])
    del case["name"]
    return case


# ------------------------------------------------------------------ shapes --
def _groups(length, W):
    G = (W + 1) // 2
    return 0 if length <= W else (length - (W + 1)) // G + 1


def _lengths(case):
    if case.get("ragged"):
        rng = np.random.default_rng(case["batch"] * 7919 + case["length"])
        low = min(1024, max(1, case["length"] // 4))
        return [int(n) for n in rng.integers(low, case["length"] + 1, size=case["batch"])]
    return [case["length"]] * case["batch"]


# ------------------------------------------------------------------ inputs --
def _tokens(B, H, L, D, dtype, seed):
    """Keys and values ``(B, H, L, D)`` of ``dtype``."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    scale = torch.exp(torch.randn((B, H, 1, D), generator=gen, device="cuda"))
    big = torch.rand((B, H, 1, D), generator=gen, device="cuda").argsort(-1) < max(1, round(0.02 * D))
    scale = torch.where(big, 10.0 * scale, scale)
    half = D // 2
    inv = 10000.0 ** (-2.0 * torch.arange(half, device="cuda", dtype=torch.float64) / D)
    k = torch.empty((B, H, L, D), dtype=dtype, device="cuda")
    v = torch.empty_like(k)
    for t in range(0, L, CHUNK):
        n = min(CHUNK, L - t)
        x = torch.randn((B, H, n, D), generator=gen, device="cuda") * scale
        ang = torch.arange(t, t + n, device="cuda", dtype=torch.float64)[:, None] * inv
        cos, sin = ang.cos().float(), ang.sin().float()
        a, b = x[..., :half], x[..., half:]
        k[:, :, t:t + n, :half] = a * cos - b * sin
        k[:, :, t:t + n, half:] = b * cos + a * sin
        v[:, :, t:t + n] = torch.randn((B, H, n, D), generator=gen, device="cuda")
    return k, v


def _queries(case, n, dtype, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed + 1)
    return torch.randn((n, case["q_heads"], case["head_dim"]), generator=gen, device="cuda").to(dtype)


def _case_tokens(case, seed):
    L = case["prompt"] + case["steps"] if case["kind"] == "chat" else case["length"]
    k, v = _tokens(case.get("batch", 1), case["kv_heads"], L, case["head_dim"],
                   getattr(torch, case.get("dtype", "float16")), seed)
    if case["kind"] == "save":
        # no two magnitudes of a channel equal where its outliers end: as many
        # outliers, and so outputs of one shape, for every seed
        mag = k.abs()
        tied = mag == mag.topk(max(1, round(0.02 * L)), dim=2).values[:, :, -1:]
        nth = tied.cumsum(2) - 1
        k = torch.where(tied & (nth > 0), k * (1.0 - nth * 2.0 ** -18), k)
    return k, v


def _pool(case, seed):
    from turboquant_pro_amd import TQKVPool
    extra = {}
    if case["page"]:
        W = case["hot_window"]
        pages = max(1, _groups(case["length"], W)) * ((W + 1) // 2) // case["page"]
        extra = dict(page_tokens=case["page"], block_table=np.random.default_rng(4).permutation(
            case["batch"] * pages).astype(np.int32))
    return TQKVPool(n_kv_heads=case["kv_heads"], n_q_heads=case["q_heads"], head_dim=case["head_dim"],
                    max_batch=case["batch"], max_seq_len=case["length"], hot_window=case["hot_window"],
                    key_bits=case["key_bits"], value_bits=case["value_bits"], outlier_frac=case["outliers"],
                    key_grid=case["grid"], input_dtype=case["dtype"], seed=seed, **extra)


class _State:
    pass


def prepare(case, seed):
    s = _State()
    s.case = case
    k, v = _case_tokens(case, seed)
    kind = case["kind"]
    if kind == "decode":
        lens = _lengths(case)
        s.pool = _pool(case, seed)
        for t in range(0, case["length"], CHUNK):
            n = min(CHUNK, case["length"] - t)
            s.pool.append(k[:, :, t:t + n], v[:, :, t:t + n], n_new=[min(n, max(0, L - t)) for L in lens])
        s.pool.check()
        s.q = _queries(case, case["batch"], s.pool.dtype, seed)
    elif kind == "prefill":
        s.pool = _pool(case, seed)
        lens = _lengths(case)
        s.chunks = []
        for t in range(0, case["length"], case["chunk"]):
            n = min(case["chunk"], case["length"] - t)
            s.chunks.append((k[:, :, t:t + n].contiguous(), v[:, :, t:t + n].contiguous(),
                             [min(n, max(0, L - t)) for L in lens]))
    elif kind == "chat":
        from turboquant_pro_amd import TurboQuantKVCache
        H, D = case["kv_heads"], case["head_dim"]
        s.cache = TurboQuantKVCache.robust(head_dim=D, n_heads=H, n_q_heads=case["q_heads"], seed=seed)
        P = case["prompt"]
        s.prompt = (k[0, :, :P].contiguous(), v[0, :, :P].contiguous())
        s.steps = [(k[0, :, P + i].contiguous(), v[0, :, P + i].contiguous()) for i in range(case["steps"])]
        s.q = list(_queries(case, case["steps"], torch.float16, seed))
    elif kind in ("save", "load"):
        from turboquant_pro_amd import plugins
        s.keys = plugins.create("per_channel", head_dim=case["head_dim"], n_heads=case["kv_heads"],
                                nf4_asym=True, outlier_frac=0.02)
        s.values = plugins.create("polar", head_dim=case["head_dim"], n_heads=case["kv_heads"],
                                  bits=case["value_bits"], seed=seed)
        s.k, s.v = k, v
        if kind == "load":
            s.k, s.v = s.keys.compress(k, packed=True), s.values.compress(v, packed=True)
    else:
        from turboquant_pro_amd.hf_cache import TurboQuantLayer
        s.layer = TurboQuantLayer(hot_window=512, key_bits=4, value_bits=case["value_bits"],
                                  outlier_frac=0.02, seed=seed)
        s.k, s.v = k, v
    return s


def run(s):
    kind = s.case["kind"]
    if kind == "decode":
        return s.pool.decode(s.q)
    if kind == "prefill":
        s.pool.reset()
        for k, v, n in s.chunks:
            s.pool.append(k, v, n_new=n)
        p = s.pool
        return {"kcodes": p.kcodes, "vcodes": p.vcodes, "vnorm": p.vnorm, "scale": p.gscale, "mean": p.gmean,
                "ocount": p.ocount, "oent": p.oent, "hot_k": p.hot_k, "hot_v": p.hot_v}
    if kind == "chat":
        s.cache.clear()
        s.cache.extend(*s.prompt)
        out = []
        for (k, v), q in zip(s.steps, s.q):
            s.cache.append(k, v)
            out.append(s.cache.fused_decode(q))
        return torch.stack(out)
    if kind == "save":
        k, v = s.keys.compress(s.k, packed=True), s.values.compress(s.v, packed=True)
        return {"kcodes": k.indices, "scale": k.nf4_scale, "mean": k.nf4_mean, "oidx": k.outlier_idx,
                "oval": k.outlier_val, "vcodes": v.indices, "norms": v.norms}
    if kind == "load":
        return {"k": s.keys.decompress(s.k), "v": s.values.decompress(s.v)}
    s.layer.reset()
    k, v = s.layer.update(s.k, s.v)
    return {"k": k, "v": v}


# -------------------------------------------------------------------- work --
def _code_bytes(case, tokens, groups):
    """Coded bytes of ``tokens`` cold tokens of one kv head in ``groups`` groups:
    codes, norms, per-channel scale and zero point, fp16 outliers with their
    positions (6 bytes each)."""
    D, kb, vb = case["head_dim"], case.get("key_bits", 4), case["value_bits"]
    G = tokens // groups if groups else 0
    out = case.get("outliers", 0.02)
    n_out = max(1, round(G * out)) * D if out and case.get("grid") != "polar" else 0
    polar = case.get("grid") == "polar"
    return (tokens * (D * kb // 8 + D * vb // 8 + 4 + (4 if polar else 0))
            + groups * ((0 if polar else 8 * D) + 6 * n_out))


def work(case):
    kind, H, D = case["kind"], case["kv_heads"], case["head_dim"]
    if kind in ("decode", "prefill"):
        W = case["hot_window"]
        G, tok = (W + 1) // 2, 4 if case["dtype"] == "float32" else 2
        nbytes = flops = 0
        for L in _lengths(case):
            ng = _groups(L, W)
            coded = _code_bytes(case, ng * G, ng)
            if kind == "decode":
                nbytes += H * (coded + (L - ng * G) * 2 * D * tok) + case["q_heads"] * D * (tok + 4)
                flops += 4 * case["q_heads"] * L * D
            else:
                nbytes += H * (L * 2 * D * tok + coded + (L - ng * G) * 2 * D * tok)
                flops += H * ng * G * 2 * D * D * (2 if case["grid"] == "polar" else 1)
        return {"bytes": nbytes, "flops": flops}
    if kind == "chat":
        P, n, Hq = case["prompt"], case["steps"], case["q_heads"]
        c = dict(case, value_bits=4)
        nbytes = H * (P + n) * 4 * D
        flops = H * _groups(P + n, 512) * 256 * 2 * D * D
        for i in range(n):
            L = P + i + 1
            ng = _groups(L, 512)
            nbytes += H * (_code_bytes(c, ng * 256, ng) + (L - ng * 256) * 4 * D) + Hq * D * 6
            flops += 4 * Hq * L * D
        return {"bytes": nbytes, "flops": flops}
    B, L = case["batch"], case["length"]
    if kind in ("save", "load"):
        dense = B * H * L * 2 * D * (4 if kind == "load" or case["dtype"] == "float32" else 2)
        return {"bytes": dense + B * H * _code_bytes(case, L, 1), "flops": B * H * L * 2 * D * D}
    ng = _groups(L, 512)
    # the prompt in, its codes out and in again, dense K/V out
    return {"bytes": B * H * (2 * L * 4 * D + 2 * _code_bytes(case, ng * 256, ng)),
            "flops": B * H * ng * 256 * 4 * D * D}


def tolerance(case):
    if case["kind"] not in ("chat", "decode"):
        return "exact"  # whole codes, and numbers that are the reference's bit for bit
    if case["head_dim"] == 128 and case.get("dtype", "float16") == "float16":
        # value centroids in fp16, softmax weights as fp16 pairs: 2.5e-4 off the exact result
        return {"rel": 1e-3}
    return {"rel": 2e-5}  # 32-bit sums over the context


# ------------------------------------------------------------------- exact --
def _rotation(seed, D):
    gauss = np.random.default_rng(seed).standard_normal((D, D)).astype(np.float32)
    return torch.from_numpy(np.linalg.qr(gauss)[0]).cuda().double()


def _polar(x, bits, seed):
    """PolarQuant of ``x (..., n, D)`` and back, with its norms."""
    D = x.shape[-1]
    cent = (torch.tensor(LLOYD_MAX[bits], dtype=torch.float64, device="cuda") / math.sqrt(D)).float()
    bnd = ((cent[:-1] + cent[1:]) / 2).double()
    pi = _rotation(seed, D)
    norm = x.square().sum(-1).sqrt()
    y = (x / norm.clamp_min(1e-30)[..., None]) @ pi.T
    code = torch.searchsorted(bnd, y.contiguous())
    return cent.double()[code] @ pi * norm[..., None], norm


def _grouped(x, grid, bits, outliers):
    """Per-channel keys ``x (..., G, D)``, one group, and back; their scale and
    zero point."""
    if grid == "uniform":
        zero = x.amin(-2, keepdim=True)
        scale = (x.amax(-2, keepdim=True) - zero).clamp_min(1e-8) / (2 ** bits - 1)
        out = zero + scale * ((x - zero) / scale).round().clamp(0, 2 ** bits - 1)
    else:
        levels = torch.tensor(NF4, dtype=torch.float64, device="cuda")
        zero = x.mean(-2, keepdim=True)
        scale = (x - zero).abs().amax(-2, keepdim=True).clamp_min(1e-8)
        code = torch.searchsorted((levels[:-1] + levels[1:]) / 2, ((x - zero) / scale).contiguous())
        out = zero + scale * levels[code]
    if outliers:
        k = max(1, round(x.shape[-2] * outliers))
        kth = x.abs().topk(k, dim=-2).values[..., -1:, :]
        out = torch.where(x.abs() >= kth, x.half().double(), out)
    return out, scale.squeeze(-2), zero.squeeze(-2)


def _coded(k, v, length, W, grid, key_bits, value_bits, outliers, seed):
    """K/V ``(H, length, D)`` as the cache holds them in 64 bits (the hot
    window as it came), with the groups' scale and zero point."""
    G, ng = (W + 1) // 2, _groups(length, W)
    k, v = k[:, :length].double(), v[:, :length].double()
    if not ng:
        return k, v, None, None
    H, D = k.shape[0], k.shape[-1]
    cold = k[:, :ng * G].reshape(H, ng, G, D)
    scale = zero = None
    if grid == "polar":
        kc = _polar(cold, key_bits, seed)[0]
    else:
        kc, scale, zero = _grouped(cold, grid, key_bits, outliers)
    vc = _polar(v[:, :ng * G], value_bits, seed)[0]
    return (torch.cat([kc.reshape(H, ng * G, D), k[:, ng * G:]], 1),
            torch.cat([vc, v[:, ng * G:]], 1), scale, zero)


def _attend(q, k, v):
    """``q (Hq, D)`` over ``k, v (H, n, D)``, each head of which serves Hq / H queries."""
    H, D = k.shape[0], k.shape[-1]
    s = q.double().reshape(H, -1, D) @ k.transpose(1, 2) / math.sqrt(D)
    return (torch.softmax(s, -1) @ v).reshape(-1, D)


def exact(case, seed):
    kind = case["kind"]
    k, v = _case_tokens(case, seed)
    if kind in ("decode", "prefill"):
        form = (case["hot_window"], case["grid"], case["key_bits"], case["value_bits"], case["outliers"], seed)
        lens = _lengths(case)
        if kind == "decode":
            q = _queries(case, case["batch"], k.dtype, seed)
            return torch.stack([_attend(q[b], *_coded(k[b], v[b], L, *form)[:2]) for b, L in enumerate(lens)])
        if case["grid"] == "polar" or case["ragged"] or not _groups(case["length"], case["hot_window"]):
            return None
        both = [_coded(k[b], v[b], L, *form)[2:] for b, L in enumerate(lens)]
        return {"kcodes": None, "vcodes": None, "vnorm": None,
                "scale": torch.cat([s.transpose(0, 1) for s, _ in both]),
                "mean": torch.cat([z.transpose(0, 1) for _, z in both]),
                "ocount": None, "oent": None, "hot_k": None, "hot_v": None}
    if kind == "chat":
        q = _queries(case, case["steps"], torch.float16, seed)
        return torch.stack([_attend(q[i], *_coded(k[0], v[0], case["prompt"] + i + 1, 512, "nf4_asym", 4, 4,
                                                  0.02, seed)[:2]) for i in range(case["steps"])])
    if kind in ("save", "load"):
        kc, scale, mean = _grouped(k.double(), "nf4_asym", 4, 0.02)
        vc, norms = _polar(v.double(), case["value_bits"], seed)
        if kind == "load":
            return {"k": kc, "v": vc}
        return {"kcodes": None, "scale": scale, "mean": mean, "oidx": None, "oval": None, "vcodes": None,
                "norms": norms}
    # the HF layer keeps fp16 tokens
    both = [_coded(k[b].half(), v[b].half(), case["length"], 512, "nf4_asym", 4, case["value_bits"], 0.02,
                   seed)[:2] for b in range(case["batch"])]
    return {"k": torch.stack([x for x, _ in both]), "v": torch.stack([x for _, x in both])}
