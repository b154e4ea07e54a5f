"""What this library is timed on: the attention and cache calls of a serving
engine and of FlashAttention-2 user code, through the public entry points.

A case names a call (`kind`), its sizes, and `shape`: the seed of its request
lengths, so that a case's work does not depend on its input values.  The
listed sizes are those of this repository's benchmark, its configurations and
the published calls of the API it implements; `draw` spreads over the same
ranges.  Values are N(0, 1) queries and keys and 0.5 N(0, 1) values; E4M3
tensors hold N(0, 1) over per-head descales U[0.01, 0.1].
"""
import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.abspath("flash-attn-mps_amd"))
import flash_attn_mps_amd as fa  # noqa: E402
from flash_attn_mps_amd import vllm  # noqa: E402

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32, "e4m3": torch.float8_e4m3fn}
BYTES = {"fp16": 2, "bf16": 2, "fp32": 4, "e4m3": 1}
DEVICE = "cuda"


def listed():
    return [
        # One token of one short chat, FlashAttention-2 style: rotary embedding, append to a dense
        # cache, attention.  The smallest call: latency and launches.
        dict(name="generate_b1", kind="generate", batch=1, capacity=2048, lo=700, hi=700, hq=16, hkv=8, dim=128,
             dtype="fp16", interleaved=False, shape=1),
        # A decode step of a small server: slot writes, then paged attention (Qwen3-0.6B heads, 256-token
        # pages), ragged contexts.
        dict(name="serve_b16", kind="serve", batch=16, page=256, lo=2048, hi=8192, hq=16, hkv=8, dim=128,
             dtype="fp16", shape=2),
        # Paged decode of a loaded server, Llama-3-8B heads, 64 requests of up to 32K keys.
        dict(name="decode_llama", kind="decode", batch=64, rows=1, page=16, lo=512, hi=32768, hq=32, hkv=8, dim=128,
             q="bf16", kv="bf16", window=-1, softcap=0.0, shape=3),
        # Paged decode over an E4M3 cache with descales, softcap and a sliding window, Gemma-2-9B heads.
        dict(name="decode_gemma_fp8", kind="decode", batch=128, rows=1, page=16, lo=1024, hi=8192, hq=16, hkv=8,
             dim=256, q="bf16", kv="e4m3", window=4095, softcap=50.0, shape=4),
        # vLLM's FP8 attention: queries quantised too, descales for q, k and v, bf16 output.
        dict(name="decode_fp8_queries", kind="decode", batch=32, rows=1, page=16, lo=256, hi=8192, hq=32, hkv=8,
             dim=128, q="e4m3", kv="e4m3", window=-1, softcap=0.0, shape=5),
        # Decode in single precision over a contiguous cache (4 requests of 2048 keys).
        dict(name="decode_fp32", kind="decode", batch=4, rows=1, page=0, lo=2048, hi=2048, hq=16, hkv=8, dim=128,
             q="fp32", kv="fp32", window=-1, softcap=0.0, shape=6),
        # Prompt processing, 16 prompts of 256..4096 tokens, Qwen3-0.6B heads.
        dict(name="prefill_qwen", kind="prefill", batch=16, lo=256, hi=4096, hq=16, hkv=8, dim=128, dtype="bf16",
             window=-1, softcap=0.0, shape=7),
        # Prompt processing with softcap and a sliding window, Gemma-2-9B heads.
        dict(name="prefill_gemma", kind="prefill", batch=4, lo=512, hi=8192, hq=16, hkv=8, dim=256, dtype="bf16",
             window=4095, softcap=50.0, shape=8),
        # Chunked prefill of one long prompt: 512 new tokens behind a long prefix in the paged cache.
        dict(name="chunk_long", kind="chunk", batch=1, chunk=512, page=16, lo=24000, hi=24000, hq=32, hkv=8, dim=128,
             q="bf16", kv="bf16", shape=9),
        # One engine step of chunks and decodes together, K wider than V (192/128), sinks, caller's output.
        dict(name="mixed_diffkv", kind="mixed", chunks=8, chunk=512, prefix=4096, decodes=120, lo=256, hi=16384,
             page=16, heads=16, shape=10),
        # Dense causal attention in single precision (the API's own precision check, model debugging).
        dict(name="dense_fp32", kind="dense", batch=2, seq=1024, hq=16, hkv=8, dim=128, dtype="fp32", causal=True,
             shape=11),
        # Quantising cache write of a long prefill, bf16 rows into E4M3 pages, scattered slots.
        dict(name="store_fp8", kind="store", tokens=262144, page=16, hkv=8, dim=256, dtype="bf16", kv="e4m3",
             shape=12),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _span(rng, lo, hi):
    a, b = sorted((_log_int(rng, lo, hi), _log_int(rng, lo, hi)))
    return dict(lo=a, hi=b)


def draw(rng):
    kind = rng.choice(["generate", "serve", "decode", "decode", "fp8q", "fp32", "prefill", "gemma", "chunk", "mixed",
                       "dense", "store"])
    shape = rng.randrange(100, 1 << 20)
    if kind == "generate":
        hkv = rng.choice([2, 4, 8])
        return dict(kind=kind, batch=rng.randint(1, 16), capacity=4096, **_span(rng, 16, 4000),
                    hq=hkv * rng.choice([1, 2, 4]), hkv=hkv, dim=rng.choice([64, 128]),
                    dtype=rng.choice(["fp16", "bf16"]), interleaved=rng.random() < 0.5, shape=shape)
    if kind == "serve":
        return dict(kind=kind, batch=rng.randint(1, 32), page=rng.choice([16, 64, 256]), **_span(rng, 128, 8192),
                    hq=16, hkv=8, dim=128, dtype=rng.choice(["fp16", "bf16"]), shape=shape)
    if kind == "decode":
        hkv, dim = rng.choice([(8, 128), (8, 128), (4, 128), (8, 64), (8, 256)])
        return dict(kind=kind, batch=rng.randint(4, 96), rows=rng.choice([1, 1, 1, 4]) if dim < 256 else 1, page=16,
                    **_span(rng, 256, 8192), hq=hkv * rng.choice([1, 2, 4, 5, 8]), hkv=hkv, dim=dim, q="bf16",
                    kv=rng.choice(["bf16", "e4m3"]), window=rng.choice([-1, -1, 1023, 4095]),
                    softcap=rng.choice([0.0, 0.0, 50.0]), shape=shape)
    if kind == "fp8q":
        hkv = rng.choice([4, 8])
        return dict(kind="decode", batch=rng.randint(1, 32), rows=1, page=16, **_span(rng, 128, 4096),
                    hq=hkv * rng.choice([1, 2, 4, 8]), hkv=hkv, dim=rng.choice([64, 128, 256]), q="e4m3", kv="e4m3",
                    window=-1, softcap=0.0, shape=shape)
    if kind == "fp32":
        return dict(kind="decode", batch=rng.randint(1, 8), rows=1, page=rng.choice([0, 16]), **_span(rng, 256, 2048),
                    hq=8 * rng.choice([1, 2]), hkv=8, dim=rng.choice([64, 128]), q="fp32", kv="fp32", window=-1,
                    softcap=0.0, shape=shape)
    if kind == "prefill":
        hkv = rng.choice([4, 8, 8])
        return dict(kind=kind, batch=rng.randint(1, 8), **_span(rng, 64, 4096), hq=hkv * rng.choice([1, 2, 4]),
                    hkv=hkv, dim=rng.choice([64, 96, 128, 128]), dtype=rng.choice(["fp16", "bf16"]), window=-1,
                    softcap=0.0, shape=shape)
    if kind == "gemma":
        return dict(kind="prefill", batch=rng.randint(1, 4), **_span(rng, 512, 8192), hq=16, hkv=8, dim=256,
                    dtype="bf16", window=rng.choice([-1, 4095]), softcap=rng.choice([0.0, 50.0]), shape=shape)
    if kind == "chunk":
        hkv = rng.choice([2, 4, 8])
        return dict(kind=kind, batch=rng.randint(1, 2), chunk=_log_int(rng, 32, 1024), page=rng.choice([16, 256]),
                    **_span(rng, 512, 32768), hq=hkv * rng.choice([1, 2, 4]), hkv=hkv, dim=rng.choice([64, 128, 128]),
                    q="bf16", kv=rng.choice(["bf16", "bf16", "e4m3"]), shape=shape)
    if kind == "mixed":
        return dict(kind=kind, chunks=rng.randint(1, 8), chunk=_log_int(rng, 64, 512), prefix=4096,
                    decodes=rng.randint(8, 100), lo=256, hi=_log_int(rng, 512, 16384), page=16, heads=rng.choice([8, 16]),
                    shape=shape)
    if kind == "dense":
        return dict(kind=kind, batch=rng.randint(1, 2), seq=_log_int(rng, 96, 1024), hq=8 * rng.choice([1, 2]), hkv=8,
                    dim=rng.choice([64, 80, 128]), dtype="fp32", causal=rng.random() < 0.7, shape=shape)
    return dict(kind="store", tokens=_log_int(rng, 64, 262144), page=rng.choice([16, 64]), hkv=rng.choice([4, 8]),
                dim=rng.choice([64, 128, 256]), dtype="bf16", kv=rng.choice(["e4m3", "bf16"]), shape=shape)


# ------------------------------------------------------------ lengths and pages

def _lengths(seed, n, lo, hi):
    r = random.Random(seed)
    return [r.randint(lo, hi) for _ in range(n)]


def _requests(case):
    """(query rows, keys after the call) per request."""
    kind = case["kind"]
    if kind == "generate":
        ctx = _lengths(case["shape"], case["batch"], case["lo"], case["hi"])
        return [1] * case["batch"], [c + 1 for c in ctx]
    if kind in ("serve", "decode"):
        rows = case.get("rows", 1)
        ctx = _lengths(case["shape"], case["batch"], case["lo"], case["hi"])
        return [rows] * case["batch"], [max(c, rows) for c in ctx]
    if kind == "prefill":
        n = _lengths(case["shape"], case["batch"], case["lo"], case["hi"])
        return n, n
    if kind == "chunk":
        ctx = _lengths(case["shape"], case["batch"], case["lo"], case["hi"])
        return [case["chunk"]] * case["batch"], [c + case["chunk"] for c in ctx]
    if kind == "mixed":
        pre = _lengths(case["shape"], case["chunks"], 0, case["prefix"])
        ctx = _lengths(case["shape"] + 1, case["decodes"], case["lo"], case["hi"])
        return ([case["chunk"]] * case["chunks"] + [1] * case["decodes"],
                [p + case["chunk"] for p in pre] + ctx)
    if kind == "dense":
        return [case["seq"]] * case["batch"], [case["seq"]] * case["batch"]
    raise ValueError(kind)


def _features(case):
    """(Hq, Hkv, Dqk, Dv, query type, K/V type, causal, left window, softcap)."""
    kind = case["kind"]
    if kind == "mixed":
        return case["heads"], case["heads"], 192, 128, "bf16", "bf16", True, -1, 0.0
    q = case.get("q", case.get("dtype"))
    return (case["hq"], case["hkv"], case["dim"], case["dim"], q, case.get("kv", q), case.get("causal", True),
            case.get("window", -1), case.get("softcap", 0.0))


def _cu(lengths):
    c = [0]
    for n in lengths:
        c.append(c[-1] + n)
    return torch.tensor(c, dtype=torch.int32, device=DEVICE)


def _i32(values):
    return torch.tensor(values, dtype=torch.int32, device=DEVICE)


def _values(g, shape, dtype, scale=1.0, descale=None):
    """scale N(0, 1) of `dtype`; E4M3 divides head h of [..., H, D] by descale[h] first."""
    if dtype != "e4m3":
        return torch.randn(shape, generator=g, device=DEVICE, dtype=DTYPES[dtype]).mul_(scale)
    out = torch.empty(shape, dtype=DTYPES["e4m3"], device=DEVICE)
    flat, step = out.flatten(0, 1) if out.ndim == 4 else out, 1 << 16
    for i in range(0, flat.shape[0], step):     # in pieces: the fp32 draw is four times the result
        part = flat[i:i + step]
        x = torch.randn(part.shape, generator=g, device=DEVICE).mul_(scale)
        part.copy_(x.div_(descale[:, None]).clamp_(-448, 448))
    return out


def _pages(g, k_lens, page):
    """A block table [B, width] over a pool of exactly the pages needed, in random order."""
    need = [-(-n // page) for n in k_lens]
    perm = torch.randperm(sum(need), generator=g, device=DEVICE).to(torch.int32)
    table = torch.zeros(len(need), max(need), dtype=torch.int32, device=DEVICE)
    at = 0
    for b, n in enumerate(need):
        table[b, :n] = perm[at:at + n]
        at += n
    return table, sum(need)


# ------------------------------------------------------------ the calls

def prepare(case, seed):
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    kind = case["kind"]
    s = dict(case=case)
    if kind == "store":
        shape = (case["tokens"], case["hkv"], case["dim"])
        pages = -(-case["tokens"] // case["page"])
        cache = (pages, case["page"], case["hkv"], case["dim"])
        s.update(k=_values(g, shape, case["dtype"]), v=_values(g, shape, case["dtype"], 0.5),
                 k_cache=torch.zeros(cache, device=DEVICE, dtype=torch.uint8).to(DTYPES[case["kv"]]),
                 v_cache=torch.zeros(cache, device=DEVICE, dtype=torch.uint8).to(DTYPES[case["kv"]]))
        pos = torch.arange(case["tokens"], device=DEVICE)
        perm = torch.randperm(pages, generator=g, device=DEVICE)
        s["slots"] = (perm[pos // case["page"]] * case["page"] + pos % case["page"]).to(torch.int32)
        s["k_scale"] = s["v_scale"] = None
        if case["kv"] == "e4m3":
            s["k_scale"], s["v_scale"] = torch.empty(2, case["hkv"], device=DEVICE).uniform_(0.01, 0.1, generator=g)
        return s

    hq, hkv, dqk, dv, qt, kvt, _, _, _ = _features(case)
    q_lens, k_lens = _requests(case)
    batch, tokens = len(q_lens), sum(q_lens)
    descale = torch.empty(3, hkv, device=DEVICE).uniform_(0.01, 0.1, generator=g)
    head_descale = descale[0].repeat_interleave(hq // hkv)
    q = _values(g, (tokens, hq, dqk), qt, 1.0, head_descale)
    s.update(max_q=max(q_lens), max_k=max(k_lens), cu_q=_cu(q_lens), lengths=_i32(k_lens), q=q)
    if kind == "dense":
        s["q"] = q.unflatten(0, (batch, -1))
        s["k"] = _values(g, (batch, case["seq"], hkv, dqk), kvt)
        s["v"] = _values(g, (batch, case["seq"], hkv, dv), kvt, 0.5)
        return s
    if kind == "prefill":
        s["k"], s["v"] = _values(g, (tokens, hkv, dqk), kvt), _values(g, (tokens, hkv, dv), kvt, 0.5)
        return s
    if kind == "generate":
        cap = case["capacity"]
        s["k_cache"] = _values(g, (batch, cap, hkv, dqk), kvt)
        s["v_cache"] = _values(g, (batch, cap, hkv, dv), kvt, 0.5)
        s["k"], s["v"] = _values(g, (batch, 1, hkv, dqk), kvt), _values(g, (batch, 1, hkv, dv), kvt, 0.5)
        s["q"] = q.unflatten(0, (batch, 1))
        inv = 10000.0 ** (-torch.arange(0, dqk, 2, device=DEVICE, dtype=torch.float32) / dqk)
        angle = torch.arange(cap, device=DEVICE, dtype=torch.float32)[:, None] * inv
        s["cos"], s["sin"] = angle.cos().to(DTYPES[kvt]), angle.sin().to(DTYPES[kvt])
        s["lengths"] = s["lengths"] - 1         # the lengths before the append
        return s
    if case["page"]:
        s["table"], pool = _pages(g, k_lens, case["page"])
        s["k_cache"] = _values(g, (pool, case["page"], hkv, dqk), kvt, 1.0, descale[1])
        s["v_cache"] = _values(g, (pool, case["page"], hkv, dv), kvt, 0.5, descale[2])
    else:
        s["table"] = None
        s["k_cache"] = _values(g, (batch, max(k_lens), hkv, dqk), kvt)
        s["v_cache"] = _values(g, (batch, max(k_lens), hkv, dv), kvt, 0.5)
    if kind == "serve":
        s["k"], s["v"] = _values(g, (batch, hkv, dqk), kvt), _values(g, (batch, hkv, dv), kvt, 0.5)
        last = [n - 1 for n in k_lens]
        pages = s["table"][torch.arange(batch, device=DEVICE), _i32([n // case["page"] for n in last]).long()]
        s["slots"] = pages * case["page"] + _i32([n % case["page"] for n in last])
    s["q_descale"], s["k_descale"], s["v_descale"] = (
        descale[i].expand(batch, hkv) if t == "e4m3" else None for i, t in enumerate((qt, kvt, kvt)))
    s["sinks"] = torch.randn(hq, generator=g, device=DEVICE) if kind == "mixed" else None
    out_type = DTYPES["bf16"] if qt == "e4m3" else DTYPES[qt]
    s["out"] = torch.empty(tokens, hq, dv, dtype=out_type, device=DEVICE)
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "store":
        fa.store_kvcache(s["k"], s["v"], s["k_cache"], s["v_cache"], s["slots"], k_scale=s["k_scale"],
                         v_scale=s["v_scale"])
        return [c.view(torch.uint8) for c in (s["k_cache"], s["v_cache"])]
    _, _, _, _, _, _, causal, window, softcap = _features(case)
    if kind == "generate":
        out, lse = fa.flash_attn_with_kvcache(
            s["q"], s["k_cache"], s["v_cache"], s["k"], s["v"], s["cos"], s["sin"], s["lengths"], causal=True,
            rotary_interleaved=case["interleaved"], return_softmax_lse=True)
        return out, lse, s["k_cache"], s["v_cache"]
    if kind == "serve":
        fa.store_kvcache(s["k"], s["v"], s["k_cache"], s["v_cache"], s["slots"])
        out = fa.flash_attn_with_kvcache(s["q"].unsqueeze(1), s["k_cache"], s["v_cache"], cache_seqlens=s["lengths"],
                                         block_table=s["table"], causal=True)
        return out, s["k_cache"], s["v_cache"]
    if kind == "dense":
        return fa.flash_attn_func(s["q"], s["k"], s["v"], causal=causal, return_softmax_lse=True)
    if kind == "prefill":
        return fa.flash_attn_varlen_func(s["q"], s["k"], s["v"], s["cu_q"], s["cu_q"], s["max_q"], s["max_q"],
                                         causal=True, window_size=(window, -1 if window < 0 else 0), softcap=softcap,
                                         return_softmax_lse=True)
    if kind == "decode" and s["table"] is None:
        return fa.flash_attn_with_kvcache(s["q"].unsqueeze(1), s["k_cache"], s["v_cache"], cache_seqlens=s["lengths"],
                                          causal=True, return_softmax_lse=True)
    return vllm.flash_attn_varlen_func(
        s["q"], s["k_cache"], s["v_cache"], s["max_q"], s["cu_q"], s["max_k"], seqused_k=s["lengths"],
        block_table=s["table"], causal=True, softcap=softcap, window_size=(window, -1 if window < 0 else 0),
        q_descale=s["q_descale"], k_descale=s["k_descale"], v_descale=s["v_descale"], s_aux=s["sinks"],
        out=s["out"], return_softmax_lse=True)


# ------------------------------------------------------------ work, tolerance, 64-bit result

def _visible(case):
    """(visible (query, key) pairs, keys that any row sees) summed over the requests."""
    _, _, _, _, _, _, causal, window, _ = _features(case)
    pairs = keys = 0
    for lq, lk in zip(*_requests(case)):
        if not causal:
            pairs, keys = pairs + lq * lk, keys + lk
            continue
        first = max(lk - lq + 1, 1)             # keys that the first row sees
        seen = range(first, lk + 1)
        if window >= 0:
            pairs += sum(min(n, window + 1) for n in seen)
            keys += min(lk, window + lq)
        else:
            pairs += (first + lk) * len(seen) // 2
            keys += lk
    return pairs, keys


def work(case):
    if case["kind"] == "store":
        return {"bytes": 2 * case["tokens"] * case["hkv"] * case["dim"] * (BYTES[case["dtype"]] + BYTES[case["kv"]])
                + 4 * case["tokens"], "flops": 0}
    hq, hkv, dqk, dv, qt, kvt, _, _, _ = _features(case)
    pairs, keys = _visible(case)
    tokens = sum(_requests(case)[0])
    out = 2 if qt == "e4m3" else BYTES[qt]
    nbytes = keys * hkv * (dqk + dv) * BYTES[kvt] + tokens * hq * (dqk * BYTES[qt] + dv * out + 4)
    if case["kind"] in ("generate", "serve"):   # the new rows: read, and written to the cache
        nbytes += 2 * tokens * hkv * (dqk + dv) * BYTES[kvt]
    return {"bytes": nbytes, "flops": pairs * hq * 2 * (dqk + dv)}


def tolerance(case):
    if case["kind"] == "store":
        return "exact"
    # About four times the measured error against float64: 5e-7 in single precision, 2.1e-4 / 2.3e-3 with
    # fp16 / bf16 probabilities and outputs (E4M3 queries write bf16).
    qt = _features(case)[4]
    return {"rel": {"fp32": 3e-6, "fp16": 1e-3, "bf16": 1e-2, "e4m3": 1e-2}[qt]}


def _attend(q, k, v, causal, window, softcap, sinks):
    """One request in float64: q [Lq, Hq, D], k/v [Lk, Hkv, D] -> (out [Lq, Hq, Dv], lse [Hq, Lq])."""
    lq, hq, _ = q.shape
    lk, hkv, _ = k.shape
    scale, group = q.shape[-1] ** -0.5, hq // hkv
    out = torch.empty(lq, hq, v.shape[-1], dtype=torch.float64, device=q.device)
    lse = torch.empty(hq, lq, dtype=torch.float64, device=q.device)
    row = torch.arange(lq, device=q.device)[:, None] + (lk - lq)
    col = torch.arange(lk, device=q.device)[None, :]
    hidden = torch.zeros(lq, lk, dtype=torch.bool, device=q.device)
    if causal:
        hidden |= col > row
    if window >= 0:
        hidden |= col < row - window
    for h in range(hq):
        kd, vd = k[:, h // group].double(), v[:, h // group].double()
        s = (q[:, h].double() @ kd.T.contiguous()) * scale
        if softcap:
            s = softcap * torch.tanh(s / softcap)
        s.masked_fill_(hidden, -math.inf)
        total = torch.logsumexp(s, -1)
        if sinks is not None:
            total = torch.logaddexp(total, sinks[h].double())
        lse[h] = total
        out[:, h] = torch.exp(s - total[:, None]) @ vd
    return out, lse


def _rotate(x, cos, sin, interleaved):
    """x [H, D] at one position, rounded to x's type as the cache holds it."""
    d, (c, s) = x.double(), (cos.double(), sin.double())
    y = torch.empty_like(d)
    a, b = (d[:, 0::2], d[:, 1::2]) if interleaved else d.chunk(2, -1)
    first, second = a * c - b * s, b * c + a * s
    if interleaved:
        y[:, 0::2], y[:, 1::2] = first, second
    else:
        y = torch.cat([first, second], -1)
    return y.to(x.dtype)


def exact(case, seed):
    if case["kind"] == "store":     # bytes: compared as they are
        return None
    s = prepare(case, seed)
    hq, hkv, dqk, dv, qt, kvt, causal, window, softcap = _features(case)
    q_lens, k_lens = _requests(case)
    kind, q = case["kind"], s["q"]
    if kind == "generate":
        q = q.clone()
        for b, n in enumerate(k_lens):
            at = n - 1
            q[b, 0] = _rotate(q[b, 0], s["cos"][at], s["sin"][at], case["interleaved"])
            s["k_cache"][b, at] = _rotate(s["k"][b, 0], s["cos"][at], s["sin"][at], case["interleaved"])
            s["v_cache"][b, at] = s["v"][b, 0]
    if kind == "serve":
        s["k_cache"].flatten(0, 1)[s["slots"].long()] = s["k"]
        s["v_cache"].flatten(0, 1)[s["slots"].long()] = s["v"]
    q = q.reshape(-1, hq, dqk)
    outs, lses, at = [], [], 0
    for b, (lq, lk) in enumerate(zip(q_lens, k_lens)):
        if kind in ("prefill", "dense"):
            keys, vals = (s[n].reshape(-1, hkv, d)[at:at + lk] for n, d in (("k", dqk), ("v", dv)))
        elif s.get("table") is not None:
            pages = s["table"][b, :-(-lk // case["page"])].long()
            keys, vals = (s[n].view(torch.uint8)[pages].view(s[n].dtype).flatten(0, 1)[:lk] for n in ("k_cache", "v_cache"))
        else:
            keys, vals = s["k_cache"][b, :lk], s["v_cache"][b, :lk]
        qb = q[at:at + lq]
        if qt == "e4m3":
            qb = qb.double() * s["q_descale"][b].double().repeat_interleave(hq // hkv)[:, None]
        if kvt == "e4m3":
            keys, vals = (t.double() * s[n][b].double()[:, None] for t, n in ((keys, "k_descale"), (vals, "v_descale")))
        o, l = _attend(qb, keys, vals, causal, window, softcap, s.get("sinks"))
        outs.append(o)
        lses.append(l)
        at += lq
    out, lse = torch.cat(outs), torch.cat(lses, 1)
    if kind == "serve":
        return out.unflatten(0, (-1, 1)), s["k_cache"].double(), s["v_cache"].double()
    if kind in ("generate", "dense") or (kind == "decode" and s["table"] is None):
        batch = len(q_lens)
        out, lse = out.unflatten(0, (batch, -1)), lse.reshape(hq, batch, -1).transpose(0, 1)
    if kind == "generate":
        return out, lse, s["k_cache"].double(), s["v_cache"].double()
    return out, lse
