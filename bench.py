"""Benchmark of the flash_attn_mps_amd hot path on one MI355X.

Headline (`value`): bf16 causal varlen prefill TFLOP/s on config 2
(16 sequences, lengths U[256, 4096], Hq/Hkv = 16/8, d = 128, Qwen3-0.6B
attention shape), one `flash_attn_varlen_func` call per step with Q/K/V
resident in HBM.  Algorithmic FLOPs = sum over visible (query, key) pairs x
Hq x 2 (Dqk + Dv), lower-right causal.

Secondary lines (same JSON object, key "secondary"): paged bf16 decode
(config 3, Llama-3-8B shape), paged FP8 decode with softcap + window
(config 4, Gemma-2-9B shape), and the mixed chunked-prefill + decode DIFFKV
call (config 5), each in algorithmic KV GB/s against 8 TB/s; store_kvcache
into config 4's E4M3 caches (GB/s); config 2 with E4M3 Q/K/V (TFLOP/s
against the 5.0 PF E4M3 peak and the 3.33 PF peak of its E4M3 + bf16 mix).

Inputs are synthetic (seeded N(0,1)); lengths/tables come from
torch.Generator().manual_seed(123 + cfg).  The CPU baseline times the fp32
CPU oracle (tests' checker) on a bounded sample of config 2.
"""
import argparse
import json
import math
import os
import sys
import time
from pathlib import Path

ROOT = Path(__file__).resolve().parent
sys.path.insert(0, str(ROOT / "flash-attn-mps_amd"))
sys.path.insert(0, str(ROOT))

PEAK_BF16_TFLOPS = 2500.0
PEAK_HBM_GBS = 8000.0
PEAK_FP8_TFLOPS = 5000.0
PEAK_FP8_BF16_MIXED_TFLOPS = 2.0 / (1.0 / 5000.0 + 1.0 / 2500.0)
# Warmup calls of every secondary line (at least the command's --warmup):
# after an idle period the GPU's clock dips and ramps back over the first
# tens of calls (a per-call trace of config 3: ~1 ms for the first call, the
# shader clock down to ~1.7 GHz for calls 2-8, back to 2.4 GHz by call ~24),
# and MFMA-bound launches settle only after ~100 of them.  Each entry states
# the warmup it used.
SECONDARY_WARMUP = 50


def parse():
    p = argparse.ArgumentParser()
    p.add_argument("--gpus", type=int, default=1)
    p.add_argument("--steps", type=int, default=20)
    p.add_argument("--warmup", type=int, default=200)
    p.add_argument("--no-secondary", action="store_true", help="only the headline prefill config")
    p.add_argument("--no-cpu-baseline", action="store_true")
    p.add_argument("--only", default="", help="comma list of secondary configs to run (3,4,5,5_fixed_order,store4,prefill_d256,prefill_fp8); "
                        "config 2 always runs")
    p.add_argument("--copy-probe", action="store_true",
                   help="first run a known-size copy kernel (reads and writes 1 GiB) that calibrates "
                        "rocprofv3 FETCH_SIZE / WRITE_SIZE")
    return p.parse_args()


def cu_lengths(lengths, device):
    import torch
    c = torch.zeros(len(lengths) + 1, dtype=torch.int32)
    c[1:] = torch.tensor(lengths, dtype=torch.int32).cumsum(0)
    return c.to(device)


def causal_pairs(q_lens, k_lens):
    """Visible (query, key) pairs under lower-right causality: row i of a
    request sees max(0, lk - lq + 1 + i) keys, consecutive integers from
    lk - lq + 1 up to lk, so a request's sum is that of the positive ones."""
    total = 0
    for lq, lk in zip(q_lens, k_lens):
        if lq <= 0 or lk <= 0:
            continue
        lo = max(lk - lq + 1, 1)
        total += (lo + lk) * (lk - lo + 1) // 2
    return total


def time_calls(fn, steps, warmup, kernel=None, defer=False):
    """Warmup, then `steps` back-to-back calls bracketed by synchronize with
    no other work in between (ms per step = the region over `steps`).  A
    second pass of `steps` calls then records a HIP event pair around every
    call, and around every launch of the C-ABI entry point `kernel` when one
    is named, on the launching stream (event records cost a few microseconds
    each, so they stay out of the first region).  Returns (ms per step, median
    ms per call, mean ms per `kernel` launch or None); with `defer`, a
    function that returns them, leaving the final synchronize (which the
    event readings need) to that function, so the caller can enqueue its next
    work before the GPU drains."""
    import torch
    for _ in range(warmup):
        fn()
    torch.cuda.synchronize()
    region0 = torch.cuda.Event(enable_timing=True)
    region1 = torch.cuda.Event(enable_timing=True)
    region0.record()
    for _ in range(steps):
        fn()
    region1.record()
    torch.cuda.synchronize()
    total = region0.elapsed_time(region1)
    starts = [torch.cuda.Event(enable_timing=True) for _ in range(steps)]
    ends = [torch.cuda.Event(enable_timing=True) for _ in range(steps)]
    with launch_events(kernel) as pairs:
        for i in range(steps):
            starts[i].record()
            fn()
            ends[i].record()

    def finish():
        torch.cuda.synchronize()
        per_call = sorted(s.elapsed_time(e) for s, e in zip(starts, ends))
        kernel_ms = sum(s.elapsed_time(e) for s, e in pairs) / len(pairs) if pairs else None
        return total / steps, per_call[len(per_call) // 2], kernel_ms

    return finish if defer else finish()


class launch_events:
    """Record a HIP event pair on the launching stream around every call of
    one C-ABI entry point (the library's only route to the GPU), so a single
    kernel's duration is timed inside the benchmark; name None records none."""

    def __init__(self, name):
        self.name = name
        self.pairs = []

    def __enter__(self):
        import torch
        from flash_attn_mps_amd import _lib
        self._lib, self._orig = _lib, _lib.call

        def call(name, args, device):
            if self.name is None or name != self.name:
                return self._orig(name, args, device)
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            rc = self._orig(name, args, device)
            end.record()
            self.pairs.append((start, end))
            return rc

        _lib.call = call
        return self.pairs

    def __exit__(self, *exc):
        self._lib.call = self._orig
        return False


def copy_probe(device):
    """torch.neg over 2^28 fp32 values: 1 GiB read + 1 GiB written per launch,
    three launches.  Under rocprofv3 --pmc its FETCH_SIZE / WRITE_SIZE give
    the factor from counter KiB to bytes moved."""
    import torch
    x = torch.ones(1 << 28, dtype=torch.float32, device=device)
    y = torch.empty_like(x)
    for _ in range(3):
        torch.neg(x, out=y)
    torch.cuda.synchronize()
    del x, y
    torch.cuda.empty_cache()


def measured_traffic():
    """HBM bytes per launch of the prefill kernel on config 2, from the
    committed rocprofv3 FETCH_SIZE / WRITE_SIZE passes (scaled by the copy
    probe), or None when that summary is absent."""
    path = ROOT / "profiles" / "prefill_config2_traffic.md"
    if not path.exists():
        return None
    for line in path.read_text().splitlines():
        if line.startswith("traffic_bytes_per_launch:"):
            return int(line.split(":", 1)[1].strip())
    return None


def config2_inputs(device):
    """Config 2: 16 sequences, lengths U[256, 4096], 0.5*N(0,1) bf16 Q/K/V, Hq/Hkv 16/8, d 128."""
    import torch
    g = torch.Generator().manual_seed(123 + 2)
    lengths = torch.randint(256, 4097, (16,), generator=g).tolist()
    total = sum(lengths)
    hq, hkv, d = 16, 8, 128
    q = (torch.randn(total, hq, d, generator=g) * 0.5).to(torch.bfloat16).to(device)
    k = (torch.randn(total, hkv, d, generator=g) * 0.5).to(torch.bfloat16).to(device)
    v = (torch.randn(total, hkv, d, generator=g) * 0.5).to(torch.bfloat16).to(device)
    return dict(lengths=lengths, q=q, k=k, v=v, cu=cu_lengths(lengths, device), heads=hq, kv_heads=hkv, dim=d,
                out=torch.empty_like(q))


def config2(device, steps, warmup, c=None):
    import torch
    import flash_attn_mps_amd as fa
    c = c or config2_inputs(device)
    q, k, v, cu, lengths = c["q"], c["k"], c["v"], c["cu"], c["lengths"]
    maxlen = max(lengths)
    out = c["out"]

    def step():
        fa.flash_attn_varlen_func(q, k, v, cu, cu, maxlen, maxlen, causal=True, out=out)

    ms, call_ms, kernel_ms = time_calls(step, steps, warmup, kernel="fa_prefill_fwd")
    flops = causal_pairs(lengths, lengths) * c["heads"] * 2 * (c["dim"] + c["dim"])
    return dict(lengths=lengths, flops=flops, ms=ms, call_ms=call_ms, kernel_ms=kernel_ms,
                tflops=flops / (ms * 1e-3) / 1e12, call_tflops=flops / (call_ms * 1e-3) / 1e12,
                kernel_tflops=flops / (kernel_ms * 1e-3) / 1e12, tensors=(q, k, v, cu))


def prefill_d256(device, steps, warmup, c=None):
    """Config 2's lengths with 256-dim heads (Gemma-like, Hq/Hkv 16/8), bf16
    0.5*N(0,1) Q/K/V, causal: the 256-dim MFMA prefill, in which two waves share
    32 query rows, each with one 128-column half of V."""
    import torch
    import flash_attn_mps_amd as fa
    c = c or config2_inputs(device)
    lengths, cu = c["lengths"], c["cu"]
    g = torch.Generator().manual_seed(123 + 256)
    total, hq, hkv, d = sum(lengths), 16, 8, 256
    q = (torch.randn(total, hq, d, generator=g) * 0.5).to(torch.bfloat16).to(device)
    k = (torch.randn(total, hkv, d, generator=g) * 0.5).to(torch.bfloat16).to(device)
    v = (torch.randn(total, hkv, d, generator=g) * 0.5).to(torch.bfloat16).to(device)
    out = torch.empty_like(q)
    maxlen = max(lengths)

    def step():
        fa.flash_attn_varlen_func(q, k, v, cu, cu, maxlen, maxlen, causal=True, out=out)

    ms, call_ms, kernel_ms = time_calls(step, steps, warmup, kernel="fa_prefill_fwd")
    flops = causal_pairs(lengths, lengths) * hq * 2 * (d + d)
    return dict(ms=ms, call_ms=call_ms, kernel_ms=kernel_ms, flops=flops, tflops=flops / (ms * 1e-3) / 1e12,
                what="config 2 lengths, Hq/Hkv 16/8, d256 bf16 causal (Gemma-like heads); "
                     "wave pairs sharing 32 rows")


def prefill_fp8(device, steps, warmup, c=None, defer=False):
    """Config 2 with E4M3 queries, keys and values (per-(request, KV head)
    descales) and bf16 output: S = Q K^T on the FP8 MFMA, P.V on the bf16
    MFMA.  Same algorithmic FLOPs as config 2; half of them (Q K^T) run at
    the 5.0 PF E4M3 rate and half (P V) at 2.5 PF bf16, so the mixed peak is
    2 / (1/5.0 + 1/2.5) = 3.33 PF."""
    import torch
    from flash_attn_mps_amd import vllm
    c = c or config2_inputs(device)
    lengths, cu, hkv = c["lengths"], c["cu"], c["kv_heads"]
    g = torch.Generator().manual_seed(123 + 20)
    desc = {n: torch.empty(len(lengths), hkv).uniform_(0.005, 0.01, generator=g).to(device) for n in "qkv"}
    per_tok = [torch.repeat_interleave(desc[n], torch.tensor(lengths, device=device), dim=0) for n in "qkv"]
    group = c["heads"] // hkv
    q = (c["q"].float() / per_tok[0].repeat_interleave(group, dim=1)[..., None]).clamp(-448, 448)
    q = q.to(torch.float8_e4m3fn)
    k = (c["k"].float() / per_tok[1][..., None]).clamp(-448, 448).to(torch.float8_e4m3fn)
    v = (c["v"].float() / per_tok[2][..., None]).clamp(-448, 448).to(torch.float8_e4m3fn)
    maxlen = max(lengths)
    out = torch.empty(q.shape, dtype=torch.bfloat16, device=device)

    def step():
        vllm.flash_attn_varlen_func(q, k, v, maxlen, cu, maxlen, cu_seqlens_k=cu, causal=True, out=out,
                                    q_descale=desc["q"], k_descale=desc["k"], v_descale=desc["v"])

    flops = causal_pairs(lengths, lengths) * 16 * 2 * (128 + 128)
    timing = time_calls(step, steps, warmup, kernel="fa_prefill_fwd", defer=True)

    def finish():
        ms, call_ms, kernel_ms = timing()
        return dict(ms=ms, call_ms=call_ms, kernel_ms=kernel_ms, flops=flops, tflops=flops / (ms * 1e-3) / 1e12,
                    what="config 2 lengths, E4M3 Q/K/V with descales, bf16 out; Q.K^T on the FP8 MFMA")

    return finish if defer else finish()


def paged_cache(ctx, page, hkv, d, dtype, device, gen_seed, scale=None, dv=None):
    """K/V caches written by store_kvcache from a slot mapping whose block
    table is a random permutation of a pool sized to the total tokens."""
    import torch
    import flash_attn_mps_amd as fa
    g = torch.Generator().manual_seed(gen_seed)
    dv = dv or d
    pages_per = [(c + page - 1) // page for c in ctx]
    pool = sum(pages_per)
    perm = torch.randperm(pool, generator=g).to(torch.int32)
    width = max(pages_per)
    table = torch.zeros(len(ctx), width, dtype=torch.int32)
    slots = []
    start = 0
    for b, (c, n) in enumerate(zip(ctx, pages_per)):
        table[b, :n] = perm[start:start + n]
        start += n
        pos = torch.arange(c)
        slots.append(table[b, pos // page] * page + pos % page)
    slots = torch.cat(slots).to(torch.int32).to(device)
    tokens = sum(ctx)
    gdev = torch.Generator(device=device).manual_seed(gen_seed)
    kx = torch.randn(tokens, hkv, d, generator=gdev, device=device, dtype=torch.float32).to(torch.bfloat16)
    vx = torch.randn(tokens, hkv, dv, generator=gdev, device=device, dtype=torch.float32).to(torch.bfloat16)
    kc = torch.empty(pool, page, hkv, d, dtype=dtype, device=device)
    vc = torch.empty(pool, page, hkv, dv, dtype=dtype, device=device)
    fa.store_kvcache(kx, vx, kc, vc, slots, k_scale=scale, v_scale=scale)
    torch.cuda.synchronize()
    del kx, vx
    return kc, vc, table.to(device), slots


def config3_inputs(device):
    """Config 3: 64 requests, contexts U[512, 32768], Hq/Hkv 32/8, d 128, bf16 cache in
    16-token pages written by store_kvcache through a permuted block table."""
    import torch
    g = torch.Generator().manual_seed(123 + 3)
    ctx = torch.randint(512, 32769, (64,), generator=g).tolist()
    hq, hkv, d, page = 32, 8, 128, 16
    kc, vc, table, slots = paged_cache(ctx, page, hkv, d, torch.bfloat16, device, 123 + 3)
    q = torch.randn(64, 1, hq, d, generator=g).to(torch.bfloat16).to(device)
    return dict(ctx=ctx, q=q, k_cache=kc, v_cache=vc, table=table, slots=slots,
                lengths=torch.tensor(ctx, dtype=torch.int32, device=device), heads=hq, kv_heads=hkv, dim=d,
                page=page, kv_bytes=sum(ctx) * hkv * 2 * d * 2)


def config3(device, steps, warmup):
    """Config 3, then on the same cache a speculative-decode step: 4 query rows per
    request (the last 4 positions, causal), whose rows share each request's K/V reads."""
    import torch
    import flash_attn_mps_amd as fa
    c = config3_inputs(device)

    def step():
        fa.flash_attn_with_kvcache(c["q"], c["k_cache"], c["v_cache"], cache_seqlens=c["lengths"],
                                   block_table=c["table"], causal=True)

    ms, call_ms, kernel_ms = time_calls(step, steps, warmup, kernel="fa_decode_fwd")
    kv_bytes = c["kv_bytes"]
    g = torch.Generator().manual_seed(123 + 30)
    q4 = torch.randn(64, 4, c["heads"], c["dim"], generator=g).to(torch.bfloat16).to(device)

    def step4():
        fa.flash_attn_with_kvcache(q4, c["k_cache"], c["v_cache"], cache_seqlens=c["lengths"],
                                   block_table=c["table"], causal=True)

    ms4, call_ms4, kernel_ms4 = time_calls(step4, steps, warmup, kernel="fa_decode_fwd")
    del c
    rows4 = dict(kv_bytes=kv_bytes, ms=ms4, call_ms=call_ms4, kernel_ms=kernel_ms4, gbs=kv_bytes / (ms4 * 1e-3) / 1e9,
                 call_gbs=kv_bytes / (call_ms4 * 1e-3) / 1e9)
    return dict(kv_bytes=kv_bytes, ms=ms, call_ms=call_ms, kernel_ms=kernel_ms, gbs=kv_bytes / (ms * 1e-3) / 1e9,
                call_gbs=kv_bytes / (call_ms * 1e-3) / 1e9, rows4=rows4)


def config4_inputs(device):
    """Config 4: 128 requests, contexts U[1024, 8192], Hq/Hkv 16/8, d 256, E4M3 cache with
    per-KV-head scales U[0.01, 0.1] (descales [B, Hkv] as a stride-0 view), softcap 50,
    window (4095, 0)."""
    import torch
    g = torch.Generator().manual_seed(123 + 4)
    ctx = torch.randint(1024, 8193, (128,), generator=g).tolist()
    hq, hkv, d, page = 16, 8, 256, 16
    scale = torch.empty(hkv).uniform_(0.01, 0.1, generator=g)
    kc, vc, table, slots = paged_cache(ctx, page, hkv, d, torch.float8_e4m3fn, device, 123 + 4,
                                       scale=scale.to(device))
    q = torch.randn(128, hq, d, generator=g).to(torch.bfloat16).to(device)
    return dict(ctx=ctx, q=q, k_cache=kc, v_cache=vc, table=table, slots=slots, scale=scale,
                cu_q=torch.arange(129, dtype=torch.int32, device=device),
                lengths=torch.tensor(ctx, dtype=torch.int32, device=device),
                descale=scale.to(device).expand(128, hkv), heads=hq, kv_heads=hkv, dim=d, page=page,
                softcap=50.0, window=(4095, 0), kv_bytes=sum(min(c, 4096) for c in ctx) * hkv * 2 * d * 1)


def config4(device, steps, warmup):
    import torch
    from flash_attn_mps_amd import vllm
    c = config4_inputs(device)
    out = torch.empty(128, c["heads"], c["dim"], dtype=torch.bfloat16, device=device)

    def step():
        vllm.flash_attn_varlen_func(c["q"], c["k_cache"], c["v_cache"], 1, c["cu_q"], max(c["ctx"]),
                                    seqused_k=c["lengths"], block_table=c["table"], causal=True,
                                    softcap=c["softcap"], window_size=c["window"], k_descale=c["descale"],
                                    v_descale=c["descale"], out=out)

    ms, call_ms, kernel_ms = time_calls(step, steps, warmup, kernel="fa_decode_fwd")
    kv_bytes = c["kv_bytes"]
    del c
    return dict(kv_bytes=kv_bytes, ms=ms, call_ms=call_ms, kernel_ms=kernel_ms, gbs=kv_bytes / (ms * 1e-3) / 1e9,
                call_gbs=kv_bytes / (call_ms * 1e-3) / 1e9)


def config5_inputs(device):
    """Config 5: one DIFFKV call (Dqk 192 / Dv 128, Hq = Hkv = 16, bf16, 16-token pages) of
    8 chunks of 512 new tokens on prefixes U[0, 4096] plus 120 decode requests with
    contexts U[256, 16384]; per-head sinks N(0,1); caller-owned out."""
    import torch
    g = torch.Generator().manual_seed(123 + 5)
    hq = hkv = 16
    dqk, dv, page = 192, 128, 16
    prefixes = torch.randint(0, 4097, (8,), generator=g).tolist()
    dec_ctx = torch.randint(256, 16385, (120,), generator=g).tolist()
    q_lens = [512] * 8 + [1] * 120
    k_lens = [p + 512 for p in prefixes] + dec_ctx
    kc, vc, table, _ = paged_cache(k_lens, page, hkv, dqk, torch.bfloat16, device, 123 + 5, dv=dv)
    q = torch.randn(sum(q_lens), hq, dqk, generator=g).to(torch.bfloat16).to(device)
    sinks = torch.randn(hq, generator=g).to(device)
    return dict(q_lens=q_lens, k_lens=k_lens, dec_ctx=dec_ctx, q=q, k_cache=kc, v_cache=vc, table=table,
                sinks=sinks, cu_q=cu_lengths(q_lens, device),
                used=torch.tensor(k_lens, dtype=torch.int32, device=device), heads=hq, kv_heads=hkv,
                dim_qk=dqk, dim_v=dv, page=page)


def config5(device, steps, warmup, splits=0):
    """Config 5; splits=1 is vLLM's fixed-order (batch-invariant) call, which
    keeps every request, single-query ones included, in the MFMA prefill."""
    import torch
    from flash_attn_mps_amd import vllm
    c = config5_inputs(device)
    q_lens, k_lens, hkv, dqk, dv = c["q_lens"], c["k_lens"], c["kv_heads"], c["dim_qk"], c["dim_v"]
    out = torch.empty(sum(q_lens), c["heads"], dv, dtype=torch.bfloat16, device=device)

    def step():
        vllm.flash_attn_varlen_func(c["q"], c["k_cache"], c["v_cache"], max(q_lens), c["cu_q"], max(k_lens),
                                    seqused_k=c["used"], block_table=c["table"], causal=True, s_aux=c["sinks"],
                                    out=out, num_splits=splits)

    ms, call_ms, _ = time_calls(step, steps, warmup)
    dec_bytes = sum(c["dec_ctx"]) * hkv * (dqk + dv) * 2
    chunk_bytes = sum(k_lens[:8]) * hkv * (dqk + dv) * 2
    flops = causal_pairs(q_lens[:8], k_lens[:8]) * c["heads"] * 2 * (dqk + dv)
    roof_ms = max(flops / (PEAK_BF16_TFLOPS * 1e12), (dec_bytes + chunk_bytes) / (PEAK_HBM_GBS * 1e9)) * 1e3
    del c
    return dict(kv_bytes=dec_bytes + chunk_bytes, flops=flops, ms=ms, call_ms=call_ms,
                gbs=(dec_bytes + chunk_bytes) / (ms * 1e-3) / 1e9, roofline_ms=roof_ms,
                frac=roof_ms / ms)


def store_fp8(device, steps, warmup):
    """store_kvcache of config 4's 590K tokens (bf16 [T, 8, 256] K and V) into
    the E4M3 caches with per-head scales: bytes = 2 x T x 8 x 256 x (2 read + 1 written)."""
    import torch
    import flash_attn_mps_amd as fa
    c = config4_inputs(device)
    tokens, hkv, d = sum(c["ctx"]), c["kv_heads"], c["dim"]
    g = torch.Generator(device=device).manual_seed(123 + 4)
    kx = torch.randn(tokens, hkv, d, generator=g, device=device, dtype=torch.float32).to(torch.bfloat16)
    vx = torch.randn(tokens, hkv, d, generator=g, device=device, dtype=torch.float32).to(torch.bfloat16)
    scale = c["scale"].to(device)

    def step():
        fa.store_kvcache(kx, vx, c["k_cache"], c["v_cache"], c["slots"], k_scale=scale, v_scale=scale)

    ms, call_ms, kernel_ms = time_calls(step, steps, min(warmup, 20), kernel="fa_store_kvcache")
    nbytes = 2 * tokens * hkv * d * (2 + 1)
    del c, kx, vx
    return dict(ms=ms, call_ms=call_ms, kernel_ms=kernel_ms, bytes=nbytes, gbs=nbytes / (ms * 1e-3) / 1e9,
                what="store_kvcache bf16 -> E4M3, config 4 tokens (590K x 8 x 256, K and V)")


def cpu_baseline(lengths, tensors):
    """fp32 CPU oracle on the first sequences of config 2 (bounded sample)."""
    import torch
    from oracle.attention import attention as oracle_attention
    q, k, v, _ = tensors
    threads = os.cpu_count() or 1
    torch.set_num_threads(threads)
    take = 2
    sample = lengths[:take]
    n = sum(sample)
    qs, ks, vs = (t[:n].cpu() for t in (q, k, v))
    cu = torch.zeros(take + 1, dtype=torch.int32)
    cu[1:] = torch.tensor(sample).cumsum(0)
    oracle_attention(qs, ks, vs, cu, cu, causal=True, dtype=torch.float32)   # warmup
    times = []
    for _ in range(3):
        t0 = time.perf_counter()
        oracle_attention(qs, ks, vs, cu, cu, causal=True, dtype=torch.float32)
        times.append(time.perf_counter() - t0)
    sec = sorted(times)[1]
    flops = causal_pairs(sample, sample) * 16 * 2 * 256
    return {"value": round(flops / sec / 1e12, 4), "unit": "TFLOP/s", "cores": threads, "kind": "port",
            "cpu": cpu_model(),
            "sample": f"config 2 sequences 0-{take - 1} (lengths {sample}), fp32 oracle, median of 3"}


def cpu_model():
    """The host CPU's model name (first 'model name' line of /proc/cpuinfo)."""
    try:
        for line in Path("/proc/cpuinfo").read_text().splitlines():
            if line.startswith("model name"):
                return line.split(":", 1)[1].strip()
    except OSError:
        pass
    import platform
    return platform.processor() or "unknown"


def secondary_entry(name, r, warmup):
    """The JSON object of one secondary line."""
    entry = {"ms_per_step": round(r["ms"], 4), "warmup": warmup}
    if name == "prefill_d256":
        entry.update(TFLOPs=round(r["tflops"], 2), frac_of_bf16_peak=round(r["tflops"] / PEAK_BF16_TFLOPS, 4),
                     kernel_event_ms=round(r["kernel_ms"], 4), flops=r["flops"], what=r["what"])
    elif name == "prefill_fp8":
        entry.update(TFLOPs=round(r["tflops"], 2), frac_of_fp8_peak=round(r["tflops"] / PEAK_FP8_TFLOPS, 4),
                     frac_of_mixed_peak=round(r["tflops"] / PEAK_FP8_BF16_MIXED_TFLOPS, 4),
                     kernel_event_ms=round(r["kernel_ms"], 4), flops=r["flops"], what=r["what"])
    elif name == "store4":
        entry.update(GBps=round(r["gbs"], 1), frac_of_hbm=round(r["gbs"] / PEAK_HBM_GBS, 4),
                     bytes=r["bytes"], what=r["what"])
    elif name.startswith("5"):
        entry.update(kv_GBps=round(r["gbs"], 1), roofline_ms=round(r["roofline_ms"], 4),
                     frac=round(r["frac"], 4), chunk_flops=r["flops"])
        if name == "5_fixed_order":
            entry["what"] = ("config 5 with num_splits=1 (batch-invariant): chunks in the MFMA prefill, "
                             "single-query requests in the decode kernel with one split")
    else:
        entry.update(kv_GBps=round(r["gbs"], 1), frac_of_hbm=round(r["gbs"] / PEAK_HBM_GBS, 4),
                     kv_bytes=r["kv_bytes"], call_median_kv_GBps=round(r["call_gbs"], 1),
                     kernel_event_ms=round(r["kernel_ms"], 4))
    return entry


def main():
    args = parse()
    if args.gpus != 1:
        print(json.dumps({"error": "this build measures one MI355X; --gpus must be 1 "
                                   "(attention shards by request or KV head, one process per GPU, "
                                   "and each GPU runs these kernels on its share)"}))
        sys.exit(2)
    import torch
    device = torch.device("cuda", 0)
    only = set(args.only.split(",")) if args.only else None
    if args.copy_probe:
        copy_probe(device)
    # The secondary configurations run first: their cache writes and timed
    # calls keep the GPU busy for seconds, so the headline configuration is
    # timed at the clock a loaded GPU holds (a cold GPU's first ~100 launches
    # run up to 15% slower while its clock ramps).  Config 2's inputs are
    # built before them (on the CPU, from its seeded generator, which takes
    # about a second), so no input building leaves the GPU idle between the
    # last secondary line and config 2's warmup.
    # The last secondary line (config 2 in E4M3, the same MFMA-bound work) is
    # read only after config 2's warmup is enqueued: a host synchronize
    # between the two would leave the GPU idle for a few milliseconds, after
    # which the first ~40 prefill launches run up to 15% slower while the
    # clock settles again (kernel traces: 505-545 us per launch without the
    # gap, 502-614 us after a 3-6 ms gap).
    c2_inputs = config2_inputs(device)
    secondary = {}
    pending = None
    if not args.no_secondary:
        for name, fn in (("3", config3), ("4", config4), ("store4", store_fp8), ("5", config5),
                         ("5_fixed_order", lambda *x: config5(*x, splits=1)),
                         ("prefill_d256", lambda *x: prefill_d256(*x, c=c2_inputs)),
                         ("prefill_fp8", lambda *x: prefill_fp8(*x, c=c2_inputs, defer=True))):
            if only and name not in only and not (name == "store4" and "4" in only):
                continue
            # Every secondary line takes at least SECONDARY_WARMUP untimed
            # calls.  For the E4M3 prefill these are MFMA-bound launches that
            # bring the clock to its loaded state (it settles over ~100
            # launches, ~55 ms), so its timed calls and config 2 after it are
            # measured there rather than in the ramp; config 2 itself takes
            # exactly --warmup untimed steps.
            warmup = max(args.warmup, SECONDARY_WARMUP)
            r = fn(device, args.steps, warmup)
            if name == "prefill_fp8":
                pending = r
                continue
            secondary["config" + name if name[0].isdigit() else name] = secondary_entry(name, r, warmup)
            if "rows4" in r:
                entry = secondary_entry(name, r["rows4"], warmup)
                entry["what"] = ("config 3's cache with 4 query rows per request (speculative decode), "
                                 "causal; KV bytes counted once per request and KV head")
                secondary["config3_rows4"] = entry
            # Each line frees its inputs into torch's caching allocator and the
            # next line's inputs reuse those blocks.  No empty_cache here: K/V
            # caches in memory freshly mapped after a release to the driver
            # made config 4's page gather 3% slower (0.339-0.358 ms against
            # 0.330-0.331 after config 3, four runs each).

    c2 = config2(device, args.steps, args.warmup, c=c2_inputs)
    if pending is not None:
        secondary["prefill_fp8"] = secondary_entry("prefill_fp8", pending(), max(args.warmup, SECONDARY_WARMUP))
    line = {
        "metric": "bf16 prefill TFLOP/s & paged-decode KV GB/s, % of MI355X roofline, 1 GPU",
        "value": round(c2["tflops"], 2),
        "unit": "TFLOP/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(c2["ms"], 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "bf16",
        "data": "synthetic: seeded 0.5*N(0,1) Q/K/V, lengths from torch.Generator().manual_seed(125)",
        "config": {"workload": "config 2: varlen causal prefill, 16 seqs L~U[256,4096], Hq/Hkv 16/8, d128 "
                               "(Qwen3-0.6B attention)", "global_batch": 16, "seq_len": max(c2["lengths"]),
                   "total_tokens": sum(c2["lengths"]), "parallelism": "single GPU"},
        # achieved/frac: algorithmic FLOPs over the timed region's time per step
        # (one launch per step); the HIP-event time of the launches alone and
        # the median call are reported beside them.
        "roofline": {"bound": "mfma", "achieved": round(c2["tflops"], 2), "peak": PEAK_BF16_TFLOPS,
                     "unit": "TFLOP/s", "frac": round(c2["tflops"] / PEAK_BF16_TFLOPS, 4),
                     "traffic": measured_traffic(),
                     "flops_per_launch": c2["flops"], "kernel": "prefill_kernel",
                     "kernel_event_ms": round(c2["kernel_ms"], 4),
                     "kernel_event_frac": round(c2["kernel_tflops"] / PEAK_BF16_TFLOPS, 4),
                     "call_median_ms": round(c2["call_ms"], 4)},
    }
    line["secondary"] = secondary
    if not args.no_cpu_baseline:
        line["cpu_baseline"] = cpu_baseline(c2["lengths"], c2["tensors"])
    print(json.dumps(line))


if __name__ == "__main__":
    main()
