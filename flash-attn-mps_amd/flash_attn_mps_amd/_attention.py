"""Route a validated Problem onto the gfx950 kernels.

Counterpart of flash_attn_mps/_attention.py:88-238.  The route depends only on
shapes, dtypes, strides, feature flags and the caller's maximum lengths --
never on device values, so a call never synchronises and can be captured in
a HIP graph:

1. one query per request, not deterministic, no vLLM mask -> split-KV decode
   (`_decode.decode`; the reference's decode route, _attention.py:134-147);
2. inputs whose feature set the MFMA prefill kernel compiles
   (fa_prefill_supported) -> fa_prefill_fwd (the reference's `fast` route,
   _attention.py:149-158, which this kernel widens to windows, sinks, FP8
   K/V, E4M3 queries, ALiBi and per-request causality); in a batch of
   several requests the single-query ones go to the decode kernel first and
   fa_prefill_fwd skips them (FA_FLAG_SKIP_SINGLE_QUERY);
3. everything else -> fa_attn_fwd: fp32 calls at its head dims on the fp32
   matrix-core kernel (split by f32_splits), the rest on the generic kernel
   with the reference's split rule: deterministic -> 1, else num_splits, else
   min(32, ceil(max_k / 256)) when the row is decode-like or d > 256
   (_attention.py:159-161).

Deterministic calls (vLLM's num_splits=1, the reference's fixed
batch-invariant path, docs/contracts.md:76-79) take route 2 for every
request, single-query ones included, or route 3 with one split.  Either
kernel computes a row from its own request alone, in a fixed order: query
blocks and key tiles are aligned to the request's first query and key, the
kernel variant depends only on dtypes, head dims and feature flags, and a
key tile that a row cannot see adds exact zeros to its sums.  So a request's
rows are bit-identical whatever else is in the batch.
"""
import math

import torch

from . import _lib


def _as(t, dtype, keep):
    """`t` as a device tensor of `dtype` (kept alive until the launch is enqueued)."""
    if t is None:
        return None
    if t.dtype != dtype:
        t = t.to(dtype)
    keep.append(t)
    return t


def _bound(x):
    """A window bound as the kernels take it: 2^30 and more (past any two
    positions' distance, sys.maxsize among them) is -1, unbounded, so that
    positions plus bounds stay in 32 bits."""
    x = int(x)
    return x if -1 <= x < 1 << 30 else -1


def _float32(x):
    """x in fp32 range (larger magnitudes become infinite)."""
    x = float(x)
    return math.copysign(math.inf, x) if abs(x) > 3.4028235e38 else x


def build_args(p, out, lse, max_q=None):
    """The fa_attn_args struct of problem `p` writing `out` / `lse`."""
    keep = p.keep
    q, k, v = p.q, p.k, p.v
    code = _lib.DTYPE_CODE
    i32, f32 = torch.int32, torch.float32
    q_shape, k_shape = q.shape, k.shape
    if len(k_shape) == 4:
        page, ks, vs = k_shape[1], k.stride(), v.stride()
    else:
        page, ks, vs = 0, (0, *k.stride()), (0, *v.stride())

    def vector(t, dtype):
        """(address, stride) of an optional vector."""
        t = _as(t, dtype, keep)
        return (0, 0) if t is None else (t.data_ptr(), t.stride(0))

    def matrix(t, dtype):
        """(address, strides) of an optional [.., ..] tensor."""
        t = _as(t, dtype, keep)
        return (0, 0, 0) if t is None else (t.data_ptr(), *t.stride())

    if torch.is_tensor(p.causal):
        flags, causal = vector(p.causal, torch.bool), 0
    else:
        flags, causal = (0, 0), int(bool(p.causal))
    kind, mask_window, mask_clamp, ranges, prefix, window_len = 0, -1, 0, (0, 0, 0), (0, 0), 0
    if p.mask is not None:
        kind, mask_window, mask_clamp = p.mask.kind, _bound(p.mask.sliding_window_left), int(bool(p.mask.clamp_prefix_to_window))
        if kind == 1:
            ranges = matrix(p.mask_aux[0], i32)
            _as(p.mask_aux[1], i32, keep)
        else:
            prefix, window_len = vector(p.mask_aux[0], i32), vector(p.mask_aux[1], i32)[0]
    alibi = (0, 0, 0)
    if p.alibi is not None:
        alibi = vector(p.alibi, f32) if p.alibi.ndim == 1 else matrix(p.alibi, f32)
        if len(alibi) == 2:
            alibi = (alibi[0], 0, alibi[1])
    window_left, window_right = p.window
    return _lib.pack_attn(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), lse.data_ptr(),
        code[q.dtype], code[k.dtype], code[v.dtype], code[out.dtype],
        q_shape[0], q_shape[1], k_shape[-2], q_shape[2], v.shape[-1], p.cu_q.numel() - 1,
        page, p.max_q if max_q is None else max_q, p.max_k,
        *q.stride(), *ks, *vs, *out.stride(), *lse.stride(),
        *vector(p.cu_q, i32), *vector(p.cu_k, i32), *vector(p.used_k, i32), *matrix(p.table, i32), *vector(p.leftpad, i32),
        causal, _bound(window_left), _bound(window_right), kind, mask_window, mask_clamp, *flags,
        *ranges, *prefix, window_len,
        q_shape[2] ** -0.5 if p.scale is None else _float32(p.scale), _float32(p.softcap),
        *alibi, *vector(p.sinks, f32), *matrix(p.q_descale, f32), *matrix(p.k_descale, f32), *matrix(p.v_descale, f32),
        1, 0, 0, 0, 0, 0)


def _fits_prefill(p, out):
    """Features the MFMA route takes at all (the kernel is asked about the rest,
    vLLM mask kinds and left padding included): 16-bit queries over same-type
    or E4M3 K/V with output in the query's type, or E4M3 queries over E4M3 K/V
    with fp16/bf16 output (S on the FP8 MFMA).  Deterministic calls qualify:
    prefill_splits keeps them, and num_splits=1, at one split."""
    if p.splits not in (0, 1):
        return False
    fp8 = torch.float8_e4m3fn
    if p.k.dtype != p.v.dtype:
        return False
    if p.q.dtype == fp8:
        return p.k.dtype == fp8 and out.dtype in (torch.float16, torch.bfloat16)
    return (p.q.dtype in (torch.float16, torch.bfloat16) and out.dtype == p.q.dtype
            and p.k.dtype in (p.q.dtype, fp8))


def _partials(p, a, shape_out, shape_lse):
    """fp32 split workspace of one call: outputs, then LSEs from the next 256-byte boundary."""
    outs = -(-math.prod(shape_out) // 64) * 64
    work = torch.empty(outs + math.prod(shape_lse), dtype=torch.float32, device=p.device)
    p.keep.append(work)
    a.partial_out = work.data_ptr()
    a.partial_lse = a.partial_out + 4 * outs


# Head dims of the fp32 matrix-core kernel (attn_f32.hip, which fa_attn_fwd
# picks by itself) and the shape of its grid: 32 (head, row) columns per
# workgroup, rounds of 128 keys.
_F32_DIMS = {(d, d) for d in (32, 64, 72, 80, 96, 128, 256)} | {(192, 128)}
_F32_COLUMNS = 32
_F32_ROUND = 128


def _rows_aligned(q, k, v):
    """Whether every 16-byte piece of these fp32 rows is aligned (mirrors
    rows_aligned in attn_f32.hip)."""
    qs, ks, vs = q.stride(), k.stride(), v.stride()
    return (qs[2] == ks[-1] == vs[-1] == 1 and not (q.data_ptr() | k.data_ptr() | v.data_ptr()) & 15
            and not (qs[0] | qs[1] | ks[0] | ks[1] | ks[-2] | vs[0] | vs[1] | vs[-2]) & 3)


def f32_splits(p):
    """Key splits of an fp32 call on the matrix-core kernel (a round of 128
    keys or more each); None for calls it does not take: other types, head
    dims or alignments (the generic kernel's rule).  One query row per request is bound by memory and
    wants two workgroups per compute unit (4 x 2048 keys, 16/8 heads: 4 / 8 /
    16 splits 39.0 / 28.6 / 28.2 us a call; 4 x 8192: 8 / 16 / 32 splits 64.4 /
    58.3 / 73.5).  More rows are bound by the matrix cores, and partials cost
    more than idle compute units until most of them idle (2 x 256 tokens, 256
    workgroups: 1 / 2 splits 19.5 / 29.4 us; 1 x 2048: 177 / 204)."""
    f32 = torch.float32
    q, k, v, max_q = p.q, p.k, p.v, p.max_q
    if not (q.dtype == k.dtype == v.dtype == f32 and (p.dim_qk, p.dim_v) in _F32_DIMS and _rows_aligned(q, k, v)):
        return None
    rows = 1
    while rows < _F32_COLUMNS and rows < max_q:
        rows *= 2
    kv_heads, batch = p.kv_heads, p.batch
    group = p.heads // kv_heads
    tiles = -(-group // min(group, _F32_COLUMNS // rows))
    row_blocks = min(batch * -(-max_q // rows), p.tokens // rows + batch)
    blocks = max(1, row_blocks * kv_heads * tiles)
    wanted = -(-512 // blocks) if max_q == 1 else 256 // blocks
    return max(1, min(wanted, -(-p.visible_max // _F32_ROUND)))


# The MFMA prefill's tiles by query head dim (PrefillTile in prefill_kernel.h):
# query rows per workgroup, workgroups a compute unit holds, workgroups per
# work item, and the time of one 64-key tile on a compute unit of its own (us).
_PREFILL_TILE = {64: (128, 3, 1, 1.0), 128: (128, 2, 1, 1.1), 192: (128, 2, 1, 1.4), 256: (256, 1, 2, 2.2)}
_COMPUTE_UNITS = 256
# Below this the estimate keeps one split but for a handful of rows at d256;
# such calls are bound by the host, where planning would cost 5 of ~27 us.
_PREFILL_SPLIT_MIN_KEYS = 1024


def prefill_splits(p):
    """Key splits of an MFMA prefill call, for grids that leave at least half
    of the GPU's workgroup slots empty (the conditions mirror split_ok in
    prefill_mfma.hip).  The cheapest count by an estimate: the tiles of a
    split, 1.45 / 1.9 times as long with two / three workgroups on a compute
    unit, plus 6 us for the merge and the partials written and read back at
    2.5 TB/s.  Measured (us, 1 split -> the chosen count, bf16, 16-token
    pages): 512 rows behind 24000 keys, 32/8 heads d128 451 -> 211 (4), 64
    rows 445 -> 46 (16), 2 x 256 behind 4096, 16/8 94 -> 44 (4); d256 16/8,
    where one split runs the wave pairs, 512 of 8192 keys 297 -> 115 (4), 1024 of
    2048 84 -> 71 (2), of 8192 294 -> 198 (2); where the estimate keeps one: 1 x
    2048 causal 16/8 44 against 56 with two, d256 85 / 94, 4 x 128 behind 1024
    35 / 38."""
    if p.max_k < _PREFILL_SPLIT_MIN_KEYS:
        return 1
    if (p.splits or p.deterministic or p.mask is not None or p.alibi is not None or torch.is_tensor(p.causal)
            or p.window[0] >= 0 or (not p.causal and p.window[1] >= 0) or p.dim_qk not in _PREFILL_TILE):
        return 1
    if p.dim_v != (128 if p.dim_qk == 192 else p.dim_qk) or (p.softcap > 0 and p.dim_qk > 128):
        return 1
    blocks = _prefill_blocks(p)
    most = min(_PREFILL_TILE[p.dim_qk][1] * _COMPUTE_UNITS // blocks, 16)
    if most < 2 or p.batch > 65535:
        return 1
    best, best_us = 1, p.max_k * _key_us(p, blocks, 1)
    for n in (2, 3, 4, 6, 8, 12, 16):
        if n > most:
            break
        us = p.max_k * _key_us(p, blocks, n) + _merge_us(p, n)
        if us < best_us:
            best, best_us = n, us
    return best


def _prefill_blocks(p):
    """Workgroups of an unsplit MFMA prefill call."""
    rows, _, parts, _ = _PREFILL_TILE[p.dim_qk]
    pair = 2 if p.heads // p.kv_heads % 2 == 0 else 1   # heads per workgroup
    requests = p.batch if p.tokens >= 2 * p.batch else 1
    return requests * -(-p.tokens // (requests * (rows // pair))) * (p.heads // pair) * parts


def _key_us(p, blocks, n):
    """Time of a key in n splits: a tile's, shared by 64 keys, stretched by the
    workgroups that then share a compute unit (one split: as many as the grid has)."""
    crowd = 1 if n == 1 else 0.55 + 0.45 * -(-blocks * n // _COMPUTE_UNITS)
    return _PREFILL_TILE[p.dim_qk][3] / 64 * crowd / n


def _merge_us(p, n):
    return 6 + n * p.tokens * p.heads * p.dim_v * 8 / 2.5e6


def prefill_split_span(p, splits):
    """Keys that a request must have per split.  max_seqlen_k may be the capacity
    of a cache, far above the lengths there are, which only the kernel sees: by
    the same estimate `splits` pay from this many keys each, and a request with
    fewer takes fewer.  Captured graphs, 32/8 heads d128, capacity 32768, us with
    one split / all planned / this many each: 512 rows planned as four, 600 keys
    20.7 / 31.9 / 24.7, 1024 27.3 / 33.1 / 32.3, 2048 46.0 / 40.8 / 43.1; 64 rows
    planned as 16, 200 keys 12.7 / 15.6 / 14.9, 600 19.7 / 15.7 / 15.9.  The merge's
    launch is what one split still loses (3-4 us)."""
    blocks = _prefill_blocks(p)
    gain_us = _key_us(p, blocks, 1) - _key_us(p, blocks, splits)
    worth = _merge_us(p, splits) / gain_us if gain_us > 0 else p.max_k
    return max(1, int(min(worth, p.max_k) / splits))


_SIDE = {}

# Below this many K/V bytes (an upper bound of what the decode pass of a
# mixed batch reads: every request at the longest visible length) the decode
# pass follows the prefill on the caller's stream: it takes a few µs of GPU
# time, less than the host time of the cross-stream fork and join (an event
# record and a stream wait each way, ~30 µs per call measured on short calls).
_SIDE_STREAM_MIN_BYTES = 64 << 20


def _side_stream(device):
    """A second stream per device (default priority) for the decode rows of a
    mixed batch, with the two events that fork and join it (reused: a stream
    wait takes the event's most recent record)."""
    index = torch.device(device).index
    side = _SIDE.get(index)
    if side is None:
        side = _SIDE[index] = (torch.cuda.Stream(device), torch.cuda.Event(), torch.cuda.Event())
    return side


def _mixed_batch(p, a, fixed_order=False):
    """A batch of several requests with single-query ones among them: the
    decode kernel takes the single-query requests (it skips the others) and
    fa_prefill_fwd the rest (FA_FLAG_SKIP_SINGLE_QUERY).  The two kernels
    write disjoint rows, so they run concurrently: the prefill is enqueued
    first on the caller's stream and the decode on a side stream that starts
    after the caller's earlier work; the caller's stream then waits for it.
    The memory-bound decode fills the CUs the compute-bound prefill leaves.
    Small calls (under _SIDE_STREAM_MIN_BYTES of K/V) run both on the
    caller's stream, one after the other.
    Returns False (nothing launched) when the decode kernel cannot take the
    single-query rows.  With `fixed_order` the decode runs one split per
    request, so each single-query row is reduced in an order of its own
    request only (the batch-invariant route)."""
    dec = _lib.AttnArgs.from_buffer_copy(a)
    dec.max_seqlen_q = 1   # the decode kernel takes the one-row requests only
    if not _lib.supported("fa_decode_supported", dec):
        return False
    from ._decode import decode_workgroups, split_plan
    groups = decode_workgroups(p, 1)
    splits, span = split_plan(p.batch, groups, p.max_k, 1 if fixed_order else 0)
    dec.num_splits, dec.split_span = splits, span
    if splits > 1:
        _partials(p, dec, (p.batch, splits, p.heads, p.dim_v), (p.batch, p.heads, splits))
    a.flags |= _lib.FLAG_SKIP_SINGLE_QUERY
    kv_bytes = p.batch * p.visible_max * p.kv_heads * (p.dim_qk + p.dim_v) * p.k.element_size()
    if kv_bytes < _SIDE_STREAM_MIN_BYTES:
        _lib.call("fa_prefill_fwd", a, p.device)
        _lib.call("fa_decode_fwd", dec, p.device)
        return True
    main = torch.cuda.current_stream(p.device)
    side, fork, join = _side_stream(p.device)
    fork.record(main)
    side.wait_event(fork)
    _lib.call("fa_prefill_fwd", a, p.device)
    with torch.cuda.stream(side):
        _lib.call("fa_decode_fwd", dec, p.device)
    join.record(side)
    main.wait_event(join)
    return True


def _fixed_order_decode(p, out):
    """A fixed-order (deterministic / vLLM num_splits=1) call whose requests
    all hold one query row: the decode kernel with one split per request, on
    paged K/V, exactly when a batch holding these requests next to longer
    ones would route them to it (_mixed_batch), so a request's result does
    not depend on its neighbours.  Packed K/V keep the MFMA prefill: the
    matrix-core decode aligns its key stages to storage rows, which move
    with a request's place in the batch.  None when this route does not
    apply (nothing launched)."""
    if not p.paged or not _fits_prefill(p, out):
        return None
    lse = torch.empty((p.heads, p.tokens), device=p.device, dtype=torch.float32)
    a = build_args(p, out, lse)
    if not (_lib.supported("fa_prefill_supported", a) and _lib.supported("fa_decode_supported", a)):
        return None
    from ._decode import decode
    return decode(p, out, splits=1)


def solve(p):
    """Run a validated Problem: returns (out [T, Hq, Dv], natural-log lse [Hq, T])."""
    out = p.out
    if out is None:
        out = torch.empty((p.tokens, p.heads, p.dim_v), dtype=p.output_dtype, device=p.device)
    if p.tokens == 0:
        return out, torch.empty((p.heads, 0), device=p.device, dtype=torch.float32)
    if p.max_q <= 0:
        raise ValueError("nonempty queries need max_seqlen_q >= 1")
    if p.batch < 1:
        raise ValueError("cu_seqlens_q needs at least two offsets")
    if p.max_q == 1 and not p.deterministic and p.mask is None:
        from ._decode import decode
        return decode(p, out)
    if p.max_q == 1 and p.deterministic and p.mask is None:
        done = _fixed_order_decode(p, out)
        if done is not None:
            return done
    if p.max_q > 1 and not p.deterministic and p.mask is None:
        # A few query rows per request (speculative / multi-token decode):
        # the matrix-core decode with (head, row) columns when it takes them.
        from ._decode import decode_rows
        done = decode_rows(p, out)
        if done is not None:
            return done
    lse = torch.empty((p.heads, p.tokens), device=p.device, dtype=torch.float32)
    a = build_args(p, out, lse)
    if _fits_prefill(p, out) and _lib.supported("fa_prefill_supported", a):
        # In a mixed chunked-prefill + decode batch the single-query requests
        # take the decode kernel: a 128-row MFMA query tile per head would be
        # almost empty for them.  Packed self-attention (queries and keys on
        # the same offsets) gives a single-query request a single key, so the
        # MFMA kernel keeps it and no decode pass runs.  Deterministic calls
        # keep every request in this kernel (the decode kernel's split count
        # follows the batch).
        self_attention = p.cu_k is p.cu_q and p.used_k is None and not p.paged
        mixed = p.batch > 1 and not self_attention and (not p.deterministic or p.paged)
        splits = prefill_splits(p)
        if splits > 1:
            _partials(p, a, (splits, p.tokens, p.heads, p.dim_v), (splits, p.heads, p.tokens))
            a.num_splits, a.split_span = splits, prefill_split_span(p, splits)
        if not (mixed and _mixed_batch(p, a, fixed_order=p.deterministic)):
            _lib.call("fa_prefill_fwd", a, p.device)
        return out, lse
    per_row = p.deterministic or p.max_q == 1 or max(p.dim_qk, p.dim_v) > 256
    if p.deterministic:
        splits = 1
    else:
        splits = p.splits or f32_splits(p) or (min(32, max(1, -(-p.max_k // 256))) if per_row else 1)
    if splits > 1:
        _partials(p, a, (splits, p.tokens, p.heads, p.dim_v), (splits, p.heads, p.tokens))
    a.num_splits = splits
    _lib.call("fa_attn_fwd", a, p.device)
    return out, lse
