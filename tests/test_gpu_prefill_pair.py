"""256-dim prefill by wave pairs against the float64 oracle: edges of the
32-row blocks and 64-key tiles, rows without keys, windows that start and end
inside tiles, and the work list's forms (many requests, odd head counts).
Values are 0.5 N(0, 1), the scale at which 16-bit probabilities meet the bar."""
import pytest
import torch

from harness import assert_parity, attention, offsets, oracle_attention, seeded

pytestmark = pytest.mark.gpu


def _run(device, q_lens, k_lens, heads, kv_heads, dtype, page=0, **kw):
    q = seeded((sum(q_lens), heads, 256), 70, dtype, device)
    cu_q = offsets(q_lens, device)
    call, okw = dict(cu_seqlens_q=cu_q, max_seqlen_q=max(q_lens), max_seqlen_k=max(k_lens)), {}
    if page:
        cols = max(1, -(-max(k_lens) // page))
        n = len(k_lens) * cols
        table = torch.randperm(n, generator=torch.Generator().manual_seed(2)).reshape(-1, cols).int()
        shape = (n, page, kv_heads, 256)
        call.update(seqused_k=torch.tensor(k_lens, dtype=torch.int32, device=device), block_table=table.to(device))
        okw.update(used_k=call["seqused_k"], block_table=table)
    else:
        shape = (sum(k_lens), kv_heads, 256)
        call.update(cu_seqlens_k=offsets(k_lens, device))
        okw.update(cu_k=call["cu_seqlens_k"])
    k, v = seeded(shape, 71, dtype, device), seeded(shape, 72, dtype, device, scale=0.5)
    names = dict(window_size="window", s_aux="sinks", softmax_scale="scale")
    okw.update({names.get(n, n): x for n, x in kw.items()})
    got, lse = attention(q, k, v, **call, **kw)
    ref, ref_lse = oracle_attention(q, k, v, cu_q, **okw)
    assert_parity(got, lse, ref, ref_lse)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("softcap", [0.0, 3.0])
@pytest.mark.parametrize("window", [None, (0, 0), (70, 0), (129, 33)])
def test_tile_edges(device, dtype, causal, softcap, window):
    """17..200 rows over 0..333 keys (fewer keys than rows among them)."""
    kw = dict(causal=causal, softcap=softcap)
    if window is not None:
        kw["window_size"] = window
    _run(device, [17, 32, 33, 128, 129, 200], [0, 31, 64, 65, 333, 192], 4, 2, dtype, **kw)


@pytest.mark.parametrize("heads,kv_heads,page", [(3, 3, 16), (6, 2, 64), (8, 8, 256), (32, 2, 16)])
def test_heads_pages_sinks_and_flags(device, heads, kv_heads, page):
    """Groups of one and odd groups (one head per workgroup), paged K/V,
    sinks, per-request causality, a negative scale."""
    flags = torch.tensor([True, False, True], device=device)
    sinks = seeded((heads,), 73, torch.float32, device)
    _run(device, [70, 40, 19], [200, 129, 19], heads, kv_heads, torch.bfloat16, page, causal=flags, s_aux=sinks,
         softmax_scale=-0.05)


@pytest.mark.parametrize("requests", [70, 300])
def test_many_requests(device, requests):
    """Over 64 (several requests per lane) and over 256 (per-pair grid)."""
    lens = [17 + (7 * i) % 50 for i in range(requests)]
    _run(device, lens, lens, 2, 1, torch.float16, causal=True)
