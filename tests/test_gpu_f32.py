"""fp32 attention on the fp32 matrix-core kernel against the float64 oracle:
edges of its 32-row blocks, 32-key stages and 128-key rounds, every head dim,
packed (head, row) columns, splits, and the features it evaluates at run time.

Tolerance: with |v| <= 5 and scores of standard deviation ~1, a score's fp32
dot product over <= 256 dims is within ~16 * 2^-24 * |q||k| / sqrt(d) ~ 2e-6,
a probability within twice that relative, and an output within 2 * 4e-6 *
max|v| = 4e-5 (softcaps and ALiBi add terms of the same size).
"""
import pytest
import torch

from flash_attn_mps_amd import vllm
from harness import assert_parity, attention, offsets, oracle_attention, seeded

pytestmark = pytest.mark.gpu

BAR = 4e-5


def _packed(device, q_lens, k_lens, heads, kv_heads, dq, dv, seed):
    q = seeded((sum(q_lens), heads, dq), seed, torch.float32, device)
    k = seeded((sum(k_lens), kv_heads, dq), seed + 1, torch.float32, device)
    v = seeded((sum(k_lens), kv_heads, dv), seed + 2, torch.float32, device)
    return q, k, v, offsets(q_lens, device), offsets(k_lens, device)


@pytest.mark.parametrize("dq,dv", [(32, 32), (64, 64), (72, 72), (80, 80), (96, 96), (128, 128), (192, 128), (256, 256)])
@pytest.mark.parametrize("causal", [True, False])
def test_head_dims_and_tile_edges(device, dq, dv, causal):
    """Row blocks of 1, 31, 32, 33 rows over 0, 1, 127, 128, 129, 300 keys."""
    q_lens, k_lens = [1, 31, 32, 33, 2, 70], [0, 1, 127, 128, 129, 300]
    q, k, v, cu_q, cu_k = _packed(device, q_lens, k_lens, 4, 2, dq, dv, 900)
    got, lse = attention(q, k, v, cu_seqlens_q=cu_q, cu_seqlens_k=cu_k, max_seqlen_q=70, max_seqlen_k=300,
                         causal=causal)
    ref, ref_lse = oracle_attention(q, k, v, cu_q, cu_k, causal=causal)
    assert_parity(got, lse, ref, ref_lse, out_bar=BAR)


@pytest.mark.parametrize("rows", [1, 2, 3, 16, 17])
@pytest.mark.parametrize("heads,kv_heads", [(2, 2), (6, 2), (80, 2)])
@pytest.mark.parametrize("splits", [0, 1, 3])
def test_head_row_columns_over_paged_cache(device, rows, heads, kv_heads, splits):
    """Groups of 1, 3 and 40 heads (tiles that a group does not fill), 1..17
    rows per request, left padding, pages of 48, unread storage NaN."""
    page, k_lens, left = 48, [max(rows, 1), 131, 700], [0, 5, 47]
    cols = -(-(max(k_lens) + max(left)) // page)
    table = torch.randperm(3 * cols, generator=torch.Generator().manual_seed(7)).reshape(3, cols).int()
    k = torch.full((3 * cols, page, kv_heads, 64), float("nan"), device=device)
    v = torch.full((3 * cols, page, kv_heads, 64), float("nan"), device=device)
    for b, (n, pad) in enumerate(zip(k_lens, left)):
        pos = torch.arange(pad, pad + n)
        at = (table[b, pos // page].long(), pos % page)
        k[at] = seeded((n, kv_heads, 64), 910 + b, torch.float32, device)
        v[at] = seeded((n, kv_heads, 64), 920 + b, torch.float32, device)
    q = seeded((3 * rows, heads, 64), 930, torch.float32, device)
    sinks = seeded((heads,), 931, torch.float32, device)
    cu_q, used = offsets([rows] * 3, device), torch.tensor(k_lens, dtype=torch.int32, device=device)
    got, lse = attention(q, k, v, cu_seqlens_q=cu_q, seqused_k=used, max_seqlen_q=rows, max_seqlen_k=700,
                         block_table=table.to(device), leftpad_k=torch.tensor(left, dtype=torch.int32, device=device),
                         causal=True, s_aux=sinks, num_splits=splits)
    ref, ref_lse = oracle_attention(q, k.nan_to_num(0), v.nan_to_num(0), cu_q, used_k=used, block_table=table,
                                    leftpad=torch.tensor(left), causal=True, sinks=sinks)
    assert_parity(got, lse, ref, ref_lse, out_bar=BAR)


@pytest.mark.parametrize("feature", ["window", "right", "softcap", "alibi", "causal_flags", "descales", "prefix", "rolling"])
def test_score_features(device, feature):
    q_lens, k_lens = [40, 1, 100, 5], [40, 260, 100, 3]
    q, k, v, cu_q, cu_k = _packed(device, q_lens, k_lens, 4, 2, 128, 128, 940)
    kw = dict(causal=True)
    if feature == "window":
        kw.update(window_size=(33, 0))
    elif feature == "right":
        kw.update(causal=False, window_size=(70, 5))
    elif feature == "softcap":
        kw.update(softcap=2.0)
    elif feature == "alibi":
        kw.update(alibi_slopes=torch.tensor([0.5, 0.25, 0.0, 1.0], device=device), softcap=3.0)
    elif feature == "causal_flags":
        kw.update(causal=torch.tensor([True, False, False, True], device=device))
    elif feature == "descales":
        kw.update({n: seeded((4, 2), 950 + i, torch.float32, device).abs() + 0.1
                   for i, n in enumerate(("q_descale", "k_descale", "v_descale"))})
    elif feature == "prefix":
        ranges = torch.full((146, 2), -1, dtype=torch.int32)
        ranges[10:30] = torch.tensor([5, 35], dtype=torch.int32)
        ranges[60:140] = torch.tensor([50, 99], dtype=torch.int32)
        kw.update(mask_mod=vllm.mm_prefix_mask(20), aux_tensors=[ranges.to(device), cu_q])
    else:
        aux = [torch.tensor([3, 100, 0, 2], dtype=torch.int32, device=device),
               torch.tensor([16], dtype=torch.int32, device=device)]
        kw.update(mask_mod=vllm.rswa_mask(), aux_tensors=aux)
    names = dict(window_size="window", alibi_slopes="alibi", mask_mod="mask", aux_tensors="aux")
    okw = {names.get(n, n): x for n, x in kw.items()}
    got, lse = attention(q, k, v, cu_seqlens_q=cu_q, cu_seqlens_k=cu_k, max_seqlen_q=100, max_seqlen_k=260, **kw)
    ref, ref_lse = oracle_attention(q, k, v, cu_q, cu_k, **okw)
    assert_parity(got, lse, ref, ref_lse, out_bar=BAR)


def test_rows_do_not_depend_on_the_batch(device):
    """num_splits=1: a windowed request's rows are bit-identical alone (8 rows,
    packed columns) and beside a longer one (32-row blocks)."""
    q, k, v, cu_q, cu_k = _packed(device, [8, 90], [500, 333], 4, 2, 64, 64, 960)
    run = dict(causal=True, window_size=(150, 0), num_splits=1, deterministic=True)
    both, lse = attention(q, k, v, cu_seqlens_q=cu_q, cu_seqlens_k=cu_k, max_seqlen_q=90, max_seqlen_k=500, **run)
    alone, lse1 = attention(q[:8], k[:500], v[:500], cu_seqlens_q=cu_q[:2], cu_seqlens_k=cu_k[:2], max_seqlen_q=8,
                            max_seqlen_k=500, **run)
    assert torch.equal(both[:8], alone) and torch.equal(lse[:, :8], lse1)


@pytest.mark.parametrize("mask", ["prefix", "rolling", "prefix_rows", "clamped"])
@pytest.mark.parametrize("splits", [1, 3])
@pytest.mark.parametrize("dim", [64, 128])
def test_masked_keys_that_no_row_sees(device, mask, splits, dim):
    """Mask kinds leave keys unseen before the first window, between a prefix
    and the windows, and between rows' own ranges: whole pages (whose table
    entries then lead elsewhere) and single keys inside a 32-key stage.  They
    hold NaN and infinities here, and no result may show them."""
    page, q_lens, k_lens = 16, [40, 3], [700, 333]
    total = sum(q_lens)
    cols = -(-max(k_lens) // page)
    cu_q, used = offsets(q_lens, device), torch.tensor(k_lens, dtype=torch.int32, device=device)
    if mask == "rolling":
        spec, aux = vllm.rswa_mask(), [torch.tensor([50, 7], dtype=torch.int32, device=device),
                                       torch.tensor([21], dtype=torch.int32, device=device)]
    else:
        ranges = torch.full((total, 2), -1, dtype=torch.int32)
        if mask == "prefix_rows":
            ranges[5:9] = torch.tensor([[300, 310], [77, 77], [0, 3], [640, 2 ** 31 - 1]], dtype=torch.int32)
        elif mask == "clamped":
            ranges[:] = torch.tensor([0, 650], dtype=torch.int32)
        ranges[41] = torch.tensor([100, 120], dtype=torch.int32)
        spec, aux = vllm.mm_prefix_mask(20, mask == "clamped"), [ranges.to(device), cu_q]
    # The keys each request's rows see, by the definition of the masks.
    seen, row = [torch.zeros(n, dtype=torch.bool) for n in k_lens], 0
    for b, (nq, nk) in enumerate(zip(q_lens, k_lens)):
        key = torch.arange(nk)
        for i in range(nq):
            diff = i + nk - nq - key
            if mask == "rolling":
                see = (diff >= 0) & ((key < int(aux[0][b])) | (diff < 21))
            else:
                first, last = ranges[row].tolist()
                see = (diff >= 0) & (diff < 20)
                if first >= 0:
                    see |= (key >= first) & (key <= last) & ((diff < 20) if mask == "clamped" else True)
            seen[b] |= see
            row += 1
    table = torch.full((2, cols), -1, dtype=torch.int64)
    poison = 2 * cols   # the page of unseen pages' table entries
    order = torch.randperm(2 * cols, generator=torch.Generator().manual_seed(5))
    k, v = (torch.full((2 * cols + 1, page, 2, dim), float(x), device=device) for x in ("nan", "inf"))
    for b, nk in enumerate(k_lens):
        for c in range(cols):
            pos = torch.arange(min(c * page, nk), min((c + 1) * page, nk))
            if not seen[b][pos].any():
                table[b, c] = poison
                continue
            table[b, c] = order[b * cols + c]
            own = pos[seen[b][pos]] % page
            for t, seed in ((k, 970), (v, 980)):
                t[table[b, c], own.to(device)] = seeded((len(own), 2, dim), seed + 100 * b + c, torch.float32, device)
    table = table.int()
    q = seeded((total, 4, dim), 990, torch.float32, device)
    got, lse = attention(q, k, v, cu_seqlens_q=cu_q, seqused_k=used, max_seqlen_q=40, max_seqlen_k=700,
                         block_table=table.to(device), causal=True, mask_mod=spec, aux_tensors=aux, num_splits=splits)
    clean = [t.nan_to_num(0, posinf=0) for t in (k, v)]
    ref, ref_lse = oracle_attention(q, *clean, cu_q, used_k=used, block_table=table, causal=True, mask=spec, aux=aux)
    assert_parity(got, lse, ref, ref_lse, out_bar=BAR)


@pytest.mark.parametrize("dq,dv", [(32, 32), (64, 64), (72, 72), (128, 128), (192, 128), (256, 256)])
@pytest.mark.parametrize("case", ["causal", "window", "rows2", "clamped", "splits"])
def test_values_that_are_not_finite_stay_with_the_rows_that_see_them(device, dq, dv, case):
    """A NaN and infinities in V at keys that only some rows of a 32-row block
    see: those rows show them in their dims, the others and the other dims
    nothing of them."""
    q_lens, k_lens = ([2, 2], [300, 131]) if case == "rows2" else ([40, 70], [45, 260])
    q, k, v, cu_q, cu_k = _packed(device, q_lens, k_lens, 6, 2, dq, dv, 995)
    total, last = sum(q_lens), max(q_lens)
    kw = dict(causal=True, num_splits=3 if case == "splits" else 1)
    if case == "window":
        kw.update(window_size=(9, 0))
    elif case == "clamped":
        ranges = torch.full((total, 2), -1, dtype=torch.int32)
        ranges[7] = torch.tensor([20, 44], dtype=torch.int32)
        kw.update(mask_mod=vllm.mm_prefix_mask(15), aux_tensors=[ranges.to(device), cu_q])
    names = dict(window_size="window", mask_mod="mask", aux_tensors="aux")
    ref, ref_lse = oracle_attention(q, k, v, cu_q, cu_k, **{names.get(n, n): x for n, x in kw.items() if n != "num_splits"})
    # (key from the request's end, dim, value); NaN in KV head 0 only.
    poison = [(1, 3, float("nan"), 0), (1, 5, float("inf"), None), (1 + last // 2, 9, float("-inf"), None)]
    bad = torch.zeros(total, 6, dv, dtype=torch.bool)
    weight = {}
    for back, dim, value, head in poison:
        probe = torch.zeros_like(v)
        for end in cu_k[1:].tolist():
            probe[end - back, slice(None) if head is None else head, dim] = 1.0
        weight[dim], _ = oracle_attention(q, k, probe, cu_q, cu_k, **{names.get(n, n): x for n, x in kw.items() if n != "num_splits"})
        bad[weight[dim] > 0] = True
        for end in cu_k[1:].tolist():
            v[end - back, slice(None) if head is None else head, dim] = value
    assert bad.any() and not bad[..., 3].all() and not bad[..., 7].any()
    got, lse = attention(q, k, v, cu_seqlens_q=cu_q, cu_seqlens_k=cu_k, max_seqlen_q=last, max_seqlen_k=max(k_lens), **kw)
    got = got.cpu()
    assert torch.equal(~got.isfinite(), bad)
    assert got[..., 3][bad[..., 3]].isnan().all() and (got[..., 5][bad[..., 5]] == float("inf")).all()
    assert (got[..., 9][bad[..., 9]] == float("-inf")).all()
    # The clean reference, without the poisoned keys' dims.
    untouched = torch.ones(dv, dtype=torch.bool)
    untouched[[3, 5, 9]] = False
    assert_parity(got[..., untouched], lse, ref[..., untouched], ref_lse, torch.float32, out_bar=BAR)
    clean = torch.where(bad, torch.zeros((), dtype=torch.float64), ref)
    for _, dim, _, head in poison:   # rows without weight on a poisoned key: as with any finite value there
        rows = ~bad[..., dim]
        assert (got[..., dim][rows].double() - clean[..., dim][rows]).abs().max() <= BAR if rows.any() else True
