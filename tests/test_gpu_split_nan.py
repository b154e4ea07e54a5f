"""A NaN among a call's inputs reaches the rows that see it whatever the number
of key splits: a split whose sum is NaN is not one without keys.

The splits' merges give such a split no weight of zero (which would drop its
whole key range from a finite, wrong row).  Expected everywhere: the rows that
see the NaN key, or have a NaN query, are NaN in every dim with LSE -inf, as
with one split, and the others equal the oracle over the clean inputs."""
import pytest
import torch

from flash_attn_mps_amd import _attention
from harness import assert_parity, attention, offsets, oracle_attention, seeded

pytestmark = pytest.mark.gpu

E4M3 = torch.float8_e4m3fn
NAN = float("nan")


def _values(shape, seed, dtype, device, scale=1.0):
    x = seeded(shape, seed, torch.float32, "cpu", scale=scale)
    return (x.clamp(-448, 448) if dtype == E4M3 else x).to(dtype).to(device)


def _poison(x, index):
    """x with NaN at `index` (E4M3: the code 0x7F)."""
    x = x.clone()
    if x.dtype == E4M3:
        x.view(torch.uint8)[index] = 0x7F
    else:
        x[index] = NAN
    return x


def _check(got, lse, ref, ref_lse, bad, out_bar=None):
    """bad [T, Hq]: rows that must be NaN."""
    bad = bad.to(got.device)
    assert got[bad].isnan().all() and torch.isneginf(lse.transpose(0, 1)[bad]).all()
    keep = ~bad.cpu()
    assert_parity(got.cpu()[keep], lse.transpose(0, 1).cpu()[keep], ref[keep], ref_lse.transpose(0, 1)[keep],
                  got.dtype, out_bar=out_bar)


@pytest.mark.parametrize("qt,kt,dq,dv", [(torch.bfloat16, torch.bfloat16, 64, 64), (torch.float16, torch.float16, 128, 128),
                                         (torch.bfloat16, torch.bfloat16, 192, 128), (torch.bfloat16, torch.bfloat16, 256, 256),
                                         (torch.bfloat16, E4M3, 128, 128), (E4M3, E4M3, 64, 64), (E4M3, E4M3, 256, 256),
                                         (torch.float32, torch.float32, 64, 64), (torch.float32, torch.float32, 256, 256)])
@pytest.mark.parametrize("splits", [1, 2, 5])
def test_rows_of_a_chunk(device, monkeypatch, qt, kt, dq, dv, splits):
    """90 and 33 rows behind 610 and 200 earlier keys; NaN in one early key of
    the first request (KV head 1 of 2), in one of its last keys, which only its
    last rows see, and in one query row of the second."""
    q_lens, k_lens = [90, 33], [700, 233]
    k, v = _values((sum(k_lens), 2, dq), 2, kt, device), _values((sum(k_lens), 2, dv), 3, kt, device, 0.5)
    q = _values((123, 4, dq), 4, qt, device)
    cu_q, cu_k = offsets(q_lens, device), offsets(k_lens, device)
    ref, ref_lse = oracle_attention(q.float() if qt == E4M3 else q, k.float(), v.float(), cu_q, cu_k, causal=True)
    monkeypatch.setattr(_attention, "prefill_splits", lambda p: splits)
    monkeypatch.setattr(_attention, "prefill_split_span", lambda p, n: 0)
    kw = dict(cu_seqlens_q=cu_q, cu_seqlens_k=cu_k, max_seqlen_q=90, max_seqlen_k=700, causal=True,
              num_splits=splits if qt == torch.float32 else 0)
    bad = torch.zeros(123, 4, dtype=torch.bool)
    bad[:90, 2:] = True            # query heads 2, 3: KV head 1
    bad[100, 1] = True
    bad[85:90, :2] = True          # the row of key 695 and those after it
    k = _poison(_poison(k, (70, 1, 5)), (695, 0, 0))
    q = _poison(q, (100, 1, 7))
    got, lse = attention(q, k, v, **kw)
    _check(got, lse, ref, ref_lse, bad, 1e-4 if qt == torch.float32 else None)


@pytest.mark.parametrize("heads,kv_heads,dim", [(12, 3, 128), (4, 4, 128), (4, 4, 256), (12, 3, 64),
                                                (16, 2, 128), (16, 4, 64), (16, 8, 128), (16, 16, 64)])
@pytest.mark.parametrize("mixed,splits", [(True, 0), (True, 1), (False, 0), (False, 1), (False, 3)])
def test_single_rows_of_e4m3_queries(device, heads, kv_heads, dim, mixed, splits):
    """Alone and beside a 40-row request; matrix-core and VALU decode."""
    k_lens = [700, 300, 257, 90]
    q_lens = [1, 1, 1, 40 if mixed else 1]
    cols, page = 44, 16
    table = torch.arange(4 * cols, dtype=torch.int32).reshape(4, cols)
    k, v = (_values((4 * cols, page, kv_heads, dim), s, E4M3, device) for s in (2, 3))
    q = _values((sum(q_lens), heads, dim), 4, E4M3, device)
    cu, used = offsets(q_lens, device), torch.tensor(k_lens, dtype=torch.int32, device=device)
    kw = dict(cu_seqlens_q=cu, seqused_k=used, max_seqlen_q=max(q_lens), max_seqlen_k=700, causal=True,
              block_table=table.to(device), num_splits=splits)
    ref, ref_lse = oracle_attention(q.float(), k.float(), v.float(), cu, used_k=used, block_table=table, causal=True)
    group = heads // kv_heads
    bad = torch.zeros(sum(q_lens), heads, dtype=torch.bool)
    bad[0, -group:] = True         # key 500 of request 0, its last KV head
    bad[2, 1] = True               # a NaN query head
    k = _poison(k, (500 // page, 500 % page, kv_heads - 1, 3))
    q = _poison(q, (2, 1, 3))
    got, lse = attention(q, k, v, **kw)
    _check(got[:3], lse[:, :3], ref[:3], ref_lse[:, :3], bad[:3])


@pytest.mark.parametrize("splits", [2, 70])
@pytest.mark.parametrize("dim", [8, 100, 256])
def test_merge_of_caller_states_with_nan_lse(device, splits, dim):
    """fa_merge_partials on its own: a NaN LSE among numbers makes the row NaN;
    a row of NaN (and -inf) LSEs alone is empty."""
    from flash_attn_mps_amd._merge import merge_partials
    part = seeded((splits, 3, 2, dim), 5, torch.float32, device)
    part_lse = seeded((splits, 2, 3), 6, torch.float32, device)
    part_lse[1, 0, 0] = NAN
    part_lse[:, 1, 2] = NAN
    part_lse[:, 0, 1] = NAN
    part_lse[0, 0, 1] = float("-inf")
    out, lse = merge_partials(part, part_lse)
    assert out[0, 0].isnan().all() and lse[0, 0].isnan()
    assert (out[2, 1] == 0).all() and torch.isneginf(lse[1, 2])
    assert (out[1, 0] == 0).all() and torch.isneginf(lse[0, 1])
    assert out[0, 1].isfinite().all() and out[2, 0].isfinite().all()


@pytest.mark.parametrize("heads,kv_heads,dim", [(16, 2, 128), (64, 4, 128), (16, 4, 64), (16, 16, 64), (16, 8, 128)])
@pytest.mark.parametrize("head", [0, 1])
@pytest.mark.parametrize("splits", [0, 1])
def test_a_nan_in_one_kv_head_stays_with_its_queries(device, heads, kv_heads, dim, head, splits):
    """E4M3 queries over neighbouring KV heads that run in pairs: a NaN in V
    (one dim) and in K (another request) of either head of a pair."""
    k_lens = [300, 131, 700]
    k, v = (_values((sum(k_lens), kv_heads, dim), s, E4M3, device) for s in (2, 3))
    q = _values((3, heads, dim), 4, E4M3, device)
    cu, cu_k = offsets([1, 1, 1], device), offsets(k_lens, device)
    ref, ref_lse = oracle_attention(q.float(), k.float(), v.float(), cu, cu_k, causal=True)
    v = _poison(v, (77, head, 9))
    k = _poison(k, (300 + 100, head, 1))
    got, lse = attention(q, k, v, cu_seqlens_q=cu, cu_seqlens_k=cu_k, max_seqlen_q=1, max_seqlen_k=700, causal=True,
                         num_splits=splits)
    group = heads // kv_heads
    own = slice(head * group, (head + 1) * group)
    assert got[0, own, 9].isnan().all()
    got[0, own, 9] = ref[0, own, 9].to(got)
    bad = torch.zeros(3, heads, dtype=torch.bool)
    bad[1, own] = True
    _check(got, lse, ref, ref_lse, bad)
