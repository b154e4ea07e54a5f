"""Key-split MFMA prefill (few query blocks over many keys) against the float64
oracle and the unsplit route: tile remainders per split, splits without tiles,
requests without keys, sinks, and mixed batches whose single-query rows the
decode kernel owns."""
import pytest
import torch

from flash_attn_mps_amd import _attention, _lib
from harness import assert_parity, attention, kernel_args, offsets, oracle_attention, problem, seeded

pytestmark = pytest.mark.gpu

E4M3 = torch.float8_e4m3fn


def _values(shape, seed, dtype, device, scale=1.0):
    if dtype == E4M3:
        return (seeded(shape, seed, torch.float32, "cpu") * scale).clamp(-448, 448).to(E4M3).to(device)
    return seeded(shape, seed, dtype, device, scale=scale)


def _paged(device, k_lens, kv_heads, dq, dv, dtype, page=16):
    cols = max(1, -(-max(k_lens) // page))
    table = torch.randperm(len(k_lens) * cols, generator=torch.Generator().manual_seed(1)).reshape(len(k_lens), cols).int()
    k = _values((table.numel(), page, kv_heads, dq), 2, dtype, device)
    v = _values((table.numel(), page, kv_heads, dv), 3, dtype, device, 0.5)
    return k, v, table


def _split_everything(monkeypatch, count):
    monkeypatch.setattr(_attention, "prefill_splits", lambda p: count)
    monkeypatch.setattr(_attention, "prefill_split_span", lambda p, splits: 0)


@pytest.mark.parametrize("qt,kt", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float16),
                                   (torch.bfloat16, E4M3), (E4M3, E4M3)])
@pytest.mark.parametrize("dq,dv", [(64, 64), (128, 128), (256, 256), (192, 128)])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("splits", [2, 5, 16])
def test_splits(device, monkeypatch, qt, kt, dq, dv, causal, splits):
    """33, 64, 130 and 3 rows over 700, 0, 131 and 64 keys, the rows under
    causality seeing from none to all of them; more splits than tiles."""
    if kt == E4M3 and dq == 192:
        pytest.skip("no E4M3 192/128 tile")
    q_lens, k_lens = [33, 64, 130, 3], [700, 0, 131, 64]
    k, v, table = _paged(device, k_lens, 2, dq, dv, kt)
    q = _values((230, 4, dq), 4, qt, device)
    sinks = seeded((4,), 5, torch.float32, device)
    _split_everything(monkeypatch, splits)
    cu, used = offsets(q_lens, device), torch.tensor(k_lens, dtype=torch.int32, device=device)
    got, lse = attention(q, k, v, cu_seqlens_q=cu, seqused_k=used, max_seqlen_q=130, max_seqlen_k=700,
                         block_table=table.to(device), causal=causal, s_aux=sinks)
    ref, ref_lse = oracle_attention(q, k.float(), v.float(), cu, used_k=used, block_table=table, causal=causal, sinks=sinks)
    assert_parity(got, lse, ref, ref_lse)


@pytest.mark.parametrize("dim,softcap,batch", [(128, 0.0, [1, 40, 1, 1]), (64, 3.0, [1, 70]), (128, 3.0, [50])])
def test_mixed_batches_and_softcap(device, monkeypatch, dim, softcap, batch):
    k_lens = [900, 513, 64, 1][:len(batch)]
    k, v, table = _paged(device, k_lens, 2, dim, dim, torch.bfloat16)
    q = _values((sum(batch), 4, dim), 6, torch.bfloat16, device)
    _split_everything(monkeypatch, 4)
    cu, used = offsets(batch, device), torch.tensor(k_lens, dtype=torch.int32, device=device)
    out = torch.full((sum(batch) + 2, 4, dim), 77.0, dtype=torch.bfloat16, device=device)
    got, lse = attention(q, k, v, cu_seqlens_q=cu, seqused_k=used, max_seqlen_q=max(batch), max_seqlen_k=900,
                         block_table=table.to(device), causal=True, softcap=softcap, out=out[1:-1])
    ref, ref_lse = oracle_attention(q, k, v, cu, used_k=used, block_table=table, causal=True, softcap=softcap)
    assert_parity(got, lse, ref, ref_lse)
    assert (out[0] == 77).all() and (out[-1] == 77).all()


@pytest.mark.parametrize("dq,dv,kt,softcap", [(64, 64, torch.bfloat16, 2.0), (128, 128, E4M3, 0.0), (192, 128, torch.bfloat16, 0.0),
                                              (256, 256, torch.bfloat16, 0.0), (256, 256, torch.bfloat16, 2.0)])
def test_the_plan_and_the_kernel_agree(device, dq, dv, kt, softcap):
    """A 64-row chunk behind 20000 keys splits exactly where the kernel has a
    split variant, and num_splits=1 / windows / ALiBi never do."""
    q = torch.zeros(64, 4, dq, dtype=torch.bfloat16, device=device)
    k, v = (torch.zeros(1250, 16, 2, d, dtype=torch.uint8, device=device).to(kt) for d in (dq, dv))
    kw = dict(cu_seqlens_q=offsets([64], device), seqused_k=torch.tensor([20000], dtype=torch.int32, device=device),
              max_seqlen_q=64, max_seqlen_k=20000, block_table=torch.arange(1250, dtype=torch.int32, device=device)[None],
              causal=True, softcap=softcap)
    out, lse = torch.empty(64, 4, dv, dtype=torch.bfloat16, device=device), torch.empty(4, 64, device=device)
    splits = _attention.prefill_splits(problem(q, k, v, **kw))
    a = kernel_args(q, k, v, out, lse, keep=[], **kw)
    a.num_splits = 4
    assert (splits > 1) == _lib.supported("fa_prefill_supported", a) == (not (dq == 256 and softcap))
    for extra in (dict(num_splits=1), dict(deterministic=True), dict(window_size=(100, 0)),
                  dict(alibi_slopes=torch.ones(4, device=device))):
        assert _attention.prefill_splits(problem(q, k, v, **{**kw, **extra})) == 1


@pytest.mark.parametrize("max_q", [40, 1 << 20, 1 << 30])
def test_a_loose_row_bound(device, monkeypatch, max_q):
    """max_seqlen_q far above any request's rows: the merge's grid follows the
    rows there are (2^30 rows of 4 heads were refused, 2^20 of 3 requests ran
    three million idle workgroups)."""
    q_lens, k_lens = [40, 3, 17], [700, 64, 131]
    k, v, table = _paged(device, k_lens, 2, 128, 128, torch.bfloat16)
    q = _values((60, 4, 128), 8, torch.bfloat16, device)
    _split_everything(monkeypatch, 4)
    cu, used = offsets(q_lens, device), torch.tensor(k_lens, dtype=torch.int32, device=device)
    got, lse = attention(q, k, v, cu_seqlens_q=cu, seqused_k=used, max_seqlen_q=max_q, max_seqlen_k=700,
                         block_table=table.to(device), causal=True)
    ref, ref_lse = oracle_attention(q, k, v, cu, used_k=used, block_table=table, causal=True)
    assert_parity(got, lse, ref, ref_lse)


@pytest.mark.parametrize("qt,kt,dq,dv", [(torch.bfloat16, torch.bfloat16, 64, 64), (torch.float16, torch.float16, 128, 128),
                                         (torch.bfloat16, torch.bfloat16, 192, 128), (torch.bfloat16, torch.bfloat16, 256, 256),
                                         (torch.bfloat16, E4M3, 128, 128), (E4M3, E4M3, 256, 256)])
@pytest.mark.parametrize("span,counts", [(0, [4, 4, 4]), (130, [1, 4, 4]), (600, [1, 1, 3]), (2300, [1, 1, 1])])
def test_requests_far_below_the_key_bound(device, qt, kt, dq, dv, span, counts):
    """130, 1100 and 2300 keys of a call planned in four splits: a request takes
    as many as leave each `span` keys, and one split writes no partials."""
    q_lens, k_lens = [40, 70, 17], [130, 1100, 2300]
    k, v = _values((sum(k_lens), 2, dq), 2, kt, device), _values((sum(k_lens), 2, dv), 3, kt, device, 0.5)
    q = _values((127, 4, dq), 4, qt, device)
    sinks = seeded((4,), 5, torch.float32, device)
    cu, cu_k = offsets(q_lens, device), offsets(k_lens, device)
    out_type = torch.bfloat16 if qt == E4M3 else qt
    out, lse = torch.empty(127, 4, dv, dtype=out_type, device=device), torch.empty(4, 127, device=device)
    keep = [torch.full((4, 127, 4, dv), 7.0, device=device), torch.full((4, 4, 127), 7.0, device=device)]
    a = kernel_args(q, k, v, out, lse, keep=keep, cu_seqlens_q=cu, cu_seqlens_k=cu_k, max_seqlen_q=70, max_seqlen_k=1 << 16,
                    causal=True, s_aux=sinks)
    a.num_splits, a.split_span = 4, span
    a.partial_out, a.partial_lse = keep[0].data_ptr(), keep[1].data_ptr()
    _lib.call("fa_prefill_fwd", a, device)
    ref, ref_lse = oracle_attention(q.float() if qt == E4M3 else q, k.float(), v.float(), cu, cu_k, causal=True, sinks=sinks)
    assert_parity(out, lse, ref, ref_lse)
    for b, count in enumerate(counts):
        rows = slice(sum(q_lens[:b]), sum(q_lens[:b + 1]))
        written = count if count > 1 else 0
        assert (keep[0][written:, rows] == 7).all() and (keep[1][written:, :, rows] == 7).all()
        assert (keep[1][:written, :, rows] != 7).all()
