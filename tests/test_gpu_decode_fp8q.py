"""Single-query decode with E4M3 queries over E4M3 K/V on the decode kernels
(matrix-core and VALU) against the float64 oracle.

Tolerance: E4M3 products are exact and probabilities are held to fp32
accuracy (as three bf16 terms on the matrix cores), so beside the output's own
rounding (half an ulp: 2^-11 |out| in fp16, 2^-8 in bf16, 2^-25 for fp16
subnormals) only fp32 sums differ: score errors of ~256 * 2^-24 * |score| <=
6e-5, twice that relative on an output of magnitude up to max|v|.
Probabilities rounded to 16 bits would err by 2^-11 max|v| beside it.
"""
import pytest
import torch

from flash_attn_mps_amd import _lib
from harness import attention, kernel_args, offsets, oracle_attention, seeded

pytestmark = pytest.mark.gpu

E4M3 = torch.float8_e4m3fn


def _e4m3(shape, seed, device, scale):
    return (seeded(shape, seed, torch.float32, "cpu") * scale).clamp(-448, 448).to(E4M3).to(device)


def _case(device, lengths, heads, kv_heads, dim, page, pad=0):
    """K/V of [pages, page, kv_heads, dim + pad] storage sliced to dim; unread storage NaN."""
    cols = max(1, -(-max(lengths) // page))
    n = len(lengths) * cols
    table = torch.randperm(n, generator=torch.Generator().manual_seed(3)).reshape(len(lengths), cols).int()
    caches = []
    for seed in (1, 2):
        c = torch.full((n, page, kv_heads, dim + pad), 0x7F, dtype=torch.uint8)
        for b, length in enumerate(lengths):
            pos = torch.arange(length)
            c[table[b, pos // page].long(), pos % page, :, :dim] = _e4m3(
                (length, kv_heads, dim), 100 * seed + b, "cpu", 20.0).view(torch.uint8)
        caches.append(c.to(device).view(E4M3)[..., :dim])
    q = _e4m3((len(lengths), heads, dim), 7, device, 20.0)
    descales = {name: (0.04 + 0.02 * seeded((len(lengths), kv_heads), 20 + i, torch.float32, "cpu").abs()).to(device)
                for i, name in enumerate(("q_descale", "k_descale", "v_descale"))}
    return q, caches, table, descales


def _check(got, lse, ref, ref_lse, vmax):
    half = 2.0 ** -11 if got.dtype == torch.float16 else 2.0 ** -8
    err = (got.cpu().double() - ref).abs() - half * ref.abs()
    assert err.max() <= 1.2e-4 * vmax + 2.0 ** -25
    seen = ~torch.isneginf(ref_lse)
    assert torch.equal(torch.isneginf(lse.cpu()), ~seen)
    assert (lse.cpu().double() - ref_lse)[seen].abs().max() <= 1e-4


@pytest.mark.parametrize("dim", [32, 64, 80, 128, 256])
@pytest.mark.parametrize("heads,kv_heads,pad", [(2, 2, 0), (8, 4, 0), (16, 4, 0), (40, 8, 0), (16, 4, 16), (64, 2, 0)])
@pytest.mark.parametrize("out_dtype", [torch.float16, torch.bfloat16])
def test_groups_dims_and_splits(device, dim, heads, kv_heads, pad, out_dtype):
    lengths = [0, 1, 31, 33, 130, 1025]
    q, (k, v), table, desc = _case(device, lengths, heads, kv_heads, dim, 16, pad)
    used = torch.tensor(lengths, dtype=torch.int32, device=device)
    cu = offsets([1] * len(lengths), device)
    out = torch.empty(len(lengths), heads, dim, dtype=out_dtype, device=device)
    kw = dict(cu_seqlens_q=cu, seqused_k=used, max_seqlen_q=1, max_seqlen_k=1025, block_table=table.to(device),
              causal=True, **desc)
    lse = torch.empty(heads, len(lengths), device=device)
    assert _lib.supported("fa_decode_supported", kernel_args(q, k, v, out, lse, keep=[], **kw))
    ref, ref_lse = oracle_attention(q, k.contiguous().float().nan_to_num(0), v.contiguous().float().nan_to_num(0), cu,
                                    used_k=used, block_table=table, causal=True, **desc)
    vmax = float((v.contiguous().float().nan_to_num(0).abs().amax() * desc["v_descale"].max()))
    for splits in (0, 1, 3):
        got, lse = attention(q, k, v, out=out, num_splits=splits, **kw)
        _check(got, lse, ref, ref_lse, vmax)


@pytest.mark.parametrize("heads,kv_heads,dim", [(16, 2, 128), (4, 4, 256), (16, 4, 64)])
@pytest.mark.parametrize("feature", ["softcap", "window", "sinks", "chunk"])
def test_features(device, heads, kv_heads, dim, feature):
    """Softcap, a left window, sinks; and single-query requests beside a
    40-row one (the mixed-batch route)."""
    lengths = [700, 1, 257, 90]
    q, (k, v), table, desc = _case(device, lengths, heads, kv_heads, dim, 32)
    q_lens = [1] * 4
    kw = {}
    if feature == "softcap":
        kw["softcap"] = 5.0
    elif feature == "window":
        kw["window_size"] = (99, 0)
    elif feature == "sinks":
        kw["s_aux"] = seeded((heads,), 9, torch.float32, device)
    else:
        q_lens = [1, 1, 1, 40]
        q = _e4m3((43, heads, dim), 8, device, 20.0)
    cu = offsets(q_lens, device)
    used = torch.tensor(lengths, dtype=torch.int32, device=device)
    got, lse = attention(q, k, v, cu_seqlens_q=cu, seqused_k=used, max_seqlen_q=max(q_lens), max_seqlen_k=700,
                         block_table=table.to(device), causal=True, **kw, **desc)
    names = dict(s_aux="sinks", window_size="window")
    ref, ref_lse = oracle_attention(q, k.float().nan_to_num(0), v.float().nan_to_num(0), cu, used_k=used,
                                    block_table=table, causal=True, **{names.get(n, n): x for n, x in kw.items()}, **desc)
    vmax = float(v.float().nan_to_num(0).abs().amax() * desc["v_descale"].max())
    _check(got[:3], lse[:, :3], ref[:3], ref_lse[:, :3], vmax)
    if feature == "chunk":
        # The 40 rows run on the prefill kernel, with probabilities rounded to
        # fp16: 2^-11 of the largest value, and the output's own rounding.
        err = (got[3:].cpu().double() - ref[3:]).abs()
        assert err.max() <= 2.0 ** -10 * vmax
        assert (lse[:, 3:].cpu().double() - ref_lse[:, 3:]).abs().max() <= 1e-4


@pytest.mark.parametrize("heads,kv_heads,dim", [(16, 2, 128), (12, 3, 128), (16, 4, 64), (4, 4, 128), (4, 4, 256)])
def test_small_probabilities_keep_their_weight(device, heads, kv_heads, dim):
    """Four keys (one of each wave's first stage) score ~18.4 above 8000
    others, whose probabilities of 2^-26.5 alone make the output: 1.4e-3 with
    |V| = 64.  Probabilities held as 16-bit fractions of the largest drop them.

    Tolerance: an output of 2^-10 is rounded to fp16 within 2^-21, and the fp32
    sums err by less than 2^-11 of it."""
    n = 8000
    k, v = torch.zeros(n, kv_heads, dim), torch.full((n, kv_heads, dim), 64.0)
    peaks = [0, 32, 64, 96]
    k[peaks] = 1.625 * (128 / dim) ** 0.5 if dim != 256 else 1.125   # both E4M3 values at 64 (2.25) and 256
    if dim == 64:
        k[peaks] = 2.25
    v[peaks] = 0.0
    q = torch.ones(1, heads, dim)
    q, k, v = (t.to(E4M3).to(device) for t in (q, k, v))
    cu, cu_k = offsets([1], device), offsets([n], device)
    got, lse = attention(q, k, v, cu_seqlens_q=cu, cu_seqlens_k=cu_k, max_seqlen_q=1, max_seqlen_k=n, num_splits=1)
    ref, ref_lse = oracle_attention(q, k.float(), v.float(), cu, cu_k)
    assert 2.0 ** -11 < ref.max() < 2.0 ** -8
    assert ((got.cpu().double() - ref).abs() <= 2.0 ** -21 + 2.0 ** -10 * ref).all()
    assert (lse.cpu().double() - ref_lse).abs().max() <= 1e-5


@pytest.mark.parametrize("heads,kv_heads,dim", [(16, 2, 128), (12, 3, 128), (16, 4, 64), (4, 4, 128), (4, 4, 256)])
def test_small_scores_under_a_large_softcap(device, heads, kv_heads, dim):
    """Scores of ~N(0, 1) under a cap of 4000: tanhf keeps their relative
    accuracy (2^-22 of |score| <= 6 beside the dot's own ~16 * 2^-24), a
    difference of nearly equal numbers only 2^-24 of the cap."""
    n = 300
    q, k, v = (_e4m3(shape, 50 + i, device, 1.0) for i, shape in
               enumerate([(1, heads, dim), (n, kv_heads, dim), (n, kv_heads, dim)]))
    cu, cu_k = offsets([1], device), offsets([n], device)
    _, lse = attention(q, k, v, cu_seqlens_q=cu, cu_seqlens_k=cu_k, max_seqlen_q=1, max_seqlen_k=n, softcap=4000.0)
    _, ref_lse = oracle_attention(q, k.float(), v.float(), cu, cu_k, softcap=4000.0)
    assert (lse.cpu().double() - ref_lse).abs().max() <= 6e-6
