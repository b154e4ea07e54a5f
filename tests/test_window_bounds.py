"""Window bounds as large as an int32 holds (and larger) bound nothing, in the
argument struct and in every kernel that adds them to positions."""
import sys

import pytest
import torch

from flash_attn_mps_amd import _lib, vllm
from harness import attention, kernel_args, offsets, seeded

FAR = 2 ** 31 - 1


@pytest.mark.parametrize("bound,packed", [(-1, -1), (0, 0), (7, 7), (2 ** 30 - 1, 2 ** 30 - 1), (2 ** 30, -1), (FAR, -1),
                                          (2 ** 32 + 5, -1), (sys.maxsize, -1)])
def test_packed_bounds(bound, packed):
    q, cu = torch.zeros(4, 2, 64), torch.tensor([0, 4], dtype=torch.int32)
    kw = dict(cu_seqlens_q=cu, cu_seqlens_k=cu, max_seqlen_q=4, max_seqlen_k=4)
    a = kernel_args(q, q, q, q, torch.zeros(2, 4), keep=[], window_size=(bound, bound), **kw)
    assert (a.window_left, a.window_right) == (packed, packed)
    if bound > 0:
        mask = dict(mask_mod=vllm.mm_prefix_mask(bound), aux_tensors=[torch.zeros(4, 2, dtype=torch.int32), cu])
        assert kernel_args(q, q, q, q, torch.zeros(2, 4), keep=[], **mask, **kw).mask_window == packed


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,dim", [(torch.float32, 64), (torch.float32, 40), (torch.bfloat16, 256), (torch.bfloat16, 128),
                                       (torch.float16, 40)])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("entry", ["python", "c"])
def test_far_bounds_equal_unbounded(device, dtype, dim, causal, entry):
    """fp32 matrix-core and generic kernels, wave pairs, the 128-dim tile; one
    request has fewer keys than rows (positions below zero).  As packed by the
    host, and set in the struct after it."""
    q_lens, k_lens = [40, 5, 70], [40, 200, 30]
    q, k, v = (seeded((sum(n), h, dim), 30 + h, dtype, device) for n, h in ((q_lens, 4), (k_lens, 2), (k_lens, 2)))
    kw = dict(cu_seqlens_q=offsets(q_lens, device), cu_seqlens_k=offsets(k_lens, device), max_seqlen_q=70,
              max_seqlen_k=200, causal=causal, num_splits=1)
    want, want_lse = attention(q, k, v, **kw)
    for window in ((FAR, FAR), (-1, FAR), (FAR, -1)):
        if entry == "python":
            got, lse = attention(q, k, v, window_size=window, **kw)
        else:
            got, lse = torch.empty_like(want), torch.empty_like(want_lse)
            a = kernel_args(q, k, v, got, lse, keep=[], **kw)
            a.window_left, a.window_right = window
            prefill = _lib.supported("fa_prefill_supported", a)
            _lib.call("fa_prefill_fwd" if prefill else "fa_attn_fwd", a, device)
        assert torch.equal(got, want) and torch.equal(lse, want_lse), window


@pytest.mark.gpu
def test_far_bounds_in_decode(device):
    q, cache = seeded((3, 1, 8, 128), 40, torch.bfloat16, device), seeded((3, 64, 2, 128), 41, torch.bfloat16, device)
    import flash_attn_mps_amd as fa
    lens = torch.tensor([0, 64, 17], dtype=torch.int32, device=device)
    want = fa.flash_attn_with_kvcache(q, cache, cache, cache_seqlens=lens)
    assert torch.equal(fa.flash_attn_with_kvcache(q, cache, cache, cache_seqlens=lens, window_size=(FAR, FAR)), want)
