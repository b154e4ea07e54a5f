"""Split plans that have to follow the kernel that runs (host arithmetic, no GPU)."""
import pytest
import torch

from flash_attn_mps_amd._attention import f32_splits, prefill_split_span, prefill_splits
from harness import offsets, problem


def _decode(view=lambda t: t, batch=64, keys=2048, dim=128):
    """64 requests of one row: one split fills the matrix-core kernel's grid."""
    q, k, v = torch.empty(batch, 16, dim), torch.empty(batch, 32, 8, dim), torch.empty(batch, 32, 8, dim)
    return q, view(k), v, dict(cu_seqlens_q=offsets([1] * batch), seqused_k=torch.full((batch,), keys, dtype=torch.int32),
                               max_seqlen_q=1, max_seqlen_k=keys, block_table=torch.zeros(batch, 64, dtype=torch.int32))


@pytest.mark.parametrize("view,splits", [
    (lambda t: t, 1),
    (lambda t: torch.empty(*t.shape[:-1], 132)[..., :128], 1),
    (lambda t: torch.empty(*t.shape[:-1], 130)[..., :128], None),            # head stride of 130
    (lambda t: torch.empty(*t.shape[:-1], 132)[..., 1:129], None),           # rows start 4 bytes into a piece
    (lambda t: torch.empty(*t.shape[:-1], 256)[..., ::2], None),             # strided dims
])
def test_fp32_plan_is_for_the_rows_its_kernel_takes(view, splits):
    """Other fp32 rows run the generic kernel, whose single-row calls need
    more splits (None: its own rule of one per 256 keys)."""
    q, k, v, kw = _decode(view)
    assert f32_splits(problem(q, k, v, **kw)) == splits
    assert f32_splits(problem(q, v, k, **kw)) == splits


@pytest.mark.parametrize("rows,heads,dim", [(17, 8, 64), (64, 32, 128), (512, 32, 128), (512, 16, 256), (100, 12, 192)])
@pytest.mark.parametrize("batch", [1, 3])
def test_key_splits_follow_the_keys_there_are(rows, heads, dim, batch):
    """max_seqlen_k may be a cache's capacity: requests that have those keys take
    every split, and the more keys the plan is for, the fewer splits a request of
    600 keys takes (512 rows: one, as before the kernel split keys)."""
    taken = []
    for keys in (1024, 2048, 8192, 32768, 1 << 20):
        k = torch.empty(1, 1 << 20, 1, 1).expand(1, 1 << 20, heads // 2, dim)
        p = problem(torch.empty(batch * rows, heads, dim), k, k[..., :128] if dim == 192 else k,
                    cu_seqlens_q=offsets([rows] * batch), seqused_k=torch.full((batch,), keys, dtype=torch.int32),
                    max_seqlen_q=rows, max_seqlen_k=keys, block_table=torch.zeros(batch, 1, dtype=torch.int32), causal=True)
        splits = prefill_splits(p)
        if splits > 1:
            span = prefill_split_span(p, splits)
            assert span >= 1 and keys // span >= splits
            taken.append(max(1, min(600 // span, splits)))
    assert (taken or batch == 3) and (rows < 512 or not taken or taken[-1] == 1)
