"""Split plans that have to follow the kernel that runs (host arithmetic, no GPU)."""
import pytest
import torch

from flash_attn_mps_amd._attention import f32_splits
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
