"""The one-launch generation step reads its per-request vectors by index, so
the host takes it only for vectors of one entry per request (checked here
without a GPU: the launch is recorded, not made)."""
import pytest
import torch

from flash_attn_mps_amd import _cache, _lib


@pytest.mark.parametrize("leftpad,launch", [([1], "fa_append_kvcache"), ([1, 2], "fa_rotary_append"),
                                            (None, "fa_rotary_append")])
def test_leftpad_of_one_value_is_not_indexed(monkeypatch, leftpad, launch):
    calls = []
    monkeypatch.setattr(_cache, "_require_gpu", lambda **tensors: None)
    monkeypatch.setattr(_lib, "call", lambda name, args, device: calls.append(name))
    q, k, cache = torch.zeros(2, 1, 4, 8), torch.zeros(2, 1, 2, 8), torch.zeros(2, 16, 2, 8)
    lengths = torch.tensor([3, 5], dtype=torch.int32)
    pad = None if leftpad is None else torch.tensor(leftpad, dtype=torch.int32)
    _, after = _cache.rotary_append(q, k, k, cache, cache, lengths, None, None, cache_leftpad=pad)
    assert calls == [launch] and after.shape == lengths.shape
    if launch == "fa_append_kvcache":   # one value for every request
        assert after.tolist() == [3, 5]


def test_leftpad_of_another_count_is_refused(monkeypatch):
    monkeypatch.setattr(_cache, "_require_gpu", lambda **tensors: None)
    monkeypatch.setattr(_lib, "call", lambda name, args, device: pytest.fail(f"{name} launched"))
    q, k, cache = torch.zeros(2, 1, 4, 8), torch.zeros(2, 1, 2, 8), torch.zeros(2, 16, 2, 8)
    with pytest.raises(ValueError, match="cache_leftpad"):
        _cache.rotary_append(q, k, k, cache, cache, torch.tensor([3, 5], dtype=torch.int32), None, None,
                             cache_leftpad=torch.tensor([1, 2, 3], dtype=torch.int32))


@pytest.mark.parametrize("v_shape,ok", [((2, 16), True), ((3, 32), True), ((1, 16), False), ((2, 8), False)])
def test_append_bounds_cover_both_caches(monkeypatch, v_shape, ok):
    """The kernel bounds both writes by the K cache's rows and capacity."""
    calls = []
    monkeypatch.setattr(_cache, "_require_gpu", lambda **tensors: None)
    monkeypatch.setattr(_lib, "call", lambda name, args, device: calls.append(name))
    k, k_cache, v_cache = torch.zeros(2, 1, 2, 8), torch.zeros(2, 16, 2, 8), torch.zeros(*v_shape, 2, 8)
    lengths = torch.tensor([3, 5], dtype=torch.int32)
    if ok:
        _cache.append_kvcache(k, k, k_cache, v_cache, lengths)
    else:
        with pytest.raises(ValueError, match="V cache"):
            _cache.append_kvcache(k, k, k_cache, v_cache, lengths)
    assert calls == ["fa_append_kvcache"] * ok
