"""Resident index tensors of the dense entry points: views of one vector that
is never freed, whatever shapes come and go, and nothing kept from a capture.
(The GPU side, a captured graph that outlives them, is in test_gpu_graph.py.)"""
import threading

import pytest
import torch

from flash_attn_mps_amd.interface import _Counting

CPU = torch.device("cpu")


@pytest.mark.parametrize("batch,length", [(0, 5), (1, 0), (3, 0), (1, 1), (1, 7), (4, 9), (10, 10), (9, 11), (1, 99), (1, 100), (50, 3)])
def test_offsets_and_rows(batch, length):
    """Inside and past a vector of 100 entries."""
    c = _Counting(entries=100, views=4)
    offsets, rows = c.offsets(batch, length, CPU), c.rows(batch, CPU)
    assert offsets.dtype == rows.dtype == torch.int32
    assert offsets.tolist() == [length * i for i in range(batch + 1)]
    assert rows.tolist() == [[i] for i in range(batch)] and rows.shape == (batch, 1)


def test_a_shape_stays_readable_after_many_others():
    """What a captured graph has read stays where it is: every tensor lies in
    one storage, which the views' eviction does not free."""
    c = _Counting(views=4)
    storage = c.offsets(8, 16, CPU).untyped_storage().data_ptr()
    for n in range(1, 200):
        assert c.offsets(n, 3, CPU).untyped_storage().data_ptr() == storage
        assert c.rows(n, CPU).untyped_storage().data_ptr() == storage
    assert len(c._views) == 4 and len(c._vectors) == 1


def test_a_capture_keeps_nothing_and_reuses_the_vector(monkeypatch):
    c = _Counting(entries=100)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)

    class Device:   # a GPU by name, whose tensors live on the CPU here
        type, index = "cuda", 0
    monkeypatch.setattr(torch, "arange", lambda n, dtype, device=None, arange=torch.arange: arange(n, dtype=dtype))
    assert c.offsets(2, 3, Device).tolist() == [0, 3, 6] and not c._vectors and not c._views
    c._vectors["cuda", 0] = torch.arange(100, dtype=torch.int32)
    assert c.offsets(2, 3, Device).untyped_storage().data_ptr() == c._vectors["cuda", 0].untyped_storage().data_ptr()


def test_threads_share_one_vector():
    c, seen = _Counting(views=2), []

    def work(seed):
        for i in range(300):
            b, n = 1 + (seed * 31 + i * 7) % 13, (seed + i) % 9
            seen.append(c.offsets(b, n, CPU).tolist() == [n * j for j in range(b + 1)])
    threads = [threading.Thread(target=work, args=(s,)) for s in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(seen) == 2400 and all(seen) and len(c._vectors) == 1


@pytest.mark.parametrize("context", ["fake", "default device"])
def test_a_mode_around_the_first_call_leaves_nothing_behind(context):
    """Under a tracer's stand-in tensors nothing is kept (they would be every
    later call's offsets), and torch's default device does not place the vector."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    c = _Counting(entries=100)
    with FakeTensorMode() if context == "fake" else torch.device("meta"):
        first = c.offsets(2, 3, CPU)
    assert (type(first) is torch.Tensor) == (context != "fake") and first.shape == (3,)
    assert c.offsets(2, 3, CPU).tolist() == [0, 3, 6]
