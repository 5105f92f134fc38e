"""The bound on the buffers that posteriors hold for their adjoints: counted per device
while something holds them, given back afterwards, from any thread."""
import threading

import pytest
import torch

from botorch_amd import gp as G


class _Hold(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, keep):
        ctx.save_for_backward(keep)
        return x * 2

    @staticmethod
    def backward(ctx, g):
        return g * 2 + 0 * len(ctx.saved_tensors), None


@pytest.fixture
def kept(monkeypatch):
    monkeypatch.setattr(G, "KEEP_BYTES", 4096)
    return G._KeptBuffers()


def test_buffers_count_until_the_graph_lets_go(kept):
    cpu = torch.device("cpu")
    assert kept.take(0, cpu) is None and kept.take(4097, cpu) is None
    x = torch.ones(3, requires_grad=True)
    ys = [_Hold.apply(x, kept.take(1024, cpu)) for _ in range(4)]
    assert kept.take(256, cpu) is None
    assert kept.take(1024, torch.device("meta")) is not None  # another device's own count
    ys[0].sum().backward(retain_graph=True)
    assert kept.take(256, cpu) is None
    ys[0].sum().backward()
    a = kept.take(1024, cpu)
    assert a is not None and kept.take(256, cpu) is None
    ys.pop()  # a graph that never runs its backward
    b = kept.take(1024, cpu)
    assert b is not None and kept.take(256, cpu) is None
    del a, b, ys
    assert kept.take(4096, cpu) is not None


def test_a_hook_that_moves_the_buffer_gives_it_back(kept):
    cpu = torch.device("cpu")
    x = torch.ones(3, requires_grad=True)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.clone(), lambda t: t):
        y = _Hold.apply(x, kept.take(4096, cpu))
    assert kept.take(4096, cpu) is not None
    y.sum().backward()


def test_a_failed_allocation_is_not_counted(kept, monkeypatch):
    def fail(*args):
        raise MemoryError
    with monkeypatch.context() as mp:
        mp.setattr(G._lib, "workspace", fail)
        with pytest.raises(MemoryError):
            kept.take(4096, torch.device("cpu"))
    assert kept.take(4096, torch.device("cpu")) is not None


def test_threads_share_one_count(kept):
    cpu, over = torch.device("cpu"), []
    alive = []

    def work():
        for _ in range(300):
            t = kept.take(1024, cpu)
            if t is not None:
                alive.append(1)
                if len(alive) > 4:
                    over.append(1)
                alive.pop()
            del t
    threads = [threading.Thread(target=work) for _ in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not over
    assert kept.take(4096, cpu) is not None
