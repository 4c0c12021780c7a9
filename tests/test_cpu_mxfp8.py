"""quantize_layers' use of memory, without a GPU: the quantiser is a stand-in that counts."""

import gc
import weakref

import torch

from prime_kernels_amd import mxfp8


def test_layers_of_an_iterator_are_taken_one_at_a_time(monkeypatch):
    """A program that loads a checkpoint layer by layer: when it makes a layer, at most the one before
    it is still held."""
    taken = []

    def matrices(ms):
        ms = list(ms)
        taken.append(len(ms))
        return [(torch.empty(1), torch.empty(1)) for _ in ms]

    monkeypatch.setattr(mxfp8, "_quantize_all", matrices)
    alive, most = weakref.WeakSet(), 0

    def load():
        nonlocal most
        for _ in range(12):
            gc.collect()
            most = max(most, len(alive))
            ws = [torch.empty(8) for _ in range(6)]
            alive.add(ws[1])
            yield tuple(ws)
            del ws

    out = mxfp8.quantize_layers(load())
    assert len(out) == 12 and all(len(x) == 10 for x in out)
    assert taken == [4] * 12 and most <= 1


def test_layers_of_a_list_go_32_at_a_time(monkeypatch):
    """One call a model, and a bound on the copies that strided matrices need."""
    taken = []

    def matrices(ms):
        ms = list(ms)
        taken.append(len(ms))
        return [(w, w) for w in ms]

    monkeypatch.setattr(mxfp8, "_quantize_all", matrices)
    layers = [tuple(torch.full((1,), 10.0 * i + k) for k in range(6)) for i in range(67)]
    for given in (layers, tuple(layers), [list(x) for x in layers]):
        taken.clear()
        out = mxfp8.quantize_layers(given)
        assert taken == [128, 128, 12] and len(out) == 67
        for x, (n1, q, _, o, _, n2, g, _, d, _) in zip(layers, out):
            assert all(a is b for a, b in zip((n1, q, o, n2, g, d), x))
    assert mxfp8.quantize_layers([]) == []
