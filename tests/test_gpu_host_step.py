"""The native check-and-launch of decode_step (csrc/host_step.cpp): what it passes gives the bits of the
Python checks' own launch, what is wrong with any argument is still refused with its message after a good
call, and new tensors (other addresses, freed and allocated again) are seen on the next call."""

import pytest
import torch

pytestmark = pytest.mark.gpu

BF16 = torch.bfloat16


def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


def _arguments(batch=3, layers=2, seed=5):
    import prime_kernels_amd as pk
    from prime_kernels_amd import workload as WL

    mod = pk.load("decode_megakernel_360m")
    dev = torch.device("cuda:0")
    embed, final_norm, lw = WL.random_weights(mod.MODEL, seed, dev, layers=layers)
    ctx = [100 + 37 * b for b in range(batch)]
    kv = WL.PagedKV(mod.MODEL, batch, 300, layers=layers, device=dev, seed=seed + 1, fill="randn")
    return mod, dict(
        input_ids=torch.arange(3, 3 + batch, device=dev), positions=torch.tensor(ctx, device=dev),
        seq_lens=torch.tensor([c + 1 for c in ctx], dtype=torch.int32, device=dev), block_table=kv.block_table,
        slot_mapping=torch.tensor([kv.slot(b, c) for b, c in enumerate(ctx)], device=dev), embed=embed, layers=lw,
        final_norm=final_norm, kv_caches=kv.caches, cos_sin_cache=WL.rope_table(512, device=dev), eps=1e-5,
        num_layers=layers, logits_out=torch.empty((batch, 49152), dtype=BF16, device=dev),
        layer_outputs=torch.empty((layers, batch, 960), dtype=BF16, device=dev))


class _Other(torch.Tensor):
    """A subclass: the native check leaves it to the Python ones."""


def _clone(kw, hidden):
    return hidden.clone(), kw["logits_out"].clone(), kw["layer_outputs"].clone()


@pytest.mark.parametrize("batch", [1, 2, 3])
def test_both_paths_give_the_same_bits(batch):
    _need_gpu()
    from prime_kernels_amd import _decode

    mod, kw = _arguments(batch)
    mod.decode_step(**kw)                                     # the device's runtime exists from here on
    native = []
    real = _decode._plain_step

    def counted(*a, **k):
        native.append(real(*a, **k))
        return native[-1]

    _decode._plain_step = counted
    try:
        one = _clone(kw, mod.decode_step(**kw))
        slow = dict(kw, positions=kw["positions"].as_subclass(_Other))
        two = _clone(kw, mod.decode_step(**slow))
    finally:
        _decode._plain_step = real
    assert native == [0, None]
    assert all(torch.equal(a, b) for a, b in zip(one, two))
    h, ids = mod.decode_step(return_token_ids=True, **{k: v for k, v in kw.items() if k != "logits_out"})
    assert torch.equal(h, one[0]) and torch.equal(ids, one[1].float().argmax(-1))


def test_without_the_host_module_the_same_bits(monkeypatch):
    """A torch that the host module was not built for: decode_step checks and launches from Python."""
    _need_gpu()
    from prime_kernels_amd import _decode, _native

    mod, kw = _arguments(3)
    mod.decode_step(**kw)
    one = _clone(kw, mod.decode_step(**kw))
    monkeypatch.setattr(_native, "_host", False)
    monkeypatch.setattr(_decode, "_runtimes", {})
    mod.decode_step(**kw)
    two = _clone(kw, mod.decode_step(**kw))
    assert all(torch.equal(a, b) for a, b in zip(one, two))
    with pytest.raises(ValueError, match="positions must have dtype"):
        mod.decode_step(**dict(kw, positions=kw["positions"].int()))


def test_every_wrong_argument_is_refused():
    _need_gpu()
    mod, kw = _arguments()
    mod.decode_step(**kw)
    torch.cuda.synchronize()

    def layer(i, k, t):
        layers = [list(x) for x in kw["layers"]]
        layers[i][k] = t
        return layers

    w = kw["layers"][1][2]
    odd = torch.empty(w.numel() + 8, dtype=BF16, device=w.device)[1:1 + w.numel()].view(w.shape)
    caches = kw["kv_caches"]
    wrong = [
        ("layer 1 o must have dtype", dict(layers=layer(1, 2, w.float()))),
        ("layer 1 o must be a CUDA tensor", dict(layers=layer(1, 2, w.cpu()))),
        ("layer 1 o must be contiguous", dict(layers=layer(1, 2, w.t()))),
        ("layer 1 o must be 16-byte aligned", dict(layers=layer(1, 2, odd))),
        ("layer 0 gate_up must have shape", dict(layers=layer(0, 4, kw["layers"][0][4][:-1]))),
        ("must contain six", dict(layers=[x[:5] for x in kw["layers"]])),
        ("expected 2 layers", dict(kv_caches=caches[:1])),
        ("must share strides", dict(kv_caches=[caches[0], caches[1].transpose(0, 1).contiguous().transpose(0, 1)])),
        ("K/V-packed", dict(kv_caches=[c[..., :64] for c in caches])),
        ("positions must have dtype", dict(positions=kw["positions"].int())),
        ("seq_lens must have shape", dict(seq_lens=kw["seq_lens"][:2])),
        ("1-D int32 or int64", dict(input_ids=kw["input_ids"].float())),
        ("block_table must be int32", dict(block_table=kw["block_table"].long())),
        ("contiguous rows", dict(block_table=kw["block_table"].t().contiguous().t())),
        ("embed must be contiguous", dict(embed=kw["embed"][:-1])),
        ("cos_sin_cache must be contiguous", dict(cos_sin_cache=kw["cos_sin_cache"][:, :32])),
        ("logits_out must have shape", dict(logits_out=kw["logits_out"][:2])),
        ("layer_outputs must have dtype", dict(layer_outputs=kw["layer_outputs"].float())),
        ("rms eps", dict(eps=1e-6)),
        ("num_layers must be", dict(num_layers=33)),
        ("debug_layer_index", dict(debug_layer_index=40)),
        ("prepared for other", dict(encoded_gu=_Encoded(kw["layers"]))),
    ]
    for message, change in wrong:
        with pytest.raises(ValueError, match=message):
            mod.decode_step(**dict(kw, **change))
    torch.cuda.synchronize()


class _Encoded:
    """An encoded cache of other gate_up tensors."""

    def __init__(self, layers):
        self.device = layers[0][4].device
        self.weights = tuple(x[4].clone() for x in layers)
        self.table = torch.zeros(64, dtype=torch.uint8, device=self.device)


def test_new_tensors_are_seen():
    _need_gpu()
    mod, kw = _arguments()
    first = _clone(kw, mod.decode_step(**kw))
    other = dict(kw, layers=[tuple(t.clone() for t in x) for x in kw["layers"]])
    other["layers"][1][4].mul_(2)
    second = _clone(kw, mod.decode_step(**other))
    assert not torch.equal(first[0], second[0])
    again = _clone(kw, mod.decode_step(**kw))
    assert all(torch.equal(a, b) for a, b in zip(first, again))
    kw["layers"][1][4].mul_(2)                                # in place: the same addresses
    assert all(torch.equal(a, b) for a, b in zip(second, _clone(kw, mod.decode_step(**kw))))
