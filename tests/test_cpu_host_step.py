"""The host module of the step's checks (csrc/host_step.cpp) without a GPU: it answers None for whatever it
does not find right, so that decode_step's own checks word the error."""

import pytest
import torch

from prime_kernels_amd import _decode, _native

MODEL = _decode.SMOLLM2_360M


def _call(n_layers):
    """step on CPU tensors, which it never finds right."""
    host = _native.host()
    spec = host.make_spec(MODEL.model_id, MODEL.hidden, MODEL.kv_heads, MODEL.head_dim, MODEL.max_batch, MODEL.max_seq,
                          MODEL.layers, _decode.VOCAB, _decode.BLOCK_SIZE,
                          [(dtype == torch.bfloat16, shape) for _, dtype, shape in MODEL.layer_spec()])
    return host.step(1, 0, spec, n_layers, *[torch.zeros(1)] * 12, False, *[0] * 4, *[None] * 5)


def test_layer_counts_of_any_size_are_left_to_the_python_checks():
    for n in (0, -1, 32, 2 ** 31, 2 ** 63, 2 ** 70, -2 ** 70):
        assert _call(n) is None, n


def test_another_torch_gets_no_host_module(monkeypatch):
    """The module is built against one torch's C++ interfaces: under another version there is none, with a
    warning and no error, and the build for this version is found by its own name."""
    assert _native.host_path(torch.__version__).is_file() and _native.host() is not None
    monkeypatch.setattr(_native, "_host", None)
    monkeypatch.setattr(torch, "__version__", "0.0.1")
    with pytest.warns(RuntimeWarning, match="checks its arguments in Python"):
        assert _native.host() is None
    assert _native.host() is None
