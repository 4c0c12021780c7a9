"""The batched step of three or more sequences (135M: on cells of XCDs, decode_cell.hip): context lengths at the
edges of its tiles, quads, chunks and shares, every number of sequences a cell can hold, and caches laid
out otherwise.  Bars as in test_gpu_batched.py (or twice the eager-GPU floor of the
same sequence)."""

import pytest
import torch

from oracle import smollm2 as O
from tests import gpu_cases as GC

pytestmark = pytest.mark.gpu

CONTEXTS = {
    "b3_an_empty_cell": [1, 17, 64],                            # 135M: four cells, three sequences
    "b5_tile_and_quad_edges": [16, 33, 65, 66, 129],
    "b7_one_long": [3000, 1, 2, 1, 15, 18, 2],                  # short pairs padded to a share of a workgroup's range
    "b9_uneven_cells": [5, 300, 41, 1025, 257, 256, 258, 1, 700],
    "b16_equal": [513] * 16,
    "b16_ragged": [1, 4097, 64, 2048, 65, 3, 1024, 129, 2, 500, 31, 32, 33, 800, 1, 16],
}


def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


@pytest.mark.parametrize("base", [O.SMOLLM2_360M, O.SMOLLM2_135M], ids=["360m", "135m"])
@pytest.mark.parametrize("name", list(CONTEXTS))
def test_contexts_against_oracle(name, base):
    _need_gpu()
    contexts = CONTEXTS[name]
    case = GC.random_kv_case(O.with_layers(base, 2), 400 + len(contexts), contexts)
    ids = [31 + 11 * b for b in range(len(contexts))]
    pos = [S - 1 for S in contexts]
    k = case.kernel_step(ids, pos, layer_outputs=True)
    f = case.eager_gpu_step(ids, pos)
    r = case.oracle_step(ids, pos, layer_outputs=True)
    GC.assert_within_floor(k, r, f, name)
    for li in range(2):
        for b, S in enumerate(contexts):
            slot = case.kv.slot(b, S - 1)
            got = case.kvd[li][slot // 16, :, slot % 16].cpu().float()
            want = case.kv.caches[li][slot // 16, :, slot % 16].float()
            assert torch.allclose(got, want, rtol=2 ** -6, atol=2e-2), (li, b)


def test_other_cache_strides_give_the_same_bits():
    """Caches whose blocks hold the tokens before the KV heads, with a gap after every block, give every
    output and appended bit of the packed layout."""
    _need_gpu()
    contexts = [300, 41, 129, 700]
    case = GC.random_kv_case(O.with_layers(O.SMOLLM2_360M, 2), 431, contexts)
    ids, pos = [1, 2, 3, 4], [S - 1 for S in contexts]
    packed = [c.clone() for c in case.kvd]
    k1 = case.kernel_step(ids, pos)
    after = [c.clone() for c in case.kvd]
    other = []
    for c in packed:
        n, h, t, d = c.shape
        store = torch.full((n, t * h * d + 64), 7.0, dtype=c.dtype, device=c.device)
        view = store[:, :t * h * d].view(n, t, h, d).permute(0, 2, 1, 3)
        view.copy_(c)
        other.append(view)
    case.kvd = other
    k2 = case.kernel_step(ids, pos)
    for key in ("hidden", "logits", "ids"):
        assert torch.equal(k1[key], k2[key]), key
    for a, b in zip(after, case.kvd):
        assert torch.equal(a, b)


@pytest.mark.parametrize("base", [O.SMOLLM2_360M, O.SMOLLM2_135M], ids=["360m", "135m"])
@pytest.mark.parametrize("capacity", [6816, 6832], ids=["whole_workgroups", "end_to_end"])
def test_both_splits_of_the_pairs_against_oracle(capacity, base):
    """The same nine sequences at the last block table capacity of the one split and the first of the other
    (9 * 6,816 <= 61,440 < 9 * 6,832): chunks of one tile, of a quad and one token more, pairs without a
    cached token."""
    _need_gpu()
    contexts = [5, 300, 41, 1025, 257, 1, 258, 17, 2100]
    case = GC.random_kv_case(O.with_layers(base, 2), 441, contexts, capacity=capacity)
    ids, pos = [7 + 5 * b for b in range(9)], [S - 1 for S in contexts]
    got, want = case.kernel_step(ids, pos), case.oracle_step(ids, pos)
    # Two layers of either end at most 1.0 % (relative norm of the logits) from the step in 64 bits, so two
    # right results at most 2.0 % from each other
    for b in range(9):
        d, r = got["logits"][b].float().cpu(), want["logits"][b].float().cpu()
        assert (d - r).norm() <= 0.02 * r.norm(), (capacity, b, ((d - r).norm() / r.norm()).item())
    for li in range(2):
        for b, S in enumerate(contexts):
            slot = case.kv.slot(b, S - 1)
            new = case.kvd[li][slot // 16, :, slot % 16].cpu().float()
            assert torch.allclose(new, case.kv.caches[li][slot // 16, :, slot % 16].float(), rtol=2 ** -6, atol=2e-2), (li, b)
