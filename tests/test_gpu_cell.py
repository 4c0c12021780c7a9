"""The batched step of three or more sequences (135M: on cells of XCDs, decode_cell.hip, with either split of its
attention; 360M: decode_kernel_b): context lengths at the edges of its tiles, quads, chunks and shares, every
number of sequences a cell can hold, caches laid out otherwise, and 135M at full depth.  Bars as in
test_gpu_batched.py (or twice the eager-GPU floor of the same sequence).  135M's failure
handling, exchange tags, arrival skew, launches and graph replays are in test_gpu_safety.py and test_gpu_graph.py."""

import numpy as np
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


# 135M with 8 sequences: the last kind of capacity for whole workgroups, and one for the end-to-end split
SPLITS = {"whole_workgroups": None, "end_to_end": 7696}


@pytest.mark.parametrize("kernel", ["360m", *SPLITS])
def test_other_cache_strides_give_the_same_bits(kernel):
    """Caches whose blocks hold the tokens before the KV heads, with a gap after every block, give every
    output and appended bit of the packed layout (360m: decode_kernel_b; 135M's two splits)."""
    _need_gpu()
    contexts = [300, 41, 129, 700] if kernel == "360m" else [300, 41, 129, 700, 1, 1500, 17, 64]
    case = GC.random_kv_case(O.with_layers(O.SMOLLM2_360M if kernel == "360m" else O.SMOLLM2_135M, 2), 431, contexts,
                             capacity=SPLITS.get(kernel))
    ids, pos = [1 + b for b in range(len(contexts))], [S - 1 for S in contexts]
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


@pytest.mark.parametrize("split", list(SPLITS))
def test_append_to_caches_of_any_alignment(split):
    """The first token of eight sequences, appended to caches that start 2 bytes past a 16-byte boundary (nothing
    is cached yet, so nothing is read from them): the rows and outputs of aligned caches, and no other byte
    changed."""
    _need_gpu()
    case = GC.random_kv_case(O.with_layers(O.SMOLLM2_135M, 2), 433, [1] * 8, capacity=SPLITS[split])
    ids, pos = [3 + 5 * b for b in range(8)], [0] * 8
    before = [c.clone() for c in case.kvd]
    k1 = case.kernel_step(ids, pos)
    after = [c.clone() for c in case.kvd]
    assert not any(torch.equal(a, b) for a, b in zip(after, before))
    shifted = []
    for c in before:
        store = torch.full((c.numel() + 8,), 7.0, dtype=c.dtype, device=c.device)
        view = store[1:1 + c.numel()].view(c.shape)
        assert view.data_ptr() % 16 == 2
        view.copy_(c)
        shifted.append((store, view))
    case.kvd = [v for _, v in shifted]
    k2 = case.kernel_step(ids, pos)
    for key in ("hidden", "logits", "ids"):
        assert torch.equal(k1[key], k2[key]), key
    for a, (store, view) in zip(after, shifted):
        assert torch.equal(a, view) and store[0] == 7.0 and (store[1 + a.numel():] == 7.0).all()


@pytest.mark.parametrize("split", list(SPLITS))
def test_same_bits_every_time_without_an_append_and_with_other_input_types(split):
    """slot_mapping < 0 skips that sequence's K/V write and leaves its result unchanged; a repeated step, and
    one with int32 ids and an fp32 cos/sin table, give the identical result."""
    _need_gpu()
    contexts = [300, 41, 129, 1200, 1, 513, 17, 64]
    case = GC.random_kv_case(O.with_layers(O.SMOLLM2_135M, 3), 435, contexts, capacity=SPLITS[split])
    ids, pos = [11 + b for b in range(8)], [S - 1 for S in contexts]
    slots = [case.kv.slot(b, p) for b, p in enumerate(pos)]
    before = [c.clone() for c in case.kvd]
    k1 = case.kernel_step(ids, pos, slot_mapping=[-1 if b in (1, 4) else s for b, s in enumerate(slots)])
    for li, (a, c) in enumerate(zip(before, case.kvd)):
        for b, s in enumerate(slots):
            assert torch.equal(a[s // 16, :, s % 16], c[s // 16, :, s % 16]) == (b in (1, 4)), (li, b)
    for kw in ({}, {}, dict(ids_dtype=torch.int32, cs_fp32=True)):
        case.sync_kv_from_oracle()
        k = case.kernel_step(ids, pos, **kw)
        assert all(torch.equal(k[key], k1[key]) for key in ("hidden", "logits", "ids")), kw


@pytest.mark.parametrize("contexts", [[12288, 3, 700], [12288] + [3 + 40 * b for b in range(7)]],
                         ids=["b3_whole_workgroups", "b8_end_to_end"])
def test_longest_context_against_oracle(contexts):
    """One sequence at the longest context, 12,288 tokens: alone in its cell, and on the line of a cell's pairs."""
    _need_gpu()
    case = GC.random_kv_case(O.with_layers(O.SMOLLM2_135M, 2), 437, contexts, capacity=12288)
    ids, pos = [5 + b for b in range(len(contexts))], [S - 1 for S in contexts]
    k = case.kernel_step(ids, pos, layer_outputs=True)
    f = case.eager_gpu_step(ids, pos)
    r = case.oracle_step(ids, pos, layer_outputs=True)
    GC.assert_within_floor(k, r, f, "longest context")


@pytest.mark.parametrize("capacity", [None, 4096], ids=["whole_workgroups", "end_to_end"])
def test_full_135m_sixteen_sequences(capacity):
    """All 30 layers, 16 sequences with contexts drawn from 1..2000: the step as near to the oracle as the eager GPU
    step is; then every layer fed the oracle's inputs for all sequences at once, within the north-star bound of
    the oracle's output and mostly bit-identical.

    Which sequences a flipped rounding hits is chance at this depth: over six such batches 0 to 3 of 16 are more than
    twice as far from the oracle as the eager step is (of decode_kernel_b's 1 to 5, of the eager step's 0 to 4 more
    than twice as far as the kernel's).  The mean over the sequences is 0.83 to 1.20 times the eager step's in the
    largest difference and 0.70 to 1.28 times in 1 - cosine, so the bar is the mean's, 1.5 times (the repository's
    factor for sets of cases)."""
    _need_gpu()
    geom = O.SMOLLM2_135M
    contexts = [int(x) for x in np.random.default_rng(46).integers(1, 2001, 16)]
    case = GC.random_kv_case(geom, 439, contexts, norm_jitter=0.0, capacity=capacity)
    ids, pos = [int(x) for x in np.random.default_rng(47).integers(16, 49152, 16)], [S - 1 for S in contexts]
    k = case.kernel_step(ids, pos)
    f = case.eager_gpu_step(ids, pos)
    r = case.oracle_step(ids, pos, layer_outputs=True)
    for what in (lambda c: c["max_abs"], lambda c: 1.0 - c["cos"]):
        got, floor = (sum(what(GC.compare_logits(x["logits"][b], r["logits"][b])) for b in range(16)) / 16 for x in (k, f))
        assert got <= GC.SEED_SET_MEAN_FACTOR * floor, (got, floor)
    lo = r["layer_outputs"]
    case.sync_kv_from_oracle()
    fracs = []
    for li in range(geom.layers):
        x_in = case.w.embed[ids] if li == 0 else lo[li - 1]
        out = GC.teacher_forced_layer_batch(case, li, x_in, pos)["out"]
        for b in range(16):
            c = GC.compare_logits(out[b], lo[li, b])
            assert c["max_abs"] <= GC.LOGIT_ATOL and c["cos"] >= GC.COS_MIN, (li, b, c)
            fracs.append(GC.identical_fraction(out[b], lo[li, b]))
    assert sum(fracs) / len(fracs) >= 0.9, sum(fracs) / len(fracs)


@pytest.mark.parametrize("base", [O.SMOLLM2_360M, O.SMOLLM2_135M], ids=["360m", "135m"])
@pytest.mark.parametrize("capacity", [6816, 6832])
def test_both_splits_of_the_pairs_against_oracle(capacity, base):
    """The same nine sequences at the last block table capacity of 135M's whole workgroups and the first of its
    end-to-end split (9 * 6,816 <= 61,440 < 9 * 6,832; 360M runs decode_kernel_b at both): chunks of one tile,
    of a quad and one token more, pairs without a cached token."""
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
