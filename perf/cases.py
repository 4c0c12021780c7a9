"""The work a program has this package do, as timed cases: decode steps and the preparation of weights.

A decode case is one greedy or sampled serving step of a SmolLM2 model through the registry's
`load(name).decode_step(...)`: the weights, the paged KV caches, the block table and the step's
metadata are in hand (as a serving loop keeps them), and the step returns the final-normed hidden
states, the logits and the K/V rows it appended.  Contexts are ragged over a batch, block tables are
shuffled, and a table is either as wide as the longest context needs or as wide as a server that
admits 8192 tokens allocates.  A weight case is what a program does when weights arrive: encode the
lossless gate/up cache again after a reload, or quantise a model's projections to MXFP8.
"""

from __future__ import annotations

import math

import torch

import prime_kernels_amd as pk
from prime_kernels_amd import workload
from prime_kernels_amd.decode_megakernel import MODEL as M135
from prime_kernels_amd.decode_megakernel_360m import MODEL as M360
from prime_kernels_amd.lossless_bf16 import EncodedGUCache
from prime_kernels_amd.mxfp8 import quantize_layers

BF16 = torch.bfloat16
VOCAB = 49152
MODELS = {"135m": M135, "360m": M360}
REGISTRY = {("135m", "bf16"): "decode_megakernel", ("360m", "bf16"): "decode_megakernel_360m",
            ("360m", "lossless"): "decode_megakernel_360m", ("360m", "mxfp8"): "decode_megakernel_360m_mxfp8"}
DEVICE = "cuda"
REFRESHED = (0, 1, 4, 7, 10, 13, 16, 19, 22, 25, 28, 31)   # layers whose encoded buffers are returned (all five of each)


def _decode(model, batch, lo, hi, layers=0, weights="bf16", wide=False, head=True, phase=0.25):
    """A decode case: `batch` sequences with lo..hi tokens already cached, `layers` of the model's
    layers (0: all), with or without the LM head, the block table tight or 8192 tokens wide."""
    return {"kind": "decode", "model": model, "batch": batch, "lo": lo, "hi": hi, "layers": layers,
            "weights": weights, "wide": wide, "head": head, "phase": phase}


def listed():
    return [
        # one decoder block with 512 cached tokens: a pipeline stage or a layer-by-layer comparison
        dict(_decode("360m", 1, 512, 512, layers=1, head=False), name="block-360m-b1-512"),
        # the first tokens of a chat turn on the small model
        dict(_decode("135m", 1, 41, 41, wide=True), name="135m-b1-41"),
        # the ordinary interactive step: one sequence, a 1024-token prompt behind it
        dict(_decode("360m", 1, 1024, 1024), name="360m-b1-1024"),
        # the same service with its gate/up weights held losslessly encoded
        dict(_decode("360m", 1, 707, 707, weights="lossless"), name="360m-lossless-b1-707"),
        # a long document on quantised weights
        dict(_decode("360m", 1, 8192, 8192, weights="mxfp8"), name="360m-mxfp8-b1-8192"),
        # the longest context the package takes, less a few tokens
        dict(_decode("360m", 1, 12003, 12003), name="360m-b1-12003"),
        # two sequences, the reference's own batch limit for this model
        dict(_decode("360m", 2, 300, 1500, wide=True), name="360m-b2-ragged"),
        # a small server: four sequences
        dict(_decode("360m", 4, 100, 2000, wide=True), name="360m-b4-ragged"),
        # an odd batch on the small model
        dict(_decode("135m", 7, 60, 1900), name="135m-b7-ragged"),
        # a loaded server: sixteen sequences with contexts of 128 to 4096 tokens
        dict(_decode("360m", 16, 128, 4095, phase=0.0), name="360m-b16-ragged"),
        # new weights reach a program that serves the lossless form
        {"kind": "lossless-refresh", "name": "lossless-refresh"},
        # a checkpoint shard of eight layers is quantised on arrival
        {"kind": "mxfp8-quantize", "layers": 8, "name": "mxfp8-quantize"},
    ]


def draw(rng):
    kind = rng.choice(["decode"] * 8 + ["mxfp8-quantize"])
    if kind == "mxfp8-quantize":
        return {"kind": kind, "layers": rng.randint(1, 8)}
    model = rng.choice(["135m", "360m", "360m"])
    batch = rng.choice([1, 1, 2, 3]) if rng.random() < 0.5 else rng.randint(2, 16)
    weights = "bf16"
    if batch == 1 and model == "360m":
        weights = rng.choice(["bf16", "bf16", "lossless", "mxfp8"])
    # contexts over the whole range; 16 long ones together stay within the largest listed case
    top = min(12200, 33000 // batch)
    a, b = (round(math.exp(rng.uniform(math.log(8), math.log(top)))) for _ in range(2))
    lo, hi = min(a, b), max(a, b)
    if batch == 1:
        lo = hi
    return _decode(model, batch, lo, hi, layers=rng.choice([0, 0, 1, 3]) if weights != "lossless" else 0,
                   weights=weights, wide=rng.random() < 0.5 and hi < 8000, head=rng.random() < 0.7,
                   phase=round(rng.random(), 3))


def contexts(case):
    """Cached tokens of each sequence: spread evenly over lo..hi, in a shuffled order."""
    n, lo, hi = case["batch"], case["lo"], case["hi"]
    if n == 1:
        return [hi]
    step = next(s for s in range(max(2, round(0.618 * n)), 4 * n) if math.gcd(s, n) == 1)
    return [lo + round((hi - lo) * (((i * step) % n) + case["phase"]) / (n - 1 + case["phase"])) for i in range(n)]


def _layers(case):
    return case["layers"] or MODELS[case["model"]].layers


def prepare(case, seed):
    if case["kind"] == "lossless-refresh":
        def matrices(seed, std):
            g = torch.Generator(device=DEVICE).manual_seed(seed)
            return [(torch.randn((5120, 960), generator=g, device=DEVICE) * std).to(BF16) for _ in range(32)]

        # one first set of weights, so that the tables' sizes are alike; the weights that arrive are the input
        old, new = matrices(0, 0.02), matrices(seed, 0.0201)
        cache = EncodedGUCache(old)
        for i in range(32):   # the tables' unused tails hold known bytes, so that they can be compared
            cache.buffers(i)["raw"].view(torch.int16).zero_()
        return {"kind": case["kind"], "cache": cache, "weights": new,
                "buffers": [list(cache.buffers(i).values()) for i in REFRESHED]}
    if case["kind"] == "mxfp8-quantize":
        _, _, layers = workload.random_weights(M360, seed, DEVICE, layers=case["layers"])
        return {"kind": case["kind"], "layers": layers}

    model = MODELS[case["model"]]
    n, batch, ctx = _layers(case), case["batch"], contexts(case)
    embed, final_norm, layers = workload.random_weights(model, seed, DEVICE, layers=n)
    encoded = EncodedGUCache([w[4] for w in layers]) if case["weights"] == "lossless" else None
    if case["weights"] == "mxfp8":
        layers = quantize_layers(layers)
    # paged caches: the blocks of all sequences shuffled over one pool, as a server's allocator leaves them
    need = [c // 16 + 1 for c in ctx]
    cpu = torch.Generator().manual_seed(seed + 1)
    pool = torch.randperm(sum(need), generator=cpu, dtype=torch.int64)
    table = torch.zeros((batch, 512 if case["wide"] else max(need)), dtype=torch.int32)
    at = 0
    for b, k in enumerate(need):
        table[b, :k] = pool[at:at + k].to(torch.int32)
        at += k
    gpu = torch.Generator(device=DEVICE).manual_seed(seed + 2)
    kv = torch.empty((n, sum(need), model.kv_heads, 16, 128), dtype=BF16, device=DEVICE)
    for i in range(n):
        kv[i] = torch.randn(kv.shape[1:], generator=gpu, device=DEVICE)
    block = [int(table[b, c // 16]) for b, c in enumerate(ctx)]
    ids = torch.randint(0, VOCAB, (batch,), generator=cpu)
    kwargs = dict(
        input_ids=ids.to(DEVICE), positions=torch.tensor(ctx, device=DEVICE),
        seq_lens=torch.tensor([c + 1 for c in ctx], dtype=torch.int32, device=DEVICE),
        block_table=table.to(DEVICE), slot_mapping=torch.tensor([16 * k + c % 16 for k, c in zip(block, ctx)],
                                                                device=DEVICE),
        embed=embed, layers=layers, final_norm=final_norm, kv_caches=list(kv.unbind(0)),
        cos_sin_cache=workload.rope_table(max(8192, max(ctx) + 1), device=DEVICE), eps=1e-5)
    if case["layers"]:
        kwargs["num_layers"] = n
    if encoded is not None:
        kwargs["encoded_gu"] = encoded
    if case["head"]:
        kwargs["logits_out"] = torch.empty((batch, VOCAB), dtype=BF16, device=DEVICE)
    return {"kind": "decode", "step": pk.load(REGISTRY[case["model"], case["weights"]]).decode_step, "kwargs": kwargs,
            "kv": kv, "appended": [kv[:, k, :, c % 16] for k, c in zip(block, ctx)]}


def run(state):
    if state["kind"] == "lossless-refresh":
        state["cache"].refresh(state["weights"])
        return state["buffers"]
    if state["kind"] == "mxfp8-quantize":
        return [[q, qs, o, os, g, gs, d, ds] for _, q, qs, o, os, _, g, gs, d, ds in quantize_layers(state["layers"])]
    hidden = state["step"](**state["kwargs"])
    out = {"hidden": hidden, "appended": state["appended"]}
    if "logits_out" in state["kwargs"]:
        out["logits"] = state["kwargs"]["logits_out"]
    return out


def _matrix_bytes(model, weights):
    """(weights of one layer's projections, bytes they take)."""
    n = sum(math.prod(s) for s in model.shapes() if len(s) == 2)
    if weights == "mxfp8":
        return n, n + n // 32
    if weights == "lossless":   # gate/up: one byte plus half a byte of header a weight, escapes left out
        gu = math.prod(model.shapes()[4])
        return n, 2 * (n - gu) + gu + gu // 2
    return n, 2 * n


def work(case):
    if case["kind"] == "lossless-refresh":
        n = 32 * 5120 * 960
        return {"bytes": 2 * n + n + n // 2, "flops": 0}
    if case["kind"] == "mxfp8-quantize":
        n = case["layers"] * _matrix_bytes(M360, "bf16")[0]
        return {"bytes": 2 * n + n + n // 32, "flops": 0}
    model, n, ctx = MODELS[case["model"]], _layers(case), contexts(case)
    params, size = _matrix_bytes(model, case["weights"])
    token = 2 * model.kv_heads * model.head_dim * 2
    moved = n * (size + 4 * model.hidden + token * sum(c + 1 for c in ctx))
    flops = n * (2 * params * case["batch"] + 4 * model.heads * model.head_dim * sum(c + 1 for c in ctx))
    if case["head"]:
        moved += VOCAB * model.hidden * 2 + VOCAB * 2 * case["batch"]
        flops += 2 * VOCAB * model.hidden * case["batch"]
    return {"bytes": moved + 4 * model.hidden * case["batch"], "flops": flops}


def tolerance(case):
    """A bf16 model rounds every activation, and one rounding that falls the other way travels through
    the layers that follow: the step is 0.007 from 64-bit arithmetic after one layer, 0.012 after three
    and 0.02 to 0.048 after 30 or 32 (relative, over batches, contexts and seeds), about
    0.007 sqrt(layers).  Four times that is stated; encoded and quantised weights are whole bytes."""
    if case["kind"] != "decode":
        return "exact"
    return {"rel": round(0.028 * math.sqrt(_layers(case)), 3)}


def _dequantised(codes, scales):
    rows, cols = codes.shape
    w = codes.view(torch.float8_e4m3fn).to(torch.float64).view(rows, cols // 32, 32)
    e = scales[:, :cols // 32].to(torch.float64) - 127.0
    return (w * torch.exp2(e)[:, :, None]).view(rows, cols)


def exact(case, seed):
    """The decode step in 64-bit arithmetic with no intermediate rounding."""
    if case["kind"] != "decode":
        return None
    state = prepare(case, seed)
    kw, kv = state["kwargs"], state["kv"]
    model, batch, ctx = MODELS[case["model"]], case["batch"], contexts(case)
    heads, groups, hd = model.heads, model.kv_heads, model.head_dim
    f64 = torch.float64

    def norm(x, w):
        return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + kw["eps"]) * w.to(f64)

    angle = kw["cos_sin_cache"][kw["positions"]].to(f64)
    cos, sin = angle[:, None, :hd // 2], angle[:, None, hd // 2:]

    def rope(t):   # [batch, heads, hd], the two halves of a head rotated against each other
        a, b = t[..., :hd // 2], t[..., hd // 2:]
        return torch.cat((a * cos - b * sin, b * cos + a * sin), dim=-1)

    x = kw["embed"][kw["input_ids"]].to(f64)
    new = []
    for layer, cache in zip(kw["layers"], kv):
        if len(layer) == 10:
            n1, q8, qs, o8, os_, n2, g8, gs, d8, ds = layer
            wqkv, wo, wgu, wd = (_dequantised(*p) for p in ((q8, qs), (o8, os_), (g8, gs), (d8, ds)))
        else:
            n1, wqkv, wo, n2, wgu, wd = layer
            wqkv, wo, wgu, wd = (t.to(f64) for t in (wqkv, wo, wgu, wd))
        qkv = (norm(x, n1) @ wqkv.t()).view(batch, heads + 2 * groups, hd)
        q, k, v = rope(qkv[:, :heads]), rope(qkv[:, heads:heads + groups]), qkv[:, heads + groups:]
        new.append(torch.cat((k, v), dim=-1))
        mixed = []
        for b in range(batch):
            blocks = kw["block_table"][b, :ctx[b] // 16 + 1].long()
            past = cache[blocks].permute(1, 0, 2, 3).reshape(groups, -1, 2 * hd)[:, :ctx[b]].to(f64)
            kk = torch.cat((past[..., :hd], k[b, :, None]), dim=1)
            vv = torch.cat((past[..., hd:], v[b, :, None]), dim=1)
            s = (q[b].view(groups, heads // groups, hd) @ kk.transpose(1, 2).contiguous()) / math.sqrt(hd)
            mixed.append((torch.softmax(s, dim=-1) @ vv).reshape(heads * hd))
        x = x + torch.stack(mixed) @ wo.t()
        gate, up = (norm(x, n2) @ wgu.t()).chunk(2, dim=-1)
        x = x + (torch.nn.functional.silu(gate) * up) @ wd.t()
    hidden = norm(x, kw["final_norm"])
    stacked = torch.stack(new)
    out = {"hidden": hidden, "appended": [stacked[:, b].contiguous() for b in range(batch)]}
    if "logits_out" in kw:
        out["logits"] = hidden @ kw["embed"].to(f64).t()
    return out
