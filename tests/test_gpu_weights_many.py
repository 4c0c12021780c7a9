"""Weight preparation over many matrices a launch: the MXFP8 quantiser on every bf16 pattern, ragged sizes
and more matrices than one launch takes, against the oracle; the lossless encoder of many layers against
the encoder of one.  Whole bytes: nothing may differ."""

import ctypes

import numpy as np
import pytest
import torch

from oracle import mxfp8 as MX

pytestmark = pytest.mark.gpu


def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


def test_quantizer_on_every_bf16_pattern():
    """Every bf16 value but NaN (infinities among them), in blocks whose largest value puts it at every depth
    of the e4m3 range: an ascending ramp, and the patterns shuffled; then NaN in blocks of their own kind."""
    _need_gpu()
    from prime_kernels_amd import mxfp8

    bits = np.arange(65536, dtype=np.uint16)
    bits = bits[(bits & 0x7FFF) <= 0x7F80]
    assert bits.size == 65282
    bits = np.concatenate([bits, bits[-30:]])                 # 2,041 whole blocks of 32
    rng = np.random.default_rng(3)
    for order in (bits, rng.permutation(bits), bits[::-1].copy()):
        w = torch.from_numpy(order.view(np.int16).copy()).view(torch.bfloat16).view(157, 416)
        q, s = mxfp8.quantize(w.cuda())
        q_ref, s_ref = MX.quantize(w)
        assert np.array_equal(q.cpu().numpy(), q_ref) and np.array_equal(s.cpu().numpy(), s_ref)
    # a quiet NaN becomes e4m3's NaN and leaves its block's scale and other codes alone
    w = torch.randn((40, 256), generator=torch.Generator().manual_seed(2)).to(torch.bfloat16)
    hit = torch.rand((40, 256), generator=torch.Generator().manual_seed(4)) < 0.02
    q, s = mxfp8.quantize(torch.where(hit, torch.tensor(float("nan"), dtype=torch.bfloat16), w).cuda())
    q_ref, s_ref = MX.quantize(torch.where(hit, torch.zeros_like(w), w))
    assert np.array_equal(s.cpu().numpy(), s_ref)
    assert ((q.cpu()[hit] & 0x7F) == 0x7F).all()
    assert np.array_equal(q.cpu().numpy()[~hit.numpy()], q_ref[~hit.numpy()])


def test_quantizer_many_matrices():
    """35 matrices (a launch takes 32) of sizes around a workgroup's 1,024 pieces, among them the layer
    shapes, through quantize_layers' path: each equal to the oracle's."""
    _need_gpu()
    from prime_kernels_amd import mxfp8

    g = torch.Generator().manual_seed(9)
    shapes = [(1, 32), (3, 64), (256, 32), (255, 32), (257, 32), (64, 960), (5, 2560), (128, 64), (1, 8192)]
    ws = [(torch.randn(shapes[i % len(shapes)], generator=g) * 0.02 * (1 + i)).to(torch.bfloat16) for i in range(35)]
    for w, (q, s) in zip(ws, mxfp8._quantize_all([w.cuda() for w in ws])):
        q_ref, s_ref = MX.quantize(w)
        assert np.array_equal(q.cpu().numpy(), q_ref) and np.array_equal(s.cpu().numpy(), s_ref), tuple(w.shape)


class _Other(torch.Tensor):
    """A subclass, as a program's own parameter type may be."""


def test_quantizer_gives_plain_tensors():
    """The codes and scales of a subclass's matrix are plain tensors, one matrix or many, strided or not."""
    _need_gpu()
    from prime_kernels_amd import mxfp8

    w = (torch.randn((64, 96), generator=torch.Generator().manual_seed(1)) * 0.02).to(torch.bfloat16).cuda()
    wide = torch.stack((w, -w), dim=2).view(64, 192)[:, ::2]
    want = mxfp8.quantize(w)
    for given in (w, wide, w.as_subclass(_Other), wide.as_subclass(_Other), torch.nn.Parameter(w, requires_grad=False)):
        layer = (None, given, given, None, given, given)
        for got in (mxfp8.quantize(given), mxfp8._quantize_all([given])[0], mxfp8.quantize_layers([layer])[0][6:8]):
            assert all(type(g) is torch.Tensor and torch.equal(g, t) for g, t in zip(got, want))


@pytest.mark.parametrize("layers", [1, 33])
def test_lossless_encode_layers_equals_one_by_one(layers):
    """Layers with few, no and only escapes, tables too small for theirs, in one call (32 layers a launch):
    plane, headers, row offsets, enabled flag, stored escapes and totals equal the one-layer encoder's."""
    _need_gpu()
    from prime_kernels_amd import _native

    lib = _native.library()
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(21)
    chunks = 5120 * 120

    def matrix(i):
        w = torch.randn((5120, 960), generator=g, device=dev) * 0.02
        if i % 4 == 1:
            w = torch.full_like(w, 0.5)                       # no escapes
        if i % 4 == 2:
            w[:, ::8] *= 2.0 ** -20                           # every chunk escapes
        if i % 4 == 3:
            w[7] = float("inf")
            w[5119, 952:] = 0.0
        return w.to(torch.bfloat16)

    def buffers():
        return dict(plane=torch.zeros((5120, 960), dtype=torch.uint8, device=dev),
                    headers=torch.zeros(chunks, dtype=torch.int32, device=dev),
                    raw=torch.zeros(chunks * 8, dtype=torch.int16, device=dev),
                    row_offsets=torch.zeros(5121, dtype=torch.int32, device=dev),
                    enabled=torch.zeros((), dtype=torch.int32, device=dev))

    kinds = min(layers, 4)                                    # as many different layers, reused
    ws = [matrix(i) for i in range(kinds)]
    caps = [chunks if i % 2 == 0 else 100 for i in range(kinds)]
    one, totals = [], []
    scan = torch.empty(lib.lossless_scan_workspace_bytes(), dtype=torch.uint8, device=dev)
    flags, prefix = (torch.empty(chunks, dtype=torch.int32, device=dev) for _ in range(2))
    stream = torch.cuda.current_stream().cuda_stream
    for w, cap in zip(ws, caps):
        b = buffers()
        assert lib.lossless_encode_layer(w.data_ptr(), b["plane"].data_ptr(), b["headers"].data_ptr(), b["raw"].data_ptr(),
                                         b["row_offsets"].data_ptr(), flags.data_ptr(), prefix.data_ptr(), scan.data_ptr(),
                                         scan.numel(), b["enabled"].data_ptr(), cap, stream) == 0
        totals.append(int(prefix[-1]))
        one.append(b)
    many = [buffers() for _ in range(layers)]
    work = torch.empty(lib.lossless_encode_workspace_bytes(layers), dtype=torch.uint8, device=dev)
    got = torch.zeros(layers, dtype=torch.int32, device=dev)

    def column(ts):
        return (ctypes.c_void_p * layers)(*[t.data_ptr() for t in ts])

    args = [column([ws[i % kinds] for i in range(layers)])] + [column([b[k] for b in many]) for k in
                                                                ("plane", "headers", "raw", "row_offsets", "enabled")]
    cap_arg = (ctypes.c_uint32 * layers)(*[caps[i % kinds] for i in range(layers)])
    assert lib.lossless_encode_layers(layers, *args, cap_arg, got.data_ptr(), work.data_ptr(), work.numel() - 1, stream) == 9108
    assert lib.lossless_encode_layers(layers, *args, cap_arg, got.data_ptr(), work.data_ptr(), work.numel(), stream) == 0
    torch.cuda.synchronize()
    for i, b in enumerate(many):
        assert int(got[i]) == totals[i % kinds], i
        for k, v in b.items():
            assert torch.equal(v, one[i % kinds][k]), (i, k)


def test_refreshes_of_one_cache_from_two_threads():
    """Each thread on its own stream with its own weights, the passes one after the other: the cache ends as
    the encoding of the weights it says it holds, and no pass is lost."""
    _need_gpu()
    import threading

    from prime_kernels_amd.lossless_bf16 import LAYERS, EncodedGUCache

    def matrices(seed, std):
        g = torch.Generator(device="cuda").manual_seed(seed)
        return [(torch.randn((5120, 960), generator=g, device="cuda") * std).to(torch.bfloat16) for _ in range(LAYERS)]

    sets = [matrices(1, 0.02), matrices(2, 0.021)]
    cache = EncodedGUCache(sets[0])
    torch.cuda.synchronize()
    errors = []

    def work(weights):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(5):
                    cache.refresh(weights)
        except Exception as e:  # noqa: BLE001 - shown by the assertion below
            errors.append(e)

    threads = [threading.Thread(target=work, args=(w,)) for w in sets]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
    assert cache.generation == 11 and cache.statistics()["active_layers"] == LAYERS
    for i in range(LAYERS):
        assert cache.enabled(i) and torch.equal(cache.decode_layer(i).view(torch.int16), cache.weights[i].view(torch.int16)), i
