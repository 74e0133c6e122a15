"""Prompt attention over Q8_0 caches on the matrix cores, on the GPU's own captured
queries and cache rows, against float64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

import rust_interference_engine_amd as R  # noqa: E402
from rust_interference_engine_amd import synth  # noqa: E402

from test_gpu_parity import Q8_0, cuda  # noqa: E402,F401


def _rows(raw, hd):
    """Q8_0 rows [..., hd/32·34] bytes → block scales [..., hd/32] and codes [..., hd]"""
    b = raw.reshape(*raw.shape[:-1], hd // 32, 34)
    d = np.ascontiguousarray(b[..., :2]).view(np.float16)[..., 0].astype(np.float64)
    return d, b[..., 2:].view(np.int8).reshape(*raw.shape[:-1], hd).astype(np.float64)


def _check(oracle, g, spec, hd, nh, nkv, n_ctx, pos0, n):
    G, qd = nh // nkv, nh * hd
    for layer in range(spec.n_layer):
        q = g.capture(layer, 3, n * qd).reshape(n, nh, hd)
        att = g.capture(layer, 2, n * qd).reshape(n, nh, hd)
        (dk, ck), (dv, cv) = (_rows(g.kv_layer(layer, w, nkv, n_ctx)[0].reshape(nkv, n_ctx, -1), hd) for w in (0, 1))
        V = np.repeat(dv, 32, axis=-1) * cv
        for t in range(n):
            p = pos0 + t
            for hq in range(nh):
                kv = hq // G
                qa = oracle.quantize_q8_0(q[t, hq])
                qs, dq = qa["qs"].reshape(-1).astype(np.float64), qa["d"].astype(np.float64)
                s = (((ck[kv, :p + 1] * qs).reshape(p + 1, hd // 32, 32).sum(2) * dk[kv, :p + 1]) * dq).sum(1)
                w = np.exp(s - s.max())
                ref = (w / w.sum()) @ V[kv, :p + 1]
                # an f32 score carries a few 2^-24·|s|, which moves each weight by that
                # much; blocks of 32 dims are judged by their own largest value
                for b in range(hd // 32):
                    sl = slice(32 * b, 32 * b + 32)
                    bound = (8 * 2.0 ** -24 * np.abs(s).max() + 5e-6) * np.abs(V[kv, :p + 1, sl]).max() + 1e-6
                    err = np.abs(att[t, hq, sl] - ref[sl]).max()
                    assert err <= bound, (layer, p, hq, b, err, bound)


# one to eight query heads per KV head, every head size with a kernel; batches at 0, 64
# and 128 end inside a tile, and the last (5 tokens) splits its positions over workgroups
@pytest.mark.parametrize("hd,nh,nkv", [(32, 4, 2), (64, 6, 2), (64, 8, 1), (96, 6, 6), (128, 8, 2), (128, 10, 2), (256, 4, 1), (256, 4, 2)])
def test_q8_0_prompt_attention_matches_f64_on_captured_rows(oracle, cuda, hd, nh, nkv):
    spec = synth.tiny("llama", Q8_0)
    spec.head_dim, spec.n_head, spec.n_head_kv, spec.rope_dim = hd, nh, nkv, hd
    g = R.HipBackend(synth.build(spec), n_ctx=160, max_batch=64, kv_type=R.KvType.Q8_0)
    g.set_capture(True)
    toks = [(i * 53 + 11) % spec.n_vocab for i in range(155)]
    for pos0, end in ((0, 64), (64, 128), (128, 150), (150, 155)):
        g.forward(toks[pos0:end], pos0)
        _check(oracle, g, spec, hd, nh, nkv, 160, pos0, end - pos0)


def test_q8_0_values_past_the_half_range(oracle, cuda):
    """Value blocks of 32 dims above 65504 (in one of four), small ones beside them."""
    from gguf_np import GGUF
    hd, nh, nkv = 128, 4, 2
    spec = synth.tiny("llama", Q8_0)
    spec.head_dim, spec.n_head, spec.n_head_kv, spec.rope_dim = hd, nh, nkv, hd
    img = bytearray(synth.build(spec))
    for name, start, size in GGUF(bytes(img)).tensor_order:
        if name == "blk.0.attn_v.weight":
            rows = np.frombuffer(img, np.uint8, size, start).reshape(nkv * hd, spec.n_embd // 32, 34)
            d = rows[32:64, :, :2].copy().view(np.float16)
            rows[32:64, :, :2] = np.full_like(d, 800).view(np.uint8)
    g = R.HipBackend(bytes(img), n_ctx=96, max_batch=64, kv_type=R.KvType.Q8_0)
    g.set_capture(True)
    toks = [(i * 53 + 11) % spec.n_vocab for i in range(90)]
    spec.n_layer = 1  # the others see this layer's output through their norms
    for pos0, end in ((0, 64), (64, 90)):
        g.forward(toks[pos0:end], pos0)
        v = _rows(g.kv_layer(0, 1, nkv, 96)[0].reshape(nkv, 96, -1), hd)[0]
        assert v[0, pos0:end, 1].max() > 516 and v[0, pos0:end, 0].max() < 1
        _check(oracle, g, spec, hd, nh, nkv, 96, pos0, end - pos0)


# heads of 128 and, in two groups, of 256; later batches split their positions over workgroups
@pytest.mark.parametrize("hd", [128, 256])
def test_q8_0_values_past_the_half_range_in_splits(oracle, cuda, hd):
    from gguf_np import GGUF
    nh, nkv = 4, 2
    spec = synth.tiny("llama", Q8_0)
    spec.head_dim, spec.n_head, spec.n_head_kv, spec.rope_dim = hd, nh, nkv, hd
    img = bytearray(synth.build(spec))
    for name, start, size in GGUF(bytes(img)).tensor_order:
        if name == "blk.0.attn_v.weight":
            rows = np.frombuffer(img, np.uint8, size, start).reshape(nkv * hd, spec.n_embd // 32, 34)
            d = rows[hd - 64:hd - 32, :, :2].copy().view(np.float16)
            rows[hd - 64:hd - 32, :, :2] = np.full_like(d, 800).view(np.uint8)
    g = R.HipBackend(bytes(img), n_ctx=160, max_batch=64, kv_type=R.KvType.Q8_0)
    g.set_capture(True)
    toks = [(i * 53 + 11) % spec.n_vocab for i in range(155)]
    spec.n_layer = 1  # the others see this layer's output through their norms
    for pos0, end in ((0, 64), (64, 128), (128, 150), (150, 155)):
        g.forward(toks[pos0:end], pos0)
        _check(oracle, g, spec, hd, nh, nkv, 160, pos0, end - pos0)
    v = _rows(g.kv_layer(0, 1, nkv, 160)[0].reshape(nkv, 160, -1), hd)[0]
    assert v[0, :155, hd // 32 - 2].max() > 516 and v[0, :155, 0].max() < 1
