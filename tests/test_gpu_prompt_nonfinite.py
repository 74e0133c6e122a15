"""Non-finite values in prompts: they reach the tokens that see them, and no others."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

import rust_interference_engine_amd as R  # noqa: E402
from rust_interference_engine_amd import synth  # noqa: E402

from test_gpu_parity import F32, Q4_0, Q5_0, Q8_0, _gemv, _quant_on_gpu, act_fmt, cuda  # noqa: E402,F401

ODD, PLAIN = 7, 9  # tokens whose embeddings differ in dim 0 alone


def _image(hd, nh, nkv):
    """Token ODD's values overflow both caches in dims 32..63 of KV head 0, infinities of
    either sign; every other token's are ordinary."""
    from gguf_np import GGUF
    spec = synth.tiny("llama", F32)
    spec.head_dim, spec.n_head, spec.n_head_kv, spec.rope_dim, spec.n_layer = hd, nh, nkv, hd, 1
    img = bytearray(synth.build(spec))
    for name, start, size in GGUF(bytes(img)).tensor_order:
        w = np.frombuffer(img, np.float32, size // 4, start).reshape(-1, spec.n_embd)
        if name == "token_embd.weight":
            w[:, 0] = 0
            w[ODD] = w[PLAIN]
            w[ODD, 0] = np.abs(w).max()
        elif name == "blk.0.attn_v.weight":
            w[32:64, 0] = np.where(np.arange(32) % 3 == 0, -1e12, 1e12)
        elif name == "blk.0.attn_q.weight" or name == "blk.0.attn_k.weight":
            w[:, 0] = 0
    return spec, bytes(img)


# the odd token inside a tile and a batch, on a tile's first and last position, and in a
# batch of few tokens behind 128 positions, whose positions are split over workgroups
@pytest.mark.parametrize("hd,nh,nkv,kv", [(64, 6, 2, 1), (128, 8, 2, 1), (256, 4, 1, 1), (256, 4, 2, 1), (256, 4, 1, 0), (256, 8, 2, 0)])
@pytest.mark.parametrize("at", [37, 64, 95, 152])
def test_values_past_the_cache_format_stay_with_the_tokens_that_see_them(cuda, hd, nh, nkv, kv, at):
    spec, img = _image(hd, nh, nkv)
    toks = [10 + (i * 53) % (spec.n_vocab - 10) for i in range(155)]
    att = {}
    for tok in (ODD, PLAIN):
        g = R.HipBackend(img, n_ctx=160, max_batch=128, kv_type=kv)
        g.set_capture(True)
        toks[at] = tok
        rows = []
        for pos0, end in ((0, 128), (128, 150), (150, 155)):
            g.forward(toks[pos0:end], pos0)
            rows.append(g.capture(0, 2, (end - pos0) * nh * hd).reshape(end - pos0, nh, hd))
        att[tok] = np.concatenate(rows)
    a, b, G = att[ODD], att[PLAIN], nh // nkv
    assert np.isfinite(b).all()
    assert np.array_equal(a[:at], b[:at])  # their sums add probability 0 times another value, if any
    # from there on: infinities of the values' signs in the 32 dims, finite everywhere else
    sign = np.where(np.arange(32) % 3 == 0, -np.inf, np.inf)
    # (the per-token kernel, which runs up to 8 tokens of 256-wide heads over an f16 cache,
    # fills idle slots of a range with its first row at probability 0: NaN for a token that
    # sees an infinity there, as ever)
    seen = a[at:, :G, 32:64]
    per_token = hd == 256 and kv == 0
    assert ((seen == sign) | (np.isnan(seen) & (per_token & (np.arange(at, 155) >= 150))[:, None, None])).all()
    rest = np.ones(a.shape[1:], bool)
    rest[:G, 32:64] = False
    assert np.isfinite(a[at:][:, rest]).all()


# K of half a stage, of one and a half, and split with half a stage at the end
@pytest.mark.parametrize("ty", [Q4_0, Q5_0, Q8_0])
@pytest.mark.parametrize("k", [64, 192, 6208])
def test_an_infinite_scale_in_the_last_block(oracle, cuda, ty, k):
    import ggml_np as G
    rows, n = 70, 33
    rb, bb = G.row_bytes(ty, k), G.row_bytes(ty, 32)
    w = np.array(oracle.Rng(31 + ty).random_weight(ty, rows, k)).view(np.uint8).reshape(rows, rb).copy()
    w[::3, rb - bb:rb - bb + 2] = np.array([0x7C00], np.uint16).view(np.uint8)
    x = (np.random.default_rng(k).uniform(-1, 1, (n, k)) * 2).astype(np.float32)
    act = _quant_on_gpu(x, act_fmt(ty), cuda)["dev"]
    got = _gemv(ty, w.reshape(-1), rows, k, act, None, n, cuda, gemm=True)
    want = _gemv(ty, w.reshape(-1), rows, k, act, None, n, cuda)  # block sum times infinity (NaN where it is 0)
    assert np.isinf(want[:, ::3]).mean() > 0.9
    np.testing.assert_array_equal(got[:, ::3], want[:, ::3])
    assert np.isfinite(got[:, 1::3]).all() and np.isfinite(got[:, 2::3]).all()
