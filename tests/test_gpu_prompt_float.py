"""Prompts through models with BF16 / F16 matrices on the 16-bit matrix cores,
against the oracle's f32 dot products."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

import rust_interference_engine_amd as R  # noqa: E402
from rust_interference_engine_amd import synth  # noqa: E402

from test_gpu_parity import BF16, F16, _pair, cuda  # noqa: E402,F401


def _compare(g, o, nv, n, tol):
    from naive_model import max_rel_err
    toks = [(i * 29 + 7) % nv for i in range(n)]
    lg, lo = g.forward(toks, 0, True), o.forward(toks, 0, True)
    for t in range(n):
        err = max_rel_err(lg[t * nv:(t + 1) * nv], lo[t * nv:(t + 1) * nv])
        assert err < tol, f"token {t} of {n}: {err}"


# three stages of K and more, one to four 64-token tiles with remainders, K splits (ff 2080: uneven stages), GELU
@pytest.mark.parametrize("arch,ty,ff,n", [("llama", BF16, 96, 9), ("llama", F16, 160, 64), ("qwen3", BF16, 2080, 70),
                                          ("gemma2", BF16, 288, 65), ("gemma2", F16, 2080, 130), ("qwen2", F16, 1056, 200)])
def test_float_prompts_match_oracle(oracle, cuda, arch, ty, ff, n):
    spec, g, o = _pair(oracle, arch, ty, 0, n_ctx=256, max_batch=n, mutate=lambda s: setattr(s, "n_ff", ff))
    _compare(g, o, spec.n_vocab, n, 3e-3)  # the whole-model tolerance of unquantized weights


@pytest.mark.parametrize("ty", [BF16, F16])
def test_extreme_weights_as_in_f32(oracle, cuda, ty):
    """Head rows with an infinity, a NaN, subnormal halves and the largest values whose
    products with activations up to 2^8 sum to a finite f32 in any order."""
    from gguf_np import GGUF
    spec = synth.tiny("llama", ty)
    img = bytearray(synth.build(spec))
    head = {name: (start, size) for name, start, size in GGUF(bytes(img)).tensor_order}
    start, size = head.get("output.weight", head["token_embd.weight"])
    w = np.frombuffer(img, np.uint16, size // 2, start).reshape(-1, spec.n_embd)
    inf, nan, big, small = (0x7F80, 0x7FC0, 0x7700, 0x0080) if ty == BF16 else (0x7C00, 0x7E00, 0x7BFF, 0x0003)
    w[1, 5], w[2, 6], w[3, 7], w[3, 8] = inf, nan, inf, inf ^ 0x8000
    w[4, ::2], w[5] = big, small + (np.arange(spec.n_embd) % 7)
    img = bytes(img)
    g = R.HipBackend(img, n_ctx=64, max_batch=33)
    o = oracle.Backend(oracle.Model(img), 64, 33, 0, n_threads=4)
    toks = [10 + (i * 29) % (spec.n_vocab - 10) for i in range(33)]  # none of the rows above
    lg, lo = (np.asarray(b.forward(toks, 0, True)).reshape(33, -1) for b in (g, o))
    assert np.array_equal(np.isnan(lg), np.isnan(lo)) and np.array_equal(np.isinf(lg), np.isinf(lo))
    assert np.isinf(lo[:, 1]).all() and np.isnan(lo[:, 2]).all()
    fin = np.isfinite(lo)
    assert np.array_equal(np.sign(lg[~fin & ~np.isnan(lo)]), np.sign(lo[~fin & ~np.isnan(lo)]))
    # each head row against its own magnitude
    for r in [i for i in range(40) if fin[:, i].all()]:
        assert np.abs(lg[:, r] - lo[:, r]).max() <= 3e-3 * np.abs(lo[:, r]).max(), r
