"""The BF16 / F16 prompt GEMM keeps the accuracy of f32 dot products: attention output and
down projections of captured f32 rows, against float64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

import rust_interference_engine_amd as R  # noqa: E402
from rust_interference_engine_amd import synth  # noqa: E402

from test_gpu_parity import BF16, F16, cuda  # noqa: E402,F401


def projection_errors(cuda, ty, nh, ff, n):
    """2-norm errors of wo·att and of down·h over their own norms (the residual row's f32
    addition, one rounding, is in them)"""
    from gguf_np import GGUF
    spec = synth.tiny("llama", ty)
    spec.head_dim, spec.n_head, spec.n_head_kv, spec.rope_dim = 128, nh, nh // 2, 128
    spec.n_embd, spec.n_ff, spec.n_layer = 640, ff, 1
    img = synth.build(spec)
    t = GGUF(img).tensors

    def rows(name):
        kind, dims, raw = t[name]
        x = np.frombuffer(raw.tobytes(), np.uint16)
        x = x.view(np.float16).astype(np.float32) if kind == F16 else (x.astype(np.uint32) << 16).view(np.float32) if kind == BF16 else np.frombuffer(raw.tobytes(), np.float32)
        return x.astype(np.float64).reshape(dims[1], dims[0])

    g = R.HipBackend(img, n_ctx=n, max_batch=n)
    g.set_capture(True)
    toks = np.random.default_rng(n).integers(0, spec.n_vocab, n)
    g.forward(toks, 0)
    E = spec.n_embd
    x0 = rows("token_embd.weight")[toks]
    x1, x2 = (g.capture(0, w, n * E).reshape(n, E).astype(np.float64) for w in (0, 1))
    att = g.capture(0, 2, n * nh * 128).reshape(n, -1).astype(np.float64)
    h = g.capture(0, 6, n * ff).reshape(n, ff).astype(np.float64)
    out = []
    for before, after, act, name in ((x0, x1, att, "blk.0.attn_output.weight"), (x1, x2, h, "blk.0.ffn_down.weight")):
        ref = act @ rows(name).T
        out.append(np.linalg.norm(after - before - ref) / np.linalg.norm(ref))
    return out


# K 1024 to 9728, with and without K splits: 0.8e-7 to 1.07e-7 measured, 0.9e-7 to 1.25e-7 in
# the batched GEMV's f32 sums.  Two parts instead of three measured 1.6e-7 (F16) and 97e-7
# (BF16), stages of one sign 1.3e-7 to 1.7e-7.
@pytest.mark.parametrize("ty", [BF16, F16])
@pytest.mark.parametrize("nh,ff,n", [(8, 9728, 70), (20, 4864, 40), (20, 9728, 600)])
def test_float_gemm_error_is_that_of_f32(cuda, ty, nh, ff, n):
    assert max(projection_errors(cuda, ty, nh, ff, n)) <= 2.0 ** -23
