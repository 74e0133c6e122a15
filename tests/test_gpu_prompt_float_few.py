"""BF16 / F16 matrices of narrow models: few tokens stay in the batched GEMV, more take the GEMM."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

import rust_interference_engine_amd as R  # noqa: E402
from rust_interference_engine_amd import synth  # noqa: E402

from test_gpu_parity import BF16, F16, cuda  # noqa: E402,F401


def _values(g, spec, toks, batch):
    """The first layer's value rows of the tokens, in batches of `batch`"""
    g.set_capture(True)
    out = []
    for i in range(0, len(toks), batch):
        b = toks[i:i + batch]
        g.forward(b, 0)
        out.append(g.capture(0, 5, len(b) * spec.n_head_kv * spec.head_dim).reshape(len(b), -1))
    return np.concatenate(out)


# the last count in the GEMV, whose rows do not depend on the batch, and the first in the GEMM
@pytest.mark.parametrize("ty", [BF16, F16])
@pytest.mark.parametrize("n_embd,n", [(512, 32), (1024, 19), (1536, 13), (2048, 9)])
def test_batch_sizes_at_the_gemms_edge(cuda, ty, n_embd, n):
    spec = synth.tiny("llama", ty)
    spec.n_embd, spec.n_layer = n_embd, 1
    g = R.HipBackend(synth.build(spec), n_ctx=64, max_batch=48)
    toks = np.random.default_rng(n).integers(0, spec.n_vocab, n + 1)
    few = _values(g, spec, toks, 4)
    assert np.array_equal(_values(g, spec, toks[:n], n), few[:n])
    gemm = _values(g, spec, toks, n + 1)
    assert np.linalg.norm(gemm - few) <= 4e-7 * np.linalg.norm(few) and not np.array_equal(gemm, few)
