"""A call's logits around the size up to which they come back through pinned memory."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

import rust_interference_engine_amd as R  # noqa: E402
from rust_interference_engine_amd import synth  # noqa: E402

from test_gpu_parity import F32, cuda  # noqa: E402,F401


# 160 * 1024 floats: 40 rows of 4096, and a row fewer and more; a vocabulary whose rows end inside 16 bytes
@pytest.mark.parametrize("n_vocab,counts", [(4096, (39, 40, 41, 1)), (4099, (39, 40, 3))])
def test_logits_of_any_size(cuda, n_vocab, counts):
    spec = synth.tiny("llama", F32)
    spec.n_vocab = n_vocab
    g = R.HipBackend(synth.build(spec), n_ctx=64, max_batch=48)
    toks = np.random.default_rng(3).integers(0, n_vocab, 48)
    # row by row: each of them a call of its own on the same cache
    want = np.stack([g.forward(toks[t:t + 1], t).copy() for t in range(max(counts))])
    for n in counts:
        for _ in range(2):
            got = g.forward(toks[:n], 0, True).reshape(n, n_vocab)
            for t in range(n):
                assert np.abs(got[t] - want[t]).max() <= 1e-4 * np.abs(want[t]).max(), (n, t)
