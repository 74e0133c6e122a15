"""Prompt GEMMs whose weights the batched GEMV multiplied before: no more error against
float64 than the GEMV's, on the same activation codes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

from test_gpu_parity import Q4_0, Q5_0, Q5_K, Q6_K, Q8_0, _gemv, _quant_on_gpu, act_fmt, cuda  # noqa: E402,F401


# Both round a few dozen partial sums to f32, in other orders: their errors are equal within
# 10 % (measured: at most 9 %).  One chain over all blocks measured 1.2 to 3.1 times the
# GEMV's; the last case
# has 56 superblocks and no K split.
@pytest.mark.parametrize("ty,k,rows,n", [(Q5_0, 896, 320, 40), (Q5_0, 4096, 2048, 300), (Q5_0, 14336, 512, 130), (Q4_0, 960, 320, 200),
                                         (Q8_0, 2880, 1152, 400), (Q5_K, 2560, 640, 70), (Q6_K, 4096, 640, 70), (Q5_K, 14336, 4096, 512)])
def test_gemm_error_is_the_gemvs(oracle, cuda, ty, k, rows, n):
    import ggml_np as G
    w = oracle.Rng(17 + ty).random_weight(ty, rows, k)
    x = np.random.default_rng(k).standard_normal((n, k)).astype(np.float32)
    q = _quant_on_gpu(x, act_fmt(ty), cuda)
    xa = torch.from_numpy(q["qs"].astype(np.float64).reshape(n, -1, k // (q["d"].size // n)) * q["d"].astype(np.float64).reshape(n, -1, 1))
    wf = torch.from_numpy(G.dequantize(ty, w, rows * k).reshape(rows, k).astype(np.float64))
    ref = (xa.reshape(n, k).to(cuda) @ wf.to(cuda).T).cpu().numpy()
    err = [np.linalg.norm(_gemv(ty, w, rows, k, q["dev"], None, n, cuda, gemm=g) - ref) / np.linalg.norm(ref) for g in (False, True)]
    assert err[1] <= 1.1 * err[0], err
