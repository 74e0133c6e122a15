"""Prompt matmuls of the weight types and widths beyond 128-multiples of Q4_0 / Q8_0 and Q4_K on the matrix cores,
against the oracle: kernels through rie_hip_k_gemm, gated and grouped forms
through small models."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

from test_gpu_parity import Q4_0, Q4_K, Q5_0, Q5_K, Q6_K, Q8_0, _gemv, _pair, _quant_on_gpu, act_fmt, cuda  # noqa: E402,F401


def _check_rows(oracle, cuda, ty, k, rows, n_tok):
    """k_gemm rows within 1e-5·Σ|w·x| + 1e-6 of the oracle's block dots (the f32 sums'
    rounding over K ≤ 2^14 terms in any order stays under 1e-5 of the magnitudes)"""
    import ggml_np as G
    w = oracle.Rng(31 + ty).random_weight(ty, rows, k)
    x = (np.random.default_rng(k + n_tok).uniform(-1, 1, (n_tok, k)) * 2).astype(np.float32)
    got = _gemv(ty, w, rows, k, _quant_on_gpu(x, act_fmt(ty), cuda)["dev"], None, n_tok, cuda, gemm=True)
    wf = G.dequantize(ty, w, rows * k).reshape(rows, k).astype(np.float64)
    rb = G.row_bytes(ty, k)
    for t in range(n_tok) if rows < 1000 else (0, 127, 128, n_tok - 1):
        a = oracle.quantize_act(ty, x[t])
        want = np.array([oracle.vec_dot(ty, w[i * rb:(i + 1) * rb], a, k) for i in range(rows)])
        mag = np.abs(wf * x[t].astype(np.float64)).sum(axis=1)
        assert np.all(np.abs(got[t] - want) <= 1e-5 * mag + 1e-6), (ty, k, rows, n_tok, t)


# one superblock, row and token remainders, a K split in two uneven parts (13 superblocks)
@pytest.mark.parametrize("k,rows,n_tok", [(256, 40, 9), (512, 200, 33), (1024, 300, 130), (3328, 96, 70)])
def test_q5_k_gemm_matches_oracle_rows(oracle, cuda, k, rows, n_tok):
    _check_rows(oracle, cuda, Q5_K, k, rows, n_tok)


# K of one whole stage, of one and a half, of half a stage, 330 tiles' worth of rows and
# tokens in 64-token tiles over an odd number of half stages, a K split in uneven parts with
# half a stage at the end (49 stages)
@pytest.mark.parametrize("ty", [Q4_0, Q5_0, Q8_0])
@pytest.mark.parametrize("k,rows,n_tok", [(128, 40, 9), (192, 70, 33), (64, 64, 65), (960, 4200, 520), (6208, 96, 70)])
def test_32_block_gemm_matches_oracle_rows(oracle, cuda, ty, k, rows, n_tok):
    _check_rows(oracle, cuda, ty, k, rows, n_tok)


# 128-token tiles with half a stage at the end (520 of them), and in four splits in planes (65 stages)
@pytest.mark.parametrize("ty", [Q4_0, Q5_0, Q8_0])
@pytest.mark.parametrize("k,rows,n_tok", [(960, 6600, 520), (8256, 4096, 130)])
def test_128_token_tiles_match_oracle_rows(oracle, cuda, ty, k, rows, n_tok):
    _check_rows(oracle, cuda, ty, k, rows, n_tok)


# 256 tiles: too many to add their splits up in the launch, so two planes of four superblocks
@pytest.mark.parametrize("ty", [Q4_K, Q5_K, Q6_K])
def test_k_quant_splits_in_planes_match_oracle_rows(oracle, cuda, ty):
    _check_rows(oracle, cuda, ty, 2048, 4096, 200)


@pytest.mark.parametrize("arch,ty", [("llama", Q5_K), ("gemma2", Q5_K), ("gemma2", Q6_K), ("qwen3moe", Q5_K), ("qwen3moe", Q6_K),
                                     ("gemma2", Q5_0), ("qwen3moe", Q5_0)])
def test_gated_and_grouped_k_quant_prompts_match_oracle(oracle, cuda, arch, ty):
    """Gate/up with SwiGLU or GELU in one launch, and experts grouped on the device."""
    from naive_model import max_rel_err
    spec, g, o = _pair(oracle, arch, ty, 0, n_ctx=96, max_batch=70)
    nv = spec.n_vocab
    toks = [(i * 29 + 3) % nv for i in range(70)]
    lg, lo = g.forward(toks, 0, True), o.forward(toks, 0, True)
    for t in range(70):
        err = max_rel_err(lg[t * nv:(t + 1) * nv], lo[t * nv:(t + 1) * nv])
        assert err < 0.03, f"{arch} {ty}: token {t}: {err}"


# hidden 1024 (8 stages of 128, 4 superblocks): every launch of these prompts but the attention
# output's (K 256) splits K and adds its partial sums up in the launch, layer after layer on
# the same counters
@pytest.mark.parametrize("arch,ty", [("llama", Q4_0), ("gemma2", Q8_0), ("qwen3", Q5_0), ("llama", Q5_K), ("gemma2", Q6_K)])
def test_prompts_with_k_splits_match_oracle(oracle, cuda, arch, ty):
    from naive_model import max_rel_err
    spec, g, o = _pair(oracle, arch, ty, 0, n_ctx=96, max_batch=40, mutate=lambda s: [setattr(s, "n_embd", 1024), setattr(s, "n_ff", 2048)])
    nv = spec.n_vocab
    toks = [(i * 29 + 3) % nv for i in range(60)]
    for pos, end in ((0, 20), (20, 60)):
        lg, lo = g.forward(toks[pos:end], pos, True), o.forward(toks[pos:end], pos, True)
        for t in range(end - pos):
            err = max_rel_err(lg[t * nv:(t + 1) * nv], lo[t * nv:(t + 1) * nv])
            assert err < 0.03, f"{arch} {ty}: token {pos + t}: {err}"
