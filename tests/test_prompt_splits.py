"""The KV splits of prompt attention launches (csrc/attn_splits.hpp), compiled for the host."""
import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rust_interference_engine_amd", "csrc")


@pytest.fixture(scope="module")
def splits(tmp_path_factory):
    d = tmp_path_factory.mktemp("splits")
    (d / "s.cpp").write_text(f'#include "{CSRC}/attn_splits.hpp"\n'
                             'extern "C" int splits(int w, int t, int q8_0) { return rie::prompt_kv_splits(w, t, q8_0 != 0); }\n')
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-o", str(d / "s.so"), str(d / "s.cpp")], check=True)
    return ctypes.CDLL(str(d / "s.so")).splits


def test_few_tokens_deep_in_a_q8_0_cache_have_the_per_token_kernels_ranges(splits):
    assert splits(8, 376, 1) == 32 and splits(4, 376, 1) == 32


@pytest.mark.parametrize("q8_0", [0, 1])
def test_splits_over_all_grids(splits, q8_0):
    for wgs in (1, 2, 5, 8, 15, 16, 31, 32, 63, 64, 65, 128, 255, 256, 511, 512, 5000):
        last = 0
        for tiles in (1, 2, 3, 4, 15, 16, 31, 32, 63, 100, 512, 4096):
            s = splits(wgs, tiles, q8_0)
            assert 1 <= s <= (32 if q8_0 else 16)  # a partial buffer holds 32 per token and head
            assert s == 1 or (tiles // s >= 2 and s * wgs <= 512), (wgs, tiles, s)
            assert s >= last, (wgs, tiles)  # longer rows never take fewer
            last = s
