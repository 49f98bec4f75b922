"""Which body reads the rows of whole sequences in place (csrc/dense_rule.h), on the host."""
import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "light-vllm_amd", "csrc")
SOURCE = r"""
#include "dense_rule.h"
extern "C" int body(int seqs, int tokens, int longest, int heads, int kv_heads, int causal) {
  return lvllm::dense_body(seqs, tokens, longest, heads, kv_heads, causal);
}
"""
WAVES, COLUMNS_128, COLUMNS_256 = 0, 1, 2


@pytest.fixture(scope="module")
def body(tmp_path_factory):
    d = tmp_path_factory.mktemp("rule")
    (d / "t.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, str(d / "t.cpp"), "-o", str(d / "t.so")], check=True)
    f = ctypes.CDLL(str(d / "t.so")).body
    return lambda lens, heads, kv_heads, causal: f(len(lens), sum(lens), max(lens), heads, kv_heads, causal)


# where the bodies for lengths alike took 1.05 to 1.7 times as long
@pytest.mark.parametrize("lens,heads,kv_heads,causal", [
    ([2000] + [100] * 8, 16, 16, 0), ([2000] + [50] * 20, 12, 12, 0), ([8000] + [300] * 4, 6, 3, 0), ([4000] + [50] * 20, 16, 16, 1),
    ([8000] + [50] * 20, 12, 12, 1), ([512 - 32 * i for i in range(16)], 16, 16, 0), ([1000] * 3, 16, 2, 0), ([512] * 8, 16, 16, 1),
    ([512] * 2, 32, 8, 1), ([512] + [64] * 40, 16, 16, 1)])
def test_lengths_that_differ(body, lens, heads, kv_heads, causal):
    assert body(lens, heads, kv_heads, causal) == WAVES


@pytest.mark.parametrize("lens,heads,kv_heads,causal,want", [
    ([512] * 32, 16, 16, 0, COLUMNS_256), ([2048] * 8, 16, 16, 0, COLUMNS_256), ([8192], 16, 2, 0, COLUMNS_256), ([400] * 24, 16, 16, 0, COLUMNS_128),
    ([128] * 128, 16, 16, 0, COLUMNS_128), ([512] * 4, 16, 16, 0, COLUMNS_128), ([2048], 16, 16, 0, COLUMNS_128), ([512] * 32, 16, 16, 1, COLUMNS_128),
    ([4096] * 2, 16, 16, 1, COLUMNS_128), ([8000 - 500 * i for i in range(16)], 16, 16, 1, COLUMNS_256), ([100] * 10, 64, 1, 1, COLUMNS_128),
    ([2000 - 125 * i for i in range(16)], 16, 16, 1, COLUMNS_128), ([512 - 8 * i for i in range(32)], 12, 12, 0, COLUMNS_256), ([512 - 8 * i for i in range(32)], 10, 10, 0, COLUMNS_128)])
def test_lengths_alike(body, lens, heads, kv_heads, causal, want):
    assert body(lens, heads, kv_heads, causal) == want
