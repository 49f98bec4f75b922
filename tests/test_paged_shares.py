"""Shares that paged decode attention cuts contexts into (csrc/paged_shares.h), on the host."""
import ctypes
import os
import random
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "light-vllm_amd", "csrc")
SOURCE = r"""
#include "paged_shares.h"
extern "C" int shares(int seqs, int heads, int kv_heads, int longest, int slots, int mfma, int fp8) {
  return lvllm::paged_shares(seqs, heads, kv_heads, longest, slots, mfma, fp8);
}
"""


@pytest.fixture(scope="module")
def shares(tmp_path_factory):
    d = tmp_path_factory.mktemp("shares")
    (d / "t.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, str(d / "t.cpp"), "-o", str(d / "t.so")], check=True)
    return ctypes.CDLL(str(d / "t.so")).shares


def test_one_long_context_among_short_ones_is_cut(shares):
    """The lengths are not known where the shares are chosen: beyond 1024 tokens one context may be the launch, and as many shares as give eight
    waves a CU are taken."""
    for seqs, want in ((1, 32), (6, 6), (9, 4), (12, 3), (17, 2), (24, 2), (31, 2), (32, 1)):
        for longest in (1025, 2000, 16000, 30000):
            slots = (longest + 511) // 512
            assert shares(seqs, 32, 8, longest, slots, 1, 0) == min(want, slots)


def test_any_size(shares):
    rng = random.Random(0)
    for _ in range(20000):
        kv = rng.choice([1, 2, 4, 8, 32])
        heads, seqs, longest = kv * rng.choice([1, 4, 7, 16, 20]), rng.randint(1, 300), rng.randint(1, 20000)
        slots, mfma, fp8 = (longest + 511) // 512 + rng.choice([0, 0, 7]), rng.random() < 0.8, rng.random() < 0.3
        n, pairs = shares(seqs, heads, kv, longest, slots, mfma, fp8), seqs * kv * ((heads // kv + 15) // 16) if mfma else seqs * heads
        if mfma and not fp8 and pairs > 128 and longest <= 1024:
            assert n == 1
        else:
            assert n == max(1, min(-(-2048 // (8 * pairs)) if mfma else -(-1024 // pairs), slots, -(-longest // 16) // 4))
