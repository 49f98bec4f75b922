"""Which kernel takes a prompt's product (csrc/prompt_product.h), on the host: at sizes that were measured, and what no size may lead to."""
import ctypes
import os
import random
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "light-vllm_amd", "csrc")
SOURCE = r"""
#include "prompt_product.h"
using namespace lvllm;
extern "C" int plan(int rows, int n, int k, int gelu, int sums, int* out) {
  const ProductPlan p = prompt_product_plan(rows, n, k, gelu, sums);
  out[0] = p.size; out[1] = p.nt; out[2] = p.shares;
  if (p.size == 0) return 0;
  out[3] = product_share(p, k);
  out[4] = product_plan_valid(p, k);
  out[5] = (int)product_units(p, rows, n);
  return 1;
}
"""
ANY, SLABS, ORDERED = 0, 1, 2


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "t.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, str(d / "t.cpp"), "-o", str(d / "t.so")], check=True)
    lib = ctypes.CDLL(str(d / "t.so"))

    def f(rows, n, k, gelu=False, sums=ANY):
        out = (ctypes.c_int * 6)()
        lib.plan(rows, n, k, gelu, sums, out)
        return list(out)
    return f


MEASURED = [  # rows, n, k, sums -> this kernel's, or the library's
    (300, 4096, 14336, SLABS, True), (700, 4096, 14336, SLABS, True), (100, 4096, 14336, SLABS, True), (300, 4096, 4096, SLABS, True),
    (300, 1024, 4096, SLABS, True), (1000, 3072, 1024, ANY, True), (100, 1024, 1024, ANY, True), (300, 2048, 8448, SLABS, True),
    (300, 2048, 2048, ORDERED, True), (300, 7680, 2048, ORDERED, True), (300, 2048, 5632, ORDERED, True), (800, 3072, 2048, ORDERED, True),
    (4096, 4096, 14336, SLABS, False), (6000, 4096, 4096, SLABS, False), (8192, 3072, 1024, ANY, False), (100, 2048, 11264, ORDERED, False),
    (64, 4096, 4096, SLABS, False), (8193, 1024, 256, SLABS, False), (2000, 7680, 2048, ORDERED, False), (300, 4100, 4096, SLABS, False),
    (300, 4096, 4128, SLABS, False)]


@pytest.mark.parametrize("rows,n,k,sums,own", MEASURED)
def test_measured_sizes(plan, rows, n, k, sums, own):
    assert (plan(rows, n, k, sums=sums)[0] != 0) == own


GELU = [  # rows, n, k -> this kernel's, or tiles with GELU behind them and the library's
    (65, 4096, 1024, True), (300, 4096, 1024, True), (600, 4096, 1024, True), (1200, 4096, 1024, True), (1500, 4096, 1024, True),
    (800, 4096, 1024, False), (1000, 4096, 1024, False), (2000, 4096, 1024, False), (1000, 3072, 768, False), (1500, 5120, 1280, False),
    (500, 8192, 2048, False), (600, 8192, 2048, True), (1171, 3072, 896, False), (716, 5248, 320, False), (1978, 896, 384, True)]


@pytest.mark.parametrize("rows,n,k,own", GELU)
def test_measured_sizes_with_gelu(plan, rows, n, k, own):
    assert (plan(rows, n, k, gelu=True)[0] != 0) == own


def test_any_size(plan):
    rng = random.Random(0)
    taken = set()
    for _ in range(20000):
        rows, n, k = int(2 ** rng.uniform(0, 15)), rng.choice([8, 16, 16, 16]) * rng.randint(1, 1000), rng.choice([8, 32, 64, 64, 64]) * rng.randint(1, 256)
        gelu, sums = rng.random() < 0.3, rng.choice([ANY, SLABS, ORDERED])
        size, nt, shares, share, valid, units = plan(rows, n, k, gelu, sums)
        if size == 0:
            continue
        taken.add(nt)
        assert valid and 64 < rows <= 8192 and n % 16 == 0 and k % 64 == 0
        assert shares == 1 or (sums == SLABS and not gelu and shares <= 8)
        assert (shares - 1) * share < k // 32 <= shares * share and share % 2 == 0  # every share has steps, and all steps a share
        assert 0 < units <= 512 and not (gelu and nt == 4)
        assert size % 16 == 0 and size <= (96 if nt == 1 else 128)
    assert taken == {1, 2, 4}
