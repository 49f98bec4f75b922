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
extern "C" int plan(int rows, int n, int k, int gelu, int slabs, int* out) {
  const ProductPlan p = prompt_product_plan(rows, n, k, gelu, slabs);
  out[0] = p.body; out[1] = p.size; out[2] = p.nt; out[3] = p.shares;
  if (p.body == kProductNone) return 0;
  out[4] = product_share(p, k);
  out[5] = product_plan_valid(p, k);
  out[6] = (int)product_units(p, rows, n);
  return 1;
}
"""
NONE, SHORT, TILE = 0, 1, 2


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "t.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, str(d / "t.cpp"), "-o", str(d / "t.so")], check=True)
    lib = ctypes.CDLL(str(d / "t.so"))

    def f(rows, n, k, gelu=False, slabs=False):
        out = (ctypes.c_int * 7)()
        lib.plan(rows, n, k, gelu, slabs, out)
        return list(out)
    return f


MEASURED = [  # rows, n, k, slabs -> this kernel's, or the library's
    (300, 4096, 14336, True, True), (1000, 4096, 14336, True, True), (100, 4096, 14336, True, True), (300, 4096, 4096, True, True),
    (300, 1024, 4096, True, True), (1000, 3072, 1024, False, True), (100, 1024, 1024, False, True), (300, 2048, 8448, True, True),
    (4096, 4096, 14336, True, False), (6000, 4096, 4096, True, False), (8192, 3072, 1024, False, False), (300, 4096, 4096, False, False),
    (64, 4096, 4096, True, False), (8193, 1024, 256, True, False), (300, 4096, 14336, False, False), (300, 4100, 4096, True, False),
    (300, 4096, 4128, True, False)]


@pytest.mark.parametrize("rows,n,k,slabs,own", MEASURED)
def test_measured_sizes(plan, rows, n, k, slabs, own):
    assert (plan(rows, n, k, slabs=slabs)[0] != NONE) == own


def test_any_size(plan):
    rng = random.Random(0)
    taken = set()
    for _ in range(20000):
        rows, n, k = int(2 ** rng.uniform(0, 15)), rng.choice([8, 16, 16, 16]) * rng.randint(1, 1000), rng.choice([8, 32, 64, 64, 64]) * rng.randint(1, 256)
        gelu, slabs = rng.random() < 0.3, rng.random() < 0.5
        body, size, nt, shares, share, valid, units = plan(rows, n, k, gelu, slabs)
        if body == NONE:
            continue
        taken.add((body, size if body == SHORT else 0, nt))
        assert valid and 64 < rows <= 8192 and n % 16 == 0 and k % 64 == 0
        assert shares == 1 or (slabs and shares <= 8)
        assert (shares - 1) * share < k // 32 <= shares * share  # every share has steps, and all steps a share
        assert 0 < units <= 512 and not (gelu and body == TILE)
        assert size % 16 == 0 and size <= (64 if body == SHORT else 128)
    assert taken == {(SHORT, 16, 4), (SHORT, 32, 4), (SHORT, 48, 4), (SHORT, 64, 4), (SHORT, 32, 8), (TILE, 0, 2), (TILE, 0, 4)}, taken
