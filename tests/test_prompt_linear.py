"""Which kernel takes a prompt's projection with an activation behind it (csrc/prompt_linear.h), on the host: at sizes that were measured,
and what no size may lead to."""
import ctypes
import os
import random
import subprocess

import pytest

from test_prompt_linear_gpu import HALF_TILES

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "light-vllm_amd", "csrc")
SOURCE = r"""
#include "prompt_linear.h"
extern "C" int plan(int rows, int outputs, int k, int act, int row_major, int packed, int* groups, int* nt) {
  const lvllm::PromptLinearPlan p = lvllm::prompt_linear_plan(rows, outputs, k, act, row_major, packed);
  *groups = p.groups;
  *nt = p.nt;
  return p.body;
}
extern "C" int dealt(int rows, int wrows, int k, int act, int* groups) {
  *groups = lvllm::tile_groups(rows);
  return lvllm::dealt_half_tiles(rows, wrows, k, act);
}
"""
GELU, SILU, RELU2, CLAMPED = 1, 2, 3, 4
NONE, WIDE, TILE = 0, 1, 2


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "t.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, str(d / "t.cpp"), "-o", str(d / "t.so")], check=True)
    lib = ctypes.CDLL(str(d / "t.so"))

    def f(rows, outputs, k, act, row_major=True, packed=True):
        g, n = ctypes.c_int(), ctypes.c_int()
        body = lib.plan(rows, outputs, k, act, row_major, packed, ctypes.byref(g), ctypes.byref(n))
        return body, g.value if body == WIDE else n.value
    f.lib = lib
    return f


MEASURED = [  # rows, outputs, k, activation -> body, groups or blocks
    (4875, 14336, 4096, SILU, WIDE, 4), (3000, 14336, 4096, SILU, WIDE, 3), (1000, 14336, 4096, SILU, WIDE, 4), (700, 14336, 4096, SILU, WIDE, 3),
    (300, 14336, 4096, SILU, WIDE, 3), (65, 14336, 4096, SILU, TILE, 2), (1000, 11264, 2048, SILU, TILE, 4), (128, 11264, 2048, SILU, TILE, 2),
    (4096, 5632, 2048, CLAMPED, TILE, 4), (300, 5632, 2048, CLAMPED, TILE, 2), (100, 5632, 2048, CLAMPED, NONE, 0),
    (4096, 8448, 2048, RELU2, WIDE, 3), (1000, 8448, 2048, RELU2, WIDE, 3), (300, 8448, 2048, RELU2, TILE, 2),
    # where the library or the stream product is faster
    (100, 8192, 8192, SILU, NONE, 0), (257, 8192, 8192, SILU, NONE, 0), (700, 4096, 12288, SILU, NONE, 0), (2000, 14336, 8192, CLAMPED, NONE, 0),
    (129, 14336, 4096, SILU, NONE, 0), (89, 18944, 3584, SILU, NONE, 0), (214, 9728, 2560, SILU, NONE, 0), (916, 5136, 3776, RELU2, NONE, 0),
    (128, 16384, 4096, RELU2, NONE, 0), (257, 16384, 4096, RELU2, NONE, 0), (221, 10064, 3456, CLAMPED, NONE, 0), (517, 17184, 1920, GELU, NONE, 0),
    (100, 8448, 2048, RELU2, NONE, 0), (16384, 4096, 1024, GELU, TILE, 4), (1000, 4096, 1024, GELU, TILE, 2), (100, 4096, 1024, GELU, NONE, 0)]


@pytest.mark.parametrize("rows,outputs,k,act,body,size", MEASURED)
def test_measured_sizes(plan, rows, outputs, k, act, body, size):
    got = plan(rows, outputs, k, act)
    assert got[0] == body and (body == NONE or got[1] == size)


@pytest.mark.parametrize("rows,wrows,k,groups,dealt", HALF_TILES)
@pytest.mark.parametrize("act", [GELU, SILU, RELU2, CLAMPED])
def test_half_tiles(plan, rows, wrows, k, act, groups, dealt):
    """The sizes at which test_prompt_linear_gpu.py runs the bodies of half tiles lead there."""
    g = ctypes.c_int()
    assert plan(rows, wrows // 2 if act in (SILU, CLAMPED) else wrows, k, act, False) == (TILE, 2)
    assert bool(plan.lib.dealt(rows, wrows, k, act, ctypes.byref(g))) == (dealt and act != GELU) and g.value == groups


def test_any_size(plan):
    rng = random.Random(0)
    for _ in range(20000):
        rows, outputs, k = rng.randint(1, 40000), rng.choice([8, 16]) * rng.randint(1, 2000), rng.choice([8, 32, 64, 65536]) * rng.randint(1, 128)
        act, row_major, packed = rng.choice([GELU, SILU, RELU2, CLAMPED]), rng.random() < 0.5, rng.random() < 0.5
        body, size = plan(rows, outputs, k, act, row_major, packed)
        if body == WIDE:
            assert row_major and act != GELU and k % 64 == 0 and outputs % 16 == 0 and 2 <= size <= 4
        elif body == TILE:
            assert packed and k % 32 == 0 and outputs % 16 == 0 and size in (2, 4)
        if body != NONE:
            assert rows > 64 and outputs * k * (2 if act in (SILU, CLAMPED) else 1) * 2 < 2 ** 31 and 256 * k * 2 < 2 ** 31
