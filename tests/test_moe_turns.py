"""Every unit of the grouped products has exactly one workgroup, and which products take half blocks of weight rows: csrc/moe_turns.h
on the host, over grids of any size, with a last expert of none to many times the others' size."""
import ctypes
import os
import random
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "light-vllm_amd", "csrc")
SOURCE = r"""
#include <vector>
#include "moe_turns.h"
using namespace lvllm;
// units without a workgroup, and with several; cus: workgroups of an XCD
extern "C" void walk(int units_first, int units_last, int cus, int* missing, int* twice) {
  std::vector<int> first(units_first), last(units_last);
  for (int xcd = 0; xcd < 8; ++xcd)
    for (int cu = 0; cu < cus; ++cu) {
      const TurnUnit u = turn_unit(units_first, units_last, xcd, cu);
      if (u.any) ++(u.last ? last : first).at(u.unit);
    }
  *missing = *twice = 0;
  for (auto* v : {&first, &last})
    for (int n : *v) { *missing += n == 0; *twice += n > 1; }
}
extern "C" long single(long units_first, long units_last) { return unit_workgroups(units_first, units_last); }
extern "C" int half(int rows, long slots, int experts, int first4, int last4, int first2, int last2, int up, int larger) {
  return takes_half_blocks(rows, slots, experts, 128, {first4, last4}, {first2, last2}, up, larger);
}
extern "C" int every(int rows, long slots, int experts, int first4, int last4) {
  return takes_every_height(rows, slots, experts, 128, {first4, last4});
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("turns")
    (d / "t.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-D__host__=", "-D__device__=", "-I", CSRC, str(d / "t.cpp"), "-o",
                    str(d / "t.so")], check=True)
    t = ctypes.CDLL(str(d / "t.so"))
    t.single.restype = ctypes.c_long
    t.half.argtypes = [ctypes.c_int, ctypes.c_long] + [ctypes.c_int] * 7
    t.every.argtypes = [ctypes.c_int, ctypes.c_long] + [ctypes.c_int] * 3
    t.single.argtypes = [ctypes.c_long] * 2
    return t


def walk(lib, first, last, workgroups):
    missing, twice = ctypes.c_int(), ctypes.c_int()
    assert workgroups % 8 == 0 and workgroups > 0
    lib.walk(first, last, workgroups // 8, ctypes.byref(missing), ctypes.byref(twice))
    return missing.value, twice.value


def test_a_unit_a_workgroup(lib):
    """Units up to what the launch was sized for."""
    r = random.Random(2)
    for _ in range(600):
        most_first, most_last = int(2 ** r.uniform(0, 14)), int(2 ** r.uniform(0, 12)) - 1
        fewer = r.randint(0, most_last)
        for first, last in ((most_first, most_last), (r.randint(0, most_first), fewer), (most_first, fewer)):
            assert walk(lib, first, last, lib.single(most_first, most_last)) == (0, 0), (first, last)


# rows, experts taken by a row, experts, their inner size, the shared one's (0: none), width; whether half blocks were ahead, going up (None:
# level) and down
HALF = [(300, 2, 32, 1408, 2816, 2048, None, True), (1000, 2, 32, 1408, 2816, 2048, None, True), (1943, 6, 64, 1408, 2816, 2048, False, False),
        (65, 2, 8, 1408, 2816, 2048, True, True), (420, 2, 8, 1408, 2816, 2048, False, True), (8192, 6, 64, 2816, 2816, 2048, False, False),
        (500, 2, 16, 1408, 0, 2048, False, True), (1000, 2, 16, 1408, 0, 2048, True, False), (1500, 4, 32, 512, 0, 1024, None, False),
        (1500, 2, 16, 512, 0, 1024, True, True), (2000, 2, 16, 512, 0, 1024, None, False), (300, 2, 16, 2816, 2816, 2048, None, False),
        (100, 4, 16, 768, 768, 2048, True, False), (700, 2, 16, 512, 512, 1024, True, True), (1000, 2, 16, 512, 512, 1024, True, True),
        (1000, 2, 8, 512, 0, 2048, True, False), (300, 2, 64, 512, 0, 1024, True, True), (65, 2, 8, 7168, 0, 4096, None, True)]


@pytest.mark.parametrize("rows,top,experts,ff,shared,width,up,down", HALF)
def test_half_blocks(lib, rows, top, experts, ff, shared, width, up, down):
    """Where measurements put the line between half and whole blocks of weight rows (gated experts)."""
    all_experts, slots, last = experts + (shared > 0), rows * (top + (shared > 0)), shared or ff
    blocks = lambda n, nt: -(-n // (4 * nt))
    for is_up, want, tiles in ((1, up, lambda f: f // 8), (0, down, lambda f: width // 16)):
        got = lib.half(rows, slots, all_experts, blocks(tiles(ff), 4), blocks(tiles(last), 4), blocks(tiles(ff), 2), blocks(tiles(last), 2),
                       is_up, last > ff)
        assert want is None or bool(got) == want


@pytest.mark.parametrize("rows,top,experts,ff,shared,up", [
    (4096, 6, 64, 2816, 0, True), (3000, 6, 64, 1408, 2816, True), (8192, 2, 32, 1408, 1408, True), (1943, 6, 64, 1408, 2816, True),
    (2500, 2, 16, 512, 0, False), (1300, 2, 8, 1024, 0, False), (1500, 4, 32, 512, 0, False), (2000, 2, 8, 512, 0, False)])
def test_bodies_of_every_height(lib, rows, top, experts, ff, shared, up):
    """Products going up (gated experts) that power bounds, and those whose launch with more code is slower."""
    blocks = lambda f: -(-f // 128)
    all_experts, slots = experts + (shared > 0), rows * (top + (shared > 0))
    assert bool(lib.every(rows, slots, all_experts, blocks(ff), blocks(shared or ff))) == up
