"""Shares that decode steps of the softmax heads cut keys into, by the workspace that they ask for (csrc/head_attention.hip), on the host."""
import ctypes
import os

import pytest
import torch  # noqa: F401  (its HIP runtime is the one that the library uses)


class Options(ctypes.Structure):
    _fields_ = [(n, ctypes.c_int) for n in ("window", "chunk", "keep_first", "maps", "min_query_len")] + \
               [(n, ctypes.c_float) for n in ("softcap", "map_weight", "map_eps")] + [("sink", ctypes.c_void_p)]


@pytest.fixture(scope="module")
def shares():
    import light_vllm_amd
    lib = ctypes.CDLL(os.path.join(os.path.dirname(light_vllm_amd.__file__), "lib", "liblvllm_heads.so"))
    lib.lvllm_head_attention_workspace_bytes.restype = ctypes.c_int64

    def f(seqs, heads, kv_heads, kpad, vpad, keys, **options):
        o = Options(maps=1, **options)
        n = lib.lvllm_head_attention_workspace_bytes(seqs, seqs, heads, kv_heads, kpad, vpad, 16, keys, ctypes.byref(o), 2)
        return n // (seqs * heads * (vpad + 2) * 4) or 1
    return f


@pytest.mark.parametrize("kpad,vpad", [(128, 64), (128, 128), (64, 256), (192, 192), (192, 256), (256, 192)])
def test_short_walks_are_not_cut(shares, kpad, vpad):
    for seqs in (1, 8, 24):
        assert [shares(seqs, 16, 4, kpad, vpad, keys) for keys in (100, 300, 512, 513)] == [1, 1, 1, 3]
        assert shares(seqs, 16, 4, kpad, vpad, 20000, window=400) == 1


def test_walks_of_wide_heads_are(shares):
    for seqs in (1, 8, 24):
        assert [shares(seqs, 16, 1, 256, 256, keys) for keys in (100, 256, 257, 300, 512, 513)] == [1, 1, 2, 2, 2, 3]
