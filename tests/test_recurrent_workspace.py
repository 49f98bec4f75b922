"""Scratch of the chunked recurrences: what short sequences need beside a longer portion."""
import ctypes
import os

import pytest


@pytest.mark.parametrize("library,name,rows_of", [("hybrid", "recurrent_mix", 1), ("local", "retention", 2)])
@pytest.mark.parametrize("singles,portion", [(255, 45), (400, 40), (255, 300), (31, 5000), (0, 300)])
def test_single_tokens_need_no_segments(library, name, rows_of, singles, portion):
    """States of segments are kept for sequences of more than one: at most two for every 16 rows, however many single tokens there are."""
    import light_vllm_amd
    lib = ctypes.CDLL(os.path.join(os.path.dirname(light_vllm_amd.__file__), "lib", f"liblvllm_{library}.so"))
    need = getattr(lib, f"lvllm_{name}_workspace_bytes")
    need.restype, heads, dk, dv = ctypes.c_int64, 8, 128, 128
    rows = singles + portion
    got = need(rows, singles + 1, heads, dk, dv, portion)
    own = 4 * rows_of * rows * heads * dk   # decays, or rotated queries and keys
    state = 4 * heads * (dk * dv + dk)
    assert own <= got <= own + (2 * (rows // 16) + 1) * state
