"""Attention of prompts over unequal caches: scores are rounded once, whatever the sign of the scale -- queries and scale with the other
sign give the same result, bit for bit (queries and keys are eighths, so that their products are exact).  Whole prompts and portions
behind a context, windows, one and two maps."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def i32(v):
    return torch.tensor(v, dtype=torch.int32, device=DEV)


@pytest.mark.parametrize("window", [0, 70])
@pytest.mark.parametrize("dim,vdim,maps", [(128, 64, 1), (128, 128, 1), (192, 128, 1), (128, 128, 2)])
def test_sign_of_the_scale(dim, vdim, maps, window):
    import light_vllm_amd._custom_ops  # noqa: F401
    heads, kv_heads, seqs = 16, 4, [(300, 0), (77, 200)]
    g = torch.Generator().manual_seed(dim + maps)
    eighths = lambda *s: (torch.randint(-16, 17, s, generator=g) / 8).bfloat16().to(DEV)
    blocks = [(n + c + 15) // 16 for n, c in seqs]
    kc, vc = eighths(sum(blocks), kv_heads, dim // 8, 16, 8), eighths(sum(blocks), kv_heads, vdim, 16)
    tables = i32([list(range(blocks[0])), list(range(blocks[0], sum(blocks))) + [0] * (blocks[0] - blocks[1])])
    starts, lens = i32([0, 300, 377]), i32([n + c for n, c in seqs])
    q, out = eighths(377, heads, dim), []
    for sign in (1, -1):
        o = torch.zeros(377, heads * vdim, dtype=torch.bfloat16, device=DEV)
        torch.ops._C_amd.head_attention(o, sign * q, kc, vc, tables, lens, starts, None, vdim, sign * 0.3, 1.0, 300, 300, window, 1, 0, 0,
                                        0.0, None, maps, 0.4, 1e-5)
        out.append(o)
    assert bool(out[0].isfinite().all()) and bool(out[0].any(1).all())
    assert torch.equal(*out)
