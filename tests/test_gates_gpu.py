"""Sigmoids of gates and activations are those of 32-bit results everywhere: what leaves in bfloat16 is bit for bit the rounded float32
result of the same inputs, and the matrix-core mixtures' activation that of the plain body.  Gates far below zero and the largest ones
among the inputs."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
F32, BF16 = torch.float32, torch.bfloat16


@pytest.fixture(scope="module")
def amd():
    import light_vllm_amd._custom_ops  # noqa: F401
    return torch.ops._C_amd


def rand(*shape, seed, scale=1.0):
    return (scale * torch.randn(*shape, generator=torch.Generator().manual_seed(seed))).bfloat16()


def gates(*shape, seed):
    """Values of every size, some of them where e^-z is near the end of the range of floats."""
    z = rand(*shape, seed=seed, scale=4.0)
    z.view(-1)[::7] = rand(z.view(-1)[::7].numel(), seed=seed + 1, scale=60.0)
    z.view(-1)[::501] = -3e38
    return z


def i32(*v):
    return torch.tensor(v, dtype=torch.int32, device=DEV)


def rounded_alike(out):
    a, b = out[BF16], out[F32].bfloat16()
    assert ((a == b) | (a.isnan() & b.isnan())).all()  # (sums beyond the range of floats have a gate of 0 times infinity)


def test_short_convolution(amd):
    rows, channels, taps = 512, 1024, 4
    x, w, out = gates(rows, channels, seed=1), torch.randn(taps, channels, generator=torch.Generator().manual_seed(2)).to(DEV), {}
    for dtype in (F32, BF16):
        state = torch.zeros(1, taps, channels, device=DEV)
        out[dtype] = amd.short_conv(x.to(dtype).to(DEV), w, state, i32(0), i32(0, rows), i32(rows), rows)
    rounded_alike(out)


def test_head_norm_gate(amd):
    rows, heads, dim = 512, 8, 128
    o, out = torch.randn(rows, heads, dim, generator=torch.Generator().manual_seed(3)).to(DEV), {}
    z, weight = gates(rows, heads * dim, seed=4), 4 * torch.randn(heads * dim, generator=torch.Generator().manual_seed(5)).to(DEV)
    for dtype in (F32, BF16):
        out[dtype] = torch.empty(rows, heads * dim, dtype=dtype, device=DEV)
        amd.head_norm_gate(out[dtype], o, z.to(dtype).to(DEV), weight, 1e-5, 0.7)
    rounded_alike(out)


def test_retention(amd):
    rows, heads, dim = 2048, 4, 128
    q, k, v = (rand(rows, heads * dim, seed=6 + i) for i in range(3))
    z, out = gates(rows, heads * dim, seed=9), {}
    decay = torch.tensor([0.999, 0.99, 0.9, 0.5], dtype=torch.float64)
    turns = torch.zeros(0, dtype=torch.float64, device=DEV)
    for dtype in (F32, BF16):
        out[dtype] = torch.empty(rows, heads * dim, dtype=dtype, device=DEV)
        t = [a.to(dtype).to(DEV) for a in (q, k, v, z)]
        amd.retention(out[dtype], *t[:3], torch.arange(rows, device=DEV), turns, torch.stack([decay, decay.log()]).float().to(DEV),
                      dim ** -0.5, t[3], None, 1e-5, 1.0, torch.zeros(1, heads, dim, dim, device=DEV), i32(0), i32(0, rows), i32(rows),
                      rows)
    rounded_alike(out)


@pytest.mark.parametrize("act", ["clamped", "silu"])
@pytest.mark.parametrize("rows,experts", [(40, 2), (300, 8), (1200, 4)], ids=["decode", "few slots", "many slots"])
def test_mixtures(amd, rows, experts, act):
    """Gate and up rows that pick one input each: both bodies' products are exact."""
    from light_vllm_amd.engine.moe import ACTIVATIONS, interleave_16
    ff, width = 512, 1024 + 32
    h = gates(rows, width, seed=12)
    of_row = torch.arange(rows) % experts
    h[:, 1024:] = 0
    h[:, 1024:1024 + experts] = torch.nn.functional.one_hot(of_row, experts).bfloat16()
    router = torch.zeros(16, width, dtype=BF16)
    router[:experts, 1024:1024 + experts] = 8 * torch.eye(experts)
    one = interleave_16(torch.eye(ff, width), torch.eye(2 * ff, width)[ff:]).bfloat16().to(DEV)
    ffs, limits = torch.full((experts,), ff, dtype=torch.int32, device=DEV), torch.full((experts,), 7.0, device=DEV)
    at = torch.arange(experts, device=DEV) * one.numel()
    got = []
    for packed in (False, True):
        r = amd.pack_weight(router.to(DEV)) if packed else router[:experts].to(DEV)
        ids, _, offsets, token, slots, tiles, _ = amd.moe_route(h.to(DEV), r, None, 1, False, packed, experts, False, 1)
        assert torch.equal(ids[:, 0].long().cpu(), of_row)
        w = (amd.pack_weight(one) if packed else one).reshape(-1).repeat(experts)
        a = amd.moe_experts(h.to(DEV), w, at, ffs, limits, offsets, token, tiles, rows, width, ff, ff, ff, True, packed, None,
                            ACTIVATIONS[act])
        got.append(a[slots[:, 0].long()])
    assert torch.equal(*got)
