"""Grouped products of prompts at the edges of their tiles: experts with 0, 1, 63 .. 65 and 127 .. 129 rows, inner sizes from one k-step on
and of unequal length, weights on what an expert reads; both bodies (few and many rows an expert)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
# rows of every expert, inner sizes (multiples of 32), width; below and above 45 rows an expert
FEW = ([0, 1, 63, 64, 65, 0, 17, 30], [32, 64, 96, 128, 160, 192, 224, 704], 352)
MANY = ([129, 128, 127, 1, 0, 65, 300], [32, 96, 160, 224, 288, 352, 736], 288)


@pytest.fixture(scope="module")
def amd():
    import light_vllm_amd._custom_ops  # noqa: F401
    return torch.ops._C_amd


def rand(*shape, seed):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).bfloat16()


@pytest.mark.parametrize("weigh", [False, True])
@pytest.mark.parametrize("act", ["clamped", "silu", "relu_squared"])
@pytest.mark.parametrize("counts,ff,width", [FEW, MANY], ids=["few", "many"])
def test_products(amd, counts, ff, width, act, weigh):
    from light_vllm_amd.engine.moe import ACTIVATIONS, interleave_16
    experts, rows, limit, gated = len(counts), sum(counts), 1.1, act != "relu_squared"
    of_row = torch.repeat_interleave(torch.arange(experts), torch.tensor(counts))[torch.randperm(rows, generator=torch.Generator().manual_seed(1))]
    h = 0.5 * rand(rows, width, seed=2)
    h[:, :experts] = 0.25 * torch.nn.functional.one_hot(of_row, experts).bfloat16()
    router = torch.zeros(16, width, dtype=torch.bfloat16)  # the expert of a row is the column that it marks
    router[:experts, :experts] = 8 * torch.eye(experts)
    gate, up = ([rand(n, width, seed=s + i) * width ** -0.5 for i, n in enumerate(ff)] for s in (10, 30))
    down = [rand(width, n, seed=50 + i) * n ** -0.5 for i, n in enumerate(ff)]

    def packed(parts):
        parts = [amd.pack_weight(p.contiguous().to(DEV)).reshape(-1) for p in parts]
        at = torch.tensor([0] + [p.numel() for p in parts[:-1]]).cumsum(0).to(DEV)
        return torch.cat(parts), at
    hd = h.to(DEV)
    ids, weights, offsets, token, slots, tiles, by_slot = amd.moe_route(hd, amd.pack_weight(router.to(DEV)), None, 1, False, True, experts,
                                                                       False, 1, weigh)
    assert torch.equal(ids[:, 0].long().cpu(), of_row)
    sizes = rows, width, max(ff), max(ff[:-1]), ff[-1]
    ffs, limits = torch.tensor(ff, dtype=torch.int32, device=DEV), torch.full((experts,), limit, device=DEV)
    w_up, up_at = packed([interleave_16(g, u) if gated else u for g, u in zip(gate, up)])
    w_down, down_at = packed(down)
    a = amd.moe_experts(hd, w_up, up_at, ffs, limits, offsets, token, tiles, *sizes, True, True, by_slot if weigh else None, ACTIVATIONS[act])
    y = amd.moe_experts(a, w_down, down_at, ffs, None, offsets, token, tiles, *sizes, False, True)
    a, y, slots, w = a.double().cpu(), y.double().cpu(), slots[:, 0].long().cpu(), weights[:, 0].double().cpu()
    for e in range(experts):
        r = (of_row == e).nonzero()[:, 0]
        x = h[r].double() * (w[r][:, None] if weigh else 1)
        g, u = x @ gate[e].double().T, x @ up[e].double().T
        if act == "clamped":
            g, u = g.clamp(max=limit), u.clamp(-limit, limit)
            want = g * torch.sigmoid(1.702 * g) * (u + 1)
        else:
            want = g * torch.sigmoid(g) * u if gated else u.clamp(min=0).square()
        # one rounding to 8 bits behind fp32 sums of at most 736 products of values around 1
        got = a[slots[r], :ff[e]]
        assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + 2e-5).all(), (e, (got - want).abs().max())
        got, want = y[slots[r]], got @ down[e].double().T
        assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + 2e-5).all(), (e, (got - want).abs().max())
