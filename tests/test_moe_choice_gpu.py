"""The choice of experts at its edges: on both sides of the line between rounds of maxima and counted places (four times the chosen ones
against the experts) and of the 64 experts that a wave holds at once; equal logits, NaN, infinities; few and many rows."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
WIDTH = 128


@pytest.mark.parametrize("scoring", [0, 1])
@pytest.mark.parametrize("rows", [1, 17, 64, 65, 100])
@pytest.mark.parametrize("experts,top", [(4, 1), (4, 2), (64, 16), (64, 17), (63, 15), (63, 16), (65, 3), (8, 8)])
def test_choice(experts, top, rows, scoring, width=WIDTH):
    import light_vllm_amd._custom_ops  # noqa: F401
    amd = torch.ops._C_amd
    g = torch.Generator().manual_seed(experts * rows + top)
    # a row's input is a unit vector: its logits are whole numbers of w without rounding, with many equal ones
    z = torch.randint(-3, 4, (rows, experts), generator=g).float()
    w, h, at = torch.zeros((experts + 15) // 16 * 16, width), torch.zeros(rows, width).bfloat16(), torch.arange(rows) * (width // WIDTH)
    w[:experts, at] = z.t()
    h[torch.arange(rows), at] = 1
    bias = torch.zeros(experts)
    if experts > 4 and top + 3 < experts:
        bias[1], bias[2], bias[experts - 1] = float("nan"), float("-inf"), float("-inf")
    ids, weights, *_ = amd.moe_route(h.to(DEV), amd.pack_weight(w.bfloat16().to(DEV)), bias.to(DEV), top, False, True, experts, False, scoring)
    v = (z + bias).nan_to_num(nan=float("-inf"), neginf=float("-inf")).double()
    want = torch.sort(v, dim=1, descending=True, stable=True).indices[:, :top]
    assert torch.equal(ids.cpu().long(), want)
    chosen = v.gather(1, want)
    p = torch.sigmoid(chosen) if scoring else torch.softmax(chosen, -1)
    torch.testing.assert_close(weights.cpu().double(), p, rtol=2e-6, atol=1e-29)  # a few fp32 roundings; -inf weighs 1e-30 a part


@pytest.mark.parametrize("width", [128, 2048, 2560, 4096])
@pytest.mark.parametrize("rows", [33, 48, 49, 64])
@pytest.mark.parametrize("experts,top", [(300, 5), (352, 8)])
def test_choice_in_batches_of_rows(experts, top, rows, width):
    """Logits of 48 rows (300 experts) and of 32 (352) are held at once, the rows behind them come second; sums of 1, 4, 5 and 8 shares."""
    test_choice(experts, top, rows, 0, width)
