"""Grouped products at the edges of their tiles: experts with 0, 1, 63 .. 65 and 127 .. 129 rows, inner sizes from one k-step on
and of unequal length, weights on what an expert reads; few and many rows an expert, tiles of 16 slots and of up to 128."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
# rows of every expert, inner sizes (multiples of 32), width; few and many rows an expert
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
    router = torch.zeros(-(-experts // 16) * 16, width, dtype=torch.bfloat16)  # the expert of a row is the column that it marks
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


@pytest.mark.parametrize("act", ["clamped", "relu_squared"])
@pytest.mark.parametrize("width", [64, 2400])
@pytest.mark.parametrize("counts,full", [([64, 0, 0, 0], True), ([0, 48, 16, 0], True), ([0, 0, 15, 48], True), ([33, 1, 30, 0], False),
                                         ([49, 1, 1, 1], False), ([0, 32, 0, 31], True)], ids=lambda v: "-".join(map(str, v)) if isinstance(v, list) else "")
def test_products_of_few_rows(amd, counts, full, width, act):
    """Up to 64 rows, tiles of 16: experts of one to four tiles.  Going up, those of three and more among full tiles read their weights
    by way of the L2 where there are workgroups for whole units, all others past it."""
    tiles = sum(-(-n // 16) for n in counts)
    assert (sum(counts) >= 14 * tiles) == full
    ff = 4480 if act == "clamped" else 8320  # a fourth of its units, for each of 8 tiles that there may be, is more than 512
    test_products(amd, counts, [ff, 96, 1408, 352], width, act, True)


@pytest.mark.parametrize("act", ["clamped", "relu_squared"])
@pytest.mark.parametrize("ff", [160, 8320, 20480], ids=["half blocks", "whole blocks", "bodies of every height"])
@pytest.mark.parametrize("tiles", [1, 2], ids=["single tiles", "two tiles"])
def test_tiles_of_every_height(amd, tiles, ff, act):
    """Tiles of 65 to 128 slots in groups of 16, at both ends of each height."""
    heights = [65, 80, 81, 96, 97, 112, 113]
    test_products(amd, [tiles * n for n in heights], [ff] * 6 + [ff + 32], 160, act, False)


@pytest.mark.parametrize("tiles", [1, 2], ids=["single tiles", "two tiles"])
def test_tiles_of_every_height_going_down(amd, tiles):
    """The same where the products going down have a body for each height (70 experts of 10 blocks)."""
    test_products(amd, [tiles * n for n in [65, 80, 81, 96, 97, 112, 113]] * 10, [96] * 70, 2400, "clamped", False)


@pytest.mark.parametrize("act", [0, 2], ids=["clamped", "relu_squared"])
@pytest.mark.parametrize("copies", [1, 70], ids=["half blocks", "whole blocks"])
def test_blocks_of_weight_rows(amd, copies, act):
    """Blocks of 128 and of 256 weight rows a workgroup (few and many units), at their edges: inner sizes around 128 and 256 outputs, walks of
    1 to 12 k-steps around the steps under way (8 and 4), experts with one tile of slots (weights past the caches) and with several."""
    g, gated = torch.Generator(device=DEV).manual_seed(copies), act == 0
    counts, ff, width = [129, 128, 127, 1, 0, 65] * copies, [32, 96, 128, 160, 288, 384] * copies, 288
    experts, rows, top = len(counts), sum(counts), 1
    # units of whole blocks, slots spread evenly: far from the lines between half and whole ones
    units = experts * -(-rows // (128 * experts)) * -(-384 // (128 if gated else 256)) + -(-rows // 128) * -(-384 // (128 if gated else 256))
    assert (units > 384) == (copies > 1)
    rand = lambda *s: torch.randn(*s, generator=g, device=DEV).bfloat16()
    of_row = torch.repeat_interleave(torch.arange(experts, device=DEV), torch.tensor(counts, device=DEV))
    of_row = of_row[torch.randperm(rows, generator=g, device=DEV)]
    # two whole numbers name an expert: 2 a x - a^2 + 2 b y - b^2 is largest at (x, y) = (a, b), and exact
    marks = torch.zeros(experts, width, device=DEV)
    e = torch.arange(experts, device=DEV)
    marks[:, 0], marks[:, 1], marks[:, 2] = 2 * (e // 21), 2 * (e % 21), -((e // 21) ** 2 + (e % 21) ** 2)
    h = torch.zeros(rows, width, device=DEV)
    h[:, 0], h[:, 1], h[:, 2] = of_row // 21, of_row % 21, 1
    assert bool((marks.bfloat16().float() == marks)[:, :2].all())
    x = 0.5 * rand(rows, width)
    hi = marks[:, 2].bfloat16().float()
    marks[:, 3], marks[:, 2], h[:, 3] = marks[:, 2] - hi, hi, 1  # (a square in two parts of 8 bits)
    router = torch.nn.functional.pad(marks, (0, 0, 0, -experts % 16)).bfloat16()
    ids, _, offsets, token, slots, tiles, _ = amd.moe_route(h.bfloat16(), amd.pack_weight(router), None, top, False, True, experts, False, 1)
    assert torch.equal(ids[:, 0].long(), of_row)
    from light_vllm_amd.engine.moe import interleave_16
    gate, up = ([rand(n, width) * width ** -0.5 for n in ff] for _ in "gu")
    down = [rand(width, n) * n ** -0.5 for n in ff]

    def packed(parts):
        parts = [amd.pack_weight(p.contiguous()).reshape(-1) for p in parts]
        return torch.cat(parts), torch.tensor([0] + [p.numel() for p in parts[:-1]]).cumsum(0).to(DEV)
    sizes = rows, width, max(ff), max(ff[:-1]), ff[-1]
    ffs, limits = torch.tensor(ff, dtype=torch.int32, device=DEV), torch.full((experts,), 1.1, device=DEV)
    w_up, up_at = packed([interleave_16(a, b) if gated else b for a, b in zip(gate, up)])
    w_down, down_at = packed(down)
    a = amd.moe_experts(x, w_up, up_at, ffs, limits, offsets, token, tiles, *sizes, True, True, None, act)
    y = amd.moe_experts(a, w_down, down_at, ffs, None, offsets, token, tiles, *sizes, False, True)
    for i in [*range(min(experts, 24)), *range(max(experts - 12, 24), experts)]:
        r = (of_row == i).nonzero()[:, 0]
        s, u = slots[r, 0].long(), x[r].double() @ up[i].double().T.contiguous()
        if gated:
            p = (x[r].double() @ gate[i].double().T.contiguous()).clamp(max=1.1)
            want = p * torch.sigmoid(1.702 * p) * (u.clamp(-1.1, 1.1) + 1)
        else:
            want = u.clamp(min=0).square()
        got = a[s, :ff[i]].double()
        # one rounding to 8 bits behind fp32 sums of at most 384 products of values around 1
        assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + 2e-5).all(), (i, (got - want).abs().max())
        want = got @ down[i].double().T.contiguous()
        assert ((y[s].double() - want).abs() <= 2.0 ** -8 * want.abs() + 2e-5).all(), (i, (y[s] - want).abs().max())


@pytest.mark.parametrize("act,weigh", [("clamped", False), ("silu", True), ("relu_squared", True)])
@pytest.mark.parametrize("width", [4096, 224, 64])
def test_few_slots_an_expert_and_a_large_shared_one(amd, width, act, weigh):
    """Single tiles of few slots, walks of 1 to 12 k-steps going down, and a shared expert of eleven times the others' size, whose
    units come first: its walks have 128 k-steps and its tiles are several."""
    from light_vllm_amd.engine.moe import ACTIVATIONS, interleave_16
    g, gated, experts, limit = torch.Generator(device=DEV).manual_seed(width), act != "relu_squared", 40, 1.1
    counts = [0, 1, 64, 65, 17, 30, 2, 63, 16, 33] * 2 + [7, 20, 11, 9] * 5
    ff = ([384, 32, 64, 160, 192, 96, 256, 384, 128, 352] * 4)[:experts] + [4096]
    rows = sum(counts)
    assert len(counts) == experts and max(counts) < 128 and 64 < rows
    rand = lambda *s: torch.randn(*s, generator=g, device=DEV).bfloat16()
    of_row = torch.repeat_interleave(torch.arange(experts, device=DEV), torch.tensor(counts, device=DEV))
    of_row = of_row[torch.randperm(rows, generator=g, device=DEV)]
    h = 0.5 * rand(rows, width)
    h[:, :experts] = 0.25 * torch.nn.functional.one_hot(of_row, experts).bfloat16()
    router = torch.zeros(48, width, dtype=torch.bfloat16, device=DEV)
    router[:experts, :experts] = 8 * torch.eye(experts)
    gate, up = ([rand(n, width) * width ** -0.5 for n in ff] for _ in "gu")
    down = [rand(width, n) * n ** -0.5 for n in ff]

    def packed(parts):
        parts = [amd.pack_weight(p.contiguous()).reshape(-1) for p in parts]
        return torch.cat(parts), torch.tensor([0] + [p.numel() for p in parts[:-1]]).cumsum(0).to(DEV)
    ids, weights, offsets, token, slots, tiles, by_slot = amd.moe_route(h, amd.pack_weight(router), None, 1, True, True, experts, False, 1,
                                                                        weigh)
    assert torch.equal(ids[:, 0].long(), of_row) and bool((ids[:, 1] == experts).all())
    sizes = rows, width, max(ff), max(ff[:-1]), ff[-1]
    ffs, limits = torch.tensor(ff, dtype=torch.int32, device=DEV), torch.full((experts + 1,), limit, device=DEV)
    w_up, up_at = packed([interleave_16(a, b) if gated else b for a, b in zip(gate, up)])
    w_down, down_at = packed(down)
    a = amd.moe_experts(h, w_up, up_at, ffs, limits, offsets, token, tiles, *sizes, True, True, by_slot if weigh else None, ACTIVATIONS[act])
    y = amd.moe_experts(a, w_down, down_at, ffs, None, offsets, token, tiles, *sizes, False, True)
    # fp32 sums of n products in steps of 32, the partial sums below 8 (going up) and 16 (down, of activations up to 6 or so),
    # then one rounding to 8 bits; the products of two sums have twice the error of one, times the other
    steps = width // 32
    atol_up, atol_down = 2.0 ** -23 * 8 * steps * 8, 2.0 ** -23 * 16 * 128
    for e in range(experts + 1):
        r = torch.arange(rows, device=DEV) if e == experts else (of_row == e).nonzero()[:, 0]
        s = slots[r, int(e == experts)].long()
        x = h[r].double() * (weights[r, int(e == experts)].double()[:, None] if weigh else 1)
        p, u = x @ gate[e].double().T.contiguous(), x @ up[e].double().T.contiguous()
        if act == "clamped":
            p, u = p.clamp(max=limit), u.clamp(-limit, limit)
            want = p * torch.sigmoid(1.702 * p) * (u + 1)
        else:
            want = p * torch.sigmoid(p) * u if gated else u.clamp(min=0).square()
        got = a[s, :ff[e]].double()
        assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + atol_up).all(), (e, (got - want).abs().max())
        want = got @ down[e].double().T.contiguous()
        got = y[s].double()
        assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + atol_down).all(), (e, (got - want).abs().max())


def test_millions_of_slots(amd):
    """More tiles of 64 slots than a dimension of a grid: rows of every part of the step against the product in 64 bits."""
    rows, top, experts, width, ff = 600_000, 8, 16, 32, 32
    g = torch.Generator(device=DEV).manual_seed(5)
    h = torch.randn(rows, width, generator=g, device=DEV).bfloat16()
    router = torch.randn(experts, width, generator=g, device=DEV).bfloat16()
    up, down = (torch.randn(experts, *s, generator=g, device=DEV).bfloat16() * 32 ** -0.5 for s in ((ff, width), (width, ff)))
    ids, _, offsets, token, slots, tiles, _ = amd.moe_route(h, amd.pack_weight(router), None, top, False, True, experts, False, 1)
    assert rows * top > 64 * 65535 and tiles.shape[0] > 65535
    sizes, at = (rows, width, ff, ff, ff), torch.arange(experts, device=DEV) * ff * width
    ffs = torch.full((experts,), ff, dtype=torch.int32, device=DEV)
    pack = lambda w: torch.cat([amd.pack_weight(e.contiguous()).reshape(-1) for e in w])
    a = amd.moe_experts(h, pack(up), at, ffs, None, offsets, token, tiles, *sizes, True, True, None, 2)
    y = amd.moe_experts(a, pack(down), at, ffs, None, offsets, token, tiles, *sizes, False, True)
    r = torch.cat([torch.arange(500, device=DEV), torch.arange(rows - 500, rows, device=DEV), torch.randint(rows, (3000,), generator=g, device=DEV)])
    e, s = ids[r].long(), slots[r].long()
    for j in range(experts):
        row, place = (e == j).nonzero(as_tuple=True)
        want = (h[r[row]].double() @ up[j].double().T.contiguous()).clamp(min=0).square()
        got = a[s[row, place]].double()
        # one k-step: fp32 sums of 32 products, then one rounding to 8 bits
        assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + 1e-5).all(), j
        want = got @ down[j].double().T.contiguous()
        assert ((y[s[row, place]].double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all(), j


@pytest.mark.parametrize("rows,experts", [(2000, 4), (300, 8), (100, 200)], ids=["many slots", "few slots", "hardly any"])
def test_tiles_of_a_plain_router(amd, rows, experts):
    """Packed products over the tiles of 16 slots that a router that is not packed makes, a shared expert of several times the others' size
    among them: what they give over the packed router's tiles."""
    width, ff, shared_ff = 256, 160, 800
    g = torch.Generator(device=DEV).manual_seed(rows)
    rand = lambda *s: torch.randn(*s, generator=g, device=DEV).bfloat16()
    h, marks = rand(rows, width), torch.zeros(experts, width, dtype=torch.bfloat16, device=DEV)
    marks[torch.arange(experts), torch.arange(experts)] = 4
    of_row = torch.zeros(rows, width, dtype=torch.bfloat16, device=DEV)  # whole numbers decide: both routers choose alike
    of_row[torch.arange(rows), torch.arange(rows) % experts] = 1
    sizes, ffs = (rows, width, shared_ff, ff, shared_ff), torch.tensor([ff] * experts + [shared_ff], dtype=torch.int32, device=DEV)
    up, down = ([rand(*(s if kind == "up" else s[::-1])) * width ** -0.5 for s in [(ff, width)] * experts + [(shared_ff, width)]]
                for kind in ("up", "down"))
    at = torch.arange(experts + 1, device=DEV) * ff * width
    pack = lambda ws: torch.cat([amd.pack_weight(w.contiguous()).reshape(-1) for w in ws])
    results = []
    for packed in (True, False):
        r = amd.pack_weight(torch.nn.functional.pad(marks, (0, 0, 0, -experts % 16))) if packed else marks
        ids, _, offsets, token, slots, tiles, _ = amd.moe_route(of_row, r, None, 1, True, packed, experts, False, 1)
        a = amd.moe_experts(h, pack(up), at, ffs, None, offsets, token, tiles, *sizes, True, True, None, 2)
        y = amd.moe_experts(a, pack(down), at, ffs, None, offsets, token, tiles, *sizes, False, True)
        results.append((ids, a[slots.long()][:, 0, :ff], a[slots.long()][:, 1], y[slots.long()]))
    for one, other in zip(*results):
        assert torch.equal(one, other)
