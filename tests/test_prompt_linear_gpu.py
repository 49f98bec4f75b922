"""Projections of prompts with an activation in the same launch: tiles with remainders of rows and outputs, every number of 64-row groups,
the smallest k, and which sizes the kernels take."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
GELU, SILU, RELU2, CLAMPED = 1, 2, 3, 4
LIMIT = 1.5


@pytest.fixture(scope="module")
def amd():
    import light_vllm_amd._custom_ops  # noqa: F401
    return torch.ops._C_amd


# rows, outputs, k: whole tiles and one row more, remainders of 1 to 4 groups of 64 rows, outputs that end inside a block and inside a
# wave's part of one, odd numbers of stages, one tile a workgroup and several
WIDE = [(769, 8464, 512), (1100, 5904, 576), (1500, 4096, 512), (3000, 2832, 640), (2113, 8192, 1088), (600, 16400, 512)]
TILE = [(300, 4096, 64), (1000, 4112, 96), (129, 6160, 1024), (2500, 4096, 160), (4097, 784, 32), (513, 4224, 2048)]


# rows, W rows, k of half tiles, the groups of 16 rows in one, and whether their loads are dealt: one tile a CU and more
HALF_TILES = [(130, 8224, 256, 5, True), (180, 8224, 256, 6, False), (220, 8224, 320, 7, True), (250, 8224, 576, 8, True), (280, 8224, 256, 6, False),
              (300, 8224, 256, 7, True), (130, 16544, 256, 5, False), (180, 16544, 256, 6, False), (400, 8736, 256, 7, True),
              (512, 8736, 320, 8, True), (220, 8224, 288, 7, False)]


def check(amd, rows, outputs, k, act, row_major, pack):
    gen = torch.Generator().manual_seed(rows + outputs + k)
    n = outputs * (2 if act in (SILU, CLAMPED) else 1)
    x = torch.randn(rows, k, generator=gen).bfloat16().to(DEV)
    w = (torch.randn(n, k, generator=gen) * 2 * k ** -0.5).bfloat16().to(DEV)
    bias = (0.2 * torch.randn(n, generator=gen)).bfloat16().to(DEV) if act == GELU else None
    got = amd.prompt_linear(x, w if row_major else None, amd.pack_weight(w) if pack else None, bias, outputs, act, LIMIT)
    assert got is not None and got.shape == (rows, outputs)
    z = x.double() @ w.double().T
    # sums of up to 2048 products of values around 1 in fp32, rounded to 8 bits behind the product (not GELU) and behind the activation,
    # SwiGLU once more between; the clamped unit of rounded gate and value grows with the gate at most 1.1 times as fast, its parts at most LIMIT
    sums, eps = 1e-5, 2.0 ** -8
    if act == GELU:
        z = z + bias.double()
        want, slack = F.gelu(z), eps * F.gelu(z).abs() + 1.13 * sums
    elif act == SILU:
        g, u = z[:, :outputs], z[:, outputs:]
        want = F.silu(g) * u
        slack = eps * (2 * want.abs() + 1.1 * g.abs() * u.abs() + F.silu(g).abs() * u.abs()) + 4 * sums * (1 + g.abs() + u.abs())
    elif act == CLAMPED:
        g, u = z[:, :outputs].clamp(max=LIMIT), z[:, outputs:].clamp(-LIMIT, LIMIT)
        want = g * torch.sigmoid(1.702 * g) * (u + 1)
        slack = eps * (want.abs() + 1.13 * g.abs() * (u + 1).abs() + 1.5 * u.abs()) + 4 * sums * (1 + LIMIT) + 1e-6
    else:
        want = z.clamp(min=0).square()
        slack = eps * 3.1 * want + 2 * sums * (z.abs() + 1)
    assert ((got.double() - want).abs() <= slack).all(), ((got.double() - want).abs() - slack).max()


@pytest.mark.parametrize("act", [SILU, RELU2, CLAMPED])
@pytest.mark.parametrize("rows,outputs,k", WIDE)
def test_wide_tiles(amd, rows, outputs, k, act):
    check(amd, rows, outputs, k, act, True, False)


@pytest.mark.parametrize("act", [GELU, SILU, RELU2, CLAMPED])
@pytest.mark.parametrize("rows,outputs,k", TILE)
def test_tiles(amd, rows, outputs, k, act):
    outputs *= 1 if act in (GELU, CLAMPED) else 3
    check(amd, rows, outputs, k, act, False, True)


@pytest.mark.parametrize("act", [GELU, SILU, RELU2, CLAMPED])
@pytest.mark.parametrize("rows,wrows,k", [h[:3] for h in HALF_TILES])
def test_half_tiles(amd, rows, wrows, k, act):
    check(amd, rows, wrows // 2 if act in (SILU, CLAMPED) else wrows, k, act, False, True)


def test_activations_of_the_largest_and_smallest_values(amd):
    """GELU and SwiGLU of products from far below to far above their bends, infinities and NaN included."""
    rows, outputs, k = 2048, 4096, 512
    v = torch.cat([torch.linspace(-120, 120, rows - 8), torch.tensor([3e38, -3e38, float("inf"), float("nan"), 1e-30, -1e-30, 0., 88.])])
    x = torch.zeros(rows, k, dtype=torch.bfloat16)
    x[:, 0] = v.bfloat16()
    w = torch.zeros(2 * outputs, k, dtype=torch.bfloat16)
    w[:, 0] = 1
    x, w = x.to(DEV), w.to(DEV)
    z = x[:, :1].double()
    gelu = amd.prompt_linear(x, None, amd.pack_weight(w[:outputs].contiguous()), torch.zeros(outputs, dtype=torch.bfloat16, device=DEV), outputs,
                             GELU)
    silu = amd.prompt_linear(x, w, None, None, outputs, SILU)
    # (SwiGLU of gates below -88.72, whose e^-x has no place in 32 bits, is 0: the largest, of -89, is 89 * 89 e^-89 = 1.8e-35, and the next gate,
    # -88.5, gives 2.9e-35)
    for got, want, floor in (gelu, F.gelu(z), 1e-6), (silu, F.silu(z) * z, 1.9e-35):
        got, want = got.double(), want.expand(rows, outputs)
        nan, big = want.isnan(), want.abs() > 3.3e38
        assert (got.isnan() == nan).all() and (got[big] == got[big].sign() * float("inf")).all()
        keep = ~nan & ~big
        # (SwiGLU: two roundings; GELU: 5.9e-7 in 32 bits)
        assert ((got - want)[keep].abs() <= 2.1 * 2.0 ** -8 * want[keep].abs() + floor).all()


def test_what_is_refused(amd):
    x = torch.randn(2048, 512, device=DEV).bfloat16()
    w = torch.randn(8192, 512, device=DEV).bfloat16()
    assert amd.prompt_linear(x, w, None, None, 4096, SILU) is not None
    assert amd.prompt_linear(x[:64].contiguous(), w, None, None, 4096, SILU) is None
    assert amd.prompt_linear(x[:, ::2], w[:, ::2].contiguous(), None, None, 4096, SILU) is None   # rows that are not back to back
    assert amd.prompt_linear(x.half(), w.half(), None, None, 4096, SILU) is None
    assert amd.prompt_linear(x, None, None, None, 4096, SILU) is None
    assert amd.prompt_linear(x, None, amd.pack_weight(w), None, 8192, GELU) is None   # no bias
    flat = torch.randn(2048 * 512 + 1, device=DEV).bfloat16()
    assert amd.prompt_linear(flat[1:].view(2048, 512), w, None, None, 4096, SILU) is None   # not aligned
    with pytest.raises(RuntimeError):
        amd.prompt_linear(x, w, None, None, 8192, SILU)


@pytest.mark.parametrize("mixture", [True, False])
@pytest.mark.parametrize("kind", ["Lizazen", "Susalorn"])
def test_dense_feed_forwards_beside_routers(amd, kind, mixture):
    """In a model with routers the sums of prompts keep the library's order; in one without, the product takes its activation along."""
    from light_vllm_amd.engine.mixers import SiluMlp, project_to_residual
    from light_vllm_amd.engine.local_layers import ClampedMlp
    from light_vllm_amd.engine.registry import model_entry
    dense, moe = {"kind": "dense", "ff": 4096}, {"kind": "moe", "router": {"experts": 8, "top": 2}, "expert": {"ff": 128}}
    if kind == "Lizazen":
        dense["limit"], moe["shared"] = 7.0, {"ff": 128}
        d = {"norm": {"eps": 1e-6}, "embedding": {}}
        mixer = {"type": "attention", "mixer": {"heads": 4, "kv_heads": 2, "dim": 64, "vdim": 64, "scale": 0.125, "rot": {"dims": 64, "base": 1e4}, "softcap": 50.0,
                                                "mask": {"size": 4096}}}
    else:
        moe["router"].update(groups={"count": 4, "keep": 2}, scale=2.5)
        d = {"norm": {"eps": 1e-5}, "streams": 4, "loop": None}
        mixer = {"type": "channel_delta", "mixer": {"heads": 4, "kv_heads": 4, "dim": 64, "vdim": 64, "conv": 4}}
    d.update(architecture=kind, vocab=512, width=512, layers=[{**mixer, "mlp": dense}, {**mixer, "mlp": moe if mixture else dense}])
    entry = model_entry(kind)
    model = entry.model_cls()(entry.config_cls().from_dict(d), entry.backend_cls().get_impl_cls()(), DEV)
    subs = [s[0] for layer in model.layers for s in layer]
    mlp = next(s for s in subs if isinstance(s, (ClampedMlp, SiluMlp)))
    assert mlp.routed == mixture
    h = torch.randn(1500, 512, device=DEV).bfloat16()
    both = F.linear(h, mlp.up.w)
    want = project_to_residual(amd.clamped_unit(both, 7.0) if kind == "Lizazen" else amd.silu_unit(both), mlp.down)
    y = mlp(h)
    y = y.y if kind == "Lizazen" else y
    assert y.dtype == want.dtype and (not mixture or torch.equal(y, want))
    assert (y.float() - want.float()).norm() < 1e-2 * want.float().norm()
