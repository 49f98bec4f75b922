"""Decays from a low-rank projection at the edges of their tiles (16 rows x 64 channels, 32 x 64 and 64 x 128 by how many there are, 64 and 32 of the
rank) and with values that have no parts of 16 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def amd():
    import light_vllm_amd._custom_ops  # noqa: F401
    return torch.ops._C_amd


def reference(u, a, b, kind):
    u, a, b = u.double(), a.double(), b.double()
    z = (torch.tanh(u) if kind else u) @ a + b
    return -torch.exp(z.clamp(max=9.0)) if kind else torch.nn.functional.logsigmoid(z) / 16


def tensors(rows, rank, channels, dtype, stride):
    g = torch.Generator().manual_seed(rows + rank)
    u = torch.randn(rows, stride, generator=g).to(dtype)[:, :rank]
    return u, torch.randn(rank, channels, generator=g) * 3 * rank ** -0.5, torch.randn(channels, generator=g)


# rows, channels of the larger tiles: the last ones end inside a wave's part, with channels that are no multiple of 4 and those that are
TILES_32 = [(2003, 387), (705, 1092)]     # 882 and 810 tiles of 16 x 64, of which 700 and fewer are taken as they are
TILES_64 = [(8003, 515), (4097, 1028)]    # 4509 and 4369, more than 3800


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("rows,channels", TILES_32 + TILES_64)
@pytest.mark.parametrize("rank,stride", [(1, 1), (31, 37), (33, 40), (63, 64), (65, 65), (129, 131)])
def test_decays_of_many_rows(amd, rows, channels, rank, stride, kind, dtype):
    test_decays(amd, rows, rank, channels, stride, kind, dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("rows,rank,channels,stride", [(1, 1, 1, 1), (63, 31, 127, 37), (64, 32, 128, 32), (65, 33, 129, 33),
                                                       (128, 127, 130, 128), (129, 129, 132, 131), (70, 512, 260, 512)])
def test_decays(amd, rows, rank, channels, stride, kind, dtype):
    u, a, b = tensors(rows, rank, channels, dtype, stride)
    got = amd.log_decay(u.to(DEV), a.to(DEV), b.to(DEV), kind, 1 / 16 if kind == 0 else 1.0).cpu().double()
    f = torch.tanh(u.double()) if kind else u.double()
    # z: rank + 1 fp32 roundings of sums up to that of the sizes (and tanh's own two); either function moves by at most z's error times
    # its value where that is an exponential, and by that / 16 else; a few roundings of its own
    off = (f.abs() @ a.double().abs() + b.double().abs()) * (rank + 4) * 2.0 ** -24
    want = reference(u, a, b, kind)
    room = (off * want.abs() if kind else off / 16) + 8 * 2.0 ** -24 * want.abs() + 1e-30
    assert ((got - want).abs() <= room).all()


@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("where,value", [("u", float("inf")), ("u", float("-inf")), ("u", float("nan")), ("a", float("inf")),
                                         ("a", float("nan")), ("a", 3.4028e38), ("b", float("-inf"))])
def test_values_without_parts(amd, where, value, kind, rows=130, channels=140, rank=40):
    t = dict(zip("uab", tensors(rows, rank, channels, torch.bfloat16, rank)))
    at = {"u": (rows // 2, 3), "a": (3, 5), "b": (5,)}[where]
    t[where][at] = value
    if where == "a" and value < float("inf"):
        t["u"][:, 3] = 2.0 ** -100  # (finite products)
    got = amd.log_decay(*(t[k].to(DEV) for k in "uab"), kind, 1 / 16 if kind == 0 else 1.0).cpu().double()
    f = torch.tanh(t["u"].double()) if kind else t["u"].double()
    z = f @ t["a"].double() + t["b"].double()
    # e^x takes no infinities: kind 0 has e^-|z|, NaN for every z that is not finite; kind 1 bounds z from above, NaN included, so that
    # only -inf is left
    nan = z == float("-inf") if kind else ~z.isfinite()
    assert torch.equal(got.isnan(), nan)
    want = reference(t["u"], t["a"], t["b"], kind)
    want[~nan & ~z.isfinite()] = -torch.exp(torch.tensor(9.0, dtype=torch.float64))
    torch.testing.assert_close(got[~nan], want[~nan], rtol=1e-4, atol=1e-5)


@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("rows,channels", TILES_32[:1] + TILES_64[:1])
@pytest.mark.parametrize("rank", [40, 129])
@pytest.mark.parametrize("where,value", [("u", float("inf")), ("u", float("nan")), ("a", float("inf")), ("a", 3.4028e38), ("b", float("-inf"))])
def test_values_without_parts_among_many_rows(amd, where, value, rank, rows, channels, kind):
    test_values_without_parts(amd, where, value, kind, rows, channels, rank)


@pytest.mark.parametrize("rows", [350, 353, 1888, 1889, 1904, 1905, 2100])
@pytest.mark.parametrize("kind", [0, 1])
def test_tiles(amd, rows, kind):
    """The same bits from each size of tile: of rows by themselves, whose tiles are the smallest, and of all of them."""
    u, a, b = (t.to(DEV) for t in tensors(rows, 72, 2000, torch.bfloat16, 72))
    got = amd.log_decay(u, a, b, kind, 1 / 16)
    want = torch.cat([amd.log_decay(part, a, b, kind, 1 / 16) for part in u.split(40)])
    assert torch.equal(got, want)
    assert ((got.double() - reference(u, a, b, kind)).abs() <= 1e-4 * (1 + got.double().abs())).all()
