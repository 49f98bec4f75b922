"""Products of prompts over packed weights (csrc/prompt_product.hip): each body at the edges of its tiles and shares, against 64 bits."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def lib():
    from light_vllm_amd import _native
    _native.load_torch_ops()
    return _native.load_hip_library()


def operands(rows, n, k):
    g = torch.Generator(device=DEV).manual_seed(rows * 31 + n + k)
    x = torch.randn(rows, k, generator=g, device=DEV).bfloat16()
    w = (torch.randn(n, k, generator=g, device=DEV) * k ** -0.5).bfloat16()
    b = torch.randn(n, generator=g, device=DEV).bfloat16()
    return x, w, torch.ops._C_amd.pack_weight(w), b


def bound(x, w, k):  # k additions in 32 bits, in any order
    return (k + 8) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())


SIZES = [(16, 128), (17, 144), (65, 16), (100, 272), (129, 240), (300, 304)]  # rows, n: remainders of tiles of rows, and of blocks of weights
PLANS = [(16, 1), (32, 1), (48, 1), (64, 1), (80, 1), (96, 1), (64, 2), (80, 2), (96, 2), (112, 2), (128, 2), (80, 4), (112, 4), (128, 4)]


@pytest.mark.parametrize("rows,n", SIZES)
@pytest.mark.parametrize("size,nt", PLANS)
@pytest.mark.parametrize("k", [256, 896, 2560])
def test_bodies(lib, rows, n, size, nt, k):
    x, w, packed, b = operands(rows, n, k)
    ld = k + 8 if size % 32 else k  # rows of x beside others
    x = torch.nn.functional.pad(x, (0, ld - k))[:, :k]
    want, err = x.double() @ w.double().t(), bound(x, w, k)
    p = lambda t: ctypes.c_void_p(0 if t is None else t.data_ptr())
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for shares in (1, 2, 3, 8):
        if -(-(k // 64) // shares) * 2 * (shares - 1) >= k // 32:
            continue  # (a share without steps: refused)
        plan = (ctypes.c_int * 3)(size, nt, shares)
        for gelu in (False, True) if shares == 1 and nt < 4 else (False,):
            out = torch.full((rows + 1, n), 7.0, dtype=torch.bfloat16, device=DEV)  # (a row behind the last: not written)
            slabs = torch.full((shares * rows + 1, n), 7.0, device=DEV) if shares > 1 else None
            bias = b if shares == 1 else None
            print(rows, n, k, size, nt, shares, gelu, flush=True)
            rc = lib.lvllm_prompt_product(p(out if shares == 1 else None), p(slabs), p(x), ctypes.c_int64(ld), ctypes.c_int64(0), p(packed), p(bias), rows, n, k, int(gelu), 1, plan, stream)
            assert rc == 0, lib.lvllm_last_error()
            if shares > 1:
                got = slabs[:-1].view(shares, rows, n).double().sum(0)
                assert bool(((got - want).abs() <= err).all()) and bool((slabs[-1] == 7).all())
                continue
            z = want + b.double()
            ref = torch.nn.functional.gelu(z) if gelu else z
            # half a step of bfloat16; GELU's slope is below 1.13, and its own error in 32 bits below 1e-6
            most = 2.0 ** -8 * ref.abs() + 1.13 * (err + 2.0 ** -23 * z.abs()) + (1e-6 if gelu else 0)
            assert bool(((out[:-1].double() - ref).abs() <= most).all()) and bool((out[-1] == 7).all())


@pytest.mark.parametrize("rows,n,k", [(65, 1024, 1024), (100, 4096, 4096), (300, 2048, 8448), (1000, 1024, 4096)])
def test_op(lib, rows, n, k):
    x, w, packed, b = operands(rows, n, k)
    want, err = x.double() @ w.double().t(), bound(x, w, k)
    y = torch.ops._C_amd.prompt_product(x, packed, None, n, False, True)
    assert y is not None
    got = y.double() if y.dim() == 2 else y.double().sum(0)
    assert bool(((got - want).abs() <= err + (2.0 ** -8 * want.abs() if y.dim() == 2 else 0)).all())
    z = torch.ops._C_amd.prompt_product(x, packed, b, n)
    if z is not None:
        assert bool(((z.double() - want - b.double()).abs() <= err + 2.0 ** -8 * (want + b.double()).abs() + 2.0 ** -23 * want.abs()).all())


@pytest.mark.parametrize("rows,n,k", [(65, 2048, 2048), (100, 1024, 512), (257, 7680, 2048), (300, 2048, 5632), (520, 3072, 1536), (800, 2048, 3072)])
@pytest.mark.parametrize("with_bias", [False, True])
def test_sums_in_order(lib, rows, n, k, with_bias):
    """Every tile adds one k-step of 32 behind the other: the same bits, whichever takes a product (ahead of routers, the last ones matter)."""
    x, w, packed, b = operands(rows, n, k)
    bias = b if with_bias else None
    y = torch.ops._C_amd.prompt_product(x, packed, bias, n, ordered=True)
    assert y is not None and y.shape == (rows, n)
    p = lambda t: ctypes.c_void_p(0 if t is None else t.data_ptr())
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for size, nt in PLANS:
        out = torch.empty_like(y)
        plan = (ctypes.c_int * 3)(size, nt, 1)
        print(rows, n, k, size, nt, flush=True)
        rc = lib.lvllm_prompt_product(p(out), None, p(x), ctypes.c_int64(k), ctypes.c_int64(0), p(packed), p(bias), rows, n, k, 0, 1, plan, stream)
        assert rc == 0 and torch.equal(out, y), (size, nt)


@pytest.mark.parametrize("rows,n,k", [(300, 2048, 2048), (300, 7680, 2048), (300, 2048, 5632), (257, 2048, 2816), (700, 3072, 2048), (500, 4096, 512)])
def test_sums_in_the_library_s_order(lib, rows, n, k):
    """Sizes of models with routers at which the library takes K in one piece: the same bits, so that tokens go to the same experts."""
    x, w, packed, _ = operands(rows, n, k)
    y = torch.ops._C_amd.prompt_product(x, packed, None, n, ordered=True)
    assert y is not None and torch.equal(y, torch.nn.functional.linear(x, w))


@pytest.mark.parametrize("rows,outputs,k,act", [(300, 5632, 2048, "clamped_unit"), (700, 5632, 2048, "clamped_unit"), (1000, 11264, 2048, "silu_and_mul"),
                                                (1536, 4096, 2048, "silu_and_mul")])
def test_activations_behind_sums_in_the_library_s_order(lib, rows, outputs, k, act):
    from light_vllm_amd.engine.mixers import ORDERED_ROWS
    from light_vllm_amd.engine.model import Weight, linear_act
    assert rows <= ORDERED_ROWS
    x, w, _, _ = operands(rows, 2 * outputs, k)
    y, both = linear_act(x, Weight(w), act, outputs, 7.0), torch.nn.functional.linear(x, w)
    want = torch.ops._C_amd.clamped_unit(both, 7.0) if act == "clamped_unit" else torch.ops._C_amd.silu_unit(both)
    assert y is not None and torch.equal(y, want)


@pytest.mark.parametrize("batch,rows,n,k", [(4, 100, 2048, 2048), (4, 300, 2048, 2048), (4, 700, 512, 512), (3, 65, 1040, 320), (5, 129, 64, 256)])
def test_batches(lib, batch, rows, n, k):
    """Several products in a launch: what each is by itself."""
    g = torch.Generator(device=DEV).manual_seed(batch)
    x = torch.randn(batch + 1, rows, k, generator=g, device=DEV).bfloat16()[:batch]
    ws = [(torch.randn(n, k, generator=g, device=DEV) * k ** -0.5).bfloat16() for _ in range(batch)]
    packed = torch.cat([torch.ops._C_amd.pack_weight(w).reshape(-1) for w in ws])
    y = torch.ops._C_amd.prompt_products(x, packed, n)
    assert y is not None and y.shape == (batch, rows, n)
    for b in range(batch):
        want = x[b].double() @ ws[b].double().t()
        assert bool(((y[b].double() - want).abs() <= bound(x[b], ws[b], k) + 2.0 ** -8 * want.abs()).all()), b


def test_operands_that_the_library_takes(lib):
    x, w, packed, b = operands(130, 1024, 1024)
    op = torch.ops._C_amd.prompt_product
    assert op(x, packed, b, 1024) is not None
    wide = torch.zeros(130, 1025, dtype=torch.bfloat16, device=DEV)
    shifted = torch.zeros(130 * 1024 + 1, dtype=torch.bfloat16, device=DEV)[1:].view(130, 1024)
    odd_bias = torch.zeros(1025, dtype=torch.bfloat16, device=DEV)[1:]
    assert op(wide[:, :1024], packed, b, 1024) is None and op(shifted, packed, b, 1024) is None
    assert op(x.half(), packed, b, 1024) is None and op(x, packed.half(), b, 1024) is None
    assert op(x, packed, odd_bias, 1024) is None and op(x, packed, b.float(), 1024) is None
    assert op(x[:64], packed, b, 1024) is None and op(x[:0], packed, b, 1024) is None
    assert op(x, packed, b[:1], 1024) is None and op(x[None], packed, b, 1024) is None  # (what the library makes of these)
    with pytest.raises(RuntimeError):
        op(x, packed, b, 1040)


@pytest.mark.parametrize("which", ["x", "bias"])
def test_gradients(lib, which):
    """Products that are differentiated are the library's."""
    from light_vllm_amd.engine.model import Weight, linear, product
    x, w, _, b = operands(300, 1024, 1024)
    x.requires_grad_(which == "x")
    b.requires_grad_(which == "bias")
    for f in (linear, product):
        y = f(x, Weight(w), b)
        g, = torch.autograd.grad(y.float().sum(), x if which == "x" else b)
        assert torch.isfinite(g).all() and g.abs().max() > 0
    with torch.no_grad():
        assert torch.ops._C_amd.prompt_product(x, torch.ops._C_amd.pack_weight(w), b, 1024) is not None


@pytest.mark.parametrize("rows", [100, 300])
def test_linear_of_several_dimensions(lib, rows):
    from light_vllm_amd.engine.model import Weight, linear
    x, w, _, b = operands(rows, 1024, 1024)
    x = torch.stack([x, 2 * x], 1)  # [rows, 2, k]
    assert torch.equal(linear(x, Weight(w), b), torch.nn.functional.linear(x, w, b))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,hidden", [(1, 8), (7, 1000), (33, 1024), (130, 2048)])
@pytest.mark.parametrize("shares", [1, 2, 4, 5, 8])
@pytest.mark.parametrize("with_bias", [False, True])
def test_add_layer_norm_slabs(lib, dtype, rows, hidden, shares, with_bias):
    """The sum and its bias rounded first, and then added and normed: the bits of that but for the order of the norm's sums."""
    g = torch.Generator(device=DEV).manual_seed(rows + hidden + shares)
    x = torch.randn(rows, hidden, generator=g, device=DEV).to(dtype)
    slabs = torch.randn(shares, rows, hidden, generator=g, device=DEV)
    w, b, yb = ((i + 0.1 * torch.randn(hidden, generator=g, device=DEV)).to(dtype) for i in (1, 0, 0))
    total = torch.zeros_like(slabs[0])
    for s in slabs:
        total = total + s
    y = (total + yb.float() if with_bias else total).to(dtype)
    want, got = torch.empty_like(x), x.clone()
    torch.ops._C_amd.add_layer_norm(want, x, y, w, b, 1e-5)
    torch.ops._C_amd.add_layer_norm_slabs(got, got, slabs, yb if with_bias else None, w, b, 1e-5)
    ref = torch.nn.functional.layer_norm((x + y).double(), (hidden,), w.double(), b.double(), 1e-5)
    # half a step of the result; mean and variance of `hidden` terms in 32 bits
    most = 2.0 ** (-8 if dtype == torch.bfloat16 else -11) * ref.abs() + hidden * 2.0 ** -23 * (ref.abs() + 1)
    assert bool(((got.double() - ref).abs() <= most).all()) and bool(((want.double() - ref).abs() <= most).all())
    for bad in (slabs.half(), slabs[:, :, ::2] if hidden > 8 else slabs[0], slabs[0]):
        with pytest.raises(RuntimeError):
            torch.ops._C_amd.add_layer_norm_slabs(got, got, bad, None, w, b, 1e-5)
