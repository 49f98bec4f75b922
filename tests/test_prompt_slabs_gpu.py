"""Prompts whose products leave fp32 slabs of shares of K: what sums them, and models that take them."""
import ctypes

import pytest
import torch
import torch.nn.functional as F

from test_engine_gpu import dense_reference_logits
from test_sasilorn_gpu import LAYOUTS, i32, layout

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
SLABS = 1  # include/lvllm_hip.h LVLLM_SUMS_SLABS


@pytest.fixture(scope="module")
def amd():
    import light_vllm_amd._custom_ops  # noqa: F401
    return torch.ops._C_amd


def rand(*shape, seed=0):
    return torch.randn(*shape, generator=torch.Generator(device=DEV).manual_seed(seed), device=DEV)


def summed(slabs, dtype):
    """In their order, rounded once."""
    total = torch.zeros_like(slabs[0])
    for s in slabs:
        total = total + s
    return total.to(dtype)


def shares_of(rows, n, k):
    from light_vllm_amd import _native
    return _native.load_hip_library().lvllm_prompt_product_plan(rows, n, k, 0, SLABS, 1, (ctypes.c_int * 3)())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,hidden", [(1, 8), (70, 1000), (300, 4096), (130, 16384)])
@pytest.mark.parametrize("shares", [1, 3, 4, 5, 8, 9, 13])
def test_add_rms_norm(amd, dtype, rows, hidden, shares):
    slabs, residual, weight = rand(shares, rows, hidden), rand(rows, hidden, seed=1).to(dtype), rand(hidden, seed=2).to(dtype)
    want, kept = summed(slabs, dtype), residual.clone()
    torch.ops._C.fused_add_rms_norm(want, kept, weight, 1e-5)
    out = torch.empty_like(want)
    amd.fused_add_rms_norm_splitk(out, residual, slabs, weight, 1e-5)
    assert torch.equal(out, want) and torch.equal(residual, kept)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("width", [96, 1024, 250])
@pytest.mark.parametrize("shares", [1, 3, 4, 5, 8])
def test_dynamic_tanh(amd, dtype, width, shares):
    slabs, x = rand(shares, 130, width), rand(130, width, seed=1)
    a, w, b = rand(1, seed=2), rand(width, seed=3), rand(width, seed=4)
    xs, xr = x.clone(), x.clone()
    assert torch.equal(amd.add_dyt(xs, slabs, a, w, b, dtype), amd.add_dyt(xr, summed(slabs, dtype), a, w, b, dtype)) and torch.equal(xs, xr)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("name", sorted(LAYOUTS))
@pytest.mark.parametrize("width", [96, 90])
@pytest.mark.parametrize("shares", [1, 3, 4, 5, 8])
def test_token_shift(amd, dtype, name, width, shares):
    seqs = LAYOUTS[name]
    qsl, lens = layout(seqs)
    rows = sum(n for n, _ in seqs)
    slabs, x, mu, carried = rand(shares, rows, width), rand(rows, width, seed=1), rand(5, width, seed=2), rand(9, width, seed=3)
    a, w, b = rand(1, seed=4), rand(width, seed=5), rand(width, seed=6)
    after = [carried.clone(), carried.clone()]
    got, want = (amd.add_dyt_shift_mix(x, y, mu, a, w, b, c, i32([7, 2, 5, 0, 8][:len(seqs)]), qsl, lens, dtype)
                 for y, c in zip((slabs, summed(slabs, dtype)), after))
    assert all(torch.equal(g, h) for g, h in zip(got, want)) and torch.equal(*after)


class DenseAttention:
    """Causal softmax over one sequence without a cache."""

    def __init__(self, cfg):
        self.cfg = cfg

    def forward(self, q, k, v, kv_cache, metadata):
        c = self.cfg
        q, k, v = (t.reshape(t.shape[0], -1, c.head_dim).transpose(0, 1) for t in (q, k, v))
        k, v = (t.repeat_interleave(c.num_attention_heads // c.num_key_value_heads, 0) for t in (k, v))
        o = F.scaled_dot_product_attention(q.float()[None], k.float()[None], v.float()[None], is_causal=True)[0]
        return o.to(q.dtype).transpose(0, 1).reshape(q.shape[1], -1)


def decoder(**sizes):
    from light_vllm_amd.engine.config import ModelConfig
    from light_vllm_amd.engine.model import DecoderModel
    cfg = ModelConfig(num_hidden_layers=2, vocab_size=512, max_position_embeddings=2048, **sizes)
    return DecoderModel(cfg, DenseAttention(cfg), DEV, 0)


@torch.inference_mode()
def run(model, tokens):
    hidden = model.forward(tokens, torch.arange(tokens.numel(), device=DEV), None, None)
    return model.compute_logits(hidden[-60:])


@pytest.mark.parametrize("rows", [65, 100, 300, 700])
def test_prompts_of_a_dense_decoder(amd, monkeypatch, rows):
    """Logits are as far from those in 32 bits as the library's products leave them."""
    import light_vllm_amd.engine.model as m
    model = decoder(hidden_size=1024, intermediate_size=4096, num_attention_heads=8, num_key_value_heads=2)
    assert shares_of(rows, 1024, 4096) > 1 and (rows > 65 or shares_of(rows, 1024, 4096) > 4)
    tokens = torch.randint(0, 512, (rows,), generator=torch.Generator().manual_seed(rows)).to(DEV)
    want = dense_reference_logits(model, tokens.tolist())[-60:]
    got = run(model, tokens).float()
    monkeypatch.setattr(m, "product", lambda x, w, bias=None, slabs=False: F.linear(x, w.w, bias))
    library = run(model, tokens).float()
    # both are roundings to 16 bits of the same sums; of thousands of logits' errors the norms agree to some percent
    off, theirs = (got - want).norm(), (library - want).norm()
    assert not torch.equal(got, library) and float(off) < 1.25 * float(theirs) and float(theirs) < 0.03 * float(want.norm())


def test_weights_laid_out_anew(amd):
    """One weight for steps of every length, and for those that were captured before."""
    from light_vllm_amd.engine.model import Weight, linear, product
    w, b = rand(2048, 1024, seed=1).bfloat16(), rand(2048, 1024, seed=2).bfloat16()
    weight, xs = Weight(w.clone()), [rand(n, 1024, seed=n).bfloat16() for n in (1, 64, 100, 300, 700, 6000)]
    outs = [linear(x, weight) for x in xs]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = linear(xs[1], weight)
    packed = weight.packed
    weight.w.copy_(b)
    weight.lay_out()
    assert weight.packed is packed
    for x, before in zip(xs, outs):
        want = x.double() @ b.double().t()
        for y in (linear(x, weight), product(x, weight)):
            assert (y.double() - want).norm() < 1e-2 * want.norm() and (before.double() - want).norm() > want.norm()
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(captured, linear(xs[1], weight))


@pytest.mark.parametrize("rows", [100, 300])
def test_norm_weights_off_16_bytes(amd, rows):
    model = decoder(hidden_size=1024, intermediate_size=4096, num_attention_heads=8, num_key_value_heads=2)
    tokens = torch.randint(0, 512, (rows,), generator=torch.Generator().manual_seed(rows)).to(DEV)
    want = run(model, tokens).float()
    for lw in model.layers:
        lw.post_norm, lw.input_norm = (torch.cat([w[:1], w])[1:] for w in (lw.post_norm, lw.input_norm))
    assert model.layers[0].post_norm.data_ptr() % 16
    got = run(model, tokens).float()
    assert (got - want).norm() < 1e-2 * want.norm()


@pytest.mark.parametrize("rows", [100, 300, 700])
def test_feed_forward_of_a_hybrid_decoder(amd, rows):
    """Slabs out of the feed-forward, into the norm behind it: the sum of both in 64 bits, and the norm's bits."""
    from light_vllm_amd.engine.mixers import DynTanhNorm, SquaredReluMlp
    t = {"m.up": rand(4096, 1024) / 32, "m.down": rand(1024, 4096, seed=1) / 64}
    mlp, h = SquaredReluMlp(lambda n: t[n].bfloat16(), "m", True), rand(rows, 1024, seed=2).bfloat16()
    y = mlp(h)
    assert y.dim() == 3 and y.shape[0] == shares_of(rows, 1024, 4096)
    a = F.relu(h.double() @ t["m.up"].bfloat16().double().t()).square()
    w = t["m.down"].bfloat16().double()
    want = a @ w.t()
    # the activation's square is of a rounded product, and is rounded: three halves of 2^-8 each way; the sums' own roundings are far below
    bound = 4 * 2.0 ** -8 * (a @ w.abs().t())
    assert bool(((y.double().sum(0) - want).abs() <= bound).all())
    norm = DynTanhNorm(lambda n: rand(1024, seed=3) if not n.endswith("alpha") else torch.tensor([0.7], device=DEV), "n")
    x = rand(rows, 1024, seed=4)
    x2 = x.clone()
    assert torch.equal(norm(x, y, torch.bfloat16), norm(x2, summed(y, torch.bfloat16), torch.bfloat16)) and torch.equal(x, x2)
