"""The prefill-only workflow.  CPU: the scheduler under the three scenarios of the reference's own
test (tests/prefill_only/test_scheduler.py:27-129: limited by the request budget, limited by the
token budget, prompts over max_model_len ignored) with the same parameters; config checks; aborts.
GPU: the encoder engine against a plain fp32 torch forward; sync == async; replicas."""
import pytest
import torch

import light_vllm_amd  # noqa: F401
from light_vllm_amd.prefill_only import (PrefillOnlyRequestOutput, PrefillOnlyScheduler,
                                         PrefillOnlySchedulerConfig as SchedulerConfig, Request,
                                         SchedulableRequest)


def processor(num_new_tokens):
    return lambda r: SchedulableRequest(request_id=r.request_id, arrival_time=r.arrival_time,
                                        prompt_token_ids=[0] * num_new_tokens)


def finished(out):
    return [PrefillOnlyRequestOutput(r.request_id, None, r.prompt_token_ids, True) for r in out.scheduled_requests]


@pytest.mark.parametrize("num_new_tokens", [9, 99, 199])
@pytest.mark.parametrize("n_request", [9, 99, 199])
@pytest.mark.parametrize("max_num_requests", [1, 2, 3, 5, 7])
def test_limited_by_max_num_requests(n_request, num_new_tokens, max_num_requests):
    max_model_len = num_new_tokens + 1
    s = PrefillOnlyScheduler(SchedulerConfig(max_num_batched_tokens=max_model_len * max_num_requests,
                                             max_model_len=max_model_len, max_num_seqs=max_num_requests),
                             processor(num_new_tokens))
    for i in range(1, n_request + 1):
        s.add_request(Request(request_id=str(i), arrival_time=0.0))
    while s.has_unfinished_requests():
        out = s.schedule()
        s.free_finished_request(finished(out))
        if s.has_unfinished_requests():
            assert len(out.scheduled_requests) == max_num_requests
        else:
            assert len(out.scheduled_requests) <= max_num_requests
        assert len(out.ignored_requests) == 0


@pytest.mark.parametrize("num_new_tokens", [9, 99, 199])
@pytest.mark.parametrize("n_request", [9, 99, 199])
@pytest.mark.parametrize("max_num_requests", [2, 3, 5, 7])
def test_limited_by_token_budget(n_request, num_new_tokens, max_num_requests):
    s = PrefillOnlyScheduler(SchedulerConfig(max_model_len=num_new_tokens + 1, max_num_seqs=max_num_requests,
                                             max_num_batched_tokens=(num_new_tokens + 1) * (max_num_requests - 1)),
                             processor(num_new_tokens))
    for i in range(1, n_request + 1):
        s.add_request(Request(request_id=str(i), arrival_time=0.0))
    n = 0
    while s.has_unfinished_requests():
        out = s.schedule()
        n += len(out.scheduled_requests)
        s.free_finished_request(finished(out))
        if s.has_unfinished_requests():
            assert len(out.scheduled_requests) == max_num_requests - 1
        else:
            assert len(out.scheduled_requests) <= max_num_requests - 1
        assert len(out.ignored_requests) == 0
    assert n == n_request


@pytest.mark.parametrize("num_new_tokens", [9, 99, 199])
@pytest.mark.parametrize("n_request", [9, 99, 199])
@pytest.mark.parametrize("max_num_requests", [2, 3, 5, 7])
def test_ignored_requests(n_request, num_new_tokens, max_num_requests):
    max_model_len = num_new_tokens // 2
    s = PrefillOnlyScheduler(SchedulerConfig(max_num_batched_tokens=max_model_len * max_num_requests,
                                             max_model_len=max_model_len, max_num_seqs=max_num_requests),
                             processor(num_new_tokens))
    for i in range(1, n_request + 1):
        s.add_request(Request(request_id=str(i), arrival_time=0.0))
    n_ignored = 0
    while s.has_unfinished_requests():
        out = s.schedule()
        assert len(out.scheduled_requests) == 0 and len(out.ignored_requests) > 0
        n_ignored += len(out.ignored_requests)
    assert n_ignored == n_request


def test_config_checks_and_aborts():
    with pytest.raises(ValueError, match="max_num_batched_tokens"):
        SchedulerConfig(max_model_len=100, max_num_batched_tokens=50, max_num_seqs=4)
    with pytest.raises(ValueError, match="max_num_on_the_fly"):
        SchedulerConfig(max_model_len=10, max_num_seqs=4, max_num_on_the_fly=1)
    with pytest.raises(ValueError, match="scheduling"):
        SchedulerConfig(max_model_len=10, max_num_seqs=4, scheduling="bogus")
    assert SchedulerConfig(max_model_len=10, max_num_seqs=4, scheduling="double_buffer").max_num_on_the_fly == 3
    cfg = SchedulerConfig(max_model_len=10, max_num_seqs=4)
    assert cfg.max_num_batched_tokens == 40 and cfg.max_num_on_the_fly == 2
    s = PrefillOnlyScheduler(cfg, processor(5))
    for i in range(6):
        s.add_request(Request(str(i)))
    s.add_request(Request("3"))  # duplicate id: ignored
    s.abort_request(["1", "4"])
    out = s.schedule()
    assert [r.request_id for r in out.scheduled_requests] == ["0", "2", "3", "5"]
    outs = s.remove_abort_request(finished(out))
    s.free_finished_request(outs)
    assert not s.has_unfinished_requests()


# ------------------------------------------------------------------ GPU: the encoder engine
DEV = "cuda:0"


def reference_hidden(model, token_ids):
    """fp32 torch forward of EncoderModel's weights on one sequence, dense bidirectional attention."""
    import torch.nn.functional as F
    cfg = model.cfg
    hid, H, D = cfg.hidden_size, cfg.num_attention_heads, cfg.head_dim
    ids = torch.tensor(token_ids, device=model.device)
    T = ids.numel()
    pos = torch.arange(T, device=model.device) + cfg.pad_token_id + 1
    f = lambda t: t.float()
    x = f(model.word_emb)[ids] + f(model.pos_emb)[pos] + f(model.type_emb)[0]
    x = F.layer_norm(x, (hid,), f(model.emb_ln[0]), f(model.emb_ln[1]), cfg.layer_norm_eps)
    for lw in model.layers:
        qkv = x @ f(lw.qkv_w).T + f(lw.qkv_b)
        q, k, v = (t.view(T, H, D).transpose(0, 1) for t in qkv.split([hid, hid, hid], dim=-1))
        att = torch.softmax(q @ k.transpose(1, 2) / D ** 0.5, dim=-1) @ v
        a = att.transpose(0, 1).reshape(T, hid)
        x = F.layer_norm(x + a @ f(lw.out_w).T + f(lw.out_b), (hid,), f(lw.attn_ln[0]), f(lw.attn_ln[1]), cfg.layer_norm_eps)
        h = F.gelu(x @ f(lw.fc1_w).T + f(lw.fc1_b))
        x = F.layer_norm(x + h @ f(lw.fc2_w).T + f(lw.fc2_b), (hid,), f(lw.out_ln[0]), f(lw.out_ln[1]), cfg.layer_norm_eps)
    return x


def make_encoder(scheduling="sync", pooling="cls", max_seqs=4, budget=None):
    from light_vllm_amd.prefill_only.engine import PrefillOnlyEngine
    from light_vllm_amd.prefill_only.model import EncoderConfig
    return PrefillOnlyEngine(EncoderConfig.tiny(), SchedulerConfig(max_model_len=512, max_num_seqs=max_seqs,
                                                                   max_num_batched_tokens=budget, scheduling=scheduling),
                             device=DEV, pooling=pooling, seed=0)


def encoder_prompts():
    g = torch.Generator().manual_seed(1)
    return [torch.randint(2, 512, (n,), generator=g).tolist() for n in (1, 5, 17, 64, 33, 100, 256, 2, 31, 129)]


@pytest.mark.gpu
@pytest.mark.parametrize("tables", ["two types", "strided", "off 16 bytes"])
def test_embedding_tables(tables):
    """A table of two types, of which the first is taken, tables that are parts of wider ones, and some that begin anywhere."""
    from light_vllm_amd.attention.prefill_only import PrefillOnlyAttentionMetadata
    from light_vllm_amd.prefill_only.model import EncoderConfig, EncoderModel
    model = EncoderModel(EncoderConfig.tiny(), DEV, 0)
    ids = torch.randint(2, 512, (100,), generator=torch.Generator().manual_seed(3)).to(DEV)
    md = PrefillOnlyAttentionMetadata(100, [100], torch.tensor([0, 100], dtype=torch.int32, device=DEV))

    def run():
        with torch.inference_mode():
            return model.forward(ids, torch.arange(100, device=DEV), md)
    first = run()
    if tables == "two types":
        model.type_emb = torch.cat([model.type_emb, model.type_emb + 1])
    elif tables == "off 16 bytes":
        for name in ("word_emb", "pos_emb", "type_emb"):
            t = getattr(model, name)
            setattr(model, name, torch.cat([t.new_zeros(3), t.flatten()])[3:].view(t.shape))
    else:
        model.word_emb, model.pos_emb = (torch.cat([t, t], dim=1)[:, :128] for t in (model.word_emb, model.pos_emb))
    assert torch.equal(run(), first)


@pytest.mark.gpu
@pytest.mark.parametrize("how", ["assigned", "copied", "in a part", "by storage"])
def test_weights_that_come_after_the_model(how):
    """Weights assigned or written into a model that has been used are the ones that its next forward takes."""
    from light_vllm_amd.attention.prefill_only import PrefillOnlyAttentionMetadata
    from light_vllm_amd.prefill_only.model import EncoderConfig, EncoderModel
    cfg = EncoderConfig(hidden_size=1024, intermediate_size=4096, num_hidden_layers=1, num_attention_heads=16, vocab_size=512,
                        max_position_embeddings=1024)
    lens = [500, 300, 400]  # (rows that the kernel with GELU behind the product takes)
    model, other = (EncoderModel(cfg, DEV, seed) for seed in (0, 1))
    ids = torch.randint(2, 512, (sum(lens),), generator=torch.Generator().manual_seed(3)).to(DEV)
    pos = torch.cat([torch.arange(n) for n in lens]).to(DEV)
    starts = torch.tensor([0, 500, 800, 1200], dtype=torch.int32, device=DEV)
    md = PrefillOnlyAttentionMetadata(max(lens), lens, starts)

    def run():
        with torch.inference_mode():
            return model.forward(ids, pos, md)
    first, lw, new = run(), model.layers[0], other.layers[0].fc1_w
    if how == "assigned":
        lw.fc1_w = new
    elif how == "copied":
        lw.fc1_w.copy_(new)
    elif how == "in a part":
        lw.fc1_w[:2048].copy_(new[:2048])
    else:
        lw.fc1_w.data = new
    got = run()
    model.cfg.fused_layer_norm = False  # (the library's product and GELU)
    want = run()
    assert not torch.equal(got, first)
    assert (got.float() - want.float()).norm() < 1e-2 * want.float().norm()
    assert (first.float() - want.float()).norm() > 5e-2 * want.float().norm()


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["qkv_w", "out_w", "fc1_w", "fc2_w"])
@pytest.mark.parametrize("how", ["assigned", "copied", "captured"])
def test_each_weight_that_comes_after_the_model(name, how):
    """... each of them, in prompts of few rows; first seen in a capture: taken there and afterwards."""
    from light_vllm_amd.attention.prefill_only import PrefillOnlyAttentionMetadata
    from light_vllm_amd.prefill_only.model import EncoderConfig, EncoderModel
    cfg = EncoderConfig(hidden_size=1024, intermediate_size=4096, num_hidden_layers=1, num_attention_heads=16, vocab_size=512,
                        max_position_embeddings=1024)
    with torch.inference_mode():  # (as users make one)
        model, other = (EncoderModel(cfg, DEV, seed) for seed in (0, 1))
    lens = [50, 70]
    ids = torch.randint(2, 512, (sum(lens),), generator=torch.Generator().manual_seed(3)).to(DEV)
    pos = torch.cat([torch.arange(n) for n in lens]).to(DEV)
    md = PrefillOnlyAttentionMetadata(max(lens), lens, torch.tensor([0, 50, 120], dtype=torch.int32, device=DEV))

    def run():
        with torch.inference_mode():
            return model.forward(ids, pos, md)
    first, lw, new = run().clone(), model.layers[0], getattr(other.layers[0], name) * 2
    if how == "assigned":
        setattr(lw, name, new)
    else:
        getattr(lw, name).copy_(new)
    if how == "captured":
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            got = run()
        for _ in range(3):
            graph.replay()
            torch.cuda.synchronize()
            assert torch.allclose(got.float(), run().float(), atol=0.1, rtol=0.02)
    got = run()
    model.cfg.fused_layer_norm = False  # (the library's)
    want = run()
    assert (got.float() - want.float()).norm() < 1e-2 * want.float().norm()
    assert (first.float() - want.float()).norm() > 5e-2 * want.float().norm()


WEIGHTS = ["qkv_w", "out_w", "fc1_w", "fc2_w"]


def one_layer(lens):
    """Two encoders of a layer, and a forward over sequences of these lengths."""
    from light_vllm_amd.attention.prefill_only import PrefillOnlyAttentionMetadata
    from light_vllm_amd.prefill_only.model import EncoderConfig, EncoderModel
    cfg = EncoderConfig(hidden_size=1024, intermediate_size=4096, num_hidden_layers=1, num_attention_heads=16, vocab_size=512,
                        max_position_embeddings=2048)
    model, other = (EncoderModel(cfg, DEV, seed) for seed in (0, 1))
    ids = torch.randint(2, 512, (sum(lens),), generator=torch.Generator().manual_seed(3)).to(DEV)
    pos = torch.cat([torch.arange(n) for n in lens]).to(DEV)
    starts = torch.tensor([sum(lens[:i]) for i in range(len(lens) + 1)], dtype=torch.int32, device=DEV)
    md = PrefillOnlyAttentionMetadata(max(lens), lens, starts)

    @torch.inference_mode()
    def run(m=model):
        return m.forward(ids, pos, md)
    return model, other, run


def close(a, b):
    return float((a.float() - b.float()).norm()) < 1e-2 * float(b.float().norm())


@pytest.mark.gpu
@pytest.mark.parametrize("name", WEIGHTS)
@pytest.mark.parametrize("how", ["data.copy_", "data.copy_ by who had it before", "from_dlpack", "vars"])
def test_writes_that_torch_does_not_count(name, how):
    """Short prompts: whoever has a weight may write to it in any way, and the next forward takes what is there."""
    model, other, run = one_layer([50, 70])
    lw, new = model.layers[0], getattr(other.layers[0], name) * 2
    first = run().clone()
    if how == "data.copy_":
        getattr(lw, name).data.copy_(new)
    elif how == "data.copy_ by who had it before":
        had = getattr(lw, name)
        run()
        had.data.copy_(new)
    elif how == "from_dlpack":
        torch.from_dlpack(torch.utils.dlpack.to_dlpack(getattr(lw, name))).copy_(new)
    else:
        vars(lw).update({name: new})
    got = run()
    model.cfg.fused_layer_norm = False  # (the library's products, of the weights themselves)
    want = run()
    assert close(got, want) and not close(first, want)


@pytest.mark.gpu
@pytest.mark.parametrize("name", WEIGHTS)
@pytest.mark.parametrize("lens", [[50, 70], [900, 700, 800]])  # (own products; GELU behind a copy that the graph makes)
def test_weights_that_come_after_a_capture(name, lens):
    """Replays take the weight as it is, before the next forward outside of the graph and after it; so do those behind an assignment, which
    leaves the graph the tensor that it was captured with."""
    model, other, run = one_layer(lens)
    lw = model.layers[0]
    run()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = run()

    def replay():
        graph.replay()
        torch.cuda.synchronize()
        return out.clone()

    def library():
        model.cfg.fused_layer_norm = False
        y = run().clone()
        model.cfg.fused_layer_norm = True
        return y
    first = replay()
    assert close(first, library())
    w = getattr(lw, name)
    w.copy_(getattr(other.layers[0], name) * 2)
    second = replay()
    want = library()
    assert close(second, want) and not close(first, want)
    for _ in range(3):
        assert close(run(), want)
        torch.full((3 * 1024, 1024), 9.0, dtype=torch.bfloat16, device=DEV)  # (memory that a copy might have left)
        assert torch.equal(replay(), second)
    setattr(lw, name, getattr(other.layers[0], name).clone())
    assert close(run(), library()) and torch.equal(replay(), second)


@pytest.mark.gpu
@pytest.mark.parametrize("name", WEIGHTS)
@pytest.mark.parametrize("rows", [100, 1200])
def test_weights_of_another_shape(name, rows):
    """A weight that is turned round is refused, laid out or not."""
    model, other, run = one_layer([rows])
    lw = model.layers[0]
    w = getattr(lw, name)
    setattr(lw, name, w.t().contiguous() if name != "out_w" else w[:, :512].reshape(512, 1024).contiguous())
    for _ in range(2):
        with pytest.raises(RuntimeError):
            run()
        lw.lay_out()


@pytest.mark.gpu
def test_copies_of_a_model():
    """A copy of an encoder takes the kernels that the encoder takes."""
    import copy
    model, _, run = one_layer([50, 70])
    first = run().clone()
    other = copy.deepcopy(model)
    assert torch.equal(run(other), first) and all(other.layers[0].packed(name) is not None for name in WEIGHTS)
    assert all(other.layers[0].packed(name) is not model.layers[0].packed(name) for name in WEIGHTS)
    other.layers[0].qkv_w.zero_()
    assert not close(run(other), first) and torch.equal(run(), first)


@pytest.mark.gpu
@pytest.mark.parametrize("how", ["data.copy_", "assigned"])
def test_weights_laid_out_anew(how):
    """Behind lay_out() a model is what one that was made with the weights is: the same kernels, the same bits; and what is written then is seen."""
    model, other, run = one_layer([50, 70])
    lw, theirs = model.layers[0], other.layers[0]
    made_with = run(other).clone()
    for name in ("word_emb", "pos_emb", "type_emb", "emb_ln"):
        setattr(model, name, getattr(other, name))
    for name in vars(theirs):
        if name.endswith(("_b", "_ln")):
            setattr(lw, name, getattr(theirs, name))
    for name in WEIGHTS:
        new = theirs.weight(name).clone()
        if how == "assigned":
            setattr(lw, name, new)
        else:
            getattr(lw, name).data.copy_(new)
    assert close(run(), made_with) and all(lw.packed(name) is None for name in WEIGHTS)
    lw.lay_out()
    assert torch.equal(run(), made_with) and all(lw.packed(name) is not None for name in WEIGHTS)
    w = lw.qkv_w
    lw.lay_out()
    w.mul_(2)  # (by one who had it before)
    got = run()
    model.cfg.fused_layer_norm = False
    assert close(got, run()) and not close(got, made_with)


@pytest.mark.gpu
def test_encoder_engine_matches_fp32_reference():
    eng = make_encoder(pooling="last_hidden_states")
    ps = encoder_prompts()
    res = eng.encode(ps, use_async=False)
    for i, p in enumerate(ps):
        want = reference_hidden(eng.model, p).cpu()
        got = res[str(i)].float()
        assert got.shape == want.shape
        cos = torch.nn.functional.cosine_similarity(got, want, dim=1)
        assert float(cos.min()) >= 0.999, (i, float(cos.min()))
        assert float((got - want).abs().max()) <= 3e-2 * float(want.abs().max())


@pytest.mark.gpu
@pytest.mark.parametrize("pooling", ["cls", "mean"])
def test_encoder_async_equals_sync_and_pooling(pooling):
    ps = encoder_prompts() + [[7] * 600]  # the last one exceeds max_model_len: ignored
    sync = make_encoder("sync", pooling).encode(ps, use_async=False)
    e = make_encoder("async", pooling, max_seqs=3)
    asyn = e.encode(ps, use_async=True)
    e.shutdown()
    assert sync[str(len(ps) - 1)] is None and asyn[str(len(ps) - 1)] is None
    for i in range(len(ps) - 1):
        a, b = sync[str(i)], asyn[str(i)]
        assert a.shape == (128,) and abs(float(a.norm()) - 1.0) < 1e-3
        # batch composition differs between the two runs; per-sequence attention does not depend on it
        assert float((a - b).abs().max()) <= 2e-2
    ref = make_encoder(pooling="last_hidden_states")
    h = ref.encode(ps[:3], use_async=False)
    for i in range(3):
        x = h[str(i)].float()
        want = torch.nn.functional.normalize(x[0] if pooling == "cls" else x.mean(0), dim=-1)
        assert float((sync[str(i)] - want).abs().max()) <= 2e-2
