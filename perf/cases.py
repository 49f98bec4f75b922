"""The work that serving has the framework do: one engine step of every model that it serves, through the model's own entry points.

  prompt   a step of whole prompts: `forward` over the paged caches and state slots, logits of each prompt's last token
  decode   a step of one token per sequence behind a context that is in the caches: the captured step that the engine replays

Models keep the real width, heads, experts and feed-forwards of the framework's benchmarks and a few layers of each kind; a step over
more layers is the same launches again.  Weights and tokens are random, caches and states are filled by the model's own prompt steps,
pages lie scattered as in a pool that has been in use.  `exact` restates every model in 64 bits."""
import math

import torch

DEVICE = "cuda:0"
PAGE, VOCAB, STEP_TOKENS = 16, 32000, 8192   # tokens a page, words, the most tokens the scheduler puts in one step
EPS = {"rotary": 1e-5, "encoder": 1e-5, "hybrid": 1e-5, "latent": 1e-5, "local": 1e-6, "stream": 1e-5}

# ---- the models: sizes of the benchmarks at their smaller width, of the headline for the rotary decoder ----
ROTARY = dict(width=4096, ff=14336, layers=4, heads=32, kv_heads=8, theta=500000.0)
ENCODER = dict(width=1024, ff=4096, layers=4, heads=16)

_HYBRID_FF = {"kind": "dense", "ff": 8448}
HYBRID = {"architecture": "Sasilorn", "vocab": VOCAB, "width": 2048, "norm": {"eps": 1e-5}, "layers": [
    {"type": "parallel", "mlp": _HYBRID_FF, "mixer": {
        "left": {"heads": 16, "kv_heads": 4, "dim": 128, "vdim": 64, "scale": 128 ** -0.5},
        "right": {"heads": 8, "dim": 128, "vdim": 128, "tau": 16.0}, "left_scale": 0.7, "right_scale": 0.7}},
    {"type": "wkv", "mlp": _HYBRID_FF, "mixer": {"heads": 32, "dim": 64}}] * 2}

_LATENT = {"heads": 16, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 512, "scale": 192 ** -0.5,
           "rot": {"dims": 64, "base": 10000.0}, "mask": {"size": 4096}}
_LATENT_MOE = {"kind": "moe", "router": {"experts": 64, "top": 6}, "expert": {"ff": 1408, "limit": 7.0},
               "shared": {"ff": 2816, "limit": 7.0}}
LATENT = {"architecture": "Lepalorn", "vocab": VOCAB, "width": 2048, "norm": {"eps": 1e-5}, "embedding": {"scale": 1.0}, "layers": [
    {"type": "latent_attention", "mixer": _LATENT, "mlp": _LATENT_MOE},
    {"type": "latent_attention", "mixer": {**_LATENT, "kv_from": 0}, "mlp": _LATENT_MOE},
    {"type": "latent_attention", "mixer": _LATENT, "mlp": _LATENT_MOE},
    {"type": "latent_attention", "mixer": {**_LATENT, "kv_from": 2}, "mlp": _LATENT_MOE}]}

_ROT = {"dims": 128, "base": 500000.0}
_HEADS = {"heads": 16, "kv_heads": 4, "dim": 128, "vdim": 128, "scale": 128 ** -0.5, "rot": _ROT, "mask": {"size": 8192}}
_TWO_MAPS = {**_HEADS, "dim": 64, "scale": 64 ** -0.5, "diff": 0.3, "rot": {"dims": 64, "base": 500000.0},
             "mask": {"size": 8192, "keep_first": 64}}
_RETENTION = {"heads": 8, "dim": 128, "vdim": 128, "rot": {"dims": 128, "base": 10000.0},
              "decay": [1 - 2.0 ** (-5 - 6 * i / 8) for i in range(8)]}
_CLAMPED = {"kind": "dense", "ff": 5632, "limit": 7.0}
_LOCAL_MOE = {"kind": "moe", "router": {"experts": 32, "top": 2}, "expert": {"ff": 1408}, "shared": {"ff": 2816}}
LOCAL = {"architecture": "Lizazen", "vocab": VOCAB, "width": 2048, "norm": {"eps": 1e-6},
         "embedding": {"bigram": {"buckets": 65536, "mul_prev": 31, "mul_cur": 7}}, "layers": [
    {"type": "parallel", "mixer": {"left": _HEADS, "right": _RETENTION}, "mlp": _CLAMPED},
    {"type": "attention", "mlp": _LOCAL_MOE, "mixer": {**_HEADS, "softcap": 50.0, "rot": {
        **_ROT, "scaling": {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 8192}}}},
    {"type": "attention_2", "mixer": _TWO_MAPS, "mlp": _CLAMPED},
    {"type": "attention_2", "mixer": _TWO_MAPS, "mlp": _LOCAL_MOE}]}

_STREAM_LATENT = {"type": "latent_attention", "mixer": {
    "heads": 16, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 512, "q_rank": 1536, "scale": 192 ** -0.5,
    "rot": {"dims": 64, "base": 10000.0, "scaling": {"factor": 4.0, "original": 4096, "fast": 32.0, "slow": 1.0}}}}
_STREAM_DELTA = {"type": "channel_delta", "mixer": {"heads": 16, "kv_heads": 16, "dim": 128, "vdim": 128, "conv": 4}}
_STREAM_MOE = {"kind": "moe", "expert": {"ff": 2816},
               "router": {"experts": 64, "top": 6, "groups": {"count": 8, "keep": 4}, "scale": 2.5}}
STREAM = {"architecture": "Susalorn", "vocab": VOCAB, "width": 2048, "norm": {"eps": 1e-5}, "streams": 4, "loop": None, "layers": [
    {**_STREAM_DELTA, "mlp": {"kind": "dense", "ff": 11264}}, {**_STREAM_LATENT, "mlp": _STREAM_MOE},
    {**_STREAM_DELTA, "mlp": _STREAM_MOE}, {**_STREAM_LATENT, "mlp": _STREAM_MOE}]}

LISTED_LAYERS = {"hybrid": HYBRID, "latent": LATENT, "local": LOCAL, "stream": STREAM}
ROUTER_SCALE, ROUTED_DOWN = 2.0, 0.25
RANDOM_RANK = {"hybrid": 64, "stream": 128}   # inner size of low-rank projections


# ---- cases ----
def case(name, model, phase, seqs, tokens, ragged=False, fp8=False):
    """`tokens`: of the longest prompt, or of the longest context with its newest token; `ragged`: the others are shorter, down to half;
    `fp8`: 8-bit projections over an 8-bit cache."""
    return dict(name=name, model=model, phase=phase, seqs=seqs, tokens=tokens, ragged=ragged, fp8=fp8)


def listed():
    return [
        # one user in conversation: the smallest step, a chain of short launches
        case("rotary decode 1x1024", "rotary", "decode", 1, 1024),
        # the headline: a full decode batch
        case("rotary decode 32x1024", "rotary", "decode", 32, 1024),
        # a larger batch of unequal contexts over 8-bit weights and an 8-bit cache
        case("rotary fp8 decode 32x1500", "rotary", "decode", 32, 1500, ragged=True, fp8=True),
        # prompts of unequal length that arrived together
        case("rotary prompt 4x1500", "rotary", "prompt", 4, 1500, ragged=True),
        # the embedding service: a batch of passages
        case("encoder prompt 32x512", "encoder", "prompt", 32, 512),
        # a long document read by the hybrid decoder, and a batch behind long contexts
        case("hybrid prompt 1x4096", "hybrid", "prompt", 1, 4096),
        case("hybrid decode 24x2000", "hybrid", "decode", 24, 2000, ragged=True),
        # questions of ordinary size, and a full decode batch over 64 experts
        case("latent prompt 3x777", "latent", "prompt", 3, 777, ragged=True),
        case("latent decode 32x1024", "latent", "decode", 32, 1024),
        # one short prompt: hundreds of rows
        case("local prompt 1x300", "local", "prompt", 1, 300),
        # the largest step the scheduler makes, and a small batch in conversation
        case("stream prompt 4x2048", "stream", "prompt", 4, 2048),
        case("stream decode 8x700", "stream", "decode", 8, 700, ragged=True),
    ]


def draw(rng):
    model = rng.choice(["rotary", "rotary", "encoder", "hybrid", "latent", "local", "stream"])
    phase = "prompt" if model == "encoder" else rng.choice(["prompt", "decode"])

    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))
    if phase == "prompt":
        rows = spread(100, (12288 if model == "encoder" else 4096))
        seqs = min(spread(1, 32 if model == "encoder" else 6), max(1, rows // 50))
        tokens = rows // seqs
    else:
        seqs, tokens = spread(1, 40), spread(60, 2000)
        tokens = min(tokens, 32768 // seqs)
    return dict(model=model, phase=phase, seqs=seqs, tokens=tokens, ragged=seqs > 1 and rng.random() < 0.7,
                fp8=model == "rotary" and phase == "decode" and rng.random() < 0.3)


def lengths(c):
    n, s = c["tokens"], c["seqs"]
    return [n - i * n // (2 * s) if c["ragged"] else n for i in range(s)]


# ---- what serving has in hand before a step ----
def generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def tokens_of(c, seed):
    """The words of all sequences, back to back."""
    return torch.randint(0, VOCAB, (sum(lengths(c)),), generator=generator(seed + 1), device=DEVICE)


def listed_layers(c):
    """(configuration, registry entry) of a decoder of listed layers."""
    from light_vllm_amd.engine.registry import model_entry
    d = LISTED_LAYERS[c["model"]]
    entry = model_entry(d["architecture"])
    cfg = entry.config_cls().from_dict(d)
    if c["model"] in RANDOM_RANK:
        cfg.random_rank = RANDOM_RANK[c["model"]]
    return cfg, entry


def tensors_of(c, seed):
    """Random weights in bfloat16, by name.  Routers are surer than random ones (a token's last expert weighs little beside its first),
    and what a mixture adds is small beside the shared expert or the stream: else one logit rounded another way, which moves a token
    from its last expert to the next one, would show as much as a mistake."""
    cfg, entry = listed_layers(c)
    cls, gen = entry.model_cls(), generator(seed)

    def scale(name):
        return ROUTER_SCALE if name.endswith(".router") else ROUTED_DOWN if ".mlp.e" in name and name.endswith(".down") else 1.0
    return {name: (scale(name) * cls.random_tensor(name, shape, gen, torch.device(DEVICE))).bfloat16()
            for name, shape in cls.tensor_shapes(cfg).items()}


def rotary_model(seed, fp8, impl=None):
    from light_vllm_amd.engine.config import ModelConfig
    from light_vllm_amd.engine.model import DecoderModel
    r = ROTARY
    cfg = ModelConfig(hidden_size=r["width"], intermediate_size=r["ff"], num_hidden_layers=r["layers"], vocab_size=VOCAB,
                      num_attention_heads=r["heads"], num_key_value_heads=r["kv_heads"], rope_theta=r["theta"],
                      quantization="fp8" if fp8 else None)
    return DecoderModel(cfg, impl, DEVICE, seed)


def encoder_model(seed):
    from light_vllm_amd.prefill_only.model import EncoderConfig, EncoderModel
    e = ENCODER
    return EncoderModel(EncoderConfig(hidden_size=e["width"], intermediate_size=e["ff"], num_hidden_layers=e["layers"],
                                      num_attention_heads=e["heads"], vocab_size=VOCAB), DEVICE, seed)


def decoder(c, seed, blocks):
    """(model, caches, every layer's matrix states)."""
    from light_vllm_amd.engine.cache_engine import CacheEngine
    from light_vllm_amd.engine.config import CacheConfig
    if c["model"] == "rotary":
        from light_vllm_amd.attention.backend import PagedAttnBackend as backend
        cache = "fp8" if c["fp8"] else "auto"
        r = ROTARY
        dim = r["width"] // r["heads"]
        impl = backend.get_impl_cls()(r["heads"], dim, dim ** -0.5, r["kv_heads"], None, None, cache)
        model = rotary_model(seed, c["fp8"], impl)
    else:
        cfg, entry = listed_layers(c)
        cache, backend = "auto", entry.backend_cls()
        model = entry.model_cls()(cfg, backend.get_impl_cls()(), DEVICE, tensors=tensors_of(c, seed))
    engine = CacheEngine(CacheConfig(block_size=PAGE, num_gpu_blocks=blocks, cache_dtype=cache, num_state_slots=c["seqs"]), model.cfg,
                         backend, DEVICE)
    return model, engine.model_caches(), [s["matrix"] for s in engine.state or [] if "matrix" in s]


def int32(values):
    return torch.tensor(values, dtype=torch.int32, device=DEVICE)


def prompt_step(tables, which, new):
    """(positions, metadata) of a step of whole prompts: sequences `which` with `new` tokens each."""
    from light_vllm_amd.attention.backend import PagedAttnMetadata
    starts = [0]
    for n in new:
        starts.append(starts[-1] + n)
    positions = torch.cat([torch.arange(n, device=DEVICE) for n in new])
    slots = torch.cat([tables[s, :-(-n // PAGE)].long().repeat_interleave(PAGE)[:n] for s, n in zip(which, new)]) * PAGE
    loc = int32(starts)
    return positions, PagedAttnMetadata(
        num_prefills=len(new), num_prefill_tokens=starts[-1], num_decode_tokens=0, slot_mapping=slots + positions % PAGE,
        seq_lens=list(new), seq_lens_tensor=int32(new), max_query_len=max(new), max_prefill_seq_len=max(new), max_decode_seq_len=0,
        query_start_loc=loc, seq_start_loc=loc, context_lens_tensor=int32([0] * len(new)),
        block_tables=tables[which[0]:which[-1] + 1], query_lens=list(new), context_lens=[0] * len(new), state_slots=int32(which))


class LogitsOnly:
    """Stands where the engine's sampler does: a captured step ends with its logits."""

    def new_scratch(self, rows, device):
        return None

    def sample(self, logits, slots, scratch=None):
        return logits


def fill_caches(model, caches, tables, tokens, lens, held):
    """Prompt steps over the first `held` tokens of each sequence, as many sequences a step as the scheduler takes."""
    begins = [sum(lens[:i]) for i in range(len(lens))]
    at = 0
    while at < len(lens):
        which, rows = [], 0
        while at < len(lens) and (not which or rows + held[at] <= STEP_TOKENS):
            which.append(at)
            rows += held[at]
            at += 1
        ids = torch.cat([tokens[begins[s]:begins[s] + held[s]] for s in which])
        positions, metadata = prompt_step(tables, which, [held[s] for s in which])
        model.forward(ids, positions, caches, metadata)


@torch.inference_mode()
def prepare(c, seed):
    import light_vllm_amd._custom_ops  # noqa: F401
    lens, tokens = lengths(c), tokens_of(c, seed)
    if c["model"] == "encoder":
        from light_vllm_amd.attention.prefill_only import PrefillOnlyAttentionMetadata
        starts = int32([sum(lens[:i]) for i in range(len(lens) + 1)])
        positions = torch.cat([torch.arange(n, device=DEVICE) for n in lens])
        return dict(case=c, model=encoder_model(seed), tokens=tokens, positions=positions,
                    metadata=PrefillOnlyAttentionMetadata(max(lens), lens, starts))
    pages = [-(-n // PAGE) for n in lens]
    width = (max(lens) + 511) // 512 * 512 // PAGE
    order = torch.randperm(sum(pages), generator=generator(seed + 2), device=DEVICE).int()
    tables = torch.zeros(len(lens), width, dtype=torch.int32, device=DEVICE)
    for i, n in enumerate(pages):
        tables[i, :n] = order[sum(pages[:i]):sum(pages[:i]) + n]
    model, caches, matrices = decoder(c, seed, sum(pages))
    state = dict(case=c, model=model, caches=caches, matrices=matrices)
    if c["phase"] == "prompt":
        state["tokens"] = tokens
        state["positions"], state["metadata"] = prompt_step(tables, list(range(len(lens))), lens)
        state["last"] = torch.tensor([sum(lens[:i + 1]) - 1 for i in range(len(lens))], device=DEVICE)
        return state
    from light_vllm_amd.engine.graph_runner import DecodeGraphPool
    graph = DecodeGraphPool(model, caches, width, PAGE, DEVICE).get(len(lens), LogitsOnly())
    fill_caches(model, caches, tables, tokens, lens, [n - 1 for n in lens])
    newest = torch.tensor([sum(lens[:i + 1]) - 1 for i in range(len(lens))], device=DEVICE)
    positions = torch.tensor([n - 1 for n in lens], device=DEVICE)
    slots = tables.gather(1, (positions // PAGE)[:, None])[:, 0].long() * PAGE + positions % PAGE
    graph.load(tokens[newest], positions, slots, tables, int32(lens), recurrent_slots=int32(list(range(len(lens)))))
    state["graph"] = graph
    return state


@torch.inference_mode()
def run(state):
    c, model = state["case"], state["model"]
    if c["model"] == "encoder":
        return {"hidden": model.forward(state["tokens"], state["positions"], state["metadata"])}
    if c["phase"] == "prompt":
        hidden = model.forward(state["tokens"], state["positions"], state["caches"], state["metadata"])
        return {"hidden": hidden, "logits": model.compute_logits(hidden[state["last"]]), "states": state["matrices"]}
    graph, n = state["graph"], c["seqs"]
    logits = graph.replay()
    return {"hidden": graph.hidden[:n], "logits": logits[:n], "states": state["matrices"]}


# ---- what a step cannot do without ----
def weights_of(c):
    """(projections that every row takes, [(experts, taken per row, numbers in one)]) of all layers, in numbers."""
    if c["model"] == "rotary":
        r = ROTARY
        return r["layers"] * r["width"] * (r["width"] * 2 + 2 * r["width"] // r["heads"] * r["kv_heads"] + 3 * r["ff"]), []
    if c["model"] == "encoder":
        return ENCODER["layers"] * ENCODER["width"] * (4 * ENCODER["width"] + 2 * ENCODER["ff"]), []
    cfg, entry = listed_layers(c)
    mixtures, dense = [], 0
    for name, shape in entry.model_cls().tensor_shapes(cfg).items():
        if ".mlp.e" not in name and name not in ("embed", "head", "bigram"):
            dense += math.prod(shape)
    for l in LISTED_LAYERS[c["model"]]["layers"]:
        if l["mlp"]["kind"] == "moe":
            m = l["mlp"]
            mixtures.append((m["router"]["experts"], m["router"]["top"], (2 if c["model"] == "stream" else 3) * 2048 * m["expert"]["ff"]))
    return dense, mixtures


def attention_of(c):
    """Per layer with attention: (multiply-adds per query and key, numbers cached per token)."""
    if c["model"] == "rotary":
        r = ROTARY
        return [(2 * r["width"], 2 * r["kv_heads"] * r["width"] // r["heads"])] * r["layers"]
    if c["model"] == "encoder":
        return [(2 * ENCODER["width"], 0)] * ENCODER["layers"]
    out = []
    for l in LISTED_LAYERS[c["model"]]["layers"]:
        m = l["mixer"].get("left", l["mixer"])
        if "kv_rank" in m:
            out.append((m["heads"] * (m["dim"] + m["rot_dim"] + m["vdim"]), m["kv_rank"] + m["rot_dim"]))
        elif l["type"] not in ("wkv", "channel_delta"):
            maps = 2 if "diff" in m else 1
            out.append((m["heads"] * (maps * m["dim"] + maps * m["vdim"]), m["kv_heads"] * (maps * m["dim"] + m["vdim"])))
    return out


def states_of(c):
    """Numbers of every matrix state of a sequence."""
    out = []
    for l in LISTED_LAYERS.get(c["model"], {"layers": []})["layers"]:
        m = l["mixer"].get("right", l["mixer"])
        if "right" in l["mixer"] or l["type"] in ("wkv", "channel_delta"):
            out.append(m["heads"] * m["dim"] * m.get("vdim", m["dim"]))
    return out


def work(c):
    lens, decode = lengths(c), c["phase"] == "decode"
    rows = len(lens) if decode else sum(lens)
    width = {"rotary": ROTARY["width"], "encoder": ENCODER["width"]}.get(c["model"], 2048)
    dense, mixtures = weights_of(c)
    size = 1 if c["fp8"] else 2
    head = 0 if c["model"] == "encoder" else VOCAB * width
    nbytes = (dense + head) * size + rows * width * 4
    flops = 2 * rows * dense + 2 * len(lens) * head
    for experts, top, numbers in mixtures:
        nbytes += experts * (1 - (1 - top / experts) ** rows) * numbers * 2
        flops += 2 * rows * top * numbers
    keys = sum(lens) if decode else sum(n * n for n in lens) * (1.0 if c["model"] == "encoder" else 0.5)
    for products, cached in attention_of(c):
        flops += 2 * keys * products
        nbytes += sum(lens) * cached * size   # read behind a context, written by a prompt
    for numbers in states_of(c):
        flops += 6 * rows * numbers
        nbytes += len(lens) * numbers * (8 if decode else 4)
    return {"bytes": nbytes, "flops": flops}


def tolerance(c):
    """bfloat16 through four layers.  Against 64 bits: hybrid 0.004, encoder 0.008, rotary 0.025 (a residual stream of 16 bits); mixtures
    as much as tokens whose last expert is another one make of it, a few of them by more than the typical value."""
    return {"rel": {"hybrid": 0.015}.get(c["model"], 0.03), "max": 1.0 - 1e-6}


# ---- 64 bits ----
def spans(c):
    lens = lengths(c)
    return [(sum(lens[:i]), sum(lens[:i + 1])) for i in range(len(lens))]


def rms(x, eps, gain=1.0):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * gain


def positions_of(segs):
    return torch.cat([torch.arange(b - a, device=DEVICE) for a, b in segs]).double()


def turn(x, angles, halves, grow=1.0):
    """Entries i and i + dims / 2 (or 2i and 2i + 1) of x [n, heads, dims + rest] turn by angles [n, dims / 2]."""
    half = angles.shape[1]
    c, s = grow * angles.cos()[:, None], grow * angles.sin()[:, None]
    u, v = (x[..., :half], x[..., half:2 * half]) if halves else (x[..., 0:2 * half:2], x[..., 1:2 * half:2])
    a, b = u * c - v * s, v * c + u * s
    turned = torch.cat([a, b], -1) if halves else torch.stack([a, b], -1).flatten(-2)
    return torch.cat([turned, x[..., 2 * half:]], -1)


def base_frequencies(rot):
    return [rot["base"] ** (-2.0 * i / rot["dims"]) for i in range(rot["dims"] // 2)]


def ramp_frequencies(rot):
    """Pairs that turn often within the original length keep their frequency, slow ones are divided, a ramp between."""
    s = rot["scaling"]

    def pair(turns):
        return rot["dims"] * math.log(s["original"] / (2 * math.pi * turns)) / (2 * math.log(rot["base"]))
    first, last = max(math.floor(pair(s["fast"])), 0), min(math.ceil(pair(s["slow"])), rot["dims"] - 1)
    out = []
    for i, f in enumerate(base_frequencies(rot)):
        slow = min(max((i - first) / max(last - first, 1e-3), 0.0), 1.0)
        out.append(f / s["factor"] * slow + f * (1 - slow))
    return out


def wave_frequencies(rot):
    """By wavelengths within the original length: kept, divided, a blend between."""
    out, s = [], rot.get("scaling")
    for f in base_frequencies(rot):
        if s is not None:
            keep = min(max((s["original"] * f / (2 * math.pi) - s["low"]) / (s["high"] - s["low"]), 0.0), 1.0)
            f = (1 - keep) * f / s["factor"] + keep * f
        out.append(f)
    return out


def angles_of(segs, frequencies):
    return positions_of(segs)[:, None] * torch.tensor(frequencies, dtype=torch.float64, device=DEVICE)[None]


def attend(q, k, v, segs, scale, window=0, chunk=0, first=0, cap=0.0, sink=None, causal=True):
    """q [n, H, d], k [n, G, d], v [n, G, e], sequence by sequence and head by head."""
    group = q.shape[1] // k.shape[1]
    out = q.new_empty(q.shape[0], q.shape[1], v.shape[2])
    for a, b in segs:
        i, j = torch.arange(b - a, device=DEVICE)[:, None], torch.arange(b - a, device=DEVICE)[None]
        hidden = (j > i) if causal else (j < 0)
        if window:
            hidden = hidden | ((i - j >= window) & (j >= first))
        if chunk:
            hidden = hidden | (i // chunk != j // chunk)
        for h in range(q.shape[1]):
            s = q[a:b, h].contiguous() @ k[a:b, h // group].t().contiguous() * scale
            s = (cap * torch.tanh(s / cap) if cap else s).masked_fill_(hidden, float("-inf"))
            m = s.amax(1, keepdim=True)
            p = torch.exp(s - m)
            total = p.sum(1, keepdim=True) + (torch.exp(sink[h] - m) if sink is not None else 0)
            out[a:b, h] = p @ v[a:b, h // group].contiguous() / total
    return out


def recur(q, k, v, decay, segs, kind, beta=None, bonus=None):
    """All sequences at once, token after token -> (read-outs [n, H, e], last states [seqs, H, d, e]).  `kind`: "after" reads the state
    that holds the token's own write, "before" reads bonus * k v^T in its place, "delta" writes what is missing of v."""
    longest, outs = max(b - a for a, b in segs), []

    def padded(x, fill):
        p = x.new_full((longest, len(segs)) + x.shape[1:], fill)
        for i, (a, b) in enumerate(segs):
            p[:b - a, i] = x[a:b]
        return p
    q, k, v, decay = padded(q, 0.0), padded(k, 0.0), padded(v, 0.0), padded(decay, 1.0)
    beta = padded(beta, 0.0) if beta is not None else None
    S = q.new_zeros(q.shape[1:] + v.shape[3:])
    for t in range(longest):
        kt, qt, u = k[t][..., None], q[t][..., None], v[t]
        if kind == "before":
            kv = kt * u[..., None, :]
            outs.append(((S + bonus[..., None] * kv) * qt).sum(-2))
            S = S * decay[t][..., None] + kv
            continue
        S = S * decay[t][..., None]
        if kind == "delta":
            u = beta[t][..., None] * (u - (S * kt).sum(-2))
        S = S + kt * u[..., None, :]
        outs.append((S * qt).sum(-2))
    o = torch.stack(outs, 1)
    return torch.cat([o[i, :b - a] for i, (a, b) in enumerate(segs)]), S


def mixture(h, get, idx, weights, expert, weigh_input=False):
    """Every row's chosen experts: idx, weights [n, top]."""
    out = torch.zeros_like(h)
    for e in range(int(idx.max()) + 1):
        rows, place = (idx == e).nonzero(as_tuple=True)
        if rows.numel():
            w, x = weights[rows, place][:, None], h[rows]
            out.index_add_(0, rows, expert(w * x, f"e{e}", get) if weigh_input else w * expert(x, f"e{e}", get))
    return out


def clamped(x, name, get, limit):
    g, u = (x @ get(name + ".gate").T).clamp(max=limit), (x @ get(name + ".up").T).clamp(-limit, limit)
    return (g * torch.sigmoid(1.702 * g) * (u + 1)) @ get(name + ".down").T


def gated_silu(x, name, get):
    g = x @ get(name + ".gate").T
    return (g * torch.sigmoid(g) * (x @ get(name + ".up").T)) @ get(name + ".down").T


def rotary_exact(c, seed):
    r, model, segs = ROTARY, rotary_model(seed, False), spans(c)
    H, G, d = r["heads"], r["kv_heads"], r["width"] // r["heads"]
    x = model.embed[tokens_of(c, seed)].double()
    # cosines and sines are kept in bfloat16
    inv = 1.0 / (r["theta"] ** (torch.arange(0, d, 2, dtype=torch.float) / d))
    a = (positions_of(segs).float().cpu()[:, None] * inv[None])
    cos, sin = (t.bfloat16().double().to(DEVICE)[:, None] for t in (a.cos(), a.sin()))

    def rotated(y):
        u, v = y[..., :d // 2], y[..., d // 2:]
        return torch.cat([u * cos - v * sin, v * cos + u * sin], -1)
    for l in model.layers:
        q, k, v = (rms(x, EPS["rotary"], l.input_norm.double()) @ l.qkv.w.double().T).split([H * d, G * d, G * d], 1)
        q, k = rotated(q.reshape(-1, H, d)), rotated(k.reshape(-1, G, d))
        x = x + attend(q, k, v.reshape(-1, G, d), segs, d ** -0.5).reshape(x.shape[0], -1) @ l.o.w.double().T
        g, u = (rms(x, EPS["rotary"], l.post_norm.double()) @ l.gate_up.w.double().T).chunk(2, 1)
        x = x + (g * torch.sigmoid(g) * u) @ l.down.w.double().T
    return rms(x, EPS["rotary"], model.final_norm.double()), lambda h: h @ model.lm_head.w.double().T, []


def encoder_exact(c, seed):
    model, segs, H = encoder_model(seed), spans(c), ENCODER["heads"]
    width = ENCODER["width"]

    def norm(x, ln):
        x = x - x.mean(-1, keepdim=True)
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS["encoder"]) * ln[0].double() + ln[1].double()

    def lin(x, w, b):
        return x @ w.double().T + b.double()
    x = model.word_emb[tokens_of(c, seed)].double() + model.pos_emb[positions_of(segs).long() + 2].double() + model.type_emb[0].double()
    x = norm(x, model.emb_ln)
    for l in model.layers:
        q, k, v = (t.reshape(-1, H, width // H) for t in lin(x, l.qkv_w, l.qkv_b).chunk(3, 1))
        o = attend(q, k, v, segs, (width // H) ** -0.5, causal=False).reshape(-1, width)
        x = norm(x + lin(o, l.out_w, l.out_b), l.attn_ln)
        x = norm(x + lin(torch.nn.functional.gelu(lin(x, l.fc1_w, l.fc1_b)), l.fc2_w, l.fc2_b), l.out_ln)
    return x, None, []


def hybrid_exact(c, seed):
    w, segs, eps, states = tensors_of(c, seed), spans(c), EPS["hybrid"], []

    def norm(x, name):
        return torch.tanh(w[name + ".alpha"].double() * x) * w[name].double() + w[name + ".b"].double()

    def parallel(h, m, get):
        n, l, r = h.shape[0], m["left"], m["right"]

        def lin(s):
            return h @ get(s).T
        q = rms(lin("left.q").view(n, l["heads"], -1), eps, get("left.q.norm"))
        k = rms(lin("left.k").view(n, l["kv_heads"], -1), eps, get("left.k.norm"))
        o = attend(q, k, lin("left.v").view(n, l["kv_heads"], -1), segs, l["scale"]) * torch.sigmoid(lin("left.g"))[:, :, None]
        decay = torch.sigmoid(lin("right.a1") @ get("right.a2").T + get("right.a2.b")) ** (1 / r["tau"])
        shape = (n, r["heads"], -1)
        y, S = recur(lin("right.q").view(shape) * r["dim"] ** -0.5, lin("right.k").view(shape), lin("right.v").view(shape),
                     decay.view(shape), segs, "after")
        states.append(S)
        g = lin("right.g")
        y = rms(y, eps, get("right.norm")).reshape(n, -1) * g * torch.sigmoid(g)
        return m["left_scale"] * (o.reshape(n, -1) @ get("left.o").T) + m["right_scale"] * (y @ get("right.o").T)

    def wkv(h, m, get):
        n, shape = h.shape[0], (h.shape[0], m["heads"], m["dim"])
        before = torch.cat([h.new_zeros(1, h.shape[1]), h[:-1]])
        before[[a for a, _ in segs]] = 0

        def mixed(s):
            return h + (before - h) * get("mu." + s)
        r, k, v = ((mixed(s) @ get(s).T).view(shape) for s in "rkv")
        g = mixed("g") @ get("g").T
        z = torch.tanh(mixed("w") @ get("w1").T) @ get("w2").T + get("w0")
        o, S = recur(r, k, v, torch.exp(-torch.exp(z)).view(shape), segs, "before", bonus=get("u"))
        states.append(S)
        return (rms(o, eps).reshape(n, -1) * get("norm") * g * torch.sigmoid(g)) @ get("o").T
    x = w["embed"][tokens_of(c, seed)].double()
    for i, l in enumerate(HYBRID["layers"]):
        mix = parallel if l["type"] == "parallel" else wkv
        x = x + mix(norm(x, f"l{i}.norm1"), l["mixer"], lambda s: w[f"l{i}.mix.{s}"].double())
        u = norm(x, f"l{i}.norm2") @ w[f"l{i}.mlp.up"].double().T
        x = x + u.clamp(min=0).square() @ w[f"l{i}.mlp.down"].double().T
    return norm(x, "final.norm"), lambda h: h @ w["head"].double().T, states


def latent_exact(c, seed):
    w, segs, eps = tensors_of(c, seed), spans(c), EPS["latent"]
    x = w["embed"][tokens_of(c, seed)].double() * LATENT["embedding"]["scale"]
    streams, cached = [x], {}
    for i, l in enumerate(LATENT["layers"]):
        def get(s):
            return w[f"l{i}.{s}"].double()
        m, n = l["mixer"], x.shape[0]
        H, d, r, rank = m["heads"], m["dim"], m["rot_dim"], m["kv_rank"]
        angles = angles_of(segs, base_frequencies(m["rot"]))
        if m.get("kv_from") is None:
            z = x @ get("mix.dkv").T
            cached[i] = rms(z[:, :rank], eps, get("mix.dkv.norm")), turn(z[:, None, rank:], angles, False)
        lat, rot = cached[m.get("kv_from", i)]
        q = (x @ get("mix.q").T).view(n, H, d + r)
        q = torch.cat([q[..., :d], turn(q[..., d:], angles, False)], -1)
        k = torch.cat([(lat @ get("mix.uk").T).view(n, H, d), rot.expand(n, H, r)], -1)
        o = attend(q, k, (lat @ get("mix.uv").T).view(n, H, -1), segs, m["scale"], window=m["mask"]["size"])
        o = (o * torch.sigmoid(x @ get("mix.g").T)[:, :, None]).reshape(n, -1) @ get("mix.o").T
        x = x + rms(o, eps, get("norm1"))
        mlp = l["mlp"]
        value, idx = torch.topk(x @ get("mlp.router").T + get("mlp.router.b"), mlp["router"]["top"], -1)

        def expert(y, name, g, limit=mlp["expert"]["limit"]):
            return clamped(y, name, g, limit)
        y = mixture(x, lambda s: get("mlp." + s), idx, torch.softmax(value, -1), expert)
        y = y + torch.sigmoid(x @ get("mlp.shared.sg").T) * expert(x, "shared", lambda s: get("mlp." + s), mlp["shared"]["limit"])
        x = x + rms(y, eps, get("norm2"))
        streams.append(x)
        x = sum(p * s for p, s in zip(get("dwa"), streams))
    return rms(x, eps, w["final.norm"].double()), lambda h: h @ w["head"].double().T, []


def local_exact(c, seed):
    w, segs, eps, states = tensors_of(c, seed), spans(c), EPS["local"], []

    def heads(h, m, get, bias, norms=False, two=False):
        n, H, G, maps = h.shape[0], m["heads"], m["kv_heads"], 2 if two else 1

        def lin(x, s):
            return x @ get(s).T + (get(s + ".b") if bias else 0)
        q, k = lin(h, "q"), lin(h, "k")
        v = k if norms else lin(h, "v")
        if norms:
            q, k = rms(q, eps, get("q.norm")), rms(k, eps, get("k.norm"))
        angles = angles_of(segs, wave_frequencies(m["rot"]))
        q, k = (turn(t.reshape(n, -1, m["dim"]), angles, True).view(n, g, maps, -1) for t, g in ((q, H), (k, G)))
        v = v.reshape(n, G, -1)
        kind = {"chunk" if bias and not norms else "window": m["mask"]["size"]}
        a = [attend(q[:, :, j], k[:, :, j], v, segs, m["scale"], first=m["mask"].get("keep_first", 0), cap=m.get("softcap", 0.0),
                    sink=get("sink") if norms else None, **kind) for j in range(maps)]
        if two:
            weight = torch.exp((get("lq1") * get("lk1")).sum()) - torch.exp((get("lq2") * get("lk2")).sum()) + m["diff"]
            a = [rms(a[0] - weight * a[1], eps) * (1 - m["diff"])]
        return lin(a[0].reshape(n, -1), "o")

    def retention(h, m, get):
        n, shape = h.shape[0], (h.shape[0], m["heads"], -1)
        angles = angles_of(segs, wave_frequencies(m["rot"]))
        q, k = (turn((h @ get(s).T).view(shape), angles, True) for s in "qk")
        decay = torch.tensor(m["decay"], dtype=torch.float64, device=DEVICE)[None, :, None].expand(n, m["heads"], m["dim"])
        # (the keys' scale may go to the queries: states hold unscaled keys)
        o, S = recur(q * m["dim"] ** -0.5, k, (h @ get("v").T).view(shape), decay, segs, "after")
        states.append(S)
        g = h @ get("g").T
        return (rms(o, eps).reshape(n, -1) * g * torch.sigmoid(g)) @ get("o").T
    ids, b = tokens_of(c, seed), LOCAL["embedding"]["bigram"]
    pair = (torch.cat([ids[:1], ids[:-1]]) * b["mul_prev"] + ids * b["mul_cur"]) % b["buckets"]
    pair[[a for a, _ in segs]] = b["buckets"]
    x = w["embed"][ids].double() + w["bigram"][pair].double()
    for i, l in enumerate(LOCAL["layers"]):
        def get(s):
            return w[f"l{i}.{s}"].double()

        def of(p):
            return lambda s: get(p + s)
        h, m = rms(x, eps, get("norm1")), l["mixer"]
        if l["type"] == "parallel":
            y = (rms(heads(h, m["left"], of("mix.left."), True), eps, get("mix.left.out"))
                 + rms(retention(h, m["right"], of("mix.right.")), eps, get("mix.right.out"))) / 2
        else:
            y = heads(h, m, of("mix."), l["type"] == "attention", norms=l["type"] == "attention", two=l["type"] == "attention_2")
        x = x + rms(y, eps, get("norm1b"))
        h, mlp = rms(x, eps, get("norm2")), l["mlp"]
        if mlp["kind"] == "dense":
            y = clamped(h, "mlp", get, mlp["limit"])
        else:
            value, idx = torch.topk(h @ get("mlp.router").T, mlp["router"]["top"], -1)
            y = mixture(h, of("mlp."), idx, torch.sigmoid(value), gated_silu, weigh_input=True) + gated_silu(h, "shared", of("mlp."))
        x = x + rms(y, eps, get("norm2b"))
    return rms(x, eps, w["final.norm"].double()), lambda h: h @ w["head"].double().T, states


def stream_exact(c, seed):
    w, segs, eps, states = tensors_of(c, seed), spans(c), EPS["stream"], []

    def latent(h, m, get):
        n, H, d, r, rank = h.shape[0], m["heads"], m["dim"], m["rot_dim"], m["kv_rank"]
        angles, grow = angles_of(segs, ramp_frequencies(m["rot"])), 0.1 * math.log(m["rot"]["scaling"]["factor"]) + 1
        q = (rms(h @ get("dq").T, eps, get("dq.norm")) @ get("uq").T).view(n, H, d + r)
        kv = h @ get("dkv").T
        lat = rms(kv[:, :rank], eps, get("dkv.norm"))
        q = torch.cat([q[..., :d], turn(q[..., d:], angles, True, grow)], -1)
        k = torch.cat([(lat @ get("uk").T).view(n, H, d), turn(kv[:, None, rank:], angles, True, grow).expand(n, H, r)], -1)
        o = attend(q, k, (lat @ get("uv").T).view(n, H, -1), segs, m["scale"], sink=get("sink"))
        return o.reshape(n, -1) @ get("o").T

    def delta(h, m, get):
        n, shape = h.shape[0], (h.shape[0], m["heads"], -1)

        def conv(s):
            y, taps = h @ get(s).T, get(s + ".conv")
            out = y * taps[:, -1]
            for back in range(1, taps.shape[1]):
                late = torch.cat([y.new_zeros(back, y.shape[1]), y[:-back]])
                for a, b in segs:
                    late[a:min(a + back, b)] = 0
                out = out + late * taps[:, -1 - back]
            return (out * torch.sigmoid(out)).view(shape)

        def unit(x):
            return x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)
        q, k, v = conv("q"), conv("k"), conv("v")
        z = (h @ get("a1").T) @ get("a2").T + get("dt_bias")
        decay = torch.exp(-torch.exp(get("A_log"))[:, None] * torch.nn.functional.softplus(z, threshold=30).view(shape))
        o, S = recur(unit(q) * m["dim"] ** -0.5, unit(k), v, decay, segs, "delta", beta=torch.sigmoid(h @ get("b").T))
        states.append(S)
        gate = torch.sigmoid((h @ get("g1").T) @ get("g2").T).view(shape)
        return (rms(o, eps, get("norm")) * gate).reshape(n, -1) @ get("o").T

    def experts(h, mlp, get):
        r = mlp["router"]
        s, count = torch.softmax(h @ get("router").T, -1), r["groups"]["count"]
        best = s.view(h.shape[0], count, -1).amax(-1).topk(r["groups"]["keep"], -1).indices
        open_ = torch.zeros(h.shape[0], count, dtype=torch.bool, device=DEVICE).scatter_(1, best, True)
        value, idx = s.masked_fill(~open_.repeat_interleave(s.shape[1] // count, 1), -1.0).topk(r["top"], -1)
        weights = value / (value.sum(-1, keepdim=True) + 1e-20) * r["scale"]
        return mixture(h, get, idx, weights, lambda x, e, g: (x @ g(e + ".up").T).clamp(min=0).square() @ g(e + ".down").T)

    def feed_forward(h, mlp, get):
        return gated_silu(h, "mlp", get) if mlp["kind"] == "dense" else experts(h, mlp, lambda s: get("mlp." + s))
    x = w["embed"][tokens_of(c, seed)].double().expand(STREAM["streams"], -1, -1)
    for i, l in enumerate(STREAM["layers"]):
        def get(s):
            return w[f"l{i}.{s}"].double()
        mixer = latent if l["type"] == "latent_attention" else delta
        for q, sub in (1, lambda h: mixer(h, l["mixer"], lambda s: get("mix." + s))), (2, lambda h: feed_forward(h, l["mlp"], get)):
            h = (get(f"hc{q}.in")[:, None, None] * x).sum(0)
            y = sub(rms(h, eps, get(f"norm{q}")))
            mix = get(f"hc{q}.mix")
            x = torch.stack([(mix[:, t, None, None] * x).sum(0) + get(f"hc{q}.out")[t] * y for t in range(x.shape[0])])
    return rms(x.sum(0), eps, w["final.norm"].double()), lambda h: h @ w["embed"].double().T, states


@torch.inference_mode()
def exact(c, seed):
    """Whole sequences from their first token; a decode step's rows are the last ones.  None where a sequence's recurrence or a large
    batch would take long, and where activations are rounded to 8 bits on the way."""
    if c["fp8"] or sum(lengths(c)) * (4 if c["model"] in ("hybrid", "local", "stream") and c["tokens"] > 3000 else 1) > 40000:
        return None
    restated = {"rotary": rotary_exact, "encoder": encoder_exact, "hybrid": hybrid_exact, "latent": latent_exact, "local": local_exact,
                "stream": stream_exact}[c["model"]]
    hidden, head, states = restated(c, seed)
    if head is None:
        return {"hidden": hidden}
    last = torch.tensor([b - 1 for _, b in spans(c)], device=DEVICE)
    return {"hidden": hidden[last] if c["phase"] == "decode" else hidden, "logits": head(hidden[last]), "states": states}
