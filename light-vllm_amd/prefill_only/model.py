"""Encoder of the encode-only workflow: the XLM-RoBERTa / BERT layer sequence of
light_vllm/encode_only/modelzoo/xlm_roberta.py (bge-m3's backbone): embeddings
(word + position + token type, LayerNorm), then per layer fused QKV projection -> bidirectional
attention -> output projection -> add & LayerNorm -> GELU MLP -> add & LayerNorm.

Attention is this package's HIP varlen kernel (AttentionType.ENCODER); the residual add and the LayerNorm
behind it are one launch (`_C_amd.add_layer_norm`; the reference leaves both to torch),
exact GELU leaves the projection in front of it (csrc/tile_linear.hip) or is an in-place kernel of this package; the other projections
are library GEMMs (prompt batches are hundreds to thousands of rows).
Weights are random-initialised: no checkpoint is available offline."""
from dataclasses import dataclass
from typing import List, Optional

import torch
import torch.nn.functional as F

from ..attention.prefill_only import AttentionType, PrefillOnlyHIPVarlenBackend
from ..engine.model import PROMPT_ACTS


@dataclass
class EncoderConfig:
    hidden_size: int = 1024
    intermediate_size: int = 4096
    num_hidden_layers: int = 24
    num_attention_heads: int = 16
    vocab_size: int = 250002
    max_position_embeddings: int = 8194
    layer_norm_eps: float = 1e-5
    pad_token_id: int = 1
    dtype: torch.dtype = torch.bfloat16
    fused_layer_norm: bool = True  # residual add + LayerNorm in one launch (lvllm_add_layer_norm); off = A/B runs
    # > 0: the MLP runs over row blocks of this many tokens (fc1 -> GELU -> fc2 per block), so that the block's
    # intermediate [rows, intermediate] is still in the L2s / the Infinity Cache when GELU and fc2 read it instead of
    # making two round trips through HBM (134 MB each way at 16 384 tokens); 0 = one pass over all tokens
    mlp_block_tokens: int = 0

    @property
    def head_dim(self) -> int:
        return self.hidden_size // self.num_attention_heads

    @staticmethod
    def bge_m3(dtype=torch.bfloat16) -> "EncoderConfig":
        return EncoderConfig(dtype=dtype)

    @staticmethod
    def tiny(dtype=torch.bfloat16) -> "EncoderConfig":
        return EncoderConfig(hidden_size=128, intermediate_size=256, num_hidden_layers=2, num_attention_heads=2,
                             vocab_size=512, max_position_embeddings=1024, dtype=dtype)


class EncoderLayerWeights:
    def __init__(self, cfg: EncoderConfig, device, gen: torch.Generator):
        hid, inter = cfg.hidden_size, cfg.intermediate_size

        def w(*shape, std=0.02):
            with torch.inference_mode(False):  # (torch counts writes to these, wherever the model is made)
                return (torch.randn(*shape, generator=gen, device=device, dtype=torch.float32) * std).to(cfg.dtype)

        def ln():
            return ((1.0 + 0.05 * torch.randn(hid, generator=gen, device=device)).to(cfg.dtype),
                    (0.02 * torch.randn(hid, generator=gen, device=device)).to(cfg.dtype))

        self.qkv_w, self.qkv_b = w(3 * hid, hid), w(3 * hid)
        self.out_w, self.out_b = w(hid, hid), w(hid)
        self.attn_ln = ln()
        self.fc1_w, self.fc1_b = w(inter, hid), w(inter)
        self.fc2_w, self.fc2_b = w(hid, inter), w(hid)
        self.out_ln = ln()
        self._fused, self._packed = cfg.fused_layer_norm, {}
        for name in self.WEIGHTS:
            self.packed(name)  # (laid out now, and not in the first forward)

    WEIGHTS = "qkv_w", "out_w", "fc1_w", "fc2_w"

    def packed(self, name: str) -> Optional[torch.Tensor]:
        """A weight once more in fragment order, for this package's kernels (None: what they do not take).  Laid out anew when the weight has been
        replaced or written to since.  Writes that torch does not count (`fc1_w.data.copy_`, or to inference tensors) are not seen: assign the
        weight behind those."""
        w = getattr(self, name)
        if not (self._fused and w.is_cuda and w.dtype == torch.bfloat16 and w.is_contiguous() and w.shape[0] % 16 == 0 and w.shape[1] % 32 == 0):
            return None
        version = -1 if w.is_inference() else w._version
        was = self._packed.get(name)  # (the weight, its memory, which nothing else can have meanwhile, and its version then, the copy)
        if was is None or was[0] is not w or was[1].data_ptr() != w.data_ptr() or was[2] != version:
            if torch.cuda.is_current_stream_capturing():  # (a copy that only the graph would write)
                return None
            was = w, w.detach(), version, torch.ops._C_amd.pack_weight(w)
            torch.cuda.current_stream(w.device).synchronize()  # (the next forward may come on another stream)
            self._packed[name] = was
        return was[3]

    @property
    def fc1_packed(self) -> Optional[torch.Tensor]:
        return self.packed("fc1_w")


class EncoderModel:
    """forward(input_ids [T], positions [T], attn_metadata) -> hidden states [T, hidden]."""

    def __init__(self, cfg: EncoderConfig, device="cuda:0", seed: int = 0):
        self.cfg = cfg
        self.device = torch.device(device)
        gen = torch.Generator(device=self.device).manual_seed(seed)

        def emb(n):
            return (torch.randn(n, cfg.hidden_size, generator=gen, device=self.device) * 0.02).to(cfg.dtype)

        self.word_emb, self.pos_emb, self.type_emb = emb(cfg.vocab_size), emb(cfg.max_position_embeddings), emb(1)
        self.emb_ln = ((1.0 + 0.05 * torch.randn(cfg.hidden_size, generator=gen, device=self.device)).to(cfg.dtype),
                       (0.02 * torch.randn(cfg.hidden_size, generator=gen, device=self.device)).to(cfg.dtype))
        self.layers: List[EncoderLayerWeights] = [EncoderLayerWeights(cfg, self.device, gen)
                                                  for _ in range(cfg.num_hidden_layers)]
        self.backend = PrefillOnlyHIPVarlenBackend(AttentionType.ENCODER)
        self.attn = self.backend.get_impl_cls()(cfg.num_attention_heads, cfg.head_dim, cfg.head_dim ** -0.5,
                                                cfg.num_attention_heads, None, None, "auto")

    def forward(self, input_ids: torch.Tensor, positions: torch.Tensor, attn_metadata) -> torch.Tensor:
        cfg = self.cfg
        eps = cfg.layer_norm_eps
        hid = cfg.hidden_size
        emb, shift = self.word_emb, cfg.pad_token_id + 1  # xlm_roberta.py: position ids start after the padding index
        fused = emb.is_cuda and hid % 8 == 0 and emb.dtype in (torch.bfloat16, torch.float16) and self.cfg.fused_layer_norm

        def add_ln(a, b, ln, b_bias=None):  # LayerNorm(a + b), b optional; slabs: without their bias
            if b is not None and b.dim() == 3:
                out = torch.empty_like(a)
                torch.ops._C_amd.add_layer_norm_slabs(out, a, b, b_bias, ln[0], ln[1], eps)
                return out
            if fused:
                out = torch.empty_like(a)
                torch.ops._C_amd.add_layer_norm(out, a, b, ln[0], ln[1], eps)
                return out
            return F.layer_norm(a if b is None else a + b, (hid,), ln[0], ln[1], eps)

        def product(a, lw, name, bias, slabs=False, gelu=False):
            """This package's kernels where they are the better ones (csrc/prompt_product.h)."""
            packed = lw.packed(name) if fused and a.shape[0] > 64 else None
            y = None
            if packed is not None:
                y = torch.ops._C_amd.prompt_product(a, packed, bias, packed.numel() // a.shape[1], gelu, slabs and hid <= 2048)
            return F.linear(a, getattr(lw, name), bias) if y is None and not gelu else y

        def fc1_gelu(a, lw):
            h = product(a, lw, "fc1_w", lw.fc1_b, gelu=True)
            packed = lw.fc1_packed if fused and h is None else None
            if packed is not None:
                h = torch.ops._C_amd.prompt_linear(a, None, packed, lw.fc1_b, cfg.intermediate_size, PROMPT_ACTS["gelu"])
            if h is not None:
                return h
            h = F.linear(a, lw.fc1_w, lw.fc1_b)
            if fused and h.numel() % 8 == 0:
                torch.ops._C_amd.gelu(h, h)  # exact GELU in place
                return h
            return F.gelu(h)

        if (fused and hid <= 2048 and input_ids.dtype == positions.dtype == torch.int64
                and all(t.is_contiguous() and t.data_ptr() % 16 == 0 for t in (self.word_emb, self.pos_emb, self.type_emb[0]))):  # (one launch)
            x = torch.ops._C_amd.embed_layer_norm(input_ids.contiguous(), positions.contiguous(), shift, self.word_emb, self.pos_emb,
                                                  self.type_emb[0], *self.emb_ln, eps)
        else:
            x = F.embedding(input_ids, self.word_emb) + F.embedding(positions + shift, self.pos_emb) + self.type_emb[0]
            x = add_ln(x, None, self.emb_ln)
        for lw in self.layers:
            qkv = product(x, lw, "qkv_w", lw.qkv_b)
            q, k, v = qkv.split([hid, hid, hid], dim=-1)  # strided views of the fused projection
            a = self.attn.forward(q, k, v, None, attn_metadata, attn_type=AttentionType.ENCODER)
            x = add_ln(x, product(a, lw, "out_w", lw.out_b, slabs=True), lw.attn_ln, lw.out_b)
            blk = cfg.mlp_block_tokens
            if blk > 0 and x.shape[0] > blk:
                y = torch.empty_like(x)
                for r0 in range(0, x.shape[0], blk):
                    hb = fc1_gelu(x[r0:r0 + blk], lw)
                    torch.addmm(lw.fc2_b, hb, lw.fc2_w.t(), out=y[r0:r0 + blk])
            else:
                y = product(fc1_gelu(x, lw), lw, "fc2_w", lw.fc2_b, slabs=True)
            x = add_ln(x, y, lw.out_ln, lw.fc2_b)
        return x
