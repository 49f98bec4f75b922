"""Encoder of the encode-only workflow: the XLM-RoBERTa / BERT layer sequence of
light_vllm/encode_only/modelzoo/xlm_roberta.py (bge-m3's backbone): embeddings
(word + position + token type, LayerNorm), then per layer fused QKV projection -> bidirectional
attention -> output projection -> add & LayerNorm -> GELU MLP -> add & LayerNorm.

Attention is this package's HIP varlen kernel (AttentionType.ENCODER); the residual add and the LayerNorm
behind it are one launch (`_C_amd.add_layer_norm`; the reference leaves both to torch),
exact GELU leaves the projection in front of it (csrc/tile_linear.hip, csrc/prompt_product.hip) or is an in-place kernel of this package; batches
of up to some thousand rows take this package's products where those are faster (csrc/prompt_product.h), the rest library GEMMs.
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
    """A layer's weights: attributes that may be read, written to and assigned at any time.

    Prompts of some hundreds of rows take this package's kernels, which read a weight in fragment order, from a copy that is made with the layer.
    It is read only as long as nobody but the model has the weight: who reads or assigns an attribute may write to the tensor from then on, also in
    ways that torch does not count (`lw.qkv_w.data.copy_`), so that the model takes the weight itself.  lay_out() behind the last write lays the
    copies out anew; prompts are as fast as before it.  A captured forward runs the same kernels as others (what it has not run before, the library
    cannot load under capture) over copies that the graph makes at each replay, which so sees every write: 20 us a layer of 1024 x 4096."""

    WEIGHTS = "qkv_w", "out_w", "fc1_w", "fc2_w"

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
        self._fused, self._kept, self._copies = cfg.fused_layer_norm, {}, {}  # _kept: weights that only the model has
        self.lay_out()

    def __getattr__(self, name: str):
        """A weight that only the model had: from now on it is an attribute as any other."""
        kept = self.__dict__.get("_kept", {})
        if name not in kept:
            raise AttributeError(name)
        self.__dict__.setdefault(name, kept[name])
        return self.__dict__[name]

    def weight(self, name: str) -> torch.Tensor:
        w = self.__dict__.get(name)
        if w is None:
            return self._kept[name]
        if self._kept.get(name, w) is not w:  # (assigned: what was there before goes)
            self._kept.pop(name, None)
            self._copies.pop(name, None)
        return w

    def lay_out(self) -> None:
        """The weights stay as they are now: prompts may take copies of them in fragment order.  Writes that torch counts, and new assignments,
        are seen after it as well; behind others it is called again.  As with a write, no forward may be under way."""
        kept = {name: self.weight(name) for name in self.WEIGHTS}
        self._copies = {name: self._copy(w) for name, w in kept.items() if self._takes(w)}
        self._kept = kept
        for name in self.WEIGHTS:
            self.__dict__.pop(name, None)

    def _takes(self, w: torch.Tensor) -> bool:
        return (self._fused and w.is_cuda and w.dtype == torch.bfloat16 and w.dim() == 2 and w.is_contiguous() and w.shape[0] % 16 == 0
                and w.shape[1] % 32 == 0)

    @staticmethod
    def _version(w: torch.Tensor) -> int:
        return -1 if w.is_inference() else w._version

    def _copy(self, w: torch.Tensor):
        """(the weight, its memory, which nothing else can have meanwhile, its version, the weight in fragment order)"""
        copy = w, w.detach(), self._version(w), torch.ops._C_amd.pack_weight(w)
        torch.cuda.synchronize(w.device)  # (the next forward may come on another stream, and one may still read the copy before)
        return copy

    def _renewed(self, name: str, w: torch.Tensor) -> Optional[torch.Tensor]:
        """`w` in fragment order (None: what the kernels do not take), laid out anew when it is another tensor or has been written to since, as far
        as torch counts that."""
        if not self._takes(w):
            return None
        was = self._copies.get(name)
        if was is None or was[0] is not w or was[1].data_ptr() != w.data_ptr() or was[2] != self._version(w):
            was = self._copies[name] = self._copy(w)
        return was[3]

    def packed(self, name: str) -> Optional[torch.Tensor]:
        """A weight in fragment order, None where somebody else has it."""
        return None if name in self.__dict__ else self._renewed(name, self._kept[name])

    @property
    def fc1_packed(self) -> Optional[torch.Tensor]:
        """fc1_w in fragment order for the kernel with GELU behind the product of long prompts.  Writes that torch does not count
        (`fc1_w.data.copy_`, or to inference tensors) are not seen: assign fc1_w or lay_out() behind those."""
        return self._renewed("fc1_w", self.weight("fc1_w"))

    def fc1_packed_in_graph(self) -> Optional[torch.Tensor]:
        """... a copy that the graph under capture makes at each replay."""
        w = self.weight("fc1_w")
        return torch.ops._C_amd.pack_weight(w) if self._takes(w) else None


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
        captured = emb.is_cuda and torch.cuda.is_current_stream_capturing()

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
            w, y = lw.weight(name), None
            if fused and a.shape[0] > 64:
                packed = w if captured else lw.packed(name)
                if packed is not None:
                    y = torch.ops._C_amd.prompt_product(a, packed, bias, w.shape[0], gelu, slabs and hid <= 2048, False, captured)
            return F.linear(a, w, bias) if y is None and not gelu else y

        def fc1_gelu(a, lw):
            h = product(a, lw, "fc1_w", lw.fc1_b, gelu=True)
            packed = (lw.fc1_packed_in_graph() if captured else lw.fc1_packed) if fused and h is None and a.shape[0] > 64 else None
            if packed is not None:
                h = torch.ops._C_amd.prompt_linear(a, None, packed, lw.fc1_b, packed.shape[0], PROMPT_ACTS["gelu"])
            if h is not None:
                return h
            h = F.linear(a, lw.weight("fc1_w"), lw.fc1_b)
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
                    torch.addmm(lw.fc2_b, hb, lw.weight("fc2_w").t(), out=y[r0:r0 + blk])
            else:
                y = product(fc1_gelu(x, lw), lw, "fc2_w", lw.fc2_b, slabs=True)
            x = add_ln(x, y, lw.out_ln, lw.fc2_b)
        return x
