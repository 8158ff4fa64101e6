"""Qwen3 (dense) over a flat continuous batch, on the HIP kernels (reference:
src/miniserve/model/qwen3.py).

Same module tree, parameter names and call signatures as the reference, so checkpoints, the
loader's fused row order ([q | k | v] and [gate | up]) and the runner plug in unchanged, and each
module's ``forward`` computes what the reference's does.

Once every linear is int8, ``Qwen3ForCausalLM.forward`` runs the layers as fused pipelines that
cross module boundaries (no workgroup ever waits on another):
  * batches up to 256 tokens (decode steps, short chunks): the token-split kernels, five
    launches per layer -- [embedding gather (layer 0) + input RMSNorm + int8 qkv + q/k-norm +
    RoPE + KV write] -> [paged attention] -> [int8 o + residual] -> [post-attention RMSNorm +
    int8 gate_up + silu * up] -> [int8 down + residual];
  * larger batches (prefill chunks): the LDS-tiled int8 GEMM with residual / silu * up epilogues,
    RMSNorm and q/k-norm + RoPE + KV write as their own kernels.
Logits are computed only for sampled rows; ``greedy`` fuses the final norm, LM head and argmax.
"""

from __future__ import annotations

import json
from dataclasses import dataclass
from pathlib import Path
from typing import Any

import torch
import torch.nn.functional as F
from torch import Tensor, nn

from miniserve_amd import kernels
from miniserve_amd.attention.backends import AttentionMetadata, attend, attend_decode_qkv
from miniserve_amd.model.layers import RMSNorm, RotaryEmbedding, SwiGLU
from miniserve_amd.quant.int8 import Int8Linear


@dataclass(frozen=True)
class Qwen3Config:
    """model/qwen3.py:18-62."""

    vocab_size: int
    hidden_size: int
    intermediate_size: int
    num_hidden_layers: int
    num_attention_heads: int
    num_key_value_heads: int
    head_dim: int
    rms_norm_eps: float
    rope_theta: float
    max_position_embeddings: int
    tie_word_embeddings: bool

    @classmethod
    def from_dict(cls, d: dict[str, Any]) -> Qwen3Config:
        rope = d.get("rope_parameters") or {}
        return cls(
            vocab_size=d["vocab_size"],
            hidden_size=d["hidden_size"],
            intermediate_size=d["intermediate_size"],
            num_hidden_layers=d["num_hidden_layers"],
            num_attention_heads=d["num_attention_heads"],
            num_key_value_heads=d["num_key_value_heads"],
            head_dim=d.get("head_dim") or d["hidden_size"] // d["num_attention_heads"],
            rms_norm_eps=d["rms_norm_eps"],
            rope_theta=float(d.get("rope_theta") or rope.get("rope_theta") or 10000.0),
            max_position_embeddings=d["max_position_embeddings"],
            tie_word_embeddings=bool(d.get("tie_word_embeddings", False)),
        )

    @classmethod
    def from_pretrained(cls, model_dir: str | Path) -> Qwen3Config:
        return cls.from_dict(json.loads((Path(model_dir) / "config.json").read_text()))

    def kv_bytes_per_token(self, dtype_bytes: int) -> int:
        """K and V for every layer: 2 x layers x kv_heads x head_dim x bytes."""
        return 2 * self.num_hidden_layers * self.num_key_value_heads * self.head_dim * dtype_bytes


class Qwen3Attention(nn.Module):
    def __init__(self, cfg: Qwen3Config) -> None:
        super().__init__()
        self.num_heads = cfg.num_attention_heads
        self.num_kv_heads = cfg.num_key_value_heads
        self.head_dim = cfg.head_dim
        self.q_size = self.num_heads * self.head_dim
        self.kv_size = self.num_kv_heads * self.head_dim
        self.scale = self.head_dim**-0.5
        self.qkv_proj: nn.Module = nn.Linear(cfg.hidden_size, self.q_size + 2 * self.kv_size, bias=False)
        self.o_proj: nn.Module = nn.Linear(self.q_size, cfg.hidden_size, bias=False)
        self.q_norm = RMSNorm(self.head_dim, cfg.rms_norm_eps)
        self.k_norm = RMSNorm(self.head_dim, cfg.rms_norm_eps)

    def forward(
        self,
        x: Tensor,
        cos: Tensor,
        sin: Tensor,
        k_cache: Tensor,
        v_cache: Tensor,
        meta: AttentionMetadata,
    ) -> Tensor:
        """model/qwen3.py:84-101: qkv -> q/k-norm -> RoPE -> paged attention -> o."""
        t = x.shape[0]
        qkv = self.qkv_proj(x)
        q = kernels.qk_norm_rope_cache(
            qkv, self.num_heads, self.num_kv_heads, self.head_dim, self.q_norm.weight, self.k_norm.weight,
            self.q_norm.eps, cos, sin, meta.slot_mapping, k_cache, v_cache,
        )
        out = attend(q, k_cache, v_cache, meta, self.scale)
        result: Tensor = self.o_proj(out.view(t, self.q_size))
        return result


class Qwen3DecoderLayer(nn.Module):
    def __init__(self, cfg: Qwen3Config) -> None:
        super().__init__()
        self.input_layernorm = RMSNorm(cfg.hidden_size, cfg.rms_norm_eps)
        self.self_attn = Qwen3Attention(cfg)
        self.post_attention_layernorm = RMSNorm(cfg.hidden_size, cfg.rms_norm_eps)
        self.mlp = SwiGLU(cfg.hidden_size, cfg.intermediate_size)

    def forward(
        self,
        x: Tensor,
        cos: Tensor,
        sin: Tensor,
        k_cache: Tensor,
        v_cache: Tensor,
        meta: AttentionMetadata,
    ) -> Tensor:
        """x += attn(norm(x)); x += mlp(norm(x))  (model/qwen3.py:112-122)."""
        a = self.self_attn(self.input_layernorm(x), cos, sin, k_cache, v_cache, meta)
        x2, h = kernels.add_rmsnorm(x, a, self.post_attention_layernorm.weight, self.post_attention_layernorm.eps)
        return self.mlp(h, residual=x2)


class Qwen3ForCausalLM(nn.Module):
    def __init__(self, cfg: Qwen3Config, max_positions: int) -> None:
        super().__init__()
        self.cfg = cfg
        self.embed_tokens = nn.Embedding(cfg.vocab_size, cfg.hidden_size)
        self.layers = nn.ModuleList(Qwen3DecoderLayer(cfg) for _ in range(cfg.num_hidden_layers))
        self.norm = RMSNorm(cfg.hidden_size, cfg.rms_norm_eps)
        self.rotary = RotaryEmbedding(cfg.head_dim, max_positions, cfg.rope_theta)
        self.lm_head: nn.Linear | None = (
            None if cfg.tie_word_embeddings else nn.Linear(cfg.hidden_size, cfg.vocab_size, bias=False)
        )
        # Token-split batches of up to DEC_MAX_TOKENS tokens run their linears on the decode kernel;
        # False keeps them on the rows kernel. Both round where the reference rounds (weights as
        # bf16(q * s), the normed activations as bf16(w * bf16(x * r))): the flag selects the kernel
        # only (a second implementation of the same values, kept for comparison).
        self.decode_linears = True

    def forward(
        self,
        input_ids: Tensor,
        positions: Tensor,
        kv_caches: list[tuple[Tensor, Tensor]],
        meta: AttentionMetadata,
    ) -> Tensor:
        """input_ids, positions: [T]. Returns final hidden states [T, hidden] (qwen3.py:140-153).
        (Decode batches whose linears are all within the token-split kernels take each row's position
        from its plan, context length - 1.)"""
        if len(kv_caches) != len(self.layers):
            raise ValueError(f"{len(kv_caches)} KV caches for {len(self.layers)} layers")
        if self._token_split_ok(input_ids.numel()):
            residual = self._token_split_layers(input_ids, positions, kv_caches, meta)
            out: Tensor = self.norm(residual)
            return out
        if self._wide_decode_ok(input_ids.numel(), meta):
            return self._wide_decode_layers(input_ids, positions, kv_caches, meta)
        x = self.embed_tokens(input_ids)
        cos, sin = self.rotary(positions)
        if self._all_int8():
            return self._fused_forward(x, cos, sin, kv_caches, meta)
        for layer, (k_cache, v_cache) in zip(self.layers, kv_caches, strict=True):
            x = layer(x, cos, sin, k_cache, v_cache, meta)
        out = self.norm(x)
        return out

    def greedy(
        self,
        input_ids: Tensor,
        positions: Tensor,
        kv_caches: list[tuple[Tensor, Tensor]],
        meta: AttentionMetadata,
        logits_rows: Tensor,
    ) -> Tensor:
        """Greedy next token of each row in ``logits_rows``: the argmax of
        ``compute_logits(forward(...)[logits_rows])`` (runner/model_runner.py:214-221 with
        runner/sampler.py:59), with the final norm, LM head and argmax in one kernel pair."""
        if len(kv_caches) != len(self.layers):
            raise ValueError(f"{len(kv_caches)} KV caches for {len(self.layers)} layers")
        weight = self.embed_tokens.weight if self.lm_head is None else self.lm_head.weight
        if self._token_split_ok(input_ids.numel()):
            residual = self._token_split_layers(input_ids, positions, kv_caches, meta)
            return kernels.lm_head_argmax(residual, logits_rows, self.norm.weight, self.norm.eps, weight)
        hidden = self.forward(input_ids, positions, kv_caches, meta)
        rows = hidden[logits_rows]
        if kernels.rows_supported(self.cfg.hidden_size) and rows.shape[0] > 0:
            all_rows = torch.arange(rows.shape[0], device=rows.device)
            return kernels.lm_head_argmax(rows, all_rows, self.norm.weight, self.norm.eps, weight, prenormed=True)
        return self.compute_logits(rows).argmax(dim=-1)

    def _all_int8(self) -> bool:
        return all(
            isinstance(m, Int8Linear)
            for layer in self.layers
            for m in (layer.self_attn.qkv_proj, layer.self_attn.o_proj, layer.mlp.gate_up_proj, layer.mlp.down_proj)
        )

    def _token_split_ok(self, tokens: int) -> bool:
        """Whether the token-split layer pipeline serves this batch: every linear int8, at most
        ROWS_MAX_TOKENS tokens, head_dim 128 and the activation tiles within LDS."""
        cfg = self.cfg
        return (
            0 < tokens <= kernels.ROWS_MAX_TOKENS
            and cfg.head_dim == 128
            and kernels.rows_supported(cfg.hidden_size)
            and kernels.rows_supported(cfg.num_attention_heads * cfg.head_dim)
            and kernels.rows_supported(cfg.intermediate_size)
            and self._all_int8()
        )

    def _wide_decode_ok(self, tokens: int, meta: AttentionMetadata) -> bool:
        """Whether a batch takes the large-weight decode layers: decode rows only, fewer than
        DEC_MAX_TOKENS (from there on the layer loop's qkv GEMM norms and rotates in its own epilogue: two
        layers of the 8B shape at 128 tokens 392.9 us here, 392.1 there; of 64 heads over 8 767.9, 745.8),
        head_dim 128, int8 linears of WIDE_MIN_WEIGHTS and more (the 8B shape). Their attention writes
        the new keys itself and attends to them from registers, which is the layer loop's write followed
        by its read only when every token is a plan row known to own its slot."""
        cfg = self.cfg
        return (
            meta.prefill is None
            and meta.decode is not None
            and meta.decode.own_slots is True
            and 0 < tokens < kernels.DEC_MAX_TOKENS
            and meta.decode.num_seqs == tokens
            and cfg.head_dim == 128
            and cfg.num_attention_heads // cfg.num_key_value_heads in (1, 2, 4, 8)
            and self.decode_linears
            and all(n * k >= kernels.WIDE_MIN_WEIGHTS and k % 64 == 0 for n, k in self._linear_shapes())
            and self._all_int8()
        )

    def _linear_shapes(self) -> tuple[tuple[int, int], ...]:
        """(out, in) features of a layer's qkv, o, gate_up and down projections."""
        c = self.cfg
        q, kv = c.num_attention_heads * c.head_dim, c.num_key_value_heads * c.head_dim
        return ((q + 2 * kv, c.hidden_size), (c.hidden_size, q), (2 * c.intermediate_size, c.hidden_size),
                (c.hidden_size, c.intermediate_size))

    def _wide_decode_layers(
        self, input_ids: Tensor, positions: Tensor, kv_caches: list[tuple[Tensor, Tensor]], meta: AttentionMetadata
    ) -> Tensor:
        """The decode layers of a model with large weights; returns the final-normed hidden states.
        Per-head norms, RoPE (by ``positions``) and the cache write run inside the decode attention. Up to
        STREAM_MAX_TOKENS tokens the RMSNorms run inside the qkv and gate_up linears (five launches a
        layer); with more, each would be repeated by every workgroup, so they join the o and down
        projections (whose split-K partials that kernel merges)."""
        cfg = self.cfg
        t = input_ids.numel()
        ids = input_ids if input_ids.dtype == torch.int64 and input_ids.is_contiguous() else input_ids.long().contiguous()
        pos = positions.to(ids.device, torch.int64).contiguous()
        # x: the residual stream, updated in place
        x, cos, sin = kernels.embed_rope_rows(ids, pos, self.embed_tokens.weight.contiguous(), self.rotary.cos,
                                              self.rotary.sin)
        inside = t <= kernels.STREAM_MAX_TOKENS and kernels.dec_supported(cfg.hidden_size)
        first = self.layers[0].input_layernorm
        h = x if inside else kernels.rmsnorm(x, first.weight, first.eps)
        for i, (k_cache, v_cache) in enumerate(kv_caches):
            layer = self.layers[i]
            attn, mlp = layer.self_attn, layer.mlp
            qkv, o, gu, dn = attn.qkv_proj, attn.o_proj, mlp.gate_up_proj, mlp.down_proj
            pre, post = layer.input_layernorm, layer.post_attention_layernorm
            if inside:
                rows = kernels.int8_linear_dec(x, qkv.qweight, qkv.kscale, norm_w=pre.weight, eps=pre.eps)
            else:
                rows = kernels.int8_linear(h, qkv.qweight, qkv.kscale)
            a = attend_decode_qkv(
                rows, attn.num_heads, attn.q_norm.weight, attn.k_norm.weight, attn.q_norm.eps, cos, sin, k_cache,
                v_cache, meta, attn.scale, rope_rows=True,
            ).view(t, attn.q_size)
            if inside:
                kernels.int8_linear(a, o.qweight, o.kscale, kernels.EPI_RESIDUAL, residual=x, out=x)
                act = kernels.int8_linear_dec(x, gu.qweight, gu.kscale, kernels.EPI_SILU_MUL, norm_w=post.weight,
                                              eps=post.eps)
                kernels.int8_linear(act, dn.qweight, dn.kscale, kernels.EPI_RESIDUAL, residual=x, out=x)
            else:
                hn = kernels.int8_linear_add_rmsnorm(a, o.qweight, o.kscale, x, post.weight, post.eps)
                act = kernels.int8_linear(hn, gu.qweight, gu.kscale, kernels.EPI_SILU_MUL)
                nxt = self.layers[i + 1].input_layernorm if i + 1 < len(self.layers) else self.norm
                h = kernels.int8_linear_add_rmsnorm(act, dn.qweight, dn.kscale, x, nxt.weight, nxt.eps)
        return kernels.rmsnorm(x, self.norm.weight, self.norm.eps) if inside else h

    def _token_split_layers(
        self, input_ids: Tensor, positions: Tensor, kv_caches: list[tuple[Tensor, Tensor]], meta: AttentionMetadata
    ) -> Tensor:
        """The layer loop on the token-split kernels (``token_split_layer`` per layer). Returns the
        residual stream after the last layer (before the final norm)."""
        t = input_ids.numel()
        ids = input_ids if input_ids.dtype == torch.int64 and input_ids.is_contiguous() else input_ids.long().contiguous()
        pos = positions if positions.dtype == torch.int64 and positions.is_contiguous() else positions.long().contiguous()
        residual = torch.empty(t, self.cfg.hidden_size, dtype=torch.bfloat16, device=ids.device)
        for i, (k_cache, v_cache) in enumerate(kv_caches):
            self.token_split_layer(i, residual, k_cache, v_cache, meta, pos, ids if i == 0 else None)
        return residual

    def token_split_layer(
        self,
        i: int,
        residual: Tensor,
        k_cache: Tensor,
        v_cache: Tensor,
        meta: AttentionMetadata,
        positions: Tensor,
        input_ids: Tensor | None = None,
    ) -> None:
        """Decoder layer ``i`` (model/qwen3.py:112-122) on the token-split kernels, four launches plus
        attention, updating the residual stream [T, hidden] in place:
          [embedding gather (``input_ids``, layer 0) + input RMSNorm + int8 qkv (+ q/k-norm + RoPE +
          KV write)] -> paged attention -> [int8 o + residual add]
          -> [post-attention RMSNorm + int8 gate_up + silu * up] -> [int8 down + residual add]
        A pure-decode batch of up to DEC_MAX_TOKENS tokens runs the qkv projection as a plain decode
        linear and the per-head norms, RoPE and KV write inside the decode attention kernel (rows known
        not to own their slots are written by the qkv kernel, before any row attends)."""
        cfg = self.cfg
        t = residual.shape[0]
        rot = self.rotary
        layer = self.layers[i]
        attn, mlp = layer.self_attn, layer.mlp
        qkv, o, gu, dn = attn.qkv_proj, attn.o_proj, mlp.gate_up_proj, mlp.down_proj

        def lin(k: int):
            # Up to DEC_MAX_TOKENS tokens the decode kernel (activations straight into MFMA
            # operands, all loads in flight at once) serves the K it supports; else the
            # token-split rows kernel.
            if t <= kernels.DEC_MAX_TOKENS and kernels.dec_supported(k) and self.decode_linears:
                return kernels.int8_linear_dec
            return kernels.int8_linear_rows

        fused_decode = (
            meta.prefill is None and meta.decode is not None and meta.decode.own_slots is not False
            and t <= kernels.DEC_MAX_TOKENS and kernels.dec_supported(cfg.hidden_size) and self.decode_linears
        )
        first = input_ids is not None
        src = self.embed_tokens.weight if first else residual
        if fused_decode:
            # [gather + input RMSNorm + int8 qkv] -> [q/k-norm + RoPE + KV write + attention]
            qkv_rows = kernels.int8_linear_dec(
                src, qkv.qweight, qkv.kscale, norm_w=layer.input_layernorm.weight, eps=layer.input_layernorm.eps,
                gather=input_ids, x_copy=residual if first else None,
            )
            a = attend_decode_qkv(
                qkv_rows, attn.num_heads, attn.q_norm.weight, attn.k_norm.weight, attn.q_norm.eps, rot.cos,
                rot.sin, k_cache, v_cache, meta, attn.scale,
            ).view(t, attn.q_size)
        else:
            q = kernels.qkv_rope_cache_rows(
                src, qkv.qweight, qkv.kscale, attn.num_heads, attn.num_kv_heads, attn.head_dim,
                attn.q_norm.weight, attn.k_norm.weight, attn.q_norm.eps, positions, rot.cos, rot.sin,
                meta.slot_mapping, k_cache, v_cache, norm_w=layer.input_layernorm.weight,
                eps=layer.input_layernorm.eps, gather=input_ids, x_copy=residual if first else None,
            )
            a = attend(q, k_cache, v_cache, meta, attn.scale).view(t, attn.q_size)
        post = layer.post_attention_layernorm
        lin(attn.q_size)(a, o.qweight, o.kscale, kernels.EPI_RESIDUAL, residual=residual, out=residual)
        act = lin(cfg.hidden_size)(residual, gu.qweight, gu.kscale, kernels.EPI_SILU_MUL, norm_w=post.weight,
                                   eps=post.eps)
        lin(cfg.intermediate_size)(act, dn.qweight, dn.kscale, kernels.EPI_RESIDUAL, residual=residual, out=residual)

    def _fused_forward(
        self, x: Tensor, cos: Tensor, sin: Tensor, kv_caches: list[tuple[Tensor, Tensor]], meta: AttentionMetadata
    ) -> Tensor:
        """The layer loop for batches above the token-split limit (prefill chunks), ``gemm_layer``
        per layer. Returns norm(x_L), the same value as the module-by-module loop; ``x`` (the
        embedding output) is updated in place as the residual stream."""
        layers = self.layers
        h = kernels.rmsnorm(x, layers[0].input_layernorm.weight, layers[0].input_layernorm.eps)
        for i, (k_cache, v_cache) in enumerate(kv_caches):
            h = self.gemm_layer(i, x, h, cos, sin, k_cache, v_cache, meta)
        return h

    def gemm_layer(
        self, i: int, x: Tensor, h: Tensor, cos: Tensor, sin: Tensor, k_cache: Tensor, v_cache: Tensor,
        meta: AttentionMetadata,
    ) -> Tensor:
        """Decoder layer ``i`` (model/qwen3.py:112-122) for prefill-sized batches: int8 linears on the
        LDS-tiled MFMA GEMM (silu * up in its epilogue; the o and down projections add the residual
        and apply the next RMSNorm, merging split-K partials in the same pass; q/k-norm + RoPE +
        KV write in the qkv GEMM's epilogue when that GEMM is unsplit, else as its own kernel). ``x`` is the residual stream (updated in place), ``h`` its
        input RMSNorm; returns the next layer's normed input (the final norm after the last layer)."""
        cfg = self.cfg
        t = x.shape[0]
        layers = self.layers
        layer = layers[i]
        attn, mlp = layer.self_attn, layer.mlp
        qkv, o, gu, dn = attn.qkv_proj, attn.o_proj, mlp.gate_up_proj, mlp.down_proj
        if kernels.qkv_gemm_fuses_norm(t, attn.num_heads, attn.num_kv_heads, attn.head_dim, h.shape[-1]):
            q = kernels.int8_linear_qk_norm_rope_cache(
                h, qkv.qweight, qkv.kscale, attn.num_heads, attn.num_kv_heads, attn.head_dim, attn.q_norm.weight,
                attn.k_norm.weight, attn.q_norm.eps, cos, sin, meta.slot_mapping, k_cache, v_cache,
            )
        else:
            q = kernels.qk_norm_rope_cache(
                kernels.int8_linear(h, qkv.qweight, qkv.kscale), attn.num_heads, attn.num_kv_heads, attn.head_dim,
                attn.q_norm.weight, attn.k_norm.weight, attn.q_norm.eps, cos, sin, meta.slot_mapping, k_cache,
                v_cache,
            )
        a = attend(q, k_cache, v_cache, meta, attn.scale).view(t, attn.q_size)
        post = layer.post_attention_layernorm
        hn = kernels.int8_linear_add_rmsnorm(a, o.qweight, o.kscale, x, post.weight, post.eps)
        act = kernels.int8_linear(hn, gu.qweight, gu.kscale, kernels.EPI_SILU_MUL)
        nxt = layers[i + 1].input_layernorm if i + 1 < len(layers) else self.norm
        return kernels.int8_linear_add_rmsnorm(act, dn.qweight, dn.kscale, x, nxt.weight,
                                               cfg.rms_norm_eps if nxt is self.norm else nxt.eps)

    def compute_logits(self, hidden: Tensor) -> Tensor:
        """[n, hidden] -> [n, vocab] float32, the product in bf16 (qwen3.py:155-158). On the GPU the
        HIP LM head (bf16 MFMA products rounded to bf16, as the reference's bf16 logits)."""
        weight = self.embed_tokens.weight if self.lm_head is None else self.lm_head.weight
        if not hidden.is_cuda:
            return F.linear(hidden, weight).float()
        if hidden.shape[0] == 0:
            return hidden.new_empty(0, weight.shape[0], dtype=torch.float32)
        rows = torch.arange(hidden.shape[0], device=hidden.device)
        return kernels.lm_head_logits(hidden.contiguous(), rows, None, 0.0, weight, prenormed=True)

    def logits(
        self,
        input_ids: Tensor,
        positions: Tensor,
        kv_caches: list[tuple[Tensor, Tensor]],
        meta: AttentionMetadata,
        logits_rows: Tensor,
    ) -> Tensor:
        """``compute_logits(forward(...)[logits_rows])`` (runner/model_runner.py:214-217): on the
        token-split path the final norm of the sampled rows runs inside the LM-head kernel."""
        if len(kv_caches) != len(self.layers):
            raise ValueError(f"{len(kv_caches)} KV caches for {len(self.layers)} layers")
        if self._token_split_ok(input_ids.numel()) and logits_rows.numel() > 0:
            weight = self.embed_tokens.weight if self.lm_head is None else self.lm_head.weight
            residual = self._token_split_layers(input_ids, positions, kv_caches, meta)
            return kernels.lm_head_logits(residual, logits_rows, self.norm.weight, self.norm.eps, weight)
        hidden = self.forward(input_ids, positions, kv_caches, meta)
        return self.compute_logits(hidden[logits_rows])
