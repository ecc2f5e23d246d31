"""LLaMA decoder path on the HIP kernels.

Counterpart of the reference's models/llama.py:30-330 with identical module and parameter names
(embed_tokens, layers.N.self_attn.{q,k,v,o}_proj, layers.N.mlp.{gate,up,down}_proj,
layers.N.{input,post_attention}_layernorm, norm, lm_head), so state dicts are interchangeable.
RMSNorm, RoPE, attention, SwiGLU and the loss are the `maltos::` custom ops; the projections run on the own
product kernels up to a size and on the vendor library through torch above it (csrc/torch/products.cpp).  Attention consumes the [B, H, S, D] views
of the projection outputs in place and keeps K/V at their native head count.
"""
from __future__ import annotations

from dataclasses import dataclass

import torch
import torch.nn as nn
import torch.nn.functional as F

from . import ops
from .attention_backend import _HIP_BACKENDS, AttentionBackend, causal_attention, hip_fallback_reason, uses_hip_kernels, validate_attention_backend
from .attn_masking_utils import canonical_position_ids, canonical_sequence_ids
from .constants import (HIDDEN_STATES_KEY, INPUT_IDS_KEY, LABELS_KEY, LOSS_WEIGHT_KEY, POSITION_IDS_KEY,
                        POSITION_OFFSET_KEY, SEQUENCE_IDS_KEY)
from ._native import native
from .losses import causal_cross_entropy


@dataclass(frozen=True)
class LlamaConfig:
    vocab_size: int
    hidden_size: int = 512
    intermediate_size: int = 2048
    num_hidden_layers: int = 8
    num_attention_heads: int = 8
    num_key_value_heads: int | None = None
    max_position_embeddings: int = 2048
    rms_norm_eps: float = 1e-6
    rope_theta: float = 10000.0
    tie_word_embeddings: bool = False
    attention_backend: str = AttentionBackend.HIP
    # each residual add is done inside the RMSNorm kernel that follows it (same values; one pass less per sublayer,
    # forward and backward); False keeps the reference's op sequence
    fuse_residual_norm: bool = True
    # when the model computes the loss itself, the loss kernel writes the logits' gradient over the logits (no second
    # buffer of their size).  Nobody else may then read the lm_head output of that forward; the model falls back to a
    # separate gradient buffer by itself while lm_head carries forward hooks (which see that output).  False: always separate
    loss_overwrites_logits: bool = True
    # q/k/v (and gate/up) projections run as one product whenever their weights are adjacent in memory (flat optimizer
    # layouts); the sums inside that product are formed in another order than in three separate ones, so results differ
    # from the separate form in the last bit.  False (or `module.fuse_projections = False` on an attention / MLP module)
    # keeps one product per projection
    fuse_projections: bool = True

    def __post_init__(self) -> None:
        validate_attention_backend(self.attention_backend)


# The projections, the MLP and the rotary + attention block are C++ autograd nodes (csrc/torch/llama.cpp).  Projections that
# share their input (q/k/v; gate/up) run as ONE product there whenever their weights are adjacent row blocks of one
# allocation (what the flat optimizer layouts make of them: MasterWeightsOptimizer(flat=True), Zero1FlatBuffers): they ARE one
# [sum of out_features, in_features] matrix.  Parameter names, shapes and values are untouched.  Otherwise the projections run
# one by one as in the reference (models/llama.py:134-142,196-206).
#
# Without adjacency, and at sizes where the own product kernels run, the products of a pass are still one launch, and their
# input gradient is formed in one sum.
def _fused_rows(holder: nn.Module, modules: list[nn.Module], params: list[nn.Parameter], x: torch.Tensor):
    """The parameters as one matrix (`weight`, and `grad` when their gradients are adjacent too) or as a group of such that
    share a launch, kept on the module until a parameter or gradient moves; None when they run one by one."""
    rows = holder.__dict__.get("_maltos_hip_fused_rows")
    if rows is None or not rows.made_for(params):
        rows = holder.__dict__["_maltos_hip_fused_rows"] = native().Adjacent(params)
    if rows.adjacent:
        return rows
    return rows if all(_plain_linear(m) for m in modules) and rows.runs_as_group(x, params) else None


def _plain_linear(m: nn.Module) -> bool:
    """Whether calling the module is the product with its weight and nothing else."""
    return (type(m) is HipLinear and HipLinear.forward is _STOCK_METHODS[HipLinear, "forward"] and "forward" not in m.__dict__
            and not (m._forward_hooks or m._forward_pre_hooks or m._backward_hooks or m._backward_pre_hooks))


def _adjacent_columns(parts: list[torch.Tensor]) -> torch.Tensor | None:
    """The [rows, sum of widths] matrix whose column ranges the given [..., width_i] tensors are, in this order, when
    they are such views of one dense buffer; None otherwise."""
    return native().adjacent_columns(parts)


def _weight_grad_splits(rows: int, out_features: int, in_features: int) -> int:
    """Number of row slices a weight gradient is computed in."""
    return native().weight_grad_splits(rows, out_features, in_features)


def _fusable(modules: list[nn.Module]) -> bool:
    return all(isinstance(m, HipLinear) and m.bias is None for m in modules)


class HipLinear(nn.Linear):
    """nn.Linear (same parameter name and init) whose weight gradient is computed as a batch of row slices when the
    output is too small to fill the chip (reference: plain nn.Linear, models/llama.py:69-75,196-198).

    `accumulate_into_grad = True` (off by default; set it on the class or on an instance) makes the backward add dW
    straight into an existing `weight.grad` and return no gradient for the weight: one pass instead of two when the
    gradients live in a flat buffer that is cleared, not dropped, between steps.  Autograd hooks on the weight see no
    gradient in that mode (they run with None), so it is for callers that read the gradients from the buffer after
    backward; whoever needs to know that the buffer was written is told through `optim.notify_grad_written`."""

    accumulate_into_grad = False

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        if self.bias is not None or not x.is_cuda:
            return F.linear(x, self.weight, self.bias)
        return native().linear(x, self.weight, bool(self.accumulate_into_grad))


class LlamaEmbedding(nn.Embedding):
    """embed_tokens (reference: nn.Embedding, models/llama.py:238).  `accumulate_into_grad` as in HipLinear, except that a
    weight with tensor hooks, or tied to the lm_head, keeps its gradient with autograd."""

    accumulate_into_grad = False

    def forward(self, input_ids: torch.Tensor) -> torch.Tensor:
        plain = self.padding_idx is None and self.max_norm is None and not self.scale_grad_by_freq and not self.sparse
        if not plain or not self.weight.is_cuda:
            return super().forward(input_ids)
        return native().embedding(self.weight, input_ids, self.accumulate_into_grad and not self.weight._backward_hooks)


class LlamaHead(nn.Linear):
    """The lm_head (reference: nn.Linear, models/llama.py:242-243).  `accumulate_into_grad` as in LlamaEmbedding."""

    accumulate_into_grad = False

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        if self.bias is not None or not x.is_cuda or torch.is_autocast_enabled("cuda"):
            return F.linear(x, self.weight, self.bias)
        return native().linear(x, self.weight, self.accumulate_into_grad and not self.weight._backward_hooks)


def set_grad_accumulation_into_buffers(model: nn.Module, enabled: bool = True) -> int:
    """Switches `HipLinear.accumulate_into_grad` on every HipLinear of `model`, and returns how many were switched.  The
    norms and, when untied, the embedding and the lm_head follow (weights with tensor hooks excepted)."""
    count = 0
    for module in model.modules():
        if isinstance(module, HipLinear):
            module.accumulate_into_grad = bool(enabled)
            count += 1
        elif isinstance(module, LlamaRMSNorm):
            module.accumulate_into_grad = bool(enabled)
        elif isinstance(module, LlamaForCausalLM):
            untied = module.lm_head.weight is not module.embed_tokens.weight
            module.lm_head.accumulate_into_grad = module.embed_tokens.accumulate_into_grad = bool(enabled) and untied
    return count


class LlamaRMSNorm(nn.Module):
    accumulate_into_grad = False   # see HipLinear; a weight with tensor hooks keeps its gradient with autograd

    def __init__(self, hidden_size: int, eps: float) -> None:
        super().__init__()
        self.weight = nn.Parameter(torch.ones(hidden_size))
        self.eps = eps

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        return native().rms_norm(x, self.weight, self.eps, self.accumulate_into_grad)


def _add_norm(norm: nn.Module, x: torch.Tensor, residual: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
    """(h, norm of h) with h = x + residual."""
    return native().add_rms_norm(x, residual, norm.weight, norm.eps, getattr(norm, "accumulate_into_grad", False))


class LlamaRotaryEmbedding(nn.Module):
    """cos/sin tables [max_position_embeddings, head_dim / 2], built in fp32 and cast with the module."""

    def __init__(self, head_dim: int, max_position_embeddings: int, base: float) -> None:
        super().__init__()
        exponents = torch.arange(0, head_dim, 2, dtype=torch.float32) / head_dim
        angles = torch.arange(max_position_embeddings, dtype=torch.float32)[:, None] * (base ** -exponents)[None, :]
        self.register_buffer("cos", torch.cos(angles), persistent=False)
        self.register_buffer("sin", torch.sin(angles), persistent=False)

    def tables(self, dtype: torch.dtype, device: torch.device) -> tuple[torch.Tensor, torch.Tensor]:
        if self.cos.dtype != dtype or self.cos.device != device:
            # fp32 -> dtype is the single rounding the reference applies (cos.to(x.dtype))
            return self.cos.to(device=device, dtype=dtype), self.sin.to(device=device, dtype=dtype)
        return self.cos, self.sin


def _one_document(positions: torch.Tensor) -> torch.Tensor:
    """Sequence ids of rows that come with positions only: one document per row."""
    return ops.derived_from(positions, "_maltos_hip_zero_ids", lambda pos: torch.zeros(pos.shape, dtype=torch.int32, device=pos.device))


class HipAttentionCore(nn.Module):
    """`attn_core` of LlamaAttention: (q, k, v, position_offset, position_ids, sequence_ids) -> out."""

    preserves_native_gqa = True

    def __init__(self, attention_backend: str = AttentionBackend.HIP) -> None:
        super().__init__()
        self.attention_backend = validate_attention_backend(attention_backend)

    def row_ids(self, q, position_offset: int, position_ids=None, sequence_ids=None):
        """(positions, sequence ids) of the rows as the attention kernels take them, or (None, None) for plain causal rows."""
        if position_ids is None and sequence_ids is None:
            return None, None
        positions = canonical_position_ids(position_ids, batch_size=q.size(0), seq_len=q.size(-2),
                                           position_offset=position_offset, device=q.device)
        return positions, canonical_sequence_ids(sequence_ids, batch_size=q.size(0), seq_len=q.size(-2), device=q.device)

    def forward(self, q, k, v, position_offset: int, position_ids=None, sequence_ids=None) -> torch.Tensor:
        positions, sequences = self.row_ids(q, position_offset, position_ids, sequence_ids)
        return causal_attention(q, k, v, attention_backend=self.attention_backend, warning_prefix="LlamaAttention",
                                q_positions=positions, k_positions=positions, q_sequence_ids=sequences,
                                k_sequence_ids=sequences, flash_varlen_mode="same_length")


class LlamaAttention(nn.Module):
    # rotary embedding and attention as one autograd node whenever `attn_core` is the stock HipAttentionCore on the HIP
    # kernels (same values; dQ, dK and dV of the backward are then head ranges of one buffer, rotated back in place there,
    # so that the gradient of q/k/v projections that run as one product arrives as one matrix).  False keeps the two ops apart
    fuse_rope_attention = True

    def __init__(self, config: LlamaConfig) -> None:
        super().__init__()
        if config.hidden_size % config.num_attention_heads != 0:
            raise ValueError("hidden_size must be divisible by num_attention_heads")
        self.num_heads = config.num_attention_heads
        self.num_kv_heads = config.num_key_value_heads or config.num_attention_heads
        if self.num_heads % self.num_kv_heads != 0:
            raise ValueError("num_attention_heads must be divisible by num_key_value_heads")
        self.head_dim = config.hidden_size // config.num_attention_heads
        self.rotary_emb = LlamaRotaryEmbedding(self.head_dim, config.max_position_embeddings, config.rope_theta)
        self.q_proj = HipLinear(config.hidden_size, self.num_heads * self.head_dim, bias=False)
        self.k_proj = HipLinear(config.hidden_size, self.num_kv_heads * self.head_dim, bias=False)
        self.v_proj = HipLinear(config.hidden_size, self.num_kv_heads * self.head_dim, bias=False)
        self.o_proj = HipLinear(config.hidden_size, config.hidden_size, bias=False)
        self.attn_core = HipAttentionCore(config.attention_backend)
        self.fuse_projections = config.fuse_projections

    def forward(self, x: torch.Tensor, *, position_offset: int = 0, position_ids: torch.Tensor | None = None,
                sequence_ids: torch.Tensor | None = None) -> torch.Tensor:
        batch, seq_len, _ = x.shape
        cos, sin = self.rotary_emb.tables(x.dtype, x.device)
        rope_pos = None
        if position_ids is not None:
            rope_pos = canonical_position_ids(position_ids, batch_size=batch, seq_len=seq_len, position_offset=0,
                                              device=x.device)
        # [B, S, H*D] -> [B, H, S, D] views; no copies until the kernels read them
        projections = [self.q_proj, self.k_proj, self.v_proj]
        fused = None
        if self.fuse_projections and x.is_cuda and _fusable(projections):
            weights = [m.weight for m in projections]
            fused = _fused_rows(self, projections, weights, x)
        if fused is not None:   # one product over the three adjacent weights, or one launch
            q, k, v = native().adjacent_linears(x, fused, weights, all(m.accumulate_into_grad for m in projections))
        else:
            q, k, v = self.q_proj(x), self.k_proj(x), self.v_proj(x)
        q = q.view(batch, seq_len, self.num_heads, self.head_dim).transpose(1, 2)
        k = k.view(batch, seq_len, self.num_kv_heads, self.head_dim).transpose(1, 2)
        v = v.view(batch, seq_len, self.num_kv_heads, self.head_dim).transpose(1, 2)
        core = self.attn_core
        if (self.fuse_rope_attention and type(core) is HipAttentionCore and uses_hip_kernels(core.attention_backend)
                and hip_fallback_reason(q) is None):
            positions, sequences = core.row_ids(q, position_offset, position_ids, sequence_ids)
            if positions is not None and sequences is None:
                sequences = _one_document(positions)
            if rope_pos is not None:
                rope_pos = ops._ids32(rope_pos, batch, seq_len, "position_ids")
            vo = native().rope_attention(q, k, v, cos, sin, rope_pos, int(position_offset), positions, sequences)
            return self.o_proj(vo.transpose(1, 2).reshape(batch, seq_len, self.num_heads * self.head_dim))
        q, k = ops.rope_pair(q, k, cos, sin, positions=rope_pos, position_offset=position_offset)
        if not getattr(self.attn_core, "preserves_native_gqa", False) and self.num_heads != self.num_kv_heads:
            rep = self.num_heads // self.num_kv_heads
            k, v = k.repeat_interleave(rep, dim=1), v.repeat_interleave(rep, dim=1)
        vo = self.attn_core(q, k, v, position_offset, position_ids, sequence_ids)
        return self.o_proj(vo.transpose(1, 2).reshape(batch, seq_len, self.num_heads * self.head_dim))


class LlamaMLP(nn.Module):
    def __init__(self, config: LlamaConfig) -> None:
        super().__init__()
        self.gate_proj = HipLinear(config.hidden_size, config.intermediate_size, bias=False)
        self.up_proj = HipLinear(config.hidden_size, config.intermediate_size, bias=False)
        self.down_proj = HipLinear(config.intermediate_size, config.hidden_size, bias=False)
        self.fuse_projections = config.fuse_projections

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        pair = [self.gate_proj, self.up_proj]
        if self.fuse_projections and x.is_cuda and _fusable(pair) and self.gate_proj.out_features % (16 // x.element_size()) == 0:
            weights = [self.gate_proj.weight, self.up_proj.weight]
            fused = _fused_rows(self, pair, weights, x)
            if fused is not None:
                return self.down_proj(native().gate_up(x, fused, weights, all(m.accumulate_into_grad for m in pair)))
        return self.down_proj(ops.swiglu(self.gate_proj(x), self.up_proj(x)))


class LlamaDecoderLayer(nn.Module):
    def __init__(self, config: LlamaConfig) -> None:
        super().__init__()
        self.self_attn = LlamaAttention(config)
        self.mlp = LlamaMLP(config)
        self.input_layernorm = LlamaRMSNorm(config.hidden_size, config.rms_norm_eps)
        self.post_attention_layernorm = LlamaRMSNorm(config.hidden_size, config.rms_norm_eps)

    def forward(self, x: torch.Tensor, position_offset: int = 0, position_ids: torch.Tensor | None = None,
                sequence_ids: torch.Tensor | None = None, pending: torch.Tensor | None = None,
                defer_residual: bool = False):
        """Reference form (:217-231): x -> x.  With `defer_residual` the layer returns (x, mlp_out) and leaves the last
        residual add to whoever normalises next, and takes such a not-yet-added `pending` from the layer before."""
        if not defer_residual:
            if pending is not None:
                x = x + pending
            x = x + self.self_attn(self.input_layernorm(x), position_offset=position_offset, position_ids=position_ids,
                                   sequence_ids=sequence_ids)
            return x + self.mlp(self.post_attention_layernorm(x))
        ln1, ln2 = self.input_layernorm, self.post_attention_layernorm
        if pending is None:
            normed = ln1(x)
        else:
            x, normed = _add_norm(ln1, x, pending)
        attn_out = self.self_attn(normed, position_offset=position_offset, position_ids=position_ids, sequence_ids=sequence_ids)
        x, normed = _add_norm(ln2, x, attn_out)
        return x, self.mlp(normed)


# what native().run_layers takes a layer apart into
_STOCK_MODULES = {"layer": LlamaDecoderLayer, "attention": LlamaAttention, "core": HipAttentionCore, "rotary": LlamaRotaryEmbedding,
                  "mlp": LlamaMLP, "norm": LlamaRMSNorm, "linear": HipLinear}
# ... as long as nobody has put another method in the place of one of theirs
_STOCK_METHODS = {(cls, name): getattr(cls, name) for cls in _STOCK_MODULES.values() for name in ("forward", "row_ids", "tables") if hasattr(cls, name)}


class LlamaForCausalLM(nn.Module):
    def __init__(self, config: LlamaConfig) -> None:
        super().__init__()
        self.config = config
        self.embed_tokens = LlamaEmbedding(config.vocab_size, config.hidden_size)
        self.layers = nn.ModuleList([LlamaDecoderLayer(config) for _ in range(config.num_hidden_layers)])
        self.norm = LlamaRMSNorm(config.hidden_size, config.rms_norm_eps)
        self.lm_head = LlamaHead(config.hidden_size, config.vocab_size, bias=False)
        if config.tie_word_embeddings:
            self.lm_head.weight = self.embed_tokens.weight

    def forward(self, batch):
        """Accepts the reference's batch forms: dict with the constants' keys, (input_ids, labels), or input_ids.
        Returns the scalar loss when labels are given (already aligned, no shift), else the logits."""
        hidden_states = position_ids = sequence_ids = loss_weight = labels = None
        position_offset = 0
        if isinstance(batch, dict):
            input_ids = batch.get(INPUT_IDS_KEY)
            hidden_states = batch.get(HIDDEN_STATES_KEY)
            labels = batch.get(LABELS_KEY)
            position_offset = int(batch.get(POSITION_OFFSET_KEY, 0))
            position_ids = batch.get(POSITION_IDS_KEY)
            sequence_ids = batch.get(SEQUENCE_IDS_KEY)
            loss_weight = batch.get(LOSS_WEIGHT_KEY)
        elif isinstance(batch, (tuple, list)):
            input_ids, labels = batch
        else:
            input_ids = batch
        if hidden_states is not None:
            x = hidden_states
        elif input_ids is None:
            raise ValueError("LlamaForCausalLM requires input_ids or hidden_states")
        else:
            x = self.embed_tokens(input_ids)
        if position_ids is not None or sequence_ids is not None:
            # canonical [batch, seq] ids once per forward: every layer's attention is then handed the SAME tensors and
            # shares what is derived from them (int32 forms, the document-mask plan), where per-layer canonicalisation
            # (models/llama.py:163-175 of the reference) makes fresh ones whenever the batch's ids are rank 1, not int64,
            # on the host, or absent.  Positions made here carry position_offset, which the rotary kernel then ignores.
            position_ids = canonical_position_ids(position_ids, batch_size=x.size(0), seq_len=x.size(1),
                                                  position_offset=position_offset, device=x.device)
            sequence_ids = canonical_sequence_ids(sequence_ids, batch_size=x.size(0), seq_len=x.size(1), device=x.device)
        if self.config.fuse_residual_norm and x.is_cuda and len(self.layers) > 0:
            done = self._layers_at_once(x, position_offset, position_ids, sequence_ids)
            if done is not None:
                x, pending = done
            else:
                pending = None
                for layer in self.layers:
                    x, pending = layer(x, position_offset=position_offset, position_ids=position_ids, sequence_ids=sequence_ids,
                                       pending=pending, defer_residual=True)
            _, normed = _add_norm(self.norm, x, pending)
        else:
            for layer in self.layers:
                x = layer(x, position_offset=position_offset, position_ids=position_ids, sequence_ids=sequence_ids)
            normed = self.norm(x)
        logits = self.lm_head(normed)
        if labels is None:
            return logits
        if input_ids is not None and labels.shape != input_ids.shape:
            raise ValueError(f"labels shape must match input_ids shape, got {labels.shape} vs {input_ids.shape}")
        # the logits are this function's own and are not returned with the loss: their gradient may take their place
        own = self.config.loss_overwrites_logits and not self.lm_head._forward_hooks
        loss = causal_cross_entropy(logits, labels, overwrite_logits=own and logits.is_cuda and logits.is_contiguous())
        return loss if loss_weight is None else loss * float(loss_weight)

    def _layers_at_once(self, x, position_offset, position_ids, sequence_ids):
        """(x, pending) after all layers without leaving C++, or None: only layers of the modules above, as they are and with
        nothing hooked into them, can be run that way."""
        if type(self.layers) is not nn.ModuleList or x.dim() != 3 or torch.nn.modules.module._has_any_global_hook():
            return None
        if any(getattr(cls, name) is not method for (cls, name), method in _STOCK_METHODS.items()):
            return None
        rope_pos = sequences = None
        if position_ids is not None:
            rope_pos = ops._ids32(position_ids, x.size(0), x.size(1), "position_ids")
            sequences = sequence_ids if sequence_ids is not None else _one_document(position_ids)
        return native().run_layers(self.layers._modules, _STOCK_MODULES, _HIP_BACKENDS, x, int(position_offset), rope_pos, position_ids, sequences)

    def context_parallel_spec(self) -> list[str]:
        """Module paths whose `attn_core` a context-parallel plugin swaps (reference :311-314)."""
        return [f"layers.{i}.self_attn" for i in range(len(self.layers))]

    def flops_per_token(self) -> float:
        """The reference's estimator (:319-330): 3 x forward, attention counted non-causal."""
        c = self.config
        h, i, s, v = c.hidden_size, c.intermediate_size, c.max_position_embeddings, c.vocab_size
        per_layer = 6 * h * h + 2 * h * h + 6 * h * i + 4 * s * h
        return float(3 * (c.num_hidden_layers * per_layer + 2 * h * v))
