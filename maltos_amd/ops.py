"""torch.library custom ops over the C ABI of libmaltos_hip.so.

Layering: `torch.ops.maltos.*` (schemas and fake kernels registered here; implementations and autograd formulas in
csrc/torch/ops.cpp, the extension `_torch_ops.so`, for the GPU only) -> `mlts_*` entry points -> HIP kernels on the
current torch stream.  The functions below call the extension directly, without a Python frame per operator in between: a
training step is hundreds of launches of a few microseconds, so what an operator costs on the host is what a small step
costs.  There is deliberately no CPU implementation: calling an op with host tensors, or without the built library, raises.
"""
from __future__ import annotations

import torch

from . import _lib
from ._lib import MASK_CAUSAL, MASK_DOC, MASK_NONE, MLTS_BF16, MLTS_F32, AttnShape, strides3
from ._native import native

# mlts_attn_bwd's accumulate_f32 modes (include/maltos_hip.h)
BWD_OVERWRITE, BWD_ACCUMULATE, BWD_DQ_ACCUMULATE, BWD_DQ_STORE = 0, 1, 2, 3

__all__ = [
    "MASK_NONE", "MASK_CAUSAL", "MASK_DOC",
    "attention", "attention_forward", "attention_backward", "attention_backward_accumulate",
    "attention_backward_ring_block", "attention_merge_",
    "rms_norm", "rope", "rope_pair", "rope_pair_", "swiglu", "cross_entropy",
    "adamw_step_", "sq_norm", "scale_", "grad_to_f32_",
]


# --------------------------------------------------------------------------------------------
# helpers
# --------------------------------------------------------------------------------------------
def _dtype_code(t: torch.Tensor) -> int:
    if t.dtype == torch.bfloat16:
        return MLTS_BF16
    if t.dtype == torch.float32:
        return MLTS_F32
    raise ValueError(f"maltos_amd kernels take float32 or bfloat16 tensors, got {t.dtype}")


def derived_from(t: torch.Tensor, attr: str, build):
    """`build(t)`, kept on the tensor object `t` until `t` is modified in place (its autograd version counter moves).
    Every layer of a model is handed the same id tensors, so what is derived from them (their int32 form, run ids, a
    zero id tensor) is formed once per batch instead of once per layer, and, being the same tensor objects in every
    call, lets the calls share one document-mask plan.  Not kept for inference tensors (no version counter) nor under
    HIP graph capture (a tensor allocated while capturing belongs to the graph's pool)."""
    if t.is_inference() or (t.is_cuda and torch.cuda.is_current_stream_capturing()):
        return build(t)
    hit = t.__dict__.get(attr)
    if hit is not None and hit[0] == t._version:
        return hit[1]
    value = build(t)
    t.__dict__[attr] = (t._version, value)
    return value


def _ids32(t: torch.Tensor | None, batch: int, seq: int, what: str) -> torch.Tensor | None:
    if t is None:
        return None
    if t.shape != (batch, seq):
        raise ValueError(f"{what} must have shape ({batch}, {seq}), got {tuple(t.shape)}")
    if t.dtype == torch.int32 and t.is_contiguous():
        return t
    return derived_from(t, "_maltos_hip_int32", lambda x: x.to(dtype=torch.int32).contiguous())


def _attn_shape(q, k, v, o, mask_mode, scale, q_pos, k_pos, q_seq, k_seq) -> AttnShape:
    s = AttnShape()
    s.B, s.Hq, s.Sq, s.D = q.size(0), q.size(1), q.size(2), q.size(3)
    s.Hkv, s.Sk = k.size(1), k.size(2)
    s.dtype = _dtype_code(q)
    s.mask_mode = int(mask_mode)
    s.scale = float(scale)
    s.q_stride = strides3(q.stride()[:3])
    s.k_stride = strides3(k.stride()[:3])
    s.v_stride = strides3(v.stride()[:3])
    s.o_stride = strides3(o.stride()[:3])
    if mask_mode == MASK_DOC:
        if q_pos is None or k_pos is None or q_seq is None or k_seq is None:
            raise ValueError("document-masked attention needs q/k positions and q/k sequence ids")
        s.q_pos, s.k_pos, s.q_seq, s.k_seq = q_pos.data_ptr(), k_pos.data_ptr(), q_seq.data_ptr(), k_seq.data_ptr()
    return s


# Document-mask plans (mlts_attn_doc_plan) are kept by the extension, keyed by the id tensors of a call (csrc/torch/ops.cpp).
class _PlanCache:
    def __len__(self) -> int:
        return native().doc_plan_cache_size()


_DOC_PLAN_CACHE = _PlanCache()


def set_doc_plan_cache_entries(n: int) -> int:
    """Number of document-mask plans kept (0: every call builds its own in its workspace).  Returns the previous value."""
    return native().set_doc_plan_cache_entries(int(n))


def clear_doc_plan_cache() -> None:
    native().clear_doc_plan_cache()


# --------------------------------------------------------------------------------------------
# raw launches (no autograd)
# --------------------------------------------------------------------------------------------
def attention_forward(q, k, v, *, mask_mode: int, scale: float | None = None, q_pos=None, k_pos=None, q_seq=None,
                      k_seq=None) -> tuple[torch.Tensor, torch.Tensor]:
    """O [B,Hq,Sq,D] (BSHD storage) and LSE [B,Hq,Sq] fp32."""
    return native().attention_forward(q, k, v, mask_mode, scale, q_pos, k_pos, q_seq, k_seq)


def attention_backward(dout, q, k, v, o, lse, *, mask_mode: int, scale: float | None = None, q_pos=None, k_pos=None,
                       q_seq=None, k_seq=None):
    """(dq, dk, dv) in the input dtype, as [B, H, S, D] views of [B, S, H, D] storage.  For self-attention (queries and
    keys of one length) the three are the head ranges [0, Hq), [Hq, Hq + Hkv), [Hq + Hkv, Hq + 2 Hkv) of ONE
    [B, S, Hq + 2 Hkv, D] buffer: next to each other exactly as the input gradient of projections that run as one
    product wants them, so that nobody has to copy them together."""
    return native().attention_backward(dout, q, k, v, o, lse, mask_mode, scale, q_pos, k_pos, q_seq, k_seq)


def attention_backward_accumulate(dout, q, k, v, o, lse, dq, dk, dv, *, mask_mode: int, scale: float | None = None,
                                  q_pos=None, k_pos=None, q_seq=None, k_seq=None) -> None:
    """dq += ..., dk += ..., dv += ... into fp32 buffers (ring schedule)."""
    native().attention_backward_accumulate(dout, q, k, v, o, lse, dq, dk, dv, mask_mode, scale, q_pos, k_pos, q_seq, k_seq)


def attention_backward_ring_block(dout, q, k, v, o, lse, dq, dk, dv, *, first: bool, mask_mode: int, scale: float | None = None,
                                  q_pos=None, k_pos=None, q_seq=None, k_seq=None) -> None:
    """One block of a ring schedule on the rank that owns the queries: dq (fp32) collects every block (`first`: this
    block overwrites it, so nobody has to clear it; later blocks add), while dk and dv of the block's keys (input
    dtype) are written once, since a K/V chunk meets the local queries in exactly one block."""
    native().attention_backward_ring_block(dout, q, k, v, o, lse, dq, dk, dv, first, mask_mode, scale, q_pos, k_pos, q_seq, k_seq)


def attention_merge_(out_acc, lse_acc, o_blk, lse_blk, q_off: int = 0) -> None:
    """In-place log-sum-exp merge of a block into rows [q_off, q_off + q_len) of the running state."""
    native().attention_merge_(out_acc, lse_acc, o_blk, lse_blk, q_off)


def swiglu_rows(gu: torch.Tensor, gate_col: int, up_col: int, cols: int) -> torch.Tensor:
    """round(silu(gate)) * up where gate = gu[..., gate_col : gate_col + cols] and up = gu[..., up_col : up_col + cols] are
    column blocks of one contiguous [..., width] projection output (no autograd: used inside the fused MLP function)."""
    return native().swiglu_rows(gu, gate_col, up_col, cols)


def swiglu_rows_backward(dh: torch.Tensor, gu: torch.Tensor, gate_col: int, up_col: int, cols: int) -> torch.Tensor:
    """d gate and d up of swiglu_rows, written into the same column blocks of a buffer shaped like `gu`; its other
    columns, if there are any, are zero."""
    return native().swiglu_rows_backward(dh, gu, gate_col, up_col, cols)


def _ce_fwd_bwd(logits, labels, ignore_index, overwrite: bool = False):
    """overwrite: the gradient replaces the logits in their own buffer (they must be contiguous)."""
    return native().ce_fwd_bwd(logits, labels, ignore_index, overwrite)


# --------------------------------------------------------------------------------------------
# torch.library registration
# --------------------------------------------------------------------------------------------
_LIBRARY = torch.library.Library("maltos", "DEF")
_IDS = "Tensor? q_pos, Tensor? k_pos, Tensor? q_seq, Tensor? k_seq"
_LIBRARY.define(f"attn_fwd(Tensor q, Tensor k, Tensor v, int mask_mode, float scale, {_IDS}) -> (Tensor, Tensor)")
_LIBRARY.define(
    f"attn_bwd(Tensor dout, Tensor q, Tensor k, Tensor v, Tensor o, Tensor lse, int mask_mode, float scale, {_IDS})"
    " -> (Tensor, Tensor, Tensor)"
)
_LIBRARY.define("rmsnorm_fwd(Tensor x, Tensor w, float eps) -> (Tensor, Tensor)")
_LIBRARY.define("rmsnorm_bwd(Tensor dy, Tensor x, Tensor w, Tensor rstd) -> (Tensor, Tensor)")
_LIBRARY.define("add_rmsnorm_fwd(Tensor x, Tensor res, Tensor w, float eps) -> (Tensor, Tensor, Tensor)")
_LIBRARY.define("add_rmsnorm_bwd(Tensor dy, Tensor dres, Tensor h, Tensor w, Tensor rstd) -> (Tensor, Tensor)")
_LIBRARY.define("rope(Tensor x, Tensor cos, Tensor sin, Tensor? positions, int position_offset, bool inverse) -> Tensor")
_LIBRARY.define("rope_pair(Tensor xa, Tensor xb, Tensor cos, Tensor sin, Tensor? positions, int position_offset, bool inverse) -> (Tensor, Tensor)")
_LIBRARY.define("swiglu_fwd(Tensor gate, Tensor up) -> Tensor")
_LIBRARY.define("swiglu_bwd(Tensor dh, Tensor gate, Tensor up) -> (Tensor, Tensor)")
_LIBRARY.define("ce_fwd_bwd(Tensor logits, Tensor labels, int ignore_index) -> (Tensor, Tensor, Tensor)")
_LIBRARY.define("scale_by_scalar(Tensor x, Tensor scale) -> Tensor")
_LIBRARY.define("scale_by_scalar_(Tensor(a!) x, Tensor scale) -> ()")


def _cpu_refusal(name: str) -> None:
    def refuse(*args, **kwargs):
        raise RuntimeError(f"maltos::{name} has no CPU implementation; move the tensors to the GPU")

    _LIBRARY.impl(name, refuse, "CPU")


for _name in ("attn_fwd", "attn_bwd", "rmsnorm_fwd", "rmsnorm_bwd", "add_rmsnorm_fwd", "add_rmsnorm_bwd", "rope", "rope_pair", "swiglu_fwd", "swiglu_bwd", "ce_fwd_bwd",
              "scale_by_scalar", "scale_by_scalar_"):
    _cpu_refusal(_name)


# fake (meta) kernels: shapes/dtypes only, so the ops can be traced or captured
@torch.library.register_fake("maltos::attn_fwd")
def _(q, k, v, mask_mode, scale, q_pos, k_pos, q_seq, k_seq):
    B, H, S, D = q.shape
    return q.new_empty((B, S, H, D)).transpose(1, 2), q.new_empty((B, H, S), dtype=torch.float32)


@torch.library.register_fake("maltos::attn_bwd")
def _(dout, q, k, v, o, lse, mask_mode, scale, q_pos, k_pos, q_seq, k_seq):
    def like(t):
        B, H, S, D = t.shape
        return t.new_empty((B, S, H, D)).transpose(1, 2)

    return like(q), like(k), like(v)


@torch.library.register_fake("maltos::rmsnorm_fwd")
def _(x, w, eps):
    return torch.empty_like(x), x.new_empty((x.numel() // max(1, x.size(-1)),), dtype=torch.float32)


@torch.library.register_fake("maltos::rmsnorm_bwd")
def _(dy, x, w, rstd):
    return torch.empty_like(x), torch.empty_like(w)


@torch.library.register_fake("maltos::add_rmsnorm_fwd")
def _(x, res, w, eps):
    return (torch.empty_like(x), torch.empty_like(x),
            x.new_empty((x.numel() // max(1, x.size(-1)),), dtype=torch.float32))


@torch.library.register_fake("maltos::add_rmsnorm_bwd")
def _(dy, dres, h, w, rstd):
    return torch.empty_like(h), torch.empty_like(w)


@torch.library.register_fake("maltos::rope")
def _(x, cos, sin, positions, position_offset, inverse):
    return torch.empty_like(x)


@torch.library.register_fake("maltos::rope_pair")
def _(xa, xb, cos, sin, positions, position_offset, inverse):
    return torch.empty_like(xa), torch.empty_like(xb)


@torch.library.register_fake("maltos::swiglu_fwd")
def _(gate, up):
    return torch.empty_like(gate)


@torch.library.register_fake("maltos::swiglu_bwd")
def _(dh, gate, up):
    return torch.empty_like(gate), torch.empty_like(up)


@torch.library.register_fake("maltos::ce_fwd_bwd")
def _(logits, labels, ignore_index):
    return (logits.new_empty((), dtype=torch.float32), torch.empty_like(logits),
            logits.new_empty((), dtype=torch.int32))


@torch.library.register_fake("maltos::scale_by_scalar")
def _(x, scale):
    return torch.empty_like(x)


@torch.library.register_fake("maltos::scale_by_scalar_")
def _(x, scale):
    return None


# --------------------------------------------------------------------------------------------
# public differentiable entry points
# --------------------------------------------------------------------------------------------
def attention(q, k, v, *, mask_mode: int = MASK_CAUSAL, scale: float | None = None, q_pos=None, k_pos=None, q_seq=None,
              k_seq=None, return_lse: bool = False):
    """Differentiable attention; k/v may have fewer heads than q (native GQA)."""
    o, lse = native().attention(q, k, v, mask_mode, scale, q_pos, k_pos, q_seq, k_seq)
    return (o, lse) if return_lse else o


def rms_norm(x: torch.Tensor, weight: torch.Tensor, eps: float) -> torch.Tensor:
    return native().rms_norm(x, weight, eps)


def add_rms_norm(x: torch.Tensor, residual: torch.Tensor, weight: torch.Tensor, eps: float) -> tuple[torch.Tensor, torch.Tensor]:
    """(h, y) with h = x + residual and y = rms_norm(h), in one pass and with the roundings of the two separate ops."""
    return native().add_rms_norm(x, residual, weight, eps)


def _rope_ids(x: torch.Tensor, positions: torch.Tensor | None) -> torch.Tensor | None:
    return None if positions is None or x.dim() != 4 else _ids32(positions, x.size(0), x.size(2), "position_ids")


def rope(x: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, *, positions: torch.Tensor | None = None,
         position_offset: int = 0) -> torch.Tensor:
    return native().rope(x, cos, sin, _rope_ids(x, positions), position_offset)


def rope_pair(xa: torch.Tensor, xb: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, *, positions: torch.Tensor | None = None,
              position_offset: int = 0) -> tuple[torch.Tensor, torch.Tensor]:
    """rope(xa), rope(xb) from one kernel launch (and one in the backward): bit-equal to two `rope` calls."""
    return native().rope_pair(xa, xb, cos, sin, _rope_ids(xa, positions), position_offset)


def rope_pair_(xa: torch.Tensor, xb: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, *, positions: torch.Tensor | None = None,
               position_offset: int = 0, inverse: bool = False) -> None:
    """`rope_pair` written over its inputs, outside autograd (`inverse` rotates back: the backward pass).  For buffers
    the caller owns, e.g. the gradients an attention backward has just produced."""
    native().rope_pair_(xa, xb, cos, sin, _rope_ids(xa, positions), position_offset, inverse)


def swiglu(gate: torch.Tensor, up: torch.Tensor) -> torch.Tensor:
    return native().swiglu(gate, up)


def cross_entropy(logits: torch.Tensor, labels: torch.Tensor, ignore_index: int = -100, *,
                  overwrite_logits: bool = False) -> torch.Tensor:
    """fp32 scalar: sum CE over supervised rows / max(1, #supervised rows).  overwrite_logits=True lets the gradient take
    the place of the (contiguous) logits, which the caller must not read afterwards."""
    if overwrite_logits:
        return native().cross_entropy_over_logits(logits, labels, ignore_index)
    return native().cross_entropy(logits, labels, ignore_index)


# --------------------------------------------------------------------------------------------
# optimizer-step launches (in place, no autograd)
# --------------------------------------------------------------------------------------------
def adamw_step_(p, g, m, v, *, lr: float, beta1: float, beta2: float, eps: float, weight_decay: float, step: int,
                p_lowp: torch.Tensor | None = None, grad_scale: float = 1.0, sq_norm: torch.Tensor | None = None,
                max_norm: float = 0.0) -> None:
    native().adamw_step_(p, g, m, v, lr, beta1, beta2, eps, weight_decay, step, p_lowp, grad_scale, sq_norm, max_norm)


def sq_norm(x: torch.Tensor, out: torch.Tensor | None = None) -> torch.Tensor:
    """float64 0-d tensor: sum of squares of a float32 tensor, accumulated in fp64."""
    return native().sq_norm(x, out)


def scale_(x: torch.Tensor, scale: float) -> torch.Tensor:
    return native().scale_(x, scale)


def list_sq_norm(xs: list[torch.Tensor]) -> torch.Tensor:
    """`sq_norm` over all of the float32 tensors together: one launch per 48 of them and one that adds the parts."""
    return native().list_sq_norm(xs)


def list_scale_(xs: list[torch.Tensor], scale: float) -> None:
    native().list_scale_(xs, scale)


def list_adamw_step_(p, g, m, v, *, lr: float, beta1: float, beta2: float, eps: float, weight_decay: float, step: int,
                     sq_norm: torch.Tensor | None = None, max_norm: float = 0.0) -> None:
    """`adamw_step_` over lists of tensors that share a step count: one launch per 48 of them."""
    native().list_adamw_step_(p, g, m, v, lr, beta1, beta2, eps, weight_decay, step, sq_norm, max_norm)


def grad_sum_slices(parts: torch.Tensor, out: torch.Tensor | None = None, *, accumulate: bool = False) -> torch.Tensor:
    """parts [slices, ...] -> sum over the slices, added in fp32 and rounded once; with `out` the result is written
    there (accumulate=True: added onto what `out` holds)."""
    return native().grad_sum_slices(parts, out, accumulate)


def grad_to_f32_(dst: torch.Tensor, src: torch.Tensor, *, accumulate: bool = False,
                 sq_out: torch.Tensor | None = None) -> torch.Tensor:
    """dst (=|+=) float(src) over flat buffers, optionally fusing the fp64 sum of squares of dst."""
    return native().grad_to_f32_(dst, src, accumulate, sq_out)
