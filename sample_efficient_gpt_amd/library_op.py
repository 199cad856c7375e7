"""`torch.library` registration of the fused QK-norm attention, so that the op survives `torch.compile`
(the reference compiles the whole model, sample_efficient_gpt/training/trainer.py:227-228) and
non-reentrant activation checkpointing (transformer/transformer.py:123-132) as ONE opaque node with a fake
(shape-only) implementation instead of being traced into.

    y = torch.ops.segpt.qknorm_attention(q, k, v, g_q, g_k, v_first, vr_coef, gate_logits,
                                         gate_scale, eps, sm_scale, causal, q_start,
                                         rope_cos, rope_sin, rope_q_pos0, rope_k_pos0, qk_norm, out_bshd,
                                         inference)[0]

or the keyword wrapper ``qknorm_attention_op(...)`` below.  Canonical layout: q ``[B,H,Sq,D]``, k / v /
v_first ``[B,Hkv,Sk,D]`` (any strides, last dim contiguous), gate_logits ``[B,Sq,H]``; the optional tensors
are ``None`` when unused (rope_q_pos0 = -1 means "q_start"); ``inference=True`` promises that no backward
follows (decode-shaped calls may then take the split-key kernels, whose key/value workspace holds no keys).  Returns ``(y, lse, kv_ws)``: the output, the fp32 log-sum-exp ``[B,H,Sq]`` and the
key/value workspace the backward reuses.  Same kernels and C ABI as ``function.py``; no fallback.
"""

from __future__ import annotations

import math
from typing import List, Optional

import torch
from torch import Tensor

from . import _native
from .function import _call_flags, _no_backward_will_follow, qknorm_attention

__all__ = ["qknorm_attention_op"]


def _empty_out(q, out_bshd):
    """Output buffer [B,H,Sq,D]: contiguous, or (out_bshd) a view of a [B,Sq,H,D] buffer, the layout the
    output projection consumes (attention.py:243)."""
    B, H, Sq, D = q.shape
    if out_bshd:
        return q.new_empty((B, Sq, H, D)).permute(0, 2, 1, 3)
    return q.new_empty((B, H, Sq, D))


@torch.library.custom_op("segpt::qknorm_attention", mutates_args=())
def _fwd_op(q: Tensor, k: Tensor, v: Tensor, g_q: Tensor, g_k: Optional[Tensor], v_first: Optional[Tensor],
            vr_coef: Optional[Tensor], gate_logits: Optional[Tensor], gate_scale: float, eps: float, sm_scale: float,
            causal: bool, q_start: int, rope_cos: Optional[Tensor], rope_sin: Optional[Tensor],
            rope_q_pos0: int, rope_k_pos0: int, qk_norm: bool, out_bshd: bool, inference: bool) -> List[Tensor]:
    y, lse, kv_ws = _native.load().op_forward(
        q, k, v, g_q, g_k, v_first, vr_coef, gate_logits, gate_scale, eps, sm_scale, causal, q_start, rope_cos, rope_sin,
        None if rope_q_pos0 < 0 else rope_q_pos0, rope_k_pos0, _call_flags(qk_norm, inference), _empty_out(q, out_bshd))
    if inference:  # no backward will read it (and after the decode kernels it holds no keys)
        kv_ws = q.new_empty((0,), dtype=torch.uint8)
    return [y, lse, kv_ws]


@_fwd_op.register_fake
def _(q, k, v, g_q, g_k, v_first, vr_coef, gate_logits, gate_scale, eps, sm_scale, causal, q_start,
      rope_cos, rope_sin, rope_q_pos0, rope_k_pos0, qk_norm, out_bshd, inference):
    B, H, Sq, D = q.shape
    y = _empty_out(q, out_bshd)
    lse = q.new_empty((B, H, Sq), dtype=torch.float32)
    # normalised keys (+ mixed values) of the bf16 path, rounded up to 256 bytes each; 256 bytes otherwise
    nbytes = 256
    if q.numel() == 0 or inference:
        nbytes = 0
    elif q.dtype == torch.bfloat16:
        piece = (k.shape[0] * k.shape[1] * k.shape[2] * D * 2 + 255) // 256 * 256
        nbytes = piece * (2 if v_first is not None else 1)
    return [y, lse, q.new_empty((nbytes,), dtype=torch.uint8)]


@torch.library.custom_op("segpt::qknorm_attention_backward", mutates_args=())
def _bwd_op(dy: Tensor, q: Tensor, k: Tensor, v: Tensor, g_q: Tensor, g_k: Optional[Tensor], v_first: Optional[Tensor],
            vr_coef: Optional[Tensor], gate_logits: Optional[Tensor], y: Tensor, lse: Tensor, kv_ws: Tensor,
            gate_scale: float, eps: float, sm_scale: float, causal: bool, q_start: int,
            rope_cos: Optional[Tensor], rope_sin: Optional[Tensor], rope_q_pos0: int, rope_k_pos0: int,
            qk_norm: bool) -> List[Tensor]:
    """Returns [dq, dk, dv, dg_q, dg_k, dv_first, dvr_coef, dgate]; absent ones are empty tensors."""
    grads = _native.load().op_backward(
        dy, q, k, v, g_q, g_k, v_first, vr_coef, gate_logits, y, lse, kv_ws, gate_scale, eps, sm_scale, causal, q_start,
        rope_cos, rope_sin, None if rope_q_pos0 < 0 else rope_q_pos0, rope_k_pos0, _call_flags(qk_norm, False))
    # an absent operand's place is a fresh tensor each: returns of a custom op must not alias one another
    return [q.new_empty((0,)) if g is None else g for g in grads]


@_bwd_op.register_fake
def _(dy, q, k, v, g_q, g_k, v_first, vr_coef, gate_logits, y, lse, kv_ws, gate_scale, eps, sm_scale, causal, q_start,
      rope_cos, rope_sin, rope_q_pos0, rope_k_pos0, qk_norm):
    none = lambda: q.new_empty((0,))
    return [torch.empty_like(q), torch.empty_like(k), torch.empty_like(v), torch.empty_like(g_q),
            none() if g_k is None else torch.empty_like(g_k),
            none() if v_first is None else torch.empty_like(v_first),
            none() if vr_coef is None else torch.empty_like(vr_coef),
            none() if gate_logits is None else torch.empty_like(gate_logits)]


def _setup_context(ctx, inputs, output):
    (q, k, v, g_q, g_k, v_first, vr_coef, gate_logits, gate_scale, eps, sm_scale, causal, q_start,
     rope_cos, rope_sin, rope_q_pos0, rope_k_pos0, qk_norm, out_bshd, _inference) = inputs
    y, lse, kv_ws = output
    ctx.save_for_backward(q, k, v, g_q, g_k, v_first, vr_coef, gate_logits, y, lse, kv_ws, rope_cos, rope_sin)
    ctx.cfg = (gate_scale, eps, sm_scale, causal, q_start, rope_q_pos0, rope_k_pos0, qk_norm)


def _autograd_backward(ctx, grads):
    dy = grads[0]
    q, k, v, g_q, g_k, v_first, vr_coef, gate_logits, y, lse, kv_ws, rope_cos, rope_sin = ctx.saved_tensors
    gate_scale, eps, sm_scale, causal, q_start, rope_q_pos0, rope_k_pos0, qk_norm = ctx.cfg
    dq, dk, dv, dg_q, dg_k, dvf, dcoef, dgate = torch.ops.segpt.qknorm_attention_backward(
        dy, q, k, v, g_q, g_k, v_first, vr_coef, gate_logits, y, lse, kv_ws, gate_scale, eps, sm_scale, causal, q_start,
        rope_cos, rope_sin, rope_q_pos0, rope_k_pos0, qk_norm)
    return (dq, dk, dv, dg_q, None if g_k is None else dg_k, None if v_first is None else dvf,
            None if vr_coef is None else dcoef, None if gate_logits is None else dgate, None, None, None, None, None,
            None, None, None, None, None, None, None)


_fwd_op.register_autograd(_autograd_backward, setup_context=_setup_context)


def _seen_as_operator(*operands):
    """Somebody looks at the call as an operator: a compiler, a tracer (torch.jit.trace), a dispatch or function mode (a
    selective-checkpoint policy, fake tensors), a function transform (vmap, torch.func.grad) or an operand of a tensor
    subclass."""
    return (torch.compiler.is_compiling() or torch.jit.is_tracing() or torch._C._len_torch_dispatch_stack() or torch._C._len_torch_function_stack()
            or torch._C._are_functorch_transforms_active()
            or any(t is not None and type(t) not in (Tensor, torch.nn.Parameter) for t in operands))


def qknorm_attention_op(q, k, v, g_q, g_k=None, *, v_first=None, vr_coef=None, gate_logits=None, gate_scale=2.0,
                        eps=1e-6, sm_scale=None, causal=True, q_start=0, return_lse=False,
                        rope_cos=None, rope_sin=None, rope_q_pos0=None, rope_k_pos0=0, qk_norm=True, out_bshd=False):
    """Keyword front end of ``torch.ops.segpt.qknorm_attention`` (same arguments as ``qknorm_attention``)."""
    if q.is_cuda and not _seen_as_operator(q, k, v, g_q, g_k, v_first, vr_coef, gate_logits, rope_cos, rope_sin):
        # the same kernels without the registered op's 45 us of Python dispatch
        return qknorm_attention(q, k, v, g_q, g_k, v_first=v_first, vr_coef=vr_coef, gate_logits=gate_logits, gate_scale=gate_scale,
                                eps=eps, sm_scale=sm_scale, causal=causal, q_start=q_start, return_lse=return_lse, rope_cos=rope_cos,
                                rope_sin=rope_sin, rope_q_pos0=rope_q_pos0, rope_k_pos0=rope_k_pos0, qk_norm=qk_norm, out_bshd=out_bshd)
    if sm_scale is None:
        sm_scale = 1.0 / math.sqrt(q.shape[-1])
    # decided here, in the caller's grad mode: a forward-only call (the reference's generate loop runs under
    # inference_mode, transformer.py:160) with few query rows takes the split-key decode kernels
    inference = _no_backward_will_follow(q, k, v, g_q, g_k, v_first, vr_coef, gate_logits)
    y, lse, _ = torch.ops.segpt.qknorm_attention(q, k, v, g_q, g_k, v_first, vr_coef, gate_logits, float(gate_scale),
                                                 float(eps), float(sm_scale), bool(causal), int(q_start),
                                                 rope_cos, rope_sin, -1 if rope_q_pos0 is None else int(rope_q_pos0),
                                                 int(rope_k_pos0), bool(qk_norm), bool(out_bshd), bool(inference))
    return (y, lse) if return_lse else y
