"""Front end of the fused QK-norm flash attention (HIP kernels behind a C ABI; checks, allocation, launch and the
autograd node are native code, csrc/torch_binding.cpp).

Two entry points share one implementation:

* ``QKNormFlashAttnFunc.apply(Q, K, V, gain, is_causal=True, q_start=0, ...)`` -- positional drop-in
  for the reference's ``TritonFlashAttnQKNormFunc``
  (sample_efficient_gpt/transformer/ops/triton_flash_attn_qknorm.py:262-343): flattened
  ``[(h b), S, d]`` tensors, gradients for ``Q, K, V, gain`` and ``None`` for the flags.  Optional
  trailing positionals switch on what the reference's caller does around the op
  (sample_efficient_gpt/transformer/attention.py:207-255): un-expanded GQA K/V, the value-residual
  mix, the per-head sigmoid gate, a k-side scale vector.
* ``qknorm_attention(q, k, v, g_q, ...)`` -- the same op on canonical ``[B, H, S, D]`` /
  ``[B, Hkv, S, D]`` views with keyword arguments.

Defaults follow the live module (attention.py:51-80): RMS normaliser, eps 1e-6 on the mean,
logits scaled by 1/sqrt(d).  ``eps=1e-8/d, sm_scale=1/d`` reproduces the fused Triton kernel's
own formula (triton_flash_attn_qknorm.py:67-91).
"""

from __future__ import annotations

import math
import threading

import torch

from . import _lib, _native

_DTYPES = {torch.bfloat16: _lib.SEGPT_DTYPE_BF16, torch.float32: _lib.SEGPT_DTYPE_FP32}


# ---- filling the C ABI's struct from Python, for callers that hold on to one (plan.py)

def _rope_arg(rope_cos, rope_sin, rope_q_pos0, rope_k_pos0, q_start, device, head_dim):
    """Normalise the rotary-embedding arguments to `(cos, sin, q_pos0, k_pos0)` (fp32 contiguous device tables
    of shape [len, head_dim // 2]) or None.  Query row i sits at position q_pos0 + i (default: q_start, as in
    the reference's caller, attention.py:191-204), key row j at k_pos0 + j."""
    if rope_cos is None and rope_sin is None:
        return None
    assert rope_cos is not None and rope_sin is not None, "rope_cos and rope_sin go together"
    cos = rope_cos.detach().to(device=device, dtype=torch.float32).contiguous()
    sin = rope_sin.detach().to(device=device, dtype=torch.float32).contiguous()
    assert cos.dim() == 2 and cos.shape == sin.shape and cos.shape[1] == head_dim // 2, "rope tables must be [len, head_dim // 2]"
    return cos, sin, int(q_start if rope_q_pos0 is None else rope_q_pos0), int(rope_k_pos0)


def _fill_common(p, q, k, v, y, lse, g_q, g_k, v_first, vr_coef, gate, gate_scale, eps, sm_scale, causal, q_start,
                 rope=None):
    B, H, Sq, D = q.shape
    p.dtype = _DTYPES[q.dtype]
    p.B, p.H, p.Hkv, p.Sq, p.Sk, p.D = B, H, k.shape[1], Sq, k.shape[2], D
    p.causal = int(bool(causal))
    p.q_start = int(q_start)
    p.gq_numel = g_q.numel()
    p.gk_numel = 0 if g_k is None else g_k.numel()
    p.eps, p.sm_scale, p.gate_scale = float(eps), float(sm_scale), float(gate_scale)
    p.q, p.k, p.v, p.o = _lib.t4(q), _lib.t4(k), _lib.t4(v), _lib.t4(y)
    p.v_first = _lib.t4(v_first)
    p.gate = _lib.t3(gate)
    p.lse = _lib.ptr(lse)
    p.g_q, p.g_k, p.vr_coef = _lib.ptr(g_q), _lib.ptr(g_k), _lib.ptr(vr_coef)
    if rope is not None:
        cos, sin, q_pos0, k_pos0 = rope
        p.rope_cos, p.rope_sin, p.rope_len = cos.data_ptr(), sin.data_ptr(), cos.shape[0]
        p.rope_q_pos0, p.rope_k_pos0 = q_pos0, k_pos0


def _no_backward_will_follow(*tensors):
    """True when nothing can ask for a gradient of this call: grad mode is off (torch.no_grad / inference_mode,
    as in the reference's generate loop, transformer.py:160) or no tensor input requires one.  Must be evaluated
    by the CALLER of an autograd Function: inside ``forward`` grad mode is always off, and
    ``ctx.needs_input_grad`` mirrors ``requires_grad`` even under no_grad (a Parameter gain keeps it True)."""
    return (not torch.is_grad_enabled()) or not any(t is not None and t.requires_grad for t in tensors)


class _GradModeAtApply:
    """Mix-in for the positional drop-in Functions: ``apply`` runs ``forward`` in the caller's grad mode (the autograd
    node is the native op's) and records there, for ``forward`` to read, whether a backward can follow."""

    _tls = threading.local()

    @classmethod
    @torch.compiler.disable  # native call and Python-side bookkeeping the compiler cannot trace: a compiled caller breaks the graph here
    def apply(cls, *args):
        outer = getattr(cls._tls, "inference", False)  # a nested apply must leave the outer call's decision in place
        cls._tls.inference = _no_backward_will_follow(*(a for a in args if isinstance(a, torch.Tensor)))
        try:
            return cls.forward(None, *args)
        finally:
            cls._tls.inference = outer

    @classmethod
    def _inference(cls):
        return bool(getattr(cls._tls, "inference", False))


def qknorm_attention(q, k, v, g_q, g_k=None, *, v_first=None, vr_coef=None, gate_logits=None, gate_scale=2.0,
                     eps=1e-6, sm_scale=None, causal=True, q_start=0, return_lse=False,
                     rope_cos=None, rope_sin=None, rope_q_pos0=None, rope_k_pos0=0, qk_norm=True, out_bshd=False):
    """Fused QK-norm attention on canonical views.

    q ``[B,H,Sq,D]``; k, v, v_first ``[B,Hkv,Sk,D]`` (any strides, last dim contiguous, rows 16 B
    aligned); g_q, g_k scale parameters of 1 or D elements; vr_coef device tensor ``[2]`` = (c1, c2)
    with ``v' = c1 v + c2 v_first``; gate_logits ``[B,Sq,H]`` with ``y = gate_scale*sigmoid(z)*o``.
    rope_cos / rope_sin ``[len, D/2]``: q and k are the UNROTATED projections and the split-half rotary
    embedding (rope.py:36-56) is applied inside the kernels' loads; query row i sits at position
    ``rope_q_pos0 + i`` (default ``q_start``), key row j at ``rope_k_pos0 + j``.
    ``qk_norm=False``: no RMS normalisation of q and k (eps unused) -- the reference's attention without QK-norm
    (attention.py:233-240); the scale vectors still apply, pass ``g_q = ones(1)`` for the plain op.
    ``out_bshd=True``: the returned ``[B,H,Sq,D]`` tensor is a view of a ``[B,Sq,H,D]`` buffer, so that
    ``y.permute(0, 2, 1, 3).reshape(B, Sq, H*D)`` is the ``b seq (h head_d)`` tensor of attention.py:243 without a copy.
    """
    inference = _no_backward_will_follow(q, k, v, g_q, g_k, v_first, vr_coef, gate_logits)
    y, lse = _attend(q, k, v, g_q, g_k, v_first, vr_coef, gate_logits, gate_scale, eps, sm_scale, causal, q_start, rope_cos, rope_sin,
                     rope_q_pos0, rope_k_pos0, qk_norm, inference, 0, 0, out_bshd, return_lse)
    return (y, lse) if return_lse else y


def _attend(q, k, v, g_q, g_k, v_first, vr_coef, gate_logits, gate_scale, eps, sm_scale, causal, q_start, rope_cos, rope_sin,
            rope_q_pos0, rope_k_pos0, qk_norm, inference, heads, kv_heads, out_bshd, with_lse):
    """The native call behind every function here: ``(y, lse)``; heads > 0: flattened ``[(h b), S, d]`` operands."""
    if torch.jit.is_tracing():
        # a tracer records operators only: the native call would leave the allocation of y in the graph and nothing that
        # fills it, so a traced caller gets the registered operator
        from . import library_op  # noqa: F401  (registers it)

        canon = (lambda t, n: None if t is None else _canon(t, n)) if heads else (lambda t, n: t)
        y, lse, _ = torch.ops.segpt.qknorm_attention(
            canon(q, heads), canon(k, kv_heads), canon(v, kv_heads), g_q, g_k, canon(v_first, kv_heads), vr_coef, gate_logits,
            float(gate_scale), float(eps), 1.0 / math.sqrt(q.shape[-1]) if sm_scale is None else float(sm_scale), bool(causal), int(q_start),
            rope_cos, rope_sin, -1 if rope_q_pos0 is None else int(rope_q_pos0), int(rope_k_pos0), bool(qk_norm), bool(out_bshd), inference)
        return (y.permute(1, 0, 2, 3).reshape(q.shape) if heads else y), lse
    return _native.load().attention(q, k, v, g_q, g_k, v_first, vr_coef, gate_logits, gate_scale, eps, sm_scale, causal, q_start, rope_cos,
                                    rope_sin, rope_q_pos0, rope_k_pos0, _call_flags(qk_norm, inference), heads, kv_heads, out_bshd, with_lse)


def _call_flags(qk_norm, inference):
    """SEGPT_FLAG_* bits of a call; `inference`: no backward will follow, so a forward with few query rows or few query
    tiles may split the keys."""
    return (0 if qk_norm else _lib.SEGPT_FLAG_NO_NORM) | (_lib.SEGPT_FLAG_DECODE if inference else 0)


def _canon(x, n_heads):
    """[(h b), S, d] -> [B, H, S, d] view (no copy): head-major flatten of attention.py:199."""
    n, S, d = x.shape
    return x.view(n_heads, n // n_heads, S, d).permute(1, 0, 2, 3)


def _flat_operands(Q, K, V, n_kv_heads, gate_logits):
    """The reference's checks on the flattened operands (triton_flash_attn_qknorm.py:273-281) and the head counts:
    ``(Q, K, V, H, Hkv)`` with 2-D tensors promoted to 3-D."""
    assert Q.is_cuda and Q.is_contiguous()
    assert K.is_cuda and K.is_contiguous()
    assert V.is_cuda and V.is_contiguous()
    if Q.ndim == 2:
        Q, K, V = Q.unsqueeze(0), K.unsqueeze(0), V.unsqueeze(0)
    nq, nk = Q.shape[0], K.shape[0]
    if n_kv_heads is None:
        assert nk == nq, "n_kv_heads is required for un-expanded GQA K/V"
        # without a gate every flattened row is its own (batch, head): plain MHA layout of the reference
        H = Hkv = 1 if gate_logits is None else gate_logits.shape[-1]
    else:
        Hkv = int(n_kv_heads)
        assert nq % nk == 0 and nk % Hkv == 0, "K/V rows must be n_kv_heads * batch"
        H = Hkv * (nq // nk)
    return Q, K, V, H, Hkv


class QKNormFlashAttnFunc(_GradModeAtApply, torch.autograd.Function):
    """Drop-in for ``TritonFlashAttnQKNormFunc`` (triton_flash_attn_qknorm.py:262-343).

    ``apply(Q, K, V, gain, is_causal=True, q_start=0, k_gain=None, v_first=None, vr_coef=None,
    gate_logits=None, gate_scale=2.0, n_kv_heads=None, eps=1e-6, sm_scale=None, rope_cos=None,
    rope_sin=None)`` -- positional only, as autograd Functions are.  With the rope tables Q and K are the
    unrotated projections (positions ``q_start + i`` for queries, ``j`` for keys, attention.py:191-204).  ``Q [(h b), Nq, d]``, ``K, V [(h b) or (hkv b), Nk, d]`` contiguous
    device tensors (2-D inputs are promoted to 3-D, the output stays 3-D, :278-281).  When K/V carry
    fewer rows than Q they are un-expanded GQA tensors and ``n_kv_heads`` is required; query row
    ``n = h*B + b`` then reads kv row ``(h // rep)*B + b`` exactly as the reference's
    ``repeat_interleave`` expansion does (attention.py:207-218).  Returns ``O`` with Q's shape and dtype.
    """

    @staticmethod
    def forward(ctx, Q, K, V, gain, is_causal=True, q_start=0, k_gain=None, v_first=None, vr_coef=None,
                gate_logits=None, gate_scale=2.0, n_kv_heads=None, eps=1e-6, sm_scale=None, rope_cos=None,
                rope_sin=None):
        promoted = Q.ndim == 2
        Q, K, V, H, Hkv = _flat_operands(Q, K, V, n_kv_heads, gate_logits)
        assert gain.is_cuda
        if v_first is not None:
            assert v_first.is_cuda and v_first.is_contiguous()
            if promoted and v_first.ndim == 2:
                v_first = v_first.unsqueeze(0)
        return _attend(Q, K, V, gain, k_gain, v_first, vr_coef, gate_logits, gate_scale, eps, sm_scale, is_causal, q_start, rope_cos,
                       rope_sin, None, 0, True, QKNormFlashAttnFunc._inference(), H, Hkv, False, False)[0]


class TritonFlashAttnQKNormFunc(QKNormFlashAttnFunc):
    """The reference's class name WITH the reference kernel's own formula as the default
    (triton_flash_attn_qknorm.py:67-91: L2 normaliser ``rsqrt(sum x^2 + 1e-8)``, logits ``gain * cos``), i.e. the
    family at ``eps = 1e-8 / d, sm_scale = 1 / d``.  ``QKNormFlashAttnFunc`` keeps the live module's defaults
    (RMS normaliser, eps 1e-6, 1/sqrt(d); attention.py:51-80).  Same positional signature; explicit ``eps`` /
    ``sm_scale`` override the defaults."""

    @staticmethod
    def forward(ctx, Q, K, V, gain, is_causal=True, q_start=0, k_gain=None, v_first=None, vr_coef=None,
                gate_logits=None, gate_scale=2.0, n_kv_heads=None, eps=None, sm_scale=None, rope_cos=None,
                rope_sin=None):
        d = Q.shape[-1]
        return QKNormFlashAttnFunc.forward(ctx, Q, K, V, gain, is_causal, q_start, k_gain, v_first, vr_coef, gate_logits,
                                           gate_scale, n_kv_heads, 1e-8 / d if eps is None else eps,
                                           1.0 / d if sm_scale is None else sm_scale, rope_cos, rope_sin)


class FlashAttnFunc(_GradModeAtApply, torch.autograd.Function):
    """Drop-in for the reference's attention WITHOUT QK-norm, ``TritonFlashAttnFunc``
    (triton_flash_attn.py:208-297; called at attention.py:240): ``apply(Q, K, V, q_start=0, is_causal=True,
    n_kv_heads=None)`` -- note the argument order, which differs from the QK-norm op's.  ``Q [(h b), Nq, d]``,
    ``K, V [(h b) or (hkv b), Nk, d]`` contiguous device tensors (2-D promoted to 3-D, :222-226); logits are
    ``Q K^T / sqrt(d)`` (:232).  Same kernels as the QK-norm op with both normalisers fixed at 1
    (SEGPT_FLAG_NO_NORM).  The reference backward's mis-masked diagonal tile (BQ=32 != BK=64,
    triton_flash_attn.py:176,292-293) is not reproduced: gradients are the exact ones."""

    @staticmethod
    def forward(ctx, Q, K, V, q_start=0, is_causal=True, n_kv_heads=None):
        Q, K, V, H, Hkv = _flat_operands(Q, K, V, n_kv_heads, None)
        one = torch.ones(1, dtype=torch.float32, device=Q.device)
        return _attend(Q, K, V, one, None, None, None, None, 1.0, 0.0, None, is_causal, q_start, None, None, None, 0, False,
                       FlashAttnFunc._inference(), H, Hkv, False, False)[0]
