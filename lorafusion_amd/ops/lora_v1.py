"""Single-adapter fused LoRA linear: ``fused_linear_lora`` / ``FusedLinearLoRA``.

Same call signature and gradient contract as lorafusion/ops/lora_v1.py:173-297; the work is one call into the host
module (csrc/host_ops.cpp: ``lf_lora_fwd`` / ``lf_lora_fwd_seeded``, and an autograd node whose backward is
``lf_lora_bwd``).

Differences from the reference, all deliberate:
 * the dropped input ``where(mask, x/(1-p), 0)`` is never stored: backward rebuilds it from
   ``x`` and the 1-byte keep-mask inside the kernels (saves an [M,K] tensor per layer);
 * 2-D ``x`` works (the reference only handles 3-D, lora_v1.py:207-232);
 * ``dropout_mask`` (keyword, optional) supplies the keep-mask explicitly; with ``None`` it is
   drawn from ``seed`` (random when ``seed`` is None, as at lora_v1.py:201-202);
 * the dropout scale is fp32 ``1/(1-p)`` in both directions (the reference rounds it to bf16
   in forward, dropout.py:58-63).
"""

from __future__ import annotations

import random

import torch

from lorafusion_amd import _lib as L
from lorafusion_amd.ops import hip_ops


def _validate_shapes(x2d, w_shape, w_dtype, lora_a, lora_b, linear_bias, dropout_p):
    """Shape / dtype checks of one LoRA linear; the base weight is given by shape and (dequantised) dtype."""
    for name, t in (("x", x2d), ("lora_a", lora_a), ("lora_b", lora_b)):
        L.require_gpu(t, name)
        if t.dtype != x2d.dtype:
            raise ValueError(f"{name} must have dtype {x2d.dtype}, but got {t.dtype}.")
    if w_dtype != x2d.dtype:
        raise ValueError(f"linear_w must have dtype {x2d.dtype}, but got {w_dtype}.")
    L.dtype_id(x2d.dtype)
    M, K = x2d.shape
    if len(w_shape) != 2 or w_shape[1] != K:
        raise ValueError(f"linear_w must have shape [N, {K}], but got {tuple(w_shape)}.")
    N = w_shape[0]
    if lora_a.ndim != 2 or lora_a.shape[1] != K:
        raise ValueError(f"lora_a must have shape [r, {K}], but got {tuple(lora_a.shape)}.")
    r = lora_a.shape[0]
    if tuple(lora_b.shape) != (N, r):
        raise ValueError(f"lora_b must have shape [{N}, {r}], but got {tuple(lora_b.shape)}.")
    if linear_bias is not None and (tuple(linear_bias.shape) != (N,) or linear_bias.dtype != x2d.dtype):
        raise ValueError(f"linear_bias must have shape [{N}] and dtype {x2d.dtype}.")
    hip_ops._check_dims(M, N, K)
    hip_ops._check_rank(r)
    hip_ops._check_p(dropout_p)
    return M, N, K, r


class FusedLinearLoRA:
    """``y = x W^T + alpha * (drop(x) A^T) B^T + bias`` with the LoRA term fused into the GEMMs."""

    @staticmethod
    def apply(x, linear_w, lora_a, lora_b, alpha, dropout_p, seed=None, linear_bias=None, dropout_mask=None):
        draw = None
        if dropout_p > 0 and dropout_mask is None:
            # the reference's default path: the keep-mask is drawn while X streams through the rank-r pass
            draw = (random.randrange(int(1e6)) if seed is None else int(seed)) & 0xFFFFFFFFFFFFFFFF  # noqa: S311
        return L.host().linear_lora(x, linear_w, lora_a, lora_b, alpha, dropout_p, draw, linear_bias, dropout_mask)


def fused_linear_lora(
    x: torch.Tensor,
    linear_w: torch.Tensor,
    lora_a: torch.Tensor,
    lora_b: torch.Tensor,
    alpha: float,
    seed: int | None = None,
    dropout_p: float = 0.0,
    linear_bias: torch.Tensor | None = None,
    dropout_mask: torch.Tensor | None = None,
) -> torch.Tensor:
    """Fused linear + LoRA (lorafusion/ops/lora_v1.py:284-297).

    ``alpha`` is the multiplier applied to the LoRA branch (PEFT's ``scaling``).
    """
    return FusedLinearLoRA.apply(x, linear_w, lora_a, lora_b, alpha, dropout_p, seed, linear_bias, dropout_mask)
