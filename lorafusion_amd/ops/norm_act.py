"""RMSNorm and SiLU-multiply on the HIP kernels: the steps either side of a decoder layer's LoRA linears.

The reference swaps HF's RMSNorm and SwiGLU MLP for the liger-kernel package's
(``apply_liger_kernel``, lorafusion/utils/module.py:41-71); the names below follow that package's
(``LigerRMSNormFunction`` / ``LigerRMSNorm``, ``LigerSiLUMulFunction`` / ``LigerSwiGLUMLP``), the arithmetic its
"llama" casting mode.  ``silu_mul_merged`` is an addition for merged gate/up projections: it reads the two halves
of one ``[M, 2I]`` tensor in place and its backward writes the gradient of that tensor directly (no split / cat
copies around the activation).
"""

from __future__ import annotations

import torch
from torch import nn

from lorafusion_amd import _lib as L


class RMSNormFunction:
    """y = round16(round16(x * rstd) * w), rstd = 1/sqrt(mean(x^2) + eps) in fp32 (HF LlamaRMSNorm's arithmetic)."""

    @staticmethod
    def apply(x: torch.Tensor, w: torch.Tensor, eps: float) -> torch.Tensor:
        return L.host().rms_norm(x, w, eps)


def rms_norm(x: torch.Tensor, weight: torch.Tensor, eps: float = 1e-6) -> torch.Tensor:
    return RMSNormFunction.apply(x, weight, eps)


class RMSNorm(nn.Module):
    """Drop-in for HF ``LlamaRMSNorm`` / liger's ``LigerRMSNorm`` (offset 0, "llama" casting)."""

    def __init__(self, hidden_size: int, eps: float = 1e-6, device=None, dtype=None) -> None:
        super().__init__()
        self.weight = nn.Parameter(torch.ones(hidden_size, device=device, dtype=dtype))
        self.variance_epsilon = eps

    def forward(self, hidden_states: torch.Tensor) -> torch.Tensor:
        return rms_norm(hidden_states, self.weight, self.variance_epsilon)

    def extra_repr(self) -> str:
        return f"{tuple(self.weight.shape)}, eps={self.variance_epsilon}"


class SiLUMulFunction:
    """c = silu(a) * b with a, b separate tensors (or views: row strides are honoured)."""

    @staticmethod
    def apply(a: torch.Tensor, b: torch.Tensor) -> torch.Tensor:
        return L.host().silu_mul(a, b)


class SiLUMulMergedFunction:
    """c = silu(gu[..., :I]) * gu[..., I:] for a merged gate/up tensor ``gu`` [.., 2I]; the backward writes d(gu)."""

    @staticmethod
    def apply(gu: torch.Tensor) -> torch.Tensor:
        return L.host().silu_mul_merged(gu)


def silu_mul(a: torch.Tensor, b: torch.Tensor) -> torch.Tensor:
    return SiLUMulFunction.apply(a, b)


def silu_mul_merged(gate_up: torch.Tensor) -> torch.Tensor:
    return SiLUMulMergedFunction.apply(gate_up)


def swiglu_mlp_forward(mlp: nn.Module, x: torch.Tensor) -> torch.Tensor:
    """``down_proj(silu(gate_proj(x)) * up_proj(x))`` of an HF Llama / Qwen2 MLP (what liger's ``LigerSwiGLUMLP``
    computes), through whatever the three projections are.  A ``down_proj`` that is a LoRA linear on the fused ops
    (a PEFT layer under ``apply_lora``, or ``LoRALinear``) takes the activation as the prologue of its first kernel."""
    from lorafusion_amd.patch import patch_lora

    gate, up = mlp.gate_proj(x), mlp.up_proj(x)
    down = mlp.down_proj
    fused = getattr(down, "use_fused", None)
    if fused is None:
        fused = getattr(type(down), "_lorafusion_use_fused", None)
    if fused and patch_lora._is_lora_linear(down) and gate.shape[-1] % 128 == 0:
        return patch_lora.swiglu_lora_forward(down, gate, up, use_fused=True)
    return down(silu_mul(gate, up))
