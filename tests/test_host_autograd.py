"""What the autograd nodes of the host module refuse or pass on: forward-mode tangents (the kernels read values alone, a tangent
would be lost without a word), inputs without columns (their row count is a division), saved-tensor hooks."""

import ctypes

import pytest
import torch
import torch.autograd.forward_ad as fwd


def _attach(x, a, b):
    from lorafusion_amd import _lib as L

    r = L.single_routing(16, 1.0, 0.0)
    return L.host().attach(torch.zeros(4, 128), [x], x.detach(), torch.zeros(128, 128), 0, [], [a], [b], None, torch.zeros(4, 16), None, [],
                           ctypes.addressof(r), [], 16, "Node")


@pytest.mark.parametrize("which", [0, 1, 2])
def test_tangents_are_refused(which):
    ops = [torch.randn(4, 128), torch.randn(16, 128), torch.randn(128, 16)]
    with fwd.dual_level():
        ops[which] = fwd.make_dual(ops[which], torch.ones_like(ops[which]))
        with pytest.raises(NotImplementedError, match="forward-mode"):
            _attach(*ops)


def test_saved_tensor_hooks_run_and_raise_through():
    class Stop(Exception):
        pass

    def pack(_):
        raise Stop

    ops = [torch.randn(s, requires_grad=True) for s in ((4, 128), (16, 128), (128, 16))]
    with pytest.raises(Stop), torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t):
        _attach(*ops)
    seen = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: seen.append(tuple(t.shape)), lambda t: t):
        assert _attach(*ops).requires_grad
    assert {(4, 128), (16, 128), (128, 16), (128, 128), (4, 16)} <= set(seen)


@pytest.mark.gpu
def test_public_functions_refuse_tangents_and_empty_rows():
    from lorafusion_amd.ops.lora_v1 import fused_linear_lora
    from lorafusion_amd.ops.norm_act import rms_norm, silu_mul, silu_mul_merged

    t = lambda *s: torch.randn(*s, device="cuda", dtype=torch.bfloat16)
    x, w, a, b = t(4, 256), t(128, 256), t(16, 256), t(128, 16)
    with fwd.dual_level():
        dual = fwd.make_dual(x, torch.ones_like(x))
        for call in (lambda: fused_linear_lora(dual, w, a, b, 1.0), lambda: rms_norm(dual, w[0].contiguous()), lambda: silu_mul(dual, x),
                     lambda: silu_mul_merged(dual)):
            with pytest.raises(NotImplementedError, match="forward-mode"):
                call()
    for call in (lambda: rms_norm(t(4, 0), t(0)), lambda: silu_mul_merged(t(4, 0))):
        with pytest.raises(RuntimeError):
            call()
