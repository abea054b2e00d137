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


def test_weight_and_bias_make_the_result_differentiable():
    from lorafusion_amd import _lib as L

    x, w, a, b = torch.randn(4, 128), torch.randn(128, 128), torch.randn(16, 128), torch.randn(128, 16)
    r = L.single_routing(16, 1.0, 0.0)
    for which in range(3):
        others = [w.clone().requires_grad_(which == 0), None if which == 2 else torch.randn(128).requires_grad_(which == 1)]
        y = L.host().attach(torch.zeros(4, 128), [x], x, w, 0, others, [a], [b], None, torch.zeros(4, 16), None, [], ctypes.addressof(r), [], 16, "Node")
        assert y.requires_grad == (which < 2)
        assert which == 2 or len(y.grad_fn.next_functions) == 5


@pytest.mark.gpu
@pytest.mark.parametrize("which", ["linear_w", "linear_bias"])
def test_backward_from_a_result_that_only_weight_or_bias_makes_differentiable(which):
    """It runs, and leaves both without a gradient."""
    from lorafusion_amd.ops.lora_v1 import fused_linear_lora
    from lorafusion_amd.ops.multi_lora import fused_linear_multi_lora, prepare_multi_lora_batch_info
    from lorafusion_amd.ops.nf4 import fused_linear_lora_nf4, quantize_nf4
    from lorafusion_amd.ops.swiglu_lora import fused_swiglu_linear_lora

    t = lambda *s: torch.randn(*s, device="cuda", dtype=torch.bfloat16)
    M, K, N, r = 128, 256, 128, 16
    x, gu, w, bias, a, b = t(M, K), t(M, 2 * K), t(N, K), t(N), t(r, K), t(N, r)
    codes, state = quantize_nf4(w)
    frozen = {"linear_w": w, "linear_bias": bias}[which].requires_grad_()
    info = prepare_multi_lora_batch_info([M], [0], [r], [0.0], [2.0], 128)
    kw = dict(lora_a_list=[a], lora_b_list=[b], seq_len_list=[M], padded_seq_len_list=[M], block_to_lookup_table=info.block_to_lookup_table,
              block_to_dropout_p=info.block_to_dropout_p, block_to_alpha=info.block_to_alpha, enable_dropout=False, same_dropout_p_value=0.0,
              max_r=r, linear_bias=bias)
    calls = [lambda: fused_linear_lora(x, w, a, b, 2.0, linear_bias=bias), lambda: fused_linear_multi_lora(x[None], w, **kw),
             lambda: fused_swiglu_linear_lora(gu, w, a, b, 2.0, linear_bias=bias)]
    if which == "linear_bias":
        calls += [lambda: fused_linear_lora_nf4(x, codes, state, a, b, 2.0, linear_bias=bias),
                  lambda: fused_linear_multi_lora(x[None], codes, quant_state=state, **kw)]
    for call in calls:
        y = call()
        y.backward(torch.ones_like(y))
        assert frozen.grad is None
        (call().sum() + frozen.sum()).backward()
        assert torch.equal(frozen.grad, torch.ones_like(frozen))
        frozen.grad = None


@pytest.mark.gpu
def test_a_mask_that_changes_before_the_backward_is_noticed():
    from lorafusion_amd.ops import hip_ops
    from lorafusion_amd.ops.lora_v1 import fused_linear_lora

    t = lambda *s: torch.randn(*s, device="cuda", dtype=torch.bfloat16)
    x, w, a, b = t(2, 64, 256).requires_grad_(), t(128, 256), t(16, 256), t(128, 16)
    bits = hip_ops.pack_mask(torch.rand(128, 256, device="cuda") >= 0.1)
    for mask in (bits, bits.view(2, 64, 32)):
        y = fused_linear_lora(x, w, a, b, 1.0, dropout_p=0.1, dropout_mask=mask)
        mask.zero_()
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            y.sum().backward()


@pytest.mark.gpu
@pytest.mark.parametrize("copied", [True, False])
def test_activation_inputs_that_change_before_the_backward(copied):
    """Inputs the kernel cannot read as they lie are copied for it, and the backward works on the copies; others are the caller's, and noticed."""
    from lorafusion_amd.ops.norm_act import silu_mul

    t = lambda: torch.randn(64, 128, device="cuda", dtype=torch.bfloat16)
    a, b = (t().t().contiguous().t() if copied else t() for _ in range(2))
    dc = t()
    grads = lambda: torch.autograd.grad(silu_mul(x, y), (x, y), dc)
    x, y = a.requires_grad_(), b.requires_grad_()
    expect = grads()
    c = silu_mul(x, y)
    with torch.no_grad():
        x.zero_(), y.zero_()
    if not copied:
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            torch.autograd.grad(c, (x, y), dc)
        return
    for g, e in zip(torch.autograd.grad(c, (x, y), dc), expect):
        assert torch.equal(g, e)


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
