"""Operands that lie at an odd element of a larger buffer (contiguous views, two bytes off a dword): the direct-to-LDS loads that fetch X, W, dY and A
give what they give at an aligned address.  Where such an operand moves a product to another kernel (the skinny operands of gemm_mid.hip, X and A
of the rank-r rings), sums differ in order only: 1e-3 of the result's norm, a few 16-bit roundings (2^-9 each in bfloat16) of its smaller values."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _off(t):
    flat = torch.zeros(t.numel() + 9, dtype=t.dtype, device="cuda")
    v = flat[1:1 + t.numel()].view(t.shape)
    assert v.data_ptr() % 4 == 2
    return v.copy_(t)


@pytest.mark.parametrize("M,K,N,r,p", [
    (6, 1024, 1024, 16, 0.0), (40, 1024, 1024, 16, 0.0),         # short forwards in one launch and in two
    (300, 1024, 1024, 16, 0.0), (300, 4096, 1024, 32, 0.0),      # the rank-r ring, the sliced pass
    (300, 4096, 1024, 16, 0.1), (300, 1024, 1024, 128, 0.0),
    (2048, 1024, 1024, 16, 0.1), (5000, 1024, 1024, 64, 0.1)])
def test_operands_at_odd_addresses(M, K, N, r, p):
    from lorafusion_amd.ops.lora_v1 import fused_linear_lora

    g = torch.Generator().manual_seed(M + r)
    rn = lambda *s, std=1.0: (torch.randn(*s, generator=g) * std).bfloat16().cuda()
    args = [rn(M, K), rn(N, K, std=0.02), rn(r, K, std=0.03), rn(N, r, std=0.05), rn(M, N)]

    def run(x, w, a, b, dy):
        x, a, b = (t.detach().requires_grad_() for t in (x, a, b))
        y = fused_linear_lora(x, w, a, b, 2.0, seed=3, dropout_p=p)
        return [y.detach(), *torch.autograd.grad(y, (x, a, b), dy)]

    ref = run(*args)
    for i, name in enumerate(("x", "w", "a", "b", "dy")):
        got = run(*[_off(t) if j == i else t for j, t in enumerate(args)])
        for t, e, out in zip(got, ref, ("y", "dx", "da", "db")):
            if name in ("w", "dy"):
                assert torch.equal(t, e), f"{name} off: {out}"
            else:
                assert float((t.float() - e.float()).norm()) <= 1e-3 * float(e.float().norm()), f"{name} off: {out}"
