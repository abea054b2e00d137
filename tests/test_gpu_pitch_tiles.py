"""Products planned on the persistent 256x256 tile that run on the eight-wave one because of their row pitch, and their neighbours that do not: which kernel ran, and
the result against float32, with a LoRA term, keep bits (NN) and ragged rows."""

import pytest
import torch

from oracle import lora_ref
from tests.util import kernels_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nn,M,N,K,kernel", [
    (False, 2800, 4096, 5120, "gemm_lora_kernel"), (False, 2800, 4096, 5248, "gemm_big_kernel"),   # a pitch of 10 KB and one beside it
    (False, 2800, 4096, 8192, "gemm_big_kernel"),                                                  # a power of two
    (True, 2800, 4096, 5120, "gemm_big_kernel"), (True, 2800, 4096, 16384, "gemm_lora_kernel")])
def test_kernel_and_result(nn, M, N, K, kernel):
    from lorafusion_amd.ops import hip_ops

    g = torch.Generator(device="cuda").manual_seed(K)
    rn = lambda *s, std=1.0: (torch.randn(*s, generator=g, device="cuda") * std).bfloat16()
    a, l = rn(M, K), rn(M, 16, std=0.1)
    if nn:
        w, r, keep = rn(K, N, std=0.02), rn(16, N, std=0.1), torch.rand(M, N, generator=g, device="cuda") >= 0.1
        out, names = kernels_of(lambda: hip_ops.fused_lora_dyw_dsa(a, w, l, r, 0.1, hip_ops.pack_mask(keep)))
        exp = a.float() @ w.float() + torch.where(keep, l.float() @ r.float() / 0.9, torch.zeros((), device="cuda"))
    else:
        w, r = rn(N, K, std=0.02), rn(N, 16, std=0.1)
        out, names = kernels_of(lambda: hip_ops.fused_lora_xw_sb(a, w, l, r, 2.0))
        exp = a.float() @ w.float().T + 2.0 * l.float() @ r.float().T
    assert [k for k in ("gemm_lora_kernel", "gemm_big_kernel", "gemm_mid_kernel") if k in names] == [kernel], names
    ok, rel, excess = lora_ref.check_close(out.float().cpu(), exp.cpu(), rtol=1e-2)
    assert ok, f"rel {rel:.3e} excess {excess:.3e}"
