"""Forwards without a keep-mask either side of the rule that slices their rank-r pass along K (up to 1024 rows: from K = 8320 at ranks to 16, above from 4096
up to 512 rows and from 8192 beyond), against fp32 sums of the same 16-bit inputs: one rounding of S and of Y (|err| <= 1e-2 (|e| + rms(e)))."""

import pytest
import torch

from oracle import lora_ref
from tests.util import kernels_of, single_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,r,dtype,sliced", [
    (129, 8192, 8, torch.bfloat16, False), (1024, 8192, 16, torch.float16, False), (1025, 8192, 16, torch.bfloat16, False), (200, 8064, 16, torch.bfloat16, False),
    (511, 4096, 32, torch.float16, True), (513, 4096, 24, torch.bfloat16, False), (130, 3968, 32, torch.bfloat16, False),
    (129, 8320, 8, torch.bfloat16, True), (1024, 8320, 16, torch.float16, True), (1025, 8320, 16, torch.bfloat16, False), (1024, 8192, 24, torch.bfloat16, True)])
def test_unmasked_pass(M, K, r, dtype, sliced):
    from lorafusion_amd.ops.lora_v1 import fused_linear_lora

    d = single_inputs(M, K, 256, r, p=0.0, seed=M + r, dtype=dtype)
    x, w, a, b = (d[k].cuda() for k in ("x", "w", "a", "b"))
    ye, _ = lora_ref.linear_lora_fwd_fp32(d["x"], d["w"], d["a"], d["b"], 2.0, None, 0.0)
    y, names = kernels_of(lambda: fused_linear_lora(x, w, a, b, 2.0))
    assert ("lora_stream_kernel" in names) == sliced and ("lora_xa_ring_kernel" in names) != sliced, names
    ok, rel, excess = lora_ref.check_close(y.float().cpu(), ye, rtol=1e-2)
    assert ok, f"Y: rel {rel:.3e} excess {excess:.3e}"
