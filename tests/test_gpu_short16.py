"""The short forward in one launch (short16_fwd_kernel, csrc/lora_stream.hip): up to 16 rows and rank 32, at the edges of its forms: fewer steps of
K than waves, uneven and many of them, groups of 16 and 64 columns and both sides of the line between them, ranks that fill the tiling and
ranks that do not, the first shapes behind its rule, and that the one launch (or the two) ran.  Against the oracle with fp32 sums from the same 16-bit inputs; tolerance |err| <= 1e-2
(|e| + rms(e)): one 16-bit rounding of S and one of Y are at most 2^-8 = 0.4 % of each in bfloat16."""

import pytest
import torch

from oracle import lora_ref
from tests.util import kernels_of, single_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,N,r,dtype,bias,launches", [
    (1, 128, 128, 8, torch.bfloat16, True, 1), (16, 128, 4224, 32, torch.float16, True, 1), (5, 640, 384, 24, torch.float16, False, 1),
    (15, 1152, 4096, 16, torch.bfloat16, True, 1), (9, 4096, 4224, 16, torch.bfloat16, False, 1), (16, 2048, 4352, 24, torch.bfloat16, True, 1),
    (6, 7168, 3072, 32, torch.float16, True, 1), (2, 6144, 256, 8, torch.bfloat16, False, 1), (3, 256, 16384, 32, torch.bfloat16, True, 1),
    (17, 256, 256, 16, torch.bfloat16, True, 2), (4, 256, 256, 40, torch.float16, False, 2), (4, 6272, 256, 8, torch.bfloat16, False, 2),
    (4, 256, 16512, 16, torch.float16, True, 2)])
def test_short16(M, K, N, r, dtype, bias, launches):
    from lorafusion_amd import _lib as L
    from lorafusion_amd.ops import hip_ops

    d = single_inputs(M, K, N, r, p=0.0, seed=M + K, dtype=dtype, bias=bias)
    # one row more on every side of what the call is given: what lies beyond must not reach the results
    x, a = (torch.cat([d[k], torch.full_like(d[k][:1], float("nan"))]).cuda()[:-1] for k in ("x", "a"))
    w, b, bias_t = d["w"].cuda(), d["b"].cuda(), d["bias"].cuda() if bias else None
    (y, s), names = kernels_of(lambda: hip_ops.lora_forward(x, w, [a], [b], L.single_routing(r, 0.5, 0.0), L.round_rank(r), None, bias_t))
    assert ("short16_fwd_kernel" in names, "short_fwd_finish_kernel" in names) == ((launches == 1), (launches == 2)), names
    ye, se = lora_ref.linear_lora_fwd_fp32(d["x"], d["w"], d["a"], d["b"], 0.5, None, 0.0, d["bias"])
    for got, exp, name in ((y, ye, "Y"), (s[:, :r], se, "S")):
        ok, rel, excess = lora_ref.check_close(got.float().cpu(), exp, rtol=1e-2)
        assert ok, f"{name}: rel {rel:.3e} excess {excess:.3e}"
    assert not s[:, r:].any()


@pytest.mark.parametrize("r", [8, 16, 24, 32])
@pytest.mark.parametrize("N", [256, 4224])
def test_infinities_stay_infinities(r, N):
    """An infinity in X against positive columns of W, A and B is an infinity in Y, at ranks below the kernel's tiling too, where the rank columns
    behind the last are zeros times X; the other rows are untouched."""
    from lorafusion_amd import _lib as L
    from lorafusion_amd.ops import hip_ops

    M, K = 5, 512
    d = single_inputs(M, K, N, r, p=0.0, seed=r)
    x, w, a, b = d["x"], d["w"], d["a"], d["b"].abs()
    x[1, 7], x[3, 400] = float("inf"), float("-inf")
    for c in (7, 400):
        w[:, c], a[:, c] = w[:, c].abs() + 0.01, a[:, c].abs() + 0.01
    y, s = hip_ops.lora_forward(x.cuda(), w.cuda(), [a.cuda()], [b.cuda()], L.single_routing(r, 0.5, 0.0), L.round_rank(r), None, None)
    y, s = y.float().cpu(), s.float().cpu()
    for row, inf in ((1, float("inf")), (3, float("-inf"))):
        assert bool((y[row] == inf).all()) and bool((s[row, :r] == inf).all())
    assert not s[:, r:].any()
    ye, _ = lora_ref.linear_lora_fwd_fp32(x, w, a, b, 0.5, None, 0.0, None)
    ok, rel, excess = lora_ref.check_close(y[[0, 2, 4]], ye[[0, 2, 4]], rtol=1e-2)
    assert ok, f"rel {rel:.3e} excess {excess:.3e}"
