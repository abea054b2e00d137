"""The rank-r product without a keep-mask in rings of direct loads (lora_xa_ring_kernel, csrc/lora_stream.hip) at its edges: row counts around its 16 rows and
the end of its range (4096), fewer and more steps of K than waves, both sides of the line to the sliced pass, ranks that fill the tiling and ranks
that do not, packed batches with padded rows.  Against float64; fp32 sums of 16-bit inputs differ by their final rounding, at most 2^-8 of a
value in bfloat16, so |err| <= 1e-2 (|e| + rms(e)) as in the other kernel tests."""

import pytest
import torch

from oracle import lora_ref
from tests.util import kernels_of

pytestmark = pytest.mark.gpu


def _close(got, exp):
    ok, rel, excess = lora_ref.check_close(got.float().cpu(), exp.float(), rtol=1e-2)
    assert ok, f"rel {rel:.3e} excess {excess:.3e}"


RING, SLICED, GENERAL = "lora_xa_ring_kernel", "lora_stream_kernel", "lora_xa_kernel"


@pytest.mark.parametrize("M,K,r,dtype,kernel", [
    (1, 128, 8, torch.bfloat16, RING), (15, 640, 16, torch.float16, RING), (17, 1152, 24, torch.bfloat16, RING), (333, 3968, 32, torch.bfloat16, RING),
    (513, 4096, 32, torch.bfloat16, RING), (333, 4096, 32, torch.float16, SLICED), (100, 8192, 16, torch.bfloat16, RING), (100, 8320, 16, torch.bfloat16, SLICED),
    (1025, 8320, 8, torch.float16, RING), (1000, 8192, 24, torch.bfloat16, SLICED), (4095, 256, 32, torch.bfloat16, RING), (4097, 256, 16, torch.bfloat16, GENERAL)])
def test_xa_ring(M, K, r, dtype, kernel):
    from lorafusion_amd import _lib as L
    from lorafusion_amd.ops import hip_ops

    g = torch.Generator().manual_seed(M + r)
    x, a = torch.randn(M + 1, K, generator=g).to(dtype), (torch.randn(r + 1, K, generator=g) * K ** -0.5).to(dtype)
    x[M], a[r] = float("nan"), float("nan")   # what lies beyond the operands must not reach the result
    xd, ad = x.cuda()[:M], a.cuda()[:r]
    s, names = kernels_of(lambda: hip_ops._xa(xd, None, [ad], L.single_routing(r, 2.0, 0.0), M, K, L.round_rank(r)))
    assert [k for k in (RING, SLICED, GENERAL) if k in names] == [kernel], names
    _close(s[:, :r], x[:M].double() @ a[:r].double().t())
    assert not s[:, r:].any()


@pytest.mark.parametrize("seq,ranks,K", [([1, 129, 64], [32, 8, 24], 512), ([130, 17], [8, 16], 1280)])
def test_xa_ring_packed(seq, ranks, K):
    from lorafusion_amd.ops import hip_ops
    from lorafusion_amd.ops.multi_lora import prepare_multi_lora_batch_info

    n = len(seq)
    info = prepare_multi_lora_batch_info(seq, list(range(n)), ranks, [0.0] * n, [1.0] * n, 128, output_dtype=torch.float32)
    routing = hip_ops.MultiRouting(info.padded_seq_len_list, ranks, info.block_to_lookup_table, info.block_to_alpha, info.block_to_dropout_p)
    g = torch.Generator().manual_seed(n)
    x = torch.randn(routing.M, K, generator=g).bfloat16()
    a = [(torch.randn(r, K, generator=g) * K ** -0.5).bfloat16() for r in ranks]
    xd, ad = x.cuda(), [t.cuda() for t in a]
    s, names = kernels_of(lambda: hip_ops._xa(xd, None, ad, routing.c, routing.M, K, routing.R))
    assert RING in names, names
    row = 0
    for q, pl, r, at in zip(seq, info.padded_seq_len_list, ranks, a):
        _close(s[row:row + q, :r], x[row:row + q].double() @ at.double().t())
        assert not s[row + q:row + pl].any() and not s[row:row + pl, r:].any(), "padded rows and rank columns are zero"
        row += pl
