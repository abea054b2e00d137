"""dA = dS^T drop(X) in one launch, without fp32 partials: short segments, where a workgroup walks all row blocks of its segment over one
or two tiles of columns.  Row blocks that end ragged, one to five blocks per segment (ring and dS buffers wrap), column tiles that
do not divide by the slices, every rank tiling, both types, no mask and a mask in both formats (the same result).  Against fp32 sums of the same 16-bit inputs (|err| <= 1e-2 (|e| + rms(e)): one 16-bit rounding of the result)."""

import pytest
import torch

from oracle import lora_ref
from tests.util import kernels_of

pytestmark = pytest.mark.gpu


def _close(got, exp, name):
    ok, rel, excess = lora_ref.check_close(got.detach().float().cpu(), exp, rtol=1e-2)
    assert ok, f"{name}: rel {rel:.3e} excess {excess:.3e}"


def _direct(fn):
    """What ``fn`` returns, from one launch: no second stage over partial sums."""
    out, names = kernels_of(fn)
    assert "lora_da_ring_kernel" in names and "reduce_segments_kernel" not in names, names
    return out


@pytest.mark.parametrize("M,K,r,dtype", [
    (1, 256, 16, torch.bfloat16), (127, 1152, 8, torch.float16), (128, 16640, 16, torch.bfloat16),   # 260 column tiles: two per workgroup
    (129, 4096, 32, torch.bfloat16), (300, 4096, 16, torch.bfloat16), (300, 8192, 64, torch.float16), (385, 14336, 48, torch.bfloat16),
    (300, 14336, 128, torch.bfloat16), (600, 14336, 64, torch.bfloat16)])
@pytest.mark.parametrize("p", [0.0, 0.2])
def test_one_segment(M, K, r, dtype, p):
    from lorafusion_amd.ops import hip_ops

    g = torch.Generator().manual_seed(M + K)
    x, ds = torch.randn(M, K, generator=g).to(dtype), (torch.randn(M, r, generator=g) * 0.1).to(dtype)
    keep = torch.rand(M, K, generator=g) >= p
    exp = ds.float().T @ torch.where(keep, x.float(), torch.zeros(())) / (1 - p)
    m = keep.cuda() if p else None
    xd, dsd, bits = x.cuda(), ds.cuda(), hip_ops.pack_mask(m) if p else None
    da = _direct(lambda: hip_ops.fused_lora_da(xd, dsd, r, p, bits))
    _close(da, exp, "bits" if p else "no mask")
    if p:
        assert torch.equal(da, _direct(lambda: hip_ops.fused_lora_da(xd, dsd, r, p, m)))


@pytest.mark.parametrize("seq,ranks,p_list,K", [
    ([100, 256, 300, 1], [8, 16, 64, 32], [0.0, 0.1, 0.2, 0.1], 4096),
    ([128, 640, 37], [128, 16, 40], [0.1, 0.1, 0.0], 8192),
    ([130] * 8, [16] * 8, [0.0] * 8, 4096),                                       # 512 tiles for 256 workgroups: two each
])
def test_segments(seq, ranks, p_list, K):
    from lorafusion_amd import _lib as L
    from lorafusion_amd.ops import hip_ops
    from lorafusion_amd.ops.multi_lora import prepare_multi_lora_batch_info

    n = len(seq)
    info = prepare_multi_lora_batch_info(seq, list(range(n)), ranks, p_list, [1.0] * n, 128)
    padded = info.padded_seq_len_list
    M, R = sum(padded), L.round_rank(max(ranks))
    routing = hip_ops.MultiRouting(padded, ranks, info.block_to_lookup_table, info.block_to_alpha, info.block_to_dropout_p)
    g = torch.Generator().manual_seed(K + n)
    x, ds = torch.randn(M, K, generator=g).bfloat16(), torch.zeros(M, R).bfloat16()
    keep = torch.rand(M, K, generator=g) >= torch.cat([torch.full((pl, 1), p) for pl, p in zip(padded, p_list)])
    exp, at = [], 0
    for m, pl, r, p in zip(seq, padded, ranks, p_list):
        ds[at:at + m, :r] = (torch.randn(m, r, generator=g) * 0.1).bfloat16()
        xs = torch.where(keep[at:at + m], x[at:at + m].float(), torch.zeros(())) / (1 - p) if p else x[at:at + m].float()
        exp.append(ds[at:at + m, :r].float().T @ xs)
        at += pl
    mask = hip_ops.pack_mask(keep.cuda()) if any(p_list) else None
    xd, dsd = x.cuda(), ds.cuda()
    for i, got in enumerate(_direct(lambda: hip_ops.fused_multi_lora_da(xd, dsd, routing, mask))):
        _close(got, exp[i], f"adapter {i}")


@pytest.mark.parametrize("M,K,r,p", [(1000, 4096, 16, 0.1), (1000, 4096, 16, 0.0), (2048, 4096, 16, 0.1), (3000, 5120, 128, 0.1)])
def test_long_segments_take_two_stages(M, K, r, p):
    """One workgroup would walk 8 blocks and more alone: chunks of blocks and a second stage are ahead (1000 x 4096 with keep bits 9.3 against 13.7 us)."""
    from lorafusion_amd.ops import hip_ops

    g = torch.Generator(device="cuda").manual_seed(M)
    x, ds = torch.randn(M, K, generator=g, device="cuda").bfloat16(), (torch.randn(M, r, generator=g, device="cuda") * 0.1).bfloat16()
    keep = torch.rand(M, K, generator=g, device="cuda") >= p
    bits = hip_ops.pack_mask(keep) if p else None
    da, names = kernels_of(lambda: hip_ops.fused_lora_da(x, ds, r, p, bits))
    assert "reduce_segments_kernel" in names, names
    _close(da, (ds.float().T @ torch.where(keep, x.float(), torch.zeros((), device="cuda")) / (1 - p)).cpu(), "dA")
