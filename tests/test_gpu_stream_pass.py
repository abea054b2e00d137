"""The pass that splits the contraction over workgroups (csrc/lora_stream.hip) at the edges of its tiles: row counts around its
64-row groups, one and several slices of K, every rank tiling, masks read and drawn, several adapters in one batch; and the
short forward built on it.  Against the oracle with fp32 sums from the same 16-bit inputs, at the tolerance of the other
kernel tests (|err| <= 1e-2 (|e| + rms(e)): one 16-bit rounding of S and of Y)."""

import numpy as np
import pytest
import torch

from oracle import dropout as od
from oracle import lora_ref
from tests.util import multi_inputs, single_inputs

pytestmark = pytest.mark.gpu


def _close(got, exp, name):
    ok, rel, excess = lora_ref.check_close(got.detach().float().cpu(), exp, rtol=1e-2)
    assert ok, f"{name}: rel {rel:.3e} excess {excess:.3e}"


@pytest.mark.parametrize("mode", ["none", "given", "drawn"])
@pytest.mark.parametrize("M,K,r,dtype", [
    (1, 128, 40, torch.bfloat16), (63, 256, 48, torch.float16), (64, 384, 64, torch.bfloat16), (65, 640, 72, torch.bfloat16),
    (127, 1152, 128, torch.float16), (300, 4096, 64, torch.bfloat16), (1025, 512, 128, torch.bfloat16),
    (1, 128, 8, torch.bfloat16), (65, 1152, 16, torch.float16), (1000, 256, 24, torch.bfloat16)])   # (ranks up to 32: the drawn mask only)
def test_rank_pass(M, K, r, dtype, mode):
    from lorafusion_amd import _lib as L
    from lorafusion_amd.ops import hip_ops

    p, R, seed = 0.0 if mode == "none" else 0.1, L.round_rank(r), 4321
    d = single_inputs(M, K, 128, r, p=p, seed=M + r, dtype=dtype)
    x, w, a, b = (d[k].cuda() for k in ("x", "w", "a", "b"))
    routing = L.single_routing(r, 2.0, p)
    mask = d["mask"]
    if mode == "drawn":
        y, s, bits = hip_ops.lora_forward_seeded(x, w, [a], [b], routing, R, seed, None)
        expect = od.keep_mask(M, K, p, seed)
        assert np.array_equal(bits.cpu().numpy(), np.packbits(expect, axis=1, bitorder="little")), "drawn mask differs from the oracle"
        mask = torch.from_numpy(expect).bool()
    else:
        y, s = hip_ops.lora_forward(x, w, [a], [b], routing, R, None if mask is None else hip_ops.pack_mask(mask.cuda()), None)
    ye, se = lora_ref.linear_lora_fwd_fp32(d["x"], d["w"], d["a"], d["b"], 2.0, mask, p)
    _close(s[:, :r], se, "S")
    _close(y, ye, "Y")
    assert not s[:, r:].any()


@pytest.mark.parametrize("mode", ["given", "drawn"])
@pytest.mark.parametrize("seq,ranks,K", [([1, 129, 64], [64, 8, 40], 512), ([200, 130], [128, 16], 1280)])
def test_rank_pass_packed(seq, ranks, K, mode):
    from lorafusion_amd.ops import hip_ops
    from lorafusion_amd.ops.multi_lora import prepare_multi_lora_batch_info

    n, p_list, scales = len(seq), [0.0, 0.1, 0.05][:len(seq)], [1.0, 2.0, 0.5][:len(seq)]
    d = multi_inputs(seq, K, 256, ranks, p_list, seed=5)
    info = prepare_multi_lora_batch_info(seq, list(range(n)), ranks, p_list, scales, 128, output_dtype=torch.float32)
    routing = hip_ops.MultiRouting(info.padded_seq_len_list, ranks, info.block_to_lookup_table, info.block_to_alpha, info.block_to_dropout_p)
    x, w = d["x"].cuda(), d["w"].cuda()
    a, b = [t.cuda() for t in d["a_list"]], [t.cuda() for t in d["b_list"]]
    mask = d["mask"]
    if mode == "drawn":
        y, s, bits = hip_ops.lora_forward_seeded(x, w, a, b, routing.c, routing.R, 99, None)
        expect = od.keep_mask(routing.M, K, np.repeat(np.asarray(p_list, np.float32), info.padded_seq_len_list), 99)
        assert np.array_equal(bits.cpu().numpy(), np.packbits(expect, axis=1, bitorder="little")), "drawn mask differs from the oracle"
        mask = torch.from_numpy(expect).bool()
    else:
        y, s = hip_ops.lora_forward(x, w, a, b, routing.c, routing.R, hip_ops.pack_mask(mask.cuda()), None)
    ye, _ = lora_ref.linear_multi_lora_fwd_fp32(d["x"], d["w"], d["a_list"], d["b_list"], seq, d["padded"], scales, p_list, mask)
    _close(y, ye, "Y")
    row = 0
    for q, pl, r in zip(seq, info.padded_seq_len_list, ranks):
        assert not s[row + q:row + pl].any() and not s[row:row + pl, r:].any(), "padded rows and rank columns are zero"
        row += pl


@pytest.mark.parametrize("M", [1, 15, 16, 17, 64, 65, 128])
@pytest.mark.parametrize("K,N,r,dtype,bias", [(128, 128, 8, torch.bfloat16, True), (1152, 384, 72, torch.float16, False), (512, 4096, 128, torch.bfloat16, True)])
def test_short_forward(M, K, N, r, dtype, bias):
    from lorafusion_amd import _lib as L
    from lorafusion_amd.ops import hip_ops

    d = single_inputs(M, K, N, r, p=0.0, seed=M, dtype=dtype, bias=bias)
    R = L.round_rank(r)
    y, s = hip_ops.lora_forward(d["x"].cuda(), d["w"].cuda(), [d["a"].cuda()], [d["b"].cuda()], L.single_routing(r, 0.5, 0.0), R, None,
                                d["bias"].cuda() if bias else None)
    ye, se = lora_ref.linear_lora_fwd_fp32(d["x"], d["w"], d["a"], d["b"], 0.5, None, 0.0, d["bias"])
    _close(y, ye, "Y")
    _close(s[:, :r], se, "S")
    assert not s[:, r:].any()


@pytest.mark.parametrize("mask_form", ["none", "bytes", "bits"])
@pytest.mark.parametrize("M,N,r,dtype", [(1, 128, 72, torch.bfloat16), (129, 640, 128, torch.float16), (700, 1152, 96, torch.bfloat16),
                                         (2500, 256, 120, torch.float16)])
def test_backward_passes_of_high_ranks(M, N, r, dtype, mask_form):
    """dS, dB and dA above 64 rank columns: one and several blocks and slices, ranks that fill the tiling and ranks that do not."""
    from lorafusion_amd import _lib as L
    from lorafusion_amd.ops import hip_ops

    g = torch.Generator().manual_seed(M + r)
    dy, s = torch.randn(M, N, generator=g).to(dtype), torch.randn(M, r, generator=g).to(dtype)
    b = (torch.randn(N, r, generator=g) * 0.05).to(dtype)
    db, ds = hip_ops.fused_lora_dys_dyb(dy.cuda(), b.cuda(), s.cuda(), 2.0)
    _close(ds[:, :r], 2.0 * (dy.float() @ b.float()), "dS")
    _close(db, 2.0 * (dy.float().T @ s.float()), "dB")
    assert not ds[:, r:].any()
    p = 0.0 if mask_form == "none" else 0.2
    mask = torch.rand(M, N, generator=g) >= p
    x = torch.where(mask, dy.float() / (1 - p), torch.zeros(())) if p else dy.float()
    md = None if p == 0 else hip_ops.pack_mask(mask.cuda()) if mask_form == "bits" else mask.cuda()
    _close(hip_ops.fused_lora_da(dy.cuda(), s.cuda(), r, p, md), s.float().T @ x, "dA")


@pytest.mark.parametrize("ranks", [[128, 72], [64, 16]])
def test_backward_passes_leave_padding_out(ranks):
    """Rows behind an adapter's tokens add nothing to its gradients, whatever S and dS hold there."""
    from lorafusion_amd.ops import hip_ops
    from lorafusion_amd.ops.multi_lora import prepare_multi_lora_batch_info

    seq, N = [200, 70], 384
    info = prepare_multi_lora_batch_info(seq, [0, 1], ranks, [0.0, 0.0], [1.0, 2.0], 128)
    routing = hip_ops.MultiRouting(info.padded_seq_len_list, ranks, info.block_to_lookup_table, info.block_to_alpha, info.block_to_dropout_p)
    g = torch.Generator().manual_seed(3)
    M, R = routing.M, routing.R
    dy, s = torch.randn(M, N, generator=g).bfloat16(), torch.randn(M, R, generator=g).bfloat16()   # (padding not zero)
    b = [(torch.randn(N, r, generator=g) * 0.05).bfloat16() for r in ranks]
    db, ds = hip_ops.fused_multi_lora_dys_dyb(dy.cuda(), s.cuda(), [t.cuda() for t in b], routing)
    da = hip_ops.fused_multi_lora_da(dy.cuda(), s.cuda(), routing)
    c = 0
    for i, (q, pl, r) in enumerate(zip(seq, info.padded_seq_len_list, ranks)):
        y, si, sc = dy[c:c + q].float(), s[c:c + q, :r].float(), [1.0, 2.0][i]
        _close(ds[c:c + q, :r], sc * (y @ b[i].float()), f"dS {i}")
        _close(db[i], sc * (y.T @ si), f"dB {i}")
        _close(da[i], si.T @ y, f"dA {i}")
        assert not ds[c + q:c + pl].any()
        c += pl
