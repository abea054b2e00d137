"""The 192x128 tile (rows and columns that end inside a tile, every form of the LoRA term and the keep-mask) and the joint choice of tile
and slice count for short products over a long contraction, each tile that it picks.  Against fp32 sums of the same 16-bit
inputs at the bound of the other kernel tests (|err| <= 1e-2 (|e| + rms(e)): one 16-bit rounding of the result)."""

import ctypes

import pytest
import torch

from oracle import lora_ref
from tests.util import kernels_of, single_inputs

pytestmark = pytest.mark.gpu


def _close(got, exp, name):
    ok, rel, excess = lora_ref.check_close(got.detach().float().cpu(), exp, rtol=1e-2)
    assert ok, f"{name}: rel {rel:.3e} excess {excess:.3e}"


def _planned(M, N, K):
    from lorafusion_amd import _lib as L

    rows, head, tail = ctypes.c_int(), ctypes.c_int(), ctypes.c_int()
    L.check(L.lib().lf_gemm_plan(M, N, K, 0, ctypes.byref(rows), ctypes.byref(head), ctypes.byref(tail)), "lf_gemm_plan")
    return rows.value, head.value, tail.value


@pytest.mark.parametrize("M,N,K,r,dtype", [
    (257, 11008, 512, 16, torch.bfloat16),    # one row in the second tile row
    (384, 11136, 512, 40, torch.float16),     # whole tile rows; rank beyond one chunk of 32 columns, not a multiple of 16
    (350, 12160, 512, 128, torch.bfloat16),   # a last wave with rows of which some lie beyond the matrix
])
def test_192_row_tile(M, N, K, r, dtype):
    from lorafusion_amd.ops import hip_ops

    assert _planned(M, N, K) == (M, 13, -1)   # (with the mask's bytes: the general kernel's tile, 9)
    d = single_inputs(M, K, N, r, p=0.0, seed=M, dtype=dtype, bias=True)
    x, w, a, b = (d[k].cuda() for k in ("x", "w", "a", "b"))
    ye, se = lora_ref.linear_lora_fwd_fp32(d["x"], d["w"], d["a"], d["b"], 2.0, None, 0.0, d["bias"])
    s = se.to(dtype).cuda()
    ye = ye + 2.0 * (s.float().cpu() - se) @ d["b"].float().T
    _close(hip_ops.fused_lora_xw_sb(x, w, s, b, 2.0, bias=d["bias"].cuda()), ye, "y")
    # the dX product of the transposed sizes: N columns over K, with no mask, its bytes and its bits
    dy, wt, p = d["x"], d["w"].T.contiguous(), 0.2
    g = torch.Generator().manual_seed(r)
    at = ((torch.rand(r, N, generator=g) * 2 - 1) / N ** 0.5).to(dtype)
    ds = (torch.randn(M, r, generator=g) * 0.1).to(dtype)
    mask = torch.rand(M, N, generator=g) >= p
    base, term = dy.float() @ wt.float(), ds.float() @ at.float()
    dev = [t.cuda() for t in (dy, wt, ds, at)]
    _close(hip_ops.fused_lora_dyw_dsa(*dev, 0.0), base + term, "dx")
    expect = base + torch.where(mask, term / (1 - p), torch.zeros(()))
    by = hip_ops.fused_lora_dyw_dsa(*dev, p, mask.cuda())
    _close(by, expect, "dx, mask bytes")
    _close(hip_ops.fused_lora_dyw_dsa(*dev, p, hip_ops.pack_mask(mask.cuda())), expect, "dx, mask bits")


@pytest.mark.parametrize("seq,ranks,p_list,N,dtype", [
    ([60, 250], [40, 16], [0.2, 0.0], 11136, torch.bfloat16),              # a wave with 32 rows of one adapter and 64 of the next
    ([128, 1, 77], [16, 128, 8], [0.0, 0.1, 0.3], 11008, torch.float16),   # every block another adapter, one rank per kind of chunk
])
def test_192_row_tile_over_routing_blocks(seq, ranks, p_list, N, dtype):
    """Waves of 96 rows that lie across two routing blocks; an adapter whose matrix holds infinities does not reach its neighbours."""
    from lorafusion_amd import _lib as L
    from lorafusion_amd.ops import hip_ops
    from lorafusion_amd.ops.multi_lora import prepare_multi_lora_batch_info

    K, n, scales = 512, len(seq), [1.0, 2.0, 0.5][:len(seq)]
    info = prepare_multi_lora_batch_info(seq, list(range(n)), ranks, p_list, scales, 128)
    padded = info.padded_seq_len_list
    M, R, starts = sum(padded), L.round_rank(max(ranks)), [sum(padded[:i]) for i in range(n)]
    rows, head, tail = ctypes.c_int(), ctypes.c_int(), ctypes.c_int()
    L.check(L.lib().lf_gemm_plan(M, N, K, 128, ctypes.byref(rows), ctypes.byref(head), ctypes.byref(tail)), "lf_gemm_plan")
    assert (rows.value, head.value) == (M, 13)
    routing = hip_ops.MultiRouting(padded, ranks, info.block_to_lookup_table, info.block_to_alpha, info.block_to_dropout_p)
    g = torch.Generator().manual_seed(N)
    x, w = torch.randn(M, K, generator=g).to(dtype), (torch.randn(N, K, generator=g) * 0.02).to(dtype)
    s = torch.zeros(M, R, dtype=dtype)
    side = [(torch.randn(N, r, generator=g) * 0.05).to(dtype) for r in ranks]   # B_i [N, r]; its transpose serves as A_i [r, N]
    mask = torch.rand(M, N, generator=g) >= torch.cat([torch.full((pl, 1), p) for pl, p in zip(padded, p_list)])
    y = x.float() @ w.float().T
    dx = y.clone()
    for i, (c, m, r) in enumerate(zip(starts, seq, ranks)):
        s[c:c + m, :r] = torch.randn(m, r, generator=g).to(dtype)
        term = s[c:c + m, :r].float() @ side[i].float().T
        y[c:c + m] += scales[i] * term
        dx[c:c + m] += torch.where(mask[c:c + m], term / (1 - p_list[i]), torch.zeros(())) if p_list[i] > 0 else term
    xd, wd, sd, bd, md = x.cuda(), w.cuda(), s.cuda(), [t.cuda() for t in side], mask.cuda()
    wt, ad = w.T.contiguous().cuda(), [t.T.contiguous().cuda() for t in side]
    _close(hip_ops.fused_multi_lora_xw_sb(xd, wd, sd, bd, routing), y, "y")
    for m, name in ((md, "bytes"), (hip_ops.pack_mask(md), "bits")):
        _close(hip_ops.fused_multi_lora_dyw_dsa(xd, wt, sd, ad, routing, dropout_mask=m), dx, f"dx, mask {name}")
    bd[1].fill_(float("inf"))
    ad[1].fill_(float("inf"))
    clean = torch.ones(M, dtype=torch.bool)
    clean[starts[1]:starts[1] + padded[1]] = False
    _close(hip_ops.fused_multi_lora_xw_sb(xd, wd, sd, bd, routing)[clean.cuda()], y[clean], "y beside infinities")
    _close(hip_ops.fused_multi_lora_dyw_dsa(xd, wt, sd, ad, routing, dropout_mask=md)[clean.cuda()], dx[clean], "dx beside infinities")


@pytest.mark.parametrize("M,K,N,slices,dtype", [
    (85, 4096, 2304, 6, torch.bfloat16), (130, 6144, 2944, 8, torch.float16), (256, 8192, 2048, 8, torch.bfloat16), (283, 6144, 1024, 6, torch.bfloat16),
    (511, 14336, 1024, 8, torch.float16), (700, 8192, 1024, 5, torch.bfloat16), (2290, 9088, 1152, 2, torch.bfloat16)])
def test_tile_and_slices_together(M, K, N, slices, dtype):
    """Forward over K and dX over K (the roles of the dimensions exchanged), cut into the slices that the size query makes room for: against
    fp32 sums, and against the same products through the entry points without a workspace, which do not split: the sums
    differ in order only, so by no more than one 16-bit step of the largest value."""
    from lorafusion_amd import _lib as L
    from lorafusion_amd.ops import hip_ops

    r, p = 16, 0.1
    R, routing = L.round_rank(r), L.single_routing(r, 2.0, p)
    size = lambda op, n, k: L.lib().lf_workspace_bytes(op, M, n, k, R, routing)
    tiles = slices * M * N * 4   # fp32 partial tiles of Y, behind the rank-r pass's slices, and of dX
    assert 0 <= size(L.LF_OP_FWD, N, K) - size(L.LF_OP_XA, 0, K) - tiles < 512 and 0 <= size(L.LF_OP_BWD, K, N) - tiles < 256
    g = torch.Generator().manual_seed(M + K)
    x = torch.randn(M, K, generator=g).to(dtype).cuda()
    w = (torch.randn(N, K, generator=g) * 0.02).to(dtype).cuda()
    a, b = (torch.randn(r, K, generator=g) * K ** -0.5).to(dtype).cuda(), (torch.randn(N, r, generator=g) * 0.01).to(dtype).cuda()
    bits = hip_ops.pack_mask((torch.rand(M, K, generator=g) >= p).cuda())
    y, s = hip_ops.lora_forward(x, w, [a], [b], routing, R, bits, None)
    y1 = hip_ops.fused_lora_xw_sb(x, w, s[:, :r].contiguous(), b, 2.0)
    _close(y, (x.float() @ w.float().T + 2.0 * s[:, :r].float() @ b.float().T).cpu(), "y")
    step = 2.0 ** (-7 if dtype == torch.bfloat16 else -10)
    assert float((y.float() - y1.float()).abs().max()) <= float(y1.float().abs().max()) * step
    # dX [M, N] over K: X takes the place of dY
    wt, at, bt = w.T.contiguous(), b.T.contiguous(), a.T.contiguous()
    xs = torch.randn(M, N, generator=g).to(dtype).cuda()
    bits = hip_ops.pack_mask((torch.rand(M, N, generator=g) >= p).cuda())
    st = (torch.randn(M, R, generator=g) * 0.1).to(dtype).cuda()
    dx = hip_ops.lora_backward(x, xs, wt, [at], [bt], st, routing, R, bits, [r])[0]
    ds = hip_ops.fused_lora_dys_dyb(x, bt, st, 2.0)[1]
    dx1 = hip_ops.fused_lora_dyw_dsa(x, wt, ds, at, p, bits)
    term = ds[:, :r].float() @ at.float() / (1 - p)
    _close(dx, (x.float() @ wt.float() + torch.where(hip_ops.unpack_mask(bits), term, torch.zeros_like(term))).cpu(), "dx")
    assert float((dx.float() - dx1.float()).abs().max()) <= float(dx1.float().abs().max()) * step


@pytest.mark.parametrize("M,N,K,nn,sliced", [
    (1408, 2176, 13312, False, True), (638, 4864, 13568, False, True), (1468, 2176, 25728, True, True),   # slices of 256x256 and 128x256 tiles
    (1921, 1920, 8576, False, False), (1408, 2176, 4224, True, False), (1408, 2176, 13312, True, False)])
def test_one_round_over_a_long_contraction(M, N, K, nn, sliced):
    """Products of one round of 128x128 tiles: cut into slices of larger tiles where K is long, earlier for Y = X W^T than for dX = dY W."""
    from lorafusion_amd import _lib as L
    from lorafusion_amd.ops import hip_ops

    r, g = 16, torch.Generator(device="cuda").manual_seed(M + K)
    randn = lambda *s, std=1.0: (torch.randn(*s, generator=g, device="cuda") * std).bfloat16()
    routing, R = L.single_routing(r, 2.0, 0.0), L.round_rank(r)
    x, w = randn(M, K), randn(N, K, std=0.02)
    a, b = randn(r, K, std=K ** -0.5), randn(N, r, std=0.05)
    if not nn:
        (got, s), names = kernels_of(lambda: hip_ops.lora_forward(x, w, [a], [b], routing, R, None, None))
        exp = x.float() @ w.float().T + 2.0 * s[:, :r].float() @ b.float().T
    else:   # x in the place of dY, w^T in the place of W: dX [M, N] over K
        wt, at, bt, xs, s = w.T.contiguous(), b.T.contiguous(), a.T.contiguous(), randn(M, N), randn(M, R, std=0.1)
        (got, _, _), names = kernels_of(lambda: hip_ops.lora_backward(x, xs, wt, [at], [bt], s, routing, R, None, [r]))
        ds = hip_ops.fused_lora_dys_dyb(x, bt, s, 2.0)[1]
        exp = x.float() @ wt.float() + ds[:, :r].float() @ at.float()
    assert ("ksplit_reduce_kernel" in names) == sliced and ("gemm_mid_kernel" in names) != sliced, names
    _close(got, exp.cpu(), "dX" if nn else "Y")


def test_left_over_rows_are_priced_in_slices_only_where_there_is_memory():
    """Rows behind whole rounds of 256x256 tiles run in slices of K in the whole forward, which has memory for them.  Without memory they would run unsliced, and one launch of
    128x256 tiles is the cheaper plan."""
    from lorafusion_amd import _lib as L
    from lorafusion_amd.ops import hip_ops

    M, N, K, r = 4882, 3200, 3584, 16
    assert _planned(M, N, K)[0] < M
    g = torch.Generator(device="cuda").manual_seed(3)
    rn = lambda *s, std=1.0: (torch.randn(*s, generator=g, device="cuda") * std).bfloat16()
    x, w, a, b = rn(M, K), rn(N, K, std=0.02), rn(r, K, std=K ** -0.5), rn(N, r, std=0.01)
    exp = x.float() @ w.float().T
    y, names = kernels_of(lambda: hip_ops.gemm(x, w))
    assert "gemm_big_kernel" in names and "gemm_lora_kernel" not in names and "gemm_mid_kernel" not in names, names
    _close(y, exp.cpu(), "alone")
    (y, s), names = kernels_of(lambda: hip_ops.lora_forward(x, w, [a], [b], L.single_routing(r, 2.0, 0.0), L.round_rank(r), None, None))
    assert "gemm_big_kernel" in names and ("gemm_lora_kernel" in names or "gemm_mid_kernel" in names) and "ksplit" in names, names
    _close(y, (exp + 2.0 * s[:, :r].float() @ b.float().T).cpu(), "forward")
